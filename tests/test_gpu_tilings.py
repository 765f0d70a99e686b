"""The tilings that a launch picks by its size: the shorter ones at the sizes where
each is picked, and the 256-row family (tall and tail tiles) in launches that fill the CUs,
which small problems no longer reach."""
import numpy as np
import pytest

from tests.gpu_helpers import Case, gpu_run, oracle_run, rel
from tests.test_gpu_parity import _check, _routing_equal
from tests.tiling_rule import dense, group_tiles, routed

pytestmark = pytest.mark.gpu


PICK_CASES = [
    # (what, expected tiling, spec): one launch of the case that takes it
    (("dense", "gateup"), "mid", dict(T=1000, H=64, E=2, k=1, I=64, S=2816)),
    (("dense", "gateup"), "small", dict(T=401, H=72, E=2, k=1, I=64, S=2808)),
    (("dense", "ddgrad"), "mid", dict(T=1500, H=64, E=2, k=1, I=64, S=2816)),
    (("dense", "down"), "small", dict(T=321, H=1032, E=2, k=1, I=64, S=72)),
    (("routed", "down"), "mid", dict(T=900, H=2816, E=2, k=2, I=64, S=0)),
    (("routed", "ddgrad"), "mid", dict(T=900, H=64, E=2, k=2, I=2816, S=0)),
    (("routed", "gateup"), "mid", dict(T=500, H=64, E=2, k=2, I=2816, S=0)),
    (("routed", "gateup"), "small", dict(T=129, H=72, E=6, k=2, I=1032, S=0)),
    (("routed", "down"), "small", dict(T=193, H=1096, E=6, k=2, I=72, S=0)),
]


@pytest.mark.parametrize("what,tiling,spec", PICK_CASES)
def test_shorter_tilings(what, tiling, spec):
    where, gemm = what
    assert (dense if where == "dense" else routed)(spec, gemm) == tiling
    # 1e-2: the bf16 bar; the oracle is fp64 on the same bf16 inputs
    case = Case(**spec, dtype="bf16", w_std=0.05)
    g = gpu_run(case, d_aux=0.01, d_z=0.001)
    o = oracle_run(case, g["logits"], d_aux=0.01, d_z=0.001)
    _routing_equal(g, o)
    _check(case, g, o, 1e-2)


@pytest.mark.parametrize("T,H,I", [(22000, 64, 72), (28000, 72, 64), (45000, 64, 296)])
def test_full_tiles_over_many_experts(T, H, I):
    # 160 experts of about 275, 350 and 562 rows: more than 200 256-row tiles in every
    # routed launch, so the 256-row tilings run, with every kind of tail among the experts
    E, k = 160, 2
    assert group_tiles(E, T * k, 256) >= 200
    case = Case(T=T, H=H, E=E, k=k, I=I, S=0, dtype="bf16", w_std=0.05)
    g = gpu_run(case, d_aux=0.01, d_z=0.001)
    o = oracle_run(case, g["logits"], d_aux=0.01, d_z=0.001)
    _routing_equal(g, o)
    counts = np.asarray(g["counts"])
    tails = counts % 256
    assert ((counts > 256) & (tails > 0) & (tails <= 64)).any(), counts   # tall tiles
    assert ((counts > 256) & (tails > 64) & (tails <= 128)).any(), counts
    assert (tails > 192).any(), counts
    _check(case, g, o, 1e-2)


# Rows per expert at the edges of the 256-row tilings: a full tile that takes a tail of at
# most 64 rows (257, 300, 320: one tall tile), tails that keep their own (321, 448, 449, 511),
# tails of 94 and 128 rows (350, 384: two 192-row tiles), less than a tile (70, 128), whole
# tiles; then the same behind two full tiles, where the half tiles run last.
EDGE_ROWS = [300, 320, 321, 350, 384, 256, 257, 70, 385, 448, 449, 511, 128, 512, 576, 640]
HALF_LAST_ROWS = [560, 576, 577, 640, 641, 700, 512, 513, 767, 768, 300, 320, 600, 832, 448, 400]
EDGE_CASES = [(EDGE_ROWS * 3, 264, 264), (EDGE_ROWS * 3, 328, 296), (HALF_LAST_ROWS * 2, 264, 264),
              (HALF_LAST_ROWS * 2, 296, 392)]


def _edge_spec(counts, H, I):
    return dict(T=sum(counts), H=H, E=len(counts), k=1, I=I, S=0)


@pytest.mark.parametrize("counts,H,I", EDGE_CASES)
def test_full_tile_edges(counts, H, I):
    # H and I of at least five k-tiles: the loops refill their stages in every launch
    spec = _edge_spec(counts, H, I)
    T, E = spec["T"], spec["E"]
    assert (T >= 512 * E) == (counts[0] == HALF_LAST_ROWS[0])  # half tiles last
    for gemm in ("gateup", "down", "ddgrad", "gdgrad"):
        assert routed(spec, gemm) == "big", gemm
    case = Case(**spec, dtype="bf16", w_std=0.05)
    # token t goes to expert e: logit e is x[t, e], 8 against N(0, 1)
    expert = np.random.default_rng(0).permutation(np.repeat(np.arange(E), counts))
    case.p["router"] = np.eye(E, H, dtype=np.float32)
    case.p["x"][np.arange(T), expert] = 8.0
    g = gpu_run(case, d_aux=0.01, d_z=0.001)
    assert list(g["counts"]) == counts
    o = oracle_run(case, g["logits"], d_aux=0.01, d_z=0.001)
    _routing_equal(g, o)
    _check(case, g, o, 1e-2)


@pytest.mark.parametrize("spec", [
    # one column block, one k-tile of one token row per wave's fragment
    dict(T=65, H=8, E=1, k=1, I=8, S=8),
    # rows, columns and tokens one vector past 64-wide tiles and 16 / 32-deep k-tiles
    dict(T=131, H=200, E=3, k=2, I=72, S=136),
    # experts of about one row: k-tiles of the weight gradients nearly empty
    dict(T=67, H=136, E=64, k=1, I=72, S=0),
    # a split dense weight gradient whose last chunk is ragged
    dict(T=1030, H=64, E=4, k=1, I=24, S=72),
])
def test_fp32_k_major_tiles(spec):
    """fp32 input and weight gradients, whose K-major operands are read as they lie in memory
    (1e-5: the fp32 bar, 32-bit sums of at most 1030 terms)."""
    case = Case(**spec, w_std=0.1)
    g = gpu_run(case, d_aux=0.01, d_z=0.001)
    o = oracle_run(case, g["logits"], d_aux=0.01, d_z=0.001)
    _routing_equal(g, o)
    _check(case, g, o, 1e-5)


def test_fp32_dense_weight_gradients_sum_in_chunks():
    """The shared expert's gate and up gradients at M = 680, N = 776, T = 1999 are three
    partial sums over 672 tokens, not one chain of 1999: with every token alike but the
    first, whose terms are 2^26 times the others' q, the first one's sum loses each q added
    to it (q is below 1/4 of its ulp), the other two lose none.  At most 671 of 2^26 + 1998
    are lost (1.0e-5; the terms themselves are 1e-6 off), 1998 in one chain (3.0e-5)."""
    T, H, S = 1999, 776, 680
    case = Case(T=T, H=H, E=2, k=1, I=8, S=S, w_std=0.1, seed=3)
    x = np.tile(case.p["x"][:1], (T, 1))
    dout = np.tile(case.p["dout"][:1], (T, 1))
    dout[0] *= 2.0 ** 26
    g = gpu_run(case, x=x, dout=dout)
    o = oracle_run(case, g["logits"], x=x, dout=dout)
    for n in ("shared_gate", "shared_up"):
        assert rel(g[n], o[n]) <= 671 / 2 ** 26 + 2e-6, n
