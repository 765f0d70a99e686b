"""The tilings that a launch picks by its size: the shorter ones at the sizes where
each is picked, and the 256-row family (tall and tail tiles) in launches that fill the CUs,
which small problems no longer reach."""
import math

import numpy as np
import pytest

from tests.gpu_helpers import Case, gpu_run, oracle_run, rel
from tests.test_gpu_parity import _check, _routing_equal

pytestmark = pytest.mark.gpu


def _group_tiles(E, rows, bm):
    return E * max(1.0, rows / E / bm + 0.5)


def _round_cost(tiles, one, two):
    full, rest = divmod(tiles, 512)
    return full * two + (0 if rest == 0 else one if rest <= 256 else two)


def _leaves_idle(spec, gemm):
    T, H, E, k, I, S = (spec[n] for n in ("T", "H", "E", "k", "I", "S"))
    bn = 128 if gemm == "gateup" else 256
    cols = -(-(H if gemm == "down" else I) // bn)
    sh = -(-(H if gemm == "down" else S) // bn) if S else 0
    tiles = _group_tiles(min(E, T * k), T * k, 256) * cols + -(-T // 256) * sh
    return tiles < 200 and (T * k * cols + T * sh) / 256 < 110


def _pick(gateup, N, tiles_of, margin, swiglu_bwd=False):
    """The rule of with_dense_tiling / with_row_tiling (csrc/moe_api.hip) for a pair that
    leaves CUs idle; tiles_of(bm): row tiles."""
    big, mid, small = ((10, (5.2, 7.0), (3.1, 4.7)) if gateup else
                       (12, (6.8, 8.2), (5.0, 6.2)) if swiglu_bwd else
                       (10, (6.8, 8.2), (4.4, 5.7)))
    bn = (128, 64, 64) if gateup else (256, 128, 128)
    cols = [-(-N // b) for b in bn]
    cost = {"big": math.ceil(tiles_of(256) * cols[0] / 256) * big / margin,
            "mid": _round_cost(tiles_of(128) * cols[1], *mid),
            "small": _round_cost(tiles_of(64) * cols[2], *small)}
    return min(cost, key=cost.get)


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
    T, E, k = spec["T"], spec["E"], spec["k"]
    assert _leaves_idle(spec, what[1])
    dense, gemm = what[0] == "dense", what[1]
    N = {"gateup": spec["S" if dense else "I"], "ddgrad": spec["S" if dense else "I"],
         "down": spec["H"]}[gemm]
    tiles = (lambda bm: -(-T // bm)) if dense else (lambda bm: _group_tiles(E, T * k, bm))
    assert _pick(gemm == "gateup", N, tiles, 1.0 if dense else 1.15, gemm == "ddgrad") == tiling
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
    assert _group_tiles(E, T * k, 256) >= 200
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
