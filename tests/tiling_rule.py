"""Which row tiles a bf16 launch takes (csrc/moe_api.hip: leaves_idle, with_dense_tiling,
with_row_tiling), so that a test can say which ones its shape reaches.  The rule's numbers
are read from the source."""
import math
import os
import re

_SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oxidizr_amd",
                    "csrc", "moe_api.hip")
_TEXT = open(_SRC).read()


def _numbers(pattern):
    return [float(v) for v in re.search(pattern, _TEXT).groups()]


BUSY_TILES, BUSY_ROWS = _numbers(r"kBusyTiles = ([\d.]+), kBusyRows = ([\d.]+);")
ROWS384_ROUNDS, = _numbers(r"kRows384Rounds = (\d+);")


def _costs(name):
    n = r"([\d.]+)"
    big, m1, m2, s1, s2 = _numbers(rf"{name}{{{n}, {{{n}, {n}}}, {{{n}, {n}}}}};")
    return big, (m1, m2), (s1, s2)


COSTS = {"gateup": _costs("kGateUpCosts"), "ddgrad": _costs("kSwigluBwdCosts"),
         "down": _costs("kGemmCosts"), "gdgrad": _costs("kGemmCosts")}


def _columns(spec, gemm, width):
    """Output columns of the routed (width "I") or shared ("S") launch."""
    return spec["H"] if gemm in ("down", "gdgrad") else spec[width]


def group_tiles(E, rows, bm):
    return E * max(1.0, rows / E / bm + 0.5)


def leaves_idle(spec, gemm):
    T, S, TK = spec["T"], spec["S"], spec["T"] * spec["k"]
    bn = 128 if gemm == "gateup" else 256
    cols = -(-_columns(spec, gemm, "I") // bn)
    sh = -(-_columns(spec, gemm, "S") // bn) if S else 0
    tiles = group_tiles(min(spec["E"], TK), TK, 256) * cols + -(-T // 256) * sh
    return tiles < BUSY_TILES and (TK * cols + T * sh) / 256 < BUSY_ROWS


def _round_cost(tiles, one, two):
    full, rest = divmod(tiles, 512)
    return full * two + (0 if rest == 0 else one if rest <= 256 else two)


def pick(gemm, N, tiles_of, margin):
    """The cheapest tiling of a launch over N columns that leaves CUs idle; tiles_of(bm): row
    tiles."""
    big, mid, small = COSTS[gemm]
    cols = [-(-N // b) for b in ((128, 64, 64) if gemm == "gateup" else (256, 128, 128))]
    cost = {"big": math.ceil(tiles_of(256) * cols[0] / 256) * big / margin,
            "mid": _round_cost(tiles_of(128) * cols[1], *mid),
            "small": _round_cost(tiles_of(64) * cols[2], *small)}
    return min(cost, key=cost.get)


def routed(spec, gemm):
    """"rows384", "big" (256-row tiles, tall and half ones among them), "mid" or "small"."""
    E, TK = spec["E"], spec["T"] * spec["k"]
    if gemm != "ddgrad" and TK >= 2 * 384 * E and 6 * TK >= ROWS384_ROUNDS * 256 * 384:
        return "rows384"
    if not leaves_idle(spec, gemm):
        return "big"
    return pick(gemm, _columns(spec, gemm, "I"), lambda bm: group_tiles(min(E, TK), TK, bm), 1.15)


def dense(spec, gemm):
    """The same of the shared expert's launch, where it takes no 384-row tiles."""
    if not leaves_idle(spec, gemm):
        return "big"
    return pick(gemm, _columns(spec, gemm, "S"), lambda bm: -(-spec["T"] // bm), 1.0)
