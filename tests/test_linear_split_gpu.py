"""The linear layer on the bf16 matrix cores (linear_split_kernel): every tile (asserted) at ragged M, N and K,
every epilogue and activation on each, rows that are not 16-byte aligned, and values that have no three
bfloat16 terms on each tile.

Tolerance: each operand is held to 24 bits and six of the nine term products are kept, so a sum of K
products differs from 64 bits by the rounding of its K/32 * 6 float32 additions, at most
6 * ceil(K/32) * 2^-24 of sum |x w| and about its square root in the 2-norm. 2e-6 covers K = 584 with
the spread of sum |x w| over |sum x w| (about sqrt(K)) taken in."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import linear as ol
from supra_attn import _lib
from supra_attn.device import Event
from supra_attn.linear_workloads import make_linear
from supra_attn.runner import StagedLinear

pytestmark = pytest.mark.gpu

TOL = 2e-6

# tile: (M, N, K) that take it on 256 CUs whatever the epilogue, ragged in M and N, K % 32 of 8, 16 and 24, K shorter
# than one k-tile and an odd and an even number of them
TILES = {
    (64, 64): [(1225, 1225, 264), (4715, 1945, 8), (3100, 570, 584)],
    (64, 96): [(1798, 1091, 336), (2767, 2202, 8), (2047, 2050, 776)],
    (128, 96): [(10355, 389, 264), (3715, 2103, 8), (3071, 1730, 584)],
    (256, 144): [(10909, 517, 272), (5841, 1574, 88)],
    (256, 192): [(11528, 775, 264), (3905, 2313, 264)],
}
CASES = [(tile, *size) for tile, sizes in TILES.items() for size in sizes]
# sizes between the tiles' classes, and two where the fp32 64 x 64 kernel takes over
SIZES = [(2047, 2050, 776), (3071, 1730, 584), (16300, 570, 40), (16300, 760, 72), (16299, 571, 24), (16299, 763, 48),
         (16333, 1729, 8)]
EPILOGUES = [
    (_lib.SA_EPI_STORE, _lib.SA_ACT_NONE, {}),
    (_lib.SA_EPI_RESID_GATE, _lib.SA_ACT_GELU_TANH, dict(gate_off=3)),  # gate not 16-byte aligned
    (_lib.SA_EPI_RESID, _lib.SA_ACT_SILU, dict(y_off=1)),               # rows of y not aligned
    (_lib.SA_EPI_STORE, _lib.SA_ACT_GELU, dict(y_off=2)),
]


def run(dev, call, tile=None):
    st = StagedLinear(dev, call)
    try:
        took = _lib.linear_tile(st.args)
        print(f"[linear split] {call.name} M={call.M} N={call.N} K={call.K} act={call.act} epi={call.epi} tile={took}", flush=True)
        assert tile is None or took == (*tile, 3)
        return st.run()
    finally:
        st.release()


@pytest.mark.parametrize("tile,M,N,K", CASES + [(None, *size) for size in SIZES])
@pytest.mark.parametrize("epi,act,kw", EPILOGUES)
def test_tiles(dev, tile, M, N, K, epi, act, kw):
    kw = dict(kw, ldy=(N + 7) // 4 * 4)
    call = make_linear(f"split_{M}x{N}x{K}", M, N, K, seed=M + N + K + epi, act=act, epi=epi, **kw)
    got = run(dev, call, tile)
    e = ol.errors(got, ol.linear_fp64(call.x, call.w, call.y0, **call.oracle_kwargs()))
    assert e["finite"] and e["rel_l2"] <= TOL and e["max_rel"] <= 1e-5, e


@pytest.mark.parametrize("tile,M,N,K", [(tile, *sizes[0]) for tile, sizes in TILES.items()] + [(None, 2047, 2050, 776), (None, 16300, 570, 40)])
@pytest.mark.parametrize("epi,act,kw", EPILOGUES[:3])
def test_values_without_three_terms(dev, tile, M, N, K, epi, act, kw):
    """Infinities, NaN, and magnitudes that round past the bfloat16 range (finite products) give what
    float32 products give: the same elements infinite, NaN or finite, and the finite ones to tolerance."""
    call = make_linear(f"special_{M}x{N}x{K}", M, N, K, seed=K, act=act, epi=epi, **dict(kw, ldy=(N + 7) // 4 * 4))
    x = call.x.reshape(-1)
    x[5 * K + 3] = np.inf
    x[700 * K + 7] = -np.inf
    x[900 * K] = np.nan
    x[(M - 1) * K + 1] = np.float32(3.4e38)
    w = call.w.reshape(-1)
    w[(N - 1) * K + 2] = np.inf
    w[40 * K + 3] = 0.0  # inf * 0
    idx = (call.y_off + np.arange(M)[:, None] * call.ldy + np.arange(N)).reshape(-1)
    got = run(dev, call, tile).reshape(-1)[idx]
    ref = ol.linear_torch_fp32(call.x, call.w, call.y0, **call.oracle_kwargs()).reshape(-1)[idx]
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(ref))
    np.testing.assert_array_equal(got[np.isinf(got)], ref[np.isinf(ref)])
    fin = np.isfinite(ref)
    rows = np.repeat(np.abs(np.where(fin, ref, 0)).reshape(M, N).max(axis=1), N)  # 3.4e38 sets its row's scale
    assert np.all(np.abs(got[fin] - ref[fin]) <= 1e-5 * rows[fin])


@pytest.mark.parametrize("up,over", [(120, 0), (138, 60)])
@pytest.mark.parametrize("what", ["x", "w"])
@pytest.mark.parametrize("M,N,K", [(2047, 2050, 776), (16300, 570, 40)])
def test_tiny_operands(dev, M, N, K, what, up, over):
    """Operands around 2^-120 have no third bfloat16 term of their own (14 of 24 bits would remain, 3e-5 in the
    2-norm), those around 2^-138 none at all: they are as exact as any others, whatever they meet."""
    call = make_linear(f"tiny_{what}_{M}x{N}x{K}", M, N, K, seed=K, bias=False)
    other = "w" if what == "x" else "x"
    setattr(call, what, np.ldexp(getattr(call, what).astype(np.float64), -up).astype(np.float32))
    setattr(call, other, getattr(call, other) * np.float32(2.0 ** over))
    got = run(dev, call)
    e = ol.errors(got, ol.linear_fp64(call.x, call.w, call.y0, **call.oracle_kwargs()))
    assert e["finite"] and e["rel_l2"] <= TOL and e["max_rel"] <= 1e-5, e


@pytest.mark.parametrize("M,N,K,fp32", [(3136, 576, 576, 3.05e-7), (3136, 576, 2304, 6.07e-7), (1344, 1536, 512, 2.89e-7)])
def test_two_sums_per_output(dev, M, N, K, fp32):
    """Calls that took the two-split fp32 kernel (fp32: its measured 2-norm error on these inputs) are no less exact
    on the split kernel's 64 x 64 tile, which sums the products of first terms apart (one sum: a fifth more than
    the fp32 kernel; two: under half)."""
    call = make_linear(f"two_sums_{M}x{N}x{K}", M, N, K, seed=1, bias=False)
    st = StagedLinear(dev, call)
    try:
        assert _lib.linear_tile(st.args) == (64, 64, 3)
        got = st.run()
    finally:
        st.release()
    e = ol.errors(got, ol.linear_fp64(call.x, call.w, call.y0, **call.oracle_kwargs()))
    print(f"[linear split] {call.name} {e['rel_l2']:.3e}", flush=True)
    assert e["rel_l2"] <= 1.02 * fp32, e


@pytest.mark.parametrize("y_off,ldy", [(0, 1108), (1, 1108), (0, 1107), (3, 1109)])
def test_store_at_any_alignment(dev, y_off, ldy):
    """Plain stores into rows at every 4-byte alignment; nothing beside the rows is written."""
    call = make_linear(f"store_{y_off}_{ldy}", 2047, 1107, 584, seed=ldy + y_off, y_off=y_off, ldy=ldy)
    got = run(dev, call)
    e = ol.errors(got, ol.linear_fp64(call.x, call.w, call.y0, **call.oracle_kwargs()))  # with the gaps of y0
    assert e["finite"] and e["rel_l2"] <= TOL and e["max_rel"] <= 1e-5, e


def test_unaligned_rows_cost_little(dev):
    """Rows of y off a 16-byte boundary take at most twice as long as aligned ones (measured about the same; element by
    element and past the L2 they took 4 times)."""
    def best(y_off, ldy):
        st = StagedLinear(dev, make_linear("rows", 5714, 1107, 56, y_off=y_off, ldy=ldy))
        a, b = Event(), Event()
        try:
            times = []
            for _ in range(6):
                a.record(dev.stream)
                for _ in range(50):
                    st.launch()
                b.record(dev.stream)
                dev.sync()
                times.append(a.elapsed_ms(b))
            return min(times)
        finally:
            st.release()

    aligned, unaligned = best(0, 1120), best(1, 1107)
    print(f"[linear split] aligned {aligned:.4f} ms, unaligned {unaligned:.4f} ms", flush=True)
    assert unaligned <= 2 * aligned
