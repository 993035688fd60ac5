"""GPU: the fp16-weight product over many rows (ql_gemv_f16w with more rows than one GEMV pass), the tiled MFMA form,
against gemmNTRef on the fp16-decoded weights (double accumulation), at the edges of its tiles."""
import numpy as np
import pytest

from tests.test_gpu_parity import GEMV_ATOL, GEMV_RTOL, assert_close, f16w_case
from webllm_amd import qlinear as ql

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ql.Context(0)
    yield c
    c.destroy()


@pytest.mark.parametrize("M,N,K,biased,spread", [
    (17, 129, 896, True, False),      # one row over the GEMV's pass; one column over a tile
    (33, 1003, 72, False, False),     # K % 64 != 0, N % 4 != 0, tile of 64 rows
    (64, 128, 64, True, False),       # one whole tile, one chunk
    (65, 2047, 904, True, True),      # two row blocks of 64, ragged K, x past fp16's range
    (129, 25001, 136, True, False),   # row blocks of 128, ragged K and N, more tiles than workgroups
    (300, 16640, 192, False, True),   # row blocks of 128, the last one with 44 rows
    (5, 300, 3584, False, False),     # K so long that a GEMV pass holds 4 rows: tile of 16 rows
    (200, 64, 12800, True, False),    # the image holds 64 rows: four passes
])
def test_many_rows_match_oracle(ctx, M, N, K, biased, spread):
    from oracle import oracle as orc
    W16, bias, x = f16w_case(M, N, K, biased, 0.01, spread)
    lay = ql.ArenaLayout()
    w_off, b_off = lay.take(W16.nbytes), lay.take(N * 4)
    w = ctx.arena(lay.used)
    w.write(w_off, W16.view(np.uint16))
    if biased:
        w.write(b_off, bias)
    alay = ql.ArenaLayout()
    x_off, y_off, end = alay.take(x.nbytes), alay.take(M * N * 4, 16), alay.take(256, 4)
    act = ctx.arena(alay.used)
    act.write(x_off, x)
    guard = np.full(64, 7.25, np.float32)
    act.write(end, guard)
    ctx.gemv_f16w(w, w_off, b_off if biased else None, act, x_off, M, N, K, y_off)
    y = act.read(y_off, (M, N), np.float32)
    assert np.array_equal(act.read(end, (64,), np.float32), guard)       # nothing past y
    assert_close(orc, y, orc.gemm_nt(x, W16.astype(np.float32), bias), GEMV_ATOL, GEMV_RTOL, f"M={M} N={N} K={K}")
    ctx.gemv_f16w(w, w_off, b_off if biased else None, act, x_off, M, N, K, y_off)
    assert np.array_equal(act.read(y_off, (M, N), np.float32).view(np.uint32), y.view(np.uint32))
    # a row with an infinity and one with a NaN stay their own rows' affair
    x[1, 3], x[2, 5] = np.inf, np.nan
    act.write(x_off, x)
    ctx.gemv_f16w(w, w_off, b_off if biased else None, act, x_off, M, N, K, y_off)
    z = act.read(y_off, (M, N), np.float32)
    assert not np.isfinite(z[1]).any() and np.isnan(z[2]).all()
    keep = [m for m in range(M) if m not in (1, 2)]
    assert np.array_equal(z[keep].view(np.uint32), y[keep].view(np.uint32))
    act.release()
    w.release()
