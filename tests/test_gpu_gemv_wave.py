"""GPU: decode linears over an image of x (ql_linear and ql_linear_batch at M >= 5, and M = 3, 4 with a narrow N and K from
2048 on, groups of 128, up to a longest K) against the oracle (double accumulation on the fp32-decoded weights) at the GEMV bar, at the edges of
the kernel's tiles: 16 or 64 columns, 8 parts of K, 8 or 16 rows."""
import numpy as np
import pytest

from tests.test_gpu_parity import GEMV_ATOL, GEMV_RTOL, assert_close
from webllm_amd import qlinear as ql
from webllm_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ql.Context(0)
    yield c
    c.destroy()


def run(ctx, M, shapes, x_dtype, same_x, biased, zeros, spread=False):
    from oracle import oracle as orc
    lay, alay, lin = ql.ArenaLayout(), ql.ArenaLayout(), []
    for i, (K, N) in enumerate(shapes):
        t = synth.gptq_linear(K, N, 128, seed=0x6E3, key=(i, K, N), stored_zero=None if zeros == "any" else 7)
        offs = [lay.take(a.nbytes) for a in (t.qweight, t.qzeros, t.scales)]
        lin.append((t, offs, lay.take(N * 4) if biased else None))
    w = ctx.arena(lay.used)
    descs, xs, xo, yo = [], [], [], []
    for i, ((K, N), (t, offs, b)) in enumerate(zip(shapes, lin)):
        for o, a in zip(offs, (t.qweight, t.qzeros, t.scales)):
            w.write(o, a)
        bias = synth.activations(1, N, seed=0x6E4, key=(i,))[0] if biased else None
        if biased:
            w.write(b, bias)
        descs.append(ql.make_desc(offs[0], None if zeros == "none" else offs[1], offs[2], K, N, 128, b))
        x = xs[0][0] if same_x and i else synth.activations(M, K, seed=0x6E5, key=(i,))
        if spread and not i:
            x[0, 5], x[1] = 1e5, x[1] * 1e-6
        x = x.astype(np.float16).astype(np.float32) if x_dtype == ql.DTYPE_F16 else x
        xs.append((x, bias))
        xo.append(xo[0] if same_x and i else alay.take(x.nbytes))
        yo.append(alay.take(M * N * 4))
    end = alay.take(256, 4)
    scratch = alay.take(max(16, ql.plan_batch(descs, M)))
    act = ctx.arena(alay.used)
    for (x, _), o in zip(xs, xo):
        act.write(o, x.astype(np.float16).view(np.uint16) if x_dtype == ql.DTYPE_F16 else x)
    guard = np.full(64, 7.25, np.float32)
    act.write(end, guard)

    def call():
        if len(descs) == 1:
            ctx.linear(descs[0], w, act, xo[0], x_dtype, M, yo[0], scratch)
        else:
            ctx.linear_batch(descs, w, act, xo, x_dtype, M, yo, scratch)
        return [act.read(o, (M, d.N), np.float32) for o, d in zip(yo, descs)]

    first = call()
    assert np.array_equal(act.read(end, (64,), np.float32), guard)
    for (t, _, _), (x, bias), y in zip(lin, xs, first):
        ref = orc.gptq_linear(t.qweight, None if zeros == "none" else t.qzeros, t.scales, x, bias)
        assert_close(orc, y, ref, GEMV_ATOL, GEMV_RTOL, f"M={M} K={t.K} N={t.N}")
    assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(first, call()))
    act.release()
    w.release()


@pytest.mark.parametrize("M,shapes,x_dtype,same_x,biased,zeros,spread", [
    (5, [(128, 4)], ql.DTYPE_F32, False, True, "any", False),            # one group for eight waves, one column piece
    (8, [(1152, 60)], ql.DTYPE_F32, False, False, "none", False),        # nine groups, columns past the last tile
    (9, [(896, 896)], ql.DTYPE_F32, False, True, "sym", True),           # two fragments; spread magnitudes
    (16, [(2048, 100)], ql.DTYPE_F16, False, False, "any", False),
    (16, [(256, 8228)], ql.DTYPE_F32, False, True, "any", False),        # 64-column tiles, ragged N
    (7, [(256, 8192)], ql.DTYPE_F16, False, False, "sym", False),
    (8, [(128, 33000)], ql.DTYPE_F32, False, True, "any", False),        # 516 tiles: a third workgroup on some CUs
    (4, [(2048, 256)], ql.DTYPE_F32, False, True, "any", False),         # M = 3, 4: narrow, long K
    (3, [(4864, 896)], ql.DTYPE_F32, False, False, "any", False),
    (6, [(896, 896), (896, 128), (896, 128)], ql.DTYPE_F32, True, True, "any", False),     # one image for three
    (12, [(384, 64), (1280, 4100)], ql.DTYPE_F32, False, False, "any", False),             # two images
])
def test_image_linears_match_oracle(ctx, M, shapes, x_dtype, same_x, biased, zeros, spread):
    run(ctx, M, shapes, x_dtype, same_x, biased, zeros, spread)


def test_replay_and_other_users_of_the_workspace(ctx):
    """A captured linear replays to the same bits with eager linears, of other sizes, between the replays."""
    rng = np.random.default_rng(5)
    K, N, M = 896, 896, 8
    t = synth.gptq_linear(K, N, 128, seed=0x6E6)
    lay, alay = ql.ArenaLayout(), ql.ArenaLayout()
    offs = [lay.take(a.nbytes) for a in (t.qweight, t.qzeros, t.scales)]
    w = ctx.arena(lay.used)
    for o, a in zip(offs, (t.qweight, t.qzeros, t.scales)):
        w.write(o, a)
    d = ql.make_desc(*offs, K, N, 128)
    x0, x1, y0, y1 = alay.take(M * K * 4), alay.take(16 * K * 4), alay.take(M * N * 4), alay.take(16 * N * 4)
    scratch = alay.take(max(ql.plan_linear(m, N, K).scratch_bytes for m in (M, 16)))
    act = ctx.arena(alay.used)
    act.write(x0, rng.standard_normal((M, K)).astype(np.float32))
    act.write(x1, rng.standard_normal((16, K)).astype(np.float32))
    ctx.linear(d, w, act, x0, ql.DTYPE_F32, M, y0, scratch)
    want = act.read(y0, (M, N), np.float32)
    ctx.graph_begin()
    ctx.linear(d, w, act, x0, ql.DTYPE_F32, M, y0, scratch)
    g = ctx.graph_end()
    for _ in range(4):
        act.write(y0, np.zeros((M, N), np.float32))
        ctx.linear(d, w, act, x1, ql.DTYPE_F32, 16, y1, scratch)
        g.launch()
        ctx.sync()
        assert np.array_equal(act.read(y0, (M, N), np.float32).view(np.uint32), want.view(np.uint32))
    g.destroy()
    act.release()
    w.release()


def test_widths_past_the_split_counters_stay_refused(ctx):
    """256 x 65536 columns is the most that one call's arrival counters cover, whichever kernel runs."""
    N = 256 * 65536 + 4
    qw, qz, sc = ql.gptq_sizes(128, N, 128)
    lay = ql.ArenaLayout()
    d = ql.make_desc(lay.take(qw), None, lay.take(sc), 128, N, 128)
    w = ctx.arena(lay.used)
    for M in (4, 8):
        alay = ql.ArenaLayout()
        x, y = alay.take(M * 128 * 4), alay.take(M * N * 4)
        scratch = alay.take(max(16, ql.plan_linear(M, N, 128).scratch_bytes))
        act = ctx.arena(alay.used)
        with pytest.raises(ql.QlError) as e:
            ctx.linear(d, w, act, x, ql.DTYPE_F32, M, y, scratch)
        assert e.value.code == -10 and "N too large" in str(e.value)
        act.release()
    # two linears of half as many columns and one strip more
    half = ql.make_desc(d.qweight_off, None, d.scales_off, 128, 256 * 32768 + 4, 128)
    alay = ql.ArenaLayout()
    x, y = alay.take(8 * 128 * 4), [alay.take(8 * half.N * 4) for _ in range(2)]
    scratch = alay.take(max(16, ql.plan_batch([half] * 2, 8)))
    act = ctx.arena(alay.used)
    with pytest.raises(ql.QlError) as e:
        ctx.linear_batch([half] * 2, w, act, [x] * 2, ql.DTYPE_F32, 8, y, scratch)
    assert e.value.code == -10 and "batch too wide" in str(e.value)
    act.release()
    w.release()


def test_image_past_the_workspace(ctx):
    """K so long that 16 rows' image outgrows the workspace's 64 MiB: the other decode kernel, at the same bar."""
    M, K, N = 16, 128 * 8200, 64
    g = np.random.default_rng(0x10A6)
    qweight = g.integers(-2**31, 2**31, (K // 8, N), dtype=np.int64).astype(np.int32)
    scales = (np.abs(g.standard_normal((K // 128, N))) * 0.01).astype(np.float16)
    x = g.standard_normal((M, K)).astype(np.float32)
    lay, alay = ql.ArenaLayout(), ql.ArenaLayout()
    d = ql.make_desc(lay.take(qweight.nbytes), None, lay.take(scales.nbytes), K, N, 128)
    w = ctx.arena(lay.used)
    w.write(d.qweight_off, qweight)
    w.write(d.scales_off, scales)
    xo, yo = alay.take(x.nbytes), alay.take(M * N * 4)
    scratch = alay.take(max(16, ql.plan_linear(M, N, K).scratch_bytes))
    act = ctx.arena(alay.used)
    act.write(xo, x)
    ctx.linear(d, w, act, xo, ql.DTYPE_F32, M, yo, scratch)
    y = act.read(yo, (M, N), np.float32)
    ref = np.zeros((M, N))
    for k in range(0, K, 128 * 200):
        n = min(128 * 200, K - k)
        q = (qweight[k // 8:(k + n) // 8, None, :] >> np.arange(0, 32, 4, dtype=np.int32)[None, :, None]) & 15
        W = (q.reshape(n, N) - 8.0) * np.repeat(scales[k // 128:(k + n) // 128].astype(np.float64), 128, 0)
        ref += x[:, k:k + n].astype(np.float64) @ W
    assert np.linalg.norm(y - ref) <= 1e-5 * np.linalg.norm(ref)
    act.release()
    w.release()


@pytest.mark.parametrize("M,K,N", [(3, 8448, 2052), (3, 8576, 2052), (9, 5760, 5124), (9, 12160, 5124)])
def test_both_sides_of_the_longest_k(ctx, M, K, N):
    run(ctx, M, [(K, N)], ql.DTYPE_F32, False, True, "any")


@pytest.mark.parametrize("M", [5, 16])
def test_eight_inputs_of_a_batch(ctx, M):
    """Eight linears on inputs of their own, of several K, images in one launch."""
    run(ctx, M, [(128 * (1 + 3 * (i % 3)), 64 + 4 * i) for i in range(8)], ql.DTYPE_F32, False, True, "any")
