"""GPU: linears of some tens of rows over fp16 images (ql_linear and ql_linear_batch at M > 16, groups of 128 or 256, up
to about a thousand 64-column x 32-row tiles), against fp16-rounded operands in float64: the edges of the tiles, of the 8
parts of K and of the dispatch."""
import numpy as np
import pytest

from webllm_amd import qlinear as ql
from webllm_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ql.Context(0)
    yield c
    c.destroy()


def weights(t, zeros):
    """f16(W) [K, N] of the packed linear, as float64: (q - z) * s rounded once to fp16."""
    shift = np.arange(0, 32, 4, dtype=np.uint32)
    q = ((t.qweight[:, None, :] >> shift[None, :, None]) & 15).reshape(-1, t.N)[:t.K].astype(np.float32)
    z = ((t.qzeros[:, :, None] >> shift) & 15).reshape(t.qzeros.shape[0], -1)[:, :t.N].astype(np.float32) + 1
    s = t.scales.view(np.float16).astype(np.float32)
    z = np.full_like(s, 8.0) if zeros == "none" else z
    rep = lambda a: np.repeat(a, t.group, 0)[:t.K]
    return ((q - rep(z)) * rep(s)).astype(np.float16).astype(np.float64)


@pytest.mark.parametrize("M,shapes,group,x_dtype,same_x,biased,zeros", [
    (17, [(128, 4)], 128, ql.DTYPE_F32, False, True, "any"),               # one chunk for eight waves, one column piece
    (32, [(896, 896)], 128, ql.DTYPE_F16, False, False, "sym"),            # one whole row block
    (33, [(1152, 100)], 128, ql.DTYPE_F32, False, True, "none"),           # a block of one row, nine chunks, ragged N
    (77, [(3584, 3584)], 128, ql.DTYPE_F32, False, False, "any"),          # long K, 168 tiles
    (65, [(512, 1184), (512, 68), (512, 64)], 128, ql.DTYPE_F16, True, True, "any"),       # one image for three
    (40, [(1024, 516), (768, 260)], 256, ql.DTYPE_F32, False, False, "any"),               # groups of 256, two images
    (400, [(640, 896)], 128, ql.DTYPE_F32, False, True, "any"),            # 182 tiles of 13 row blocks
])
def test_few_rows_match_fp16_operands(ctx, M, shapes, group, x_dtype, same_x, biased, zeros):
    lay, alay, lin = ql.ArenaLayout(), ql.ArenaLayout(), []
    for i, (K, N) in enumerate(shapes):
        t = synth.gptq_linear(K, N, group, seed=0xFE3, key=(i, K, N), stored_zero=None if zeros == "any" else 7)
        lin.append((t, [lay.take(a.nbytes) for a in (t.qweight, t.qzeros, t.scales)], lay.take(N * 4) if biased else None))
    w = ctx.arena(lay.used)
    descs, xs, xo, yo, bs = [], [], [], [], []
    for i, ((K, N), (t, offs, b)) in enumerate(zip(shapes, lin)):
        for o, a in zip(offs, (t.qweight, t.qzeros, t.scales)):
            w.write(o, a)
        bs.append(synth.activations(1, N, seed=0xFE4, key=(i,))[0] if biased else np.zeros(N, np.float32))
        if biased:
            w.write(b, bs[-1])
        descs.append(ql.make_desc(offs[0], None if zeros == "none" else offs[1], offs[2], K, N, group, b))
        x = xs[0] if same_x and i else synth.activations(M, K, seed=0xFE5, key=(i,))
        xs.append(x)
        xo.append(xo[0] if same_x and i else alay.take(x.nbytes))
        yo.append(alay.take(M * N * 4))
    end = alay.take(256, 4)
    scratch = alay.take(max(16, ql.plan_batch(descs, M)))
    act = ctx.arena(alay.used)
    for x, o in zip(xs, xo):
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
    for (t, _, _), x, b, y in zip(lin, xs, bs, first):
        x16, W = x.astype(np.float16).astype(np.float64), weights(t, zeros)
        ref = x16 @ W + b
        # fp32 sums of K products: each addition rounds to 2^-24 of a partial sum, at most sum |x w|
        assert np.all(np.abs(y - ref) <= 2.0 ** -24 * (t.K / 8 + 16) * (np.abs(x16) @ np.abs(W) + np.abs(b)) + 1e-30)
        assert np.linalg.norm(y - ref) <= 2e-6 * np.linalg.norm(ref)
    assert all(np.array_equal(a.view(np.uint32), c.view(np.uint32)) for a, c in zip(first, call()))
    act.release()
    w.release()


def test_eight_inputs_of_a_batch(ctx):
    """Eight linears on inputs of their own, of several K, images in one launch."""
    test_few_rows_match_fp16_operands(ctx, 35, [(128 * (1 + 3 * (i % 3)), 64 + 4 * i) for i in range(8)], 128, ql.DTYPE_F32, False, True, "any")
