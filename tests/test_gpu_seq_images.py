"""GPU: chained decode sequences that run their passes as products over activation images (ql_seq_get_info variant 2:
M = 5..16, or 2..4 with 16 MiB of weights a pass), every linear against the oracle on the GPU's own inputs, as the tiles'
tests check them; repeats and graph replays give the same bits."""
import numpy as np
import pytest

from tests.test_gpu_fused import FusedModel, _sample, check_fused
from tests.test_gpu_seq import SeqModel, check_all
from webllm_amd import qlinear as ql
from webllm_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ql.Context(0)
    yield c
    c.destroy()


@pytest.mark.parametrize("M,layers,C,I,KV", [
    (5, 2, 256, 640, 128),        # the fewest rows; two layers: residuals and norms of produced rows
    (8, 1, 896, 4864, 128),       # one fragment, full
    (9, 1, 384, 128, 128),        # two fragments, one group of K in the down linear
    (16, 1, 4224, 256, 128),      # RMSNorm rows longer than a workgroup keeps in registers
    (2, 1, 3584, 18944, 512),     # few rows, large passes
])
def test_image_passes_match_oracle(ctx, M, layers, C, I, KV):
    from oracle import oracle as orc
    m = FusedModel(ql, ctx, M, layers, C, I, KV)
    info = m.seq.info
    assert info.kernel == ql.SEQ_TILES and info.variant == 2 and info.passes == 4 * layers
    assert info.launches == 8 * layers          # an image and a product per pass: norm, q, norm, SiLU-mul
    m.seq.run()
    m.seq.status()
    first = m.outputs()
    check_fused(orc, m, first, f"M={M} C={C} I={I}", **({"cols_for": _sample} if C == 3584 else {}))
    ctx.graph_begin()
    m.seq.run()
    g = ctx.graph_end()
    for _ in range(3):
        g.launch()
        m.seq.run()
        ctx.sync()
        assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(first, m.outputs()))
    g.destroy()


@pytest.mark.parametrize("M,C,I,variant", [(1, 896, 4864, 0), (4, 896, 4864, 0), (5, 896, 4864, 2)])
def test_small_passes_of_few_rows_keep_the_tiles(ctx, M, C, I, variant):
    m = FusedModel(ql, ctx, M, 1, C, I, 128)
    assert m.seq.info.variant == variant


@pytest.mark.parametrize("M,layers,C,I,KV", [(5, 1, 896, 4864, 128), (8, 2, 896, 4864, 128), (16, 2, 896, 4864, 128), (16, 1, 3584, 18944, 512)])
def test_fused_tiles_of_many_rows(ctx, monkeypatch, M, layers, C, I, KV):
    """The dependency-ordered tiles at M >= 5, which chained sequences with other groups, fp16 x or QL_SEQ_PASSES=0 run."""
    from oracle import oracle as orc
    monkeypatch.setenv("QL_SEQ_PASSES", "0")
    m = FusedModel(ql, ctx, M, layers, C, I, KV)
    info = m.seq.info
    assert info.kernel == ql.SEQ_TILES and info.variant == 0 and info.launches == 1
    m.seq.run()
    m.seq.status()
    first = m.outputs()
    check_fused(orc, m, first, f"tiles M={M} C={C}", **({"cols_for": _sample} if C == 3584 else {}))
    m.seq.run()
    m.seq.status()
    assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(first, m.outputs()))
    m.release()


def test_chained_tiles_of_16_rows(ctx, monkeypatch):
    """The same without fused work."""
    from oracle import oracle as orc
    monkeypatch.setenv("QL_SEQ_PASSES", "0")
    m = SeqModel(ql, ctx, 16, layers=2, C=896, I=4864, KV=128)
    assert m.seq.info.kernel == ql.SEQ_TILES and m.seq.info.variant == 0
    m.seq.run()
    m.seq.status()
    check_all(orc, m, m.outputs(), "tiles M=16")
    m.release()


@pytest.mark.parametrize("env,variant", [("0", 0), ("1", 2)])
def test_external_second_operand(ctx, monkeypatch, env, variant):
    """test_fused_silu_mul_external_operand's sequence at M = 16, as tiles and over images."""
    from oracle import oracle as orc
    from tests.test_gpu_fused import test_fused_silu_mul_external_operand as check
    monkeypatch.setenv("QL_SEQ_PASSES", env)
    seen, run = [], ql.Seq.run

    def noted(seq):
        seen.append(seq.info.variant)
        run(seq)

    monkeypatch.setattr(ql.Seq, "run", noted)
    check(ql, ctx, orc, 16)
    assert seen == [variant]


@pytest.mark.parametrize("M,K,N,variant", [(2, 8320, 4224, 0), (3, 8320, 4224, 0), (4, 8320, 4224, 2), (2, 8192, 4224, 2), (2, 8320, 4096, 2)])
def test_deep_wide_passes_of_two_and_three_rows_keep_the_tiles(ctx, M, K, N, variant):
    """N -> K -> N in two passes of 16 MiB and more: at 2 and 3 rows a K above 8192 needs one workgroup a CU at most."""
    lay, alay = ql.ArenaLayout(), ql.ArenaLayout()
    descs = [ql.make_desc(*[lay.take(b) for b in ql.gptq_sizes(k, n, 128)], k, n, 128) for k, n in ((N, K), (K, N))]
    w = ctx.arena(lay.used)
    x, h, y = alay.take(M * N * 4), alay.take(M * K * 4), alay.take(M * N * 4)
    act = ctx.arena(alay.used)
    seq = ctx.seq(descs, w, act, [x, h], ql.DTYPE_F32, M, [h, y])
    assert seq.info.variant == variant and seq.info.kernel == ql.SEQ_TILES
    seq.destroy()
    act.release()
    w.release()


def test_inputs_of_a_pass_share_launches(ctx):
    """Ten linears on inputs of their own and one on an RMSNorm in one pass, a twelfth on the first one's output: a launch
    holds up to eight images of a kind."""
    from oracle import oracle as orc
    M, shapes = 6, [(256 if i % 2 else 384, 128 if i else 256) for i in range(10)] + [(640, 64), (256, 132)]
    g = [synth.gptq_linear(K, N, 128, seed=0x5E7, key=(i,)) for i, (K, N) in enumerate(shapes)]
    norm = 1 + 0.1 * synth.activations(1, 640, seed=0x5E8)[0]
    lay, alay = ql.ArenaLayout(), ql.ArenaLayout()
    offs = [[lay.take(a.nbytes) for a in (t.qweight, t.qzeros, t.scales)] for t in g]
    norm_off = lay.take(norm.nbytes)
    w = ctx.arena(lay.used)
    for t, o in zip(g, offs):
        for at, a in zip(o, (t.qweight, t.qzeros, t.scales)):
            w.write(at, a)
    w.write(norm_off, norm.astype(np.float32))
    x = [synth.activations(M, K, seed=0x5E9, key=(i,)) for i, (K, N) in enumerate(shapes[:11])]
    xo = [alay.take(a.nbytes) for a in x]
    yo = [alay.take(M * N * 4) for _, N in shapes]
    act = ctx.arena(alay.used)
    for o, a in zip(xo, x):
        act.write(o, a)
    fuse = [ql.make_fuse(norm_w_off=norm_off if i == 10 else None) for i in range(12)]
    descs = [ql.make_desc(*o, K, N, 128) for o, (K, N) in zip(offs, shapes)]
    seq = ctx.seq(descs, w, act, xo + [yo[0]], ql.DTYPE_F32, M, yo, fuse=fuse)
    assert seq.info.variant == 2 and seq.info.passes == 2
    assert seq.info.launches == 2 + 1 + 2 + 1 + 1        # images (plain, norm), products; then one of each
    for _ in range(2):
        seq.run()
        seq.status()
    y = [act.read(o, (M, N), np.float32) for o, (_, N) in zip(yo, shapes)]
    x[10] = orc.add_rmsnorm(x[10], norm.astype(np.float32), 1e-6)[1]
    for t, a, b in zip(g, x + [y[0]], y):
        ref = orc.gptq_linear(t.qweight, t.qzeros, t.scales, a, None, 128)
        ok, ma, mr = orc.check_tolerance(b, ref, 1e-5 * max(1.0, float(np.sqrt(np.mean(a.astype(np.float64) ** 2)))), 1e-4)
        assert ok, (ma, mr)
    seq.destroy()
    act.release()
    w.release()
