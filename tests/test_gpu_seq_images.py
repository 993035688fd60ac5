"""GPU: chained decode sequences that run their passes as products over activation images (ql_seq_get_info variant 2:
M = 5..16, or 2..4 with 16 MiB of weights a pass), every linear against the oracle on the GPU's own inputs, as the tiles'
tests check them; repeats and graph replays give the same bits."""
import numpy as np
import pytest

from tests.test_gpu_fused import FusedModel, _sample, check_fused
from tests.test_gpu_seq import SeqModel, check_all
from webllm_amd import qlinear as ql

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
