"""GPU: chained prefill sequences in which fused inputs (RMSNorm, SiLU-mul) that only all-fused passes read are held in
fp16, and others in fp32: a pass that mixes fused and plain inputs, an input shared with such a pass, and all-fused
passes before and after. Every linear against the oracle on the GPU's own inputs, as test_prefill_chained_step."""
import numpy as np
import pytest

from tests.test_gpu_prefill import RTOL, flip_bound, x16
from webllm_amd import qlinear as ql
from webllm_amd import synth

pytestmark = pytest.mark.gpu

EPS = 1e-6


@pytest.fixture(scope="module")
def ctx():
    c = ql.Context(0)
    yield c
    c.destroy()


# name: (K, N, reads, norm weight, second operand, residual); h is the external input
LINEARS = {
    "a": (384, 256, "h", 0, None, None),          # all fused: fp16
    "b": (256, 512, "a", 1, None, None),          # beside c, which reads a as it is: a's RMSNorm stays fp32
    "c": (256, 512, "a", None, None, None),
    "d": (256, 512, "a", 1, None, "b"),           # a later pass, all fused, on the same RMSNorm of a: fp32 too
    "e": (512, 128, "d", None, "c", None),        # SiLU-mul, all fused: fp16
    "f": (128, 384, "e", 2, None, "h"),           # RMSNorm of e: fp16
}


@pytest.mark.parametrize("M", [17, 40, 300])
def test_mixed_passes(ctx, M):
    from oracle import oracle as orc
    lay, alay = ql.ArenaLayout(), ql.ArenaLayout()
    t = {n: synth.gptq_linear(K, N, 128, seed=0x4A1F, key=(i,), stored_zero=None if i % 2 else 7)
         for i, (n, (K, N, *_)) in enumerate(LINEARS.items())}
    offs = {n: [lay.take(v.nbytes) for v in (l.qweight, l.qzeros, l.scales)] for n, l in t.items()}
    norms = [1 + 0.1 * synth.activations(1, C, seed=0x4A20, key=(C,))[0] for C in (384, 256, 128)]
    norm_off = [lay.take(v.nbytes) for v in norms]
    w = ctx.arena(lay.used)
    for n, l in t.items():
        for o, v in zip(offs[n], (l.qweight, l.qzeros, l.scales)):
            w.write(o, v)
    for o, v in zip(norm_off, norms):
        w.write(o, v.astype(np.float32))
    at = {"h": alay.take(M * 384 * 4)}
    for n, (K, N, *_) in LINEARS.items():
        at[n] = alay.take(M * N * 4)
    act = ctx.arena(alay.used)
    act.write(at["h"], synth.activations(M, 384, seed=0x4A21))
    fuse = [ql.make_fuse(norm_w_off=None if nw is None else norm_off[nw], norm_eps=EPS, x2_off=None if x2 is None else at[x2],
                         res_off=None if r is None else at[r]) for _, _, _, nw, x2, r in LINEARS.values()]
    descs = [ql.make_desc(*offs[n], K, N, 128) for n, (K, N, *_) in LINEARS.items()]
    seq = ctx.seq(descs, w, act, [at[l[2]] for l in LINEARS.values()], ql.DTYPE_F32, M, [at[n] for n in LINEARS], fuse=fuse)
    assert seq.info.kernel == ql.SEQ_PREFILL_PASSES and seq.info.passes == 5
    seq.run()
    seq.status()
    y = {"h": act.read(at["h"], (M, 384), np.float32)}
    for n, (K, N, *_) in LINEARS.items():
        y[n] = act.read(at[n], (M, N), np.float32)
    for n, (K, N, src, nw, x2, r) in LINEARS.items():
        x = y[src]
        if nw is not None:
            x = orc.add_rmsnorm(x, norms[nw].astype(np.float32), EPS)[1]
        if x2 is not None:
            x = orc.silu_mul(x, y[x2])
        ref = orc.gptq_linear_cols(t[n].qweight, t[n].qzeros, t[n].scales, x16(x), np.arange(N, dtype=np.int32), None, 128, w_f16=True)
        if r is not None:
            ref = ref + y[r]
        w16 = orc.f16_bits_to_f32(orc.dequantize_gptq_int4_f16(t[n].qweight, t[n].qzeros, t[n].scales, K, N, 128))
        bar = 1e-5 * max(1.0, float(np.sqrt(np.mean(x.astype(np.float64) ** 2)))) + RTOL * np.abs(ref) + flip_bound(x, w16)
        err = np.abs(y[n].astype(np.float64) - ref)
        assert np.isfinite(y[n]).all() and (err <= bar).all(), f"M={M} {n}: {float((err - bar).max()):.3e} over"
    first = {n: v.copy() for n, v in y.items()}
    seq.run()
    seq.status()
    for n, (K, N, *_) in LINEARS.items():
        assert np.array_equal(act.read(at[n], (M, N), np.float32).view(np.uint32), first[n].view(np.uint32))
    seq.destroy()
    act.release()
    w.release()
