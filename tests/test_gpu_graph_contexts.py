"""GPU: graphs whose calls pass data through a workspace (images of x, attention splits), launched on another context's
stream beside the capturing context's own work, and after that context is gone. Every replay has the eager call's bits."""
import numpy as np
import pytest

from webllm_amd import qlinear as ql
from webllm_amd import synth

pytestmark = pytest.mark.gpu


class Work:
    """A call on buffers of its own, in two versions (inputs 0 and 1); the arenas are the second context's."""

    def __init__(self, owner, arrays, out_shape, call):
        lay = ql.ArenaLayout()
        self.offs = [[lay.take(a.nbytes) for a in arrays(v)] for v in (0, 1)]
        n = int(np.prod(out_shape)) * 4
        self.out = [lay.take(n) for _ in (0, 1)]
        scratch = lay.take(8 << 20)
        self.arena, self.shape = owner.arena(lay.used), out_shape
        for v in (0, 1):
            for o, a in zip(self.offs[v], arrays(v)):
                self.arena.write(o, a)
        self.call = lambda c, v: call(c, self.arena, self.offs[v], self.out[v], scratch)

    def read(self, v):
        return self.arena.read(self.out[v], self.shape, np.float32).view(np.uint32)


def attention(owner, M, H, KV, D, past):
    T = past + M
    def arrays(v):
        g = np.random.default_rng(90 + v)
        return [g.standard_normal((M, H, D)).astype(np.float32)] + [g.standard_normal((T, KV * D)).astype(np.float32) for _ in range(2)]
    return Work(owner, arrays, (M, H * D), lambda c, a, o, y, s: c.attention_decode(a, o[0], a, o[1], o[2], T, M, H, KV, D, past, y))


def head(owner, M, K, N):
    def arrays(v):
        g = np.random.default_rng(70 + v)
        return [g.standard_normal((M, K)).astype(np.float32), (0.02 * g.standard_normal((N, K))).astype(np.float16)]
    return Work(owner, arrays, (M, N), lambda c, a, o, y, s: c.gemv_f16w(a, o[1], None, a, o[0], M, N, K, y))


def linear(owner, M, K, N, noalloc=False):
    t = synth.gptq_linear(K, N, 128, seed=0x6A7)
    def arrays(v):
        return [np.random.default_rng(50 + v).standard_normal((M, K)).astype(np.float32), t.qweight, t.qzeros, t.scales]
    def call(c, a, o, y, s):
        d = ql.make_desc(o[1], o[2], o[3], K, N, 128)
        if noalloc:
            c.linear_noalloc(d, a, a, o[0], ql.DTYPE_F32, M, y)
        else:
            c.linear(d, a, a, o[0], ql.DTYPE_F32, M, y, s)
    return Work(owner, arrays, (M, N), call)


KINDS = {
    "linear_image": lambda c: [linear(c, 8, 896, 896)],
    "linear_rows": lambda c: [linear(c, 77, 896, 1024)],
    "noalloc": lambda c: [linear(c, 8, 896, 896, noalloc=True)],
    "head": lambda c: [head(c, 64, 896, 2048)],
    "attention_split": lambda c: [attention(c, 1, 4, 2, 64, 2000)],
    "attention_tiles": lambda c: [attention(c, 96, 6, 6, 64, 900)],
    # small, large and small workspaces in one graph
    "several": lambda c: [linear(c, 8, 896, 896), head(c, 64, 896, 2048), attention(c, 96, 6, 6, 64, 900), linear(c, 77, 896, 1024),
                          attention(c, 1, 4, 2, 64, 2000)],
}


@pytest.mark.parametrize("kind", list(KINDS))
def test_graph_on_another_context(kind):
    a, b = ql.Context(0), ql.Context(0)
    works = KINDS[kind](b)
    want = []
    for w in works:
        for v in (0, 1):
            w.call(b, v)
        b.sync()
        want.append([w.read(v) for v in (0, 1)])
    a.graph_begin()
    for w in works:
        w.call(a, 0)
    g = a.graph_end()
    a._owned.discard(g)
    def clear():
        for w in works:
            for v in (0, 1):
                w.arena.write(w.out[v], np.zeros(w.shape, np.float32))
    def check(versions):
        for w, e in zip(works, want):
            for v in versions:
                assert np.array_equal(w.read(v), e[v])
    for _ in range(6):
        clear()
        ql._check(ql.lib().ql_graph_launch(b.handle, g.handle))
        if kind != "noalloc":                                  # its calls share one array: they must not overlap
            for w in works:
                w.call(a, 1)
        else:
            b.sync()
            for w in works:
                w.call(a, 1)
        a.sync()
        b.sync()
        check((0, 1))
    a.destroy()
    for _ in range(2):
        clear()
        ql._check(ql.lib().ql_graph_launch(b.handle, g.handle))
        b.sync()
        check((0,))
    ql._check(ql.lib().ql_graph_destroy(g.handle))
    g.handle = None
    for w in works:
        w.arena.release()
    b.destroy()
