"""GPU: attention of many query rows (ql_attention_decode's tiled form: M >= 96, past + M / 2 >= 896, D 64 or 128)
against the oracle's attentionGqaRef restatement, at the reference's attention bar, at the edges of its tiles (blocks of
64 keys, 128 (row, head) pairs, key splits) and with infinities and NaN in keys that only later rows see."""
import numpy as np
import pytest

from webllm_amd import qlinear as ql

pytestmark = pytest.mark.gpu

ATOL, RTOL = 1e-5, 1e-4


@pytest.fixture(scope="module")
def ctx():
    c = ql.Context(0)
    yield c
    c.destroy()


def attend(ctx, q, k, v, past, max_t):
    M, H, D = q.shape
    KV = k.shape[1] // D
    lay = ql.ArenaLayout()
    q_off, o_off, end = lay.take(q.nbytes), lay.take(q.nbytes), lay.take(256)
    act = ctx.arena(lay.used)
    act.write(q_off, q)
    guard = np.full(64, 7.25, np.float32)
    act.write(end, guard)
    clay = ql.ArenaLayout()
    k_off, v_off = clay.take(max_t * KV * D * 4), clay.take(max_t * KV * D * 4)
    cache = ctx.arena(clay.used)
    junk = np.full((max_t, KV * D), np.nan, np.float32)      # positions past the context hold anything
    for off, t in ((k_off, k), (v_off, v)):
        junk[:len(t)] = t
        cache.write(off, junk)
    ctx.attention_decode(act, q_off, cache, k_off, v_off, max_t, M, H, KV, D, past, o_off)
    out = act.read(o_off, (M, H, D), np.float32)
    ctx.attention_decode(act, q_off, cache, k_off, v_off, max_t, M, H, KV, D, past, o_off)
    assert np.array_equal(act.read(o_off, (M, H, D), np.float32).view(np.uint32), out.view(np.uint32))
    assert np.array_equal(act.read(end, (64,), np.float32), guard)
    act.release()
    cache.release()
    return out


def close(got, ref):
    return np.all(np.abs(got - ref) <= ATOL + RTOL * np.abs(ref))


def make(M, H, KV, D, past, seed):
    rng = np.random.default_rng(seed)
    T = past + M
    return (rng.standard_normal((M, H, D)).astype(np.float32), rng.standard_normal((T, KV * D)).astype(np.float32),
            rng.standard_normal((T, KV * D)).astype(np.float32))


CASES = [
    # (M, H, KV, D, past)
    (96, 7, 1, 128, 848),      # the smallest call of the tiled form; seven heads; 96 * 7 = 5.25 row blocks
    (97, 2, 2, 64, 863),       # no grouping, ragged row block, T = 960 whole blocks
    (128, 8, 1, 64, 833),      # T = 961: one key in the last block
    (200, 3, 3, 128, 1000),    # several key splits
    (1793, 1, 1, 64, 0),       # from position 0: first rows see one key, splits without a visible key
    (130, 14, 2, 64, 2000),
]


@pytest.mark.parametrize("M,H,KV,D,past", CASES)
def test_tiled_attention_matches_oracle(ctx, M, H, KV, D, past):
    from oracle import oracle as orc
    q, k, v = make(M, H, KV, D, past, 0xA77 + M)
    k[5] *= 1e-4                                              # a key and a value far below their block's
    v[:, 3] *= 1e-6
    v[:, 4] *= 1e6
    got = attend(ctx, q, k, v, past, past + M + 3)
    ref = orc.attention_gqa_cache(q, k, v, H, KV, D, past)
    plain = [d for d in range(D) if d not in (3, 4)]
    assert close(got[..., plain], ref[..., plain])            # the bar is one of values of order 1
    for d in (3, 4):                                          # the small and the large column by their own size
        assert np.linalg.norm(got[..., d] - ref[..., d]) <= 1e-5 * np.linalg.norm(ref[..., d])


def test_rows_do_not_see_later_keys_values(ctx):
    """An infinity or a NaN in a key or value is seen by its own and later rows only, as in the row-per-workgroup form."""
    from oracle import oracle as orc
    M, H, KV, D, past = 100, 6, 2, 64, 900
    q, k, v = make(M, H, KV, D, past, 0xBAD)
    clean = orc.attention_gqa_cache(q, k, v, H, KV, D, past)
    v[past + 40, 7], v[past + 60, D + 2], k[past + 80, 1] = np.inf, np.nan, np.nan
    got = attend(ctx, q, k, v, past, 1024)
    assert close(got[:40], clean[:40])
    assert not np.isfinite(got[40:, :3, 7]).any() and close(got[40:80, :3, :7], clean[40:80, :3, :7])
    assert np.isnan(got[60:, 3:, 2]).all() and close(got[:, 3:, 3:], clean[:, 3:, 3:])
    assert np.isnan(got[80:, :3]).all()


@pytest.mark.parametrize("keys", [slice(0, 1), slice(256, 257), slice(256, 384), slice(0, 1000)],
                         ids=["first_key", "first_of_a_split", "a_whole_split", "all"])
def test_nan_key_reaches_every_row_that_sees_it(ctx, keys):
    """A NaN score makes its row NaN wherever the key lies: as the first key of all or of a key split (of 128 keys here),
    where no other score has been seen yet, and where a split has no other."""
    M, H, KV, D, past = 100, 6, 2, 64, 900
    q, k, v = make(M, H, KV, D, past, 0xF1)
    k[keys, 5] = np.nan                                       # of kv head 0
    got = attend(ctx, q, k, v, past, 1024)
    assert np.isnan(got[:, :3]).all()
    from oracle import oracle as orc
    clean = orc.attention_gqa_cache(q[:, 3:], np.ascontiguousarray(k[:, D:]), np.ascontiguousarray(v[:, D:]), 3, 1, D, past)
    assert close(got[:, 3:], clean)
