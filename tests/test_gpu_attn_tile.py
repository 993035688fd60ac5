"""GPU: attention of many query rows (ql_attention_decode's tiled form: M >= 96, D 64 or 128, past + M / 2
>= 896 for every key split that the other form would take, of which a few small heads have several)
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
    from oracle import oracle as orc
    M, H, KV, D, past = 100, 12, 6, 64, 900
    q, k, v = make(M, H, KV, D, past, 0xF1)
    clean = orc.attention_gqa_cache(q, k, v, H, KV, D, past)
    k[keys, 5] = np.nan                                       # of kv head 0
    got = attend(ctx, q, k, v, past, 1024)
    assert np.isnan(got[:, :2]).all()
    assert close(got[:, 2:], clean[:, 2:])


def attend64(q, k, v, past, rows):
    """Query rows `rows` in 64 bits."""
    M, H, D = q.shape
    KV = k.shape[1] // D
    out = np.empty((len(rows), H, D))
    for j, m in enumerate(rows):
        T = past + m + 1
        for h in range(H):
            g = h // (H // KV)
            s = k[:T, g * D:(g + 1) * D].astype(np.float64) @ q[m, h].astype(np.float64) / np.sqrt(D)
            p = np.exp(s - s.max())
            out[j, h] = p @ v[:T, g * D:(g + 1) * D].astype(np.float64) / p.sum()
    return out


# What two fp16 parts under a shared exponent cannot hold. With 900 cached positions rows below 50 see nothing of
# position 950 on, which lies in a block (896 .. 959) with keys that they see.
def _channel(q, k, f):
    q[..., 3] /= np.float32(f)
    k[:, 3] *= np.float32(f)


def _unweighted(q, k, v):
    q[..., 0], k[300, 0], v[300] = 1.0, -1e3, 1e9


def _small_weight(q, k, v):
    """The first block's values 2^30 larger under weights 2^-30 smaller."""
    q[..., 0], k[:64, 0] = 1.0, -30 * np.log(2) * np.sqrt(q.shape[-1])
    v[:64] *= np.float32(2.0 ** 30)


def _extremes(q, k, v):
    q *= np.float32(2.0 ** 90)
    k *= np.float32(2.0 ** -90)
    v *= np.float32(1e-30)


SPREADS = {
    "later_key": (lambda q, k, v: k.__setitem__((950, 5), 1e10), 50),
    "later_key_all": (lambda q, k, v: k.__setitem__(950, 1e8), 50),
    "later_value": (lambda q, k, v: v.__setitem__((950, 7), 1e9), 50),
    "later_values": (lambda q, k, v: v.__setitem__(slice(950, None), 1e8), 50),
    "unweighted_value": (_unweighted, 100),
    "key_channel": (lambda q, k, v: _channel(q, k, 1e8), 100),
    "query_channel": (lambda q, k, v: _channel(q, k, 1e-8), 100),
    "large_under_small_weight": (_small_weight, 100),
    "far_keys": (lambda q, k, v: k.__imul__(np.exp2(np.arange(len(k)) % 64 - 63).astype(np.float32)[:, None]), 100),
    "extremes": (_extremes, 100),
}


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("name", list(SPREADS))
def test_wide_ranges_keep_fp32_accuracy(ctx, name, D):
    """A row is as accurate beside values far from its own as without them: at most 1e-6 of its 2-norm from 64 bits, where
    fp32 sums of a thousand terms are about 2e-7 and lost parts 1e-5 and more."""
    M, H, KV, past = 100, 12, 6, 900
    q, k, v = make(M, H, KV, D, past, 0x5EED)
    change, upto = SPREADS[name]
    change(q, k, v)
    rows = range(0, upto, 7)
    got = attend(ctx, q, k, v, past, 1100)[list(rows)]
    ref = attend64(q, k, v, past, rows)
    err = np.linalg.norm(got - ref, axis=-1) / np.linalg.norm(ref, axis=-1)
    assert err.max() <= 1e-6, err.max()


def test_infinite_and_nan_values_stay_with_rows_that_see_them(ctx):
    """As test_rows_do_not_see_later_keys_values, in blocks that are computed in fp32, at a block's first key too."""
    from oracle import oracle as orc
    M, H, KV, D, past = 130, 12, 6, 128, 900
    q, k, v = make(M, H, KV, D, past, 0xBAD)
    clean = orc.attention_gqa_cache(q, k, v, H, KV, D, past)
    v[past + 40, 7], v[960, D + 2], k[past + 80, 2 * D + 1], k[past + 90, 3 * D] = np.inf, np.nan, np.nan, -np.inf
    got = attend(ctx, q, k, v, past, 1100)
    others = [d for d in range(D) if d not in (2, 7)]
    assert close(got[:, :4][..., others], clean[:, :4][..., others])
    assert close(got[:40, :2, 7], clean[:40, :2, 7]) and np.isposinf(got[40:, :2, 7]).all()
    assert close(got[:60, 2:4, 2], clean[:60, 2:4, 2]) and np.isnan(got[60:, 2:4, 2]).all()
    assert close(got[:80, 4:6], clean[:80, 4:6]) and np.isnan(got[80:, 4:6]).all()
    # a key of -inf: its score is -inf (weight 0) or +inf (NaN) by the sign of q; before it nothing shows
    assert close(got[:90, 6:8], clean[:90, 6:8])
    down = q[90:, 6:8, 0] > 0
    assert np.isfinite(got[90:, 6:8][down]).all() and np.isnan(got[90:, 6:8][~down]).all()
    assert close(got[:, 8:], clean[:, 8:])


@pytest.mark.parametrize("M,H,KV,D,past", [
    (96, 42, 6, 128, 848),     # the smallest call of the tiled form; seven heads; 96 * 7 = 5.25 row blocks
    (97, 6, 6, 64, 863),       # no grouping, ragged row block, T = 960 whole blocks
    (128, 32, 4, 64, 833),     # T = 961: one key in the last block
])
def test_tiled_attention_matches_oracle_where_keys_are_not_split(ctx, M, H, KV, D, past):
    assert ql.plan_attention(past + M, M, H, KV, D, past).nsplit == 1
    test_tiled_attention_matches_oracle(ctx, M, H, KV, D, past)


def test_few_rows_are_as_exact_as_the_general_form(ctx):
    """96 rows of 14 / 2 heads: the general form splits the keys in three, which makes its sums more exact (1.75e-7 from 64
    bits) than the tiles' (1.85e-7)."""
    M, H, KV, D, past = 96, 14, 2, 64, 912
    q, k, v = make(M, H, KV, D, past, 0xE44)
    ref = attend64(q, k, v, past, range(M))
    err = np.linalg.norm(attend(ctx, q, k, v, past, past + M) - ref) / np.linalg.norm(ref)
    assert err <= 1.8e-7, err
