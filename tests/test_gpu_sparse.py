"""Sparse selection on the GPU: MiniMax-M3's block lists and indexer, GLM's cell pools - against the oracle (pinned in
tests/test_oracle_sparse.py). Attention within max-abs 2e-3 / relative L2 1e-3 of the oracle's float32 result; the
selection itself (comparisons only) bit for bit."""
import time

import numpy as np
import pytest

from nextsycl_amd import DevBuf, Error
from oracle import orc

pytestmark = pytest.mark.gpu


def close(got, want):
    err = np.abs(got - want).max()
    rel = np.linalg.norm((got - want).ravel()) / max(np.linalg.norm(want.ravel()), 1e-30)
    assert err <= 2e-3 and rel <= 1e-3, (err, rel)


@pytest.mark.parametrize("T,H,G,pos0,K", [(1, 8, 2, 2000, 6), (3, 64, 4, 5000, 16), (2, 16, 1, 300, 4)])
def test_minimaxm3_block_lists(ops, T, H, G, pos0, K):
    g = ops.gpu
    n = pos0 + T
    nblk = (n + 127) // 128
    q = orc.randn(41, (T, H * 128))
    kc, _ = orc.randn_f16(42, (n, G, 128)); vc, _ = orc.randn_f16(43, (n, G, 128))
    rng = np.random.default_rng(5)
    sel = np.stack([np.stack([rng.permutation(nblk)[:K] if K <= nblk else np.r_[rng.permutation(nblk), [-1] * (K - nblk)] for _ in range(G)])
                    for _ in range(T)]).astype(np.int32)
    sel[0, 0, 1] = -1                                   # a hole
    sel[-1, -1, 0] = nblk - 1                           # the block the row's own position cuts
    scale = 0.0884
    out = DevBuf(g, T * H * 128 * 4); out.fill(0xFF)
    ops.minimaxm3_attend(DevBuf.of(g, q), DevBuf.of(g, kc), DevBuf.of(g, vc), out, T, H, G, pos0, scale, sel=DevBuf.of(g, sel), K=K)
    want = orc.mm3_attend(q, kc, vc, T, H, G, pos0, scale, sel=sel, K=K)
    close(out.read(np.float32).reshape(T, H * 128), want)
    # every block listed in order = the dense pass
    allb = np.tile(np.arange(nblk, dtype=np.int32), (T, G, 1))
    out2 = DevBuf(g, T * H * 128 * 4)
    ops.minimaxm3_attend(DevBuf.of(g, q), DevBuf.of(g, kc), DevBuf.of(g, vc), out2, T, H, G, pos0, scale, sel=DevBuf.of(g, allb), K=nblk)
    close(out2.read(np.float32).reshape(T, H * 128), orc.mm3_attend(q, kc, vc, T, H, G, pos0, scale))
    # nothing listed: zeros
    none = np.full((T, G, 2), -1, np.int32)
    ops.minimaxm3_attend(DevBuf.of(g, q), DevBuf.of(g, kc), DevBuf.of(g, vc), out2, T, H, G, pos0, scale, sel=DevBuf.of(g, none), K=2)
    assert not out2.read(np.float32).any()


@pytest.mark.parametrize("T,H,G,pos0,K", [(40, 32, 2, 3000, 5), (300, 64, 4, 700, 16), (8200, 64, 4, 1000, 2)])
def test_minimaxm3_block_lists_of_a_prompt(ops, tune, T, H, G, pos0, K):
    """A prompt pass with block lists: every (row, key group) is a unit of one launch, the rows' keys are cut only while
    the units are few, and a pass whose partials outgrow the library's scratch (the last case: 8200 rows x 64 heads with
    256 MiB of it to plan with) goes in several launches. Sampled rows against the oracle's one-row pass at their positions."""
    g = ops.gpu
    if T > 8000:
        tune(6, 256)
    n = pos0 + T
    q = orc.randn(51, (T, H * 128))
    kc, _ = orc.randn_f16(52, (n, G, 128)); vc, _ = orc.randn_f16(53, (n, G, 128))
    rng = np.random.default_rng(9)
    sel = np.full((T, G, K), -1, np.int32)
    for t in range(T):
        nb = (pos0 + t) // 128 + 1                                    # blocks the row can see, its own included
        for gi in range(G):
            pick = rng.permutation(nb)[:K]
            sel[t, gi, :len(pick)] = pick
    sel[T // 2, 0, 0] = -1                                            # a hole
    out = DevBuf(g, T * H * 128 * 4); out.fill(0xFF)
    ops.minimaxm3_attend(DevBuf.of(g, q), DevBuf.of(g, kc), DevBuf.of(g, vc), out, T, H, G, pos0, 0.0884, sel=DevBuf.of(g, sel), K=K)
    got = out.read(np.float32).reshape(T, H * 128)
    assert np.isfinite(got).all()
    rows = sorted(set([0, 1, T // 2, T - 2, T - 1] + [int(t) for t in rng.integers(0, T, 12)]))
    for t in rows:
        want = orc.mm3_attend(q[t:t + 1], kc[:pos0 + t + 1], vc[:pos0 + t + 1], 1, H, G, pos0 + t, 0.0884, sel=sel[t:t + 1], K=K)
        close(got[t:t + 1], want)


@pytest.mark.parametrize("T,H,G,pos0,K", [(17, 8, 2, 0, 3), (18, 48, 3, 1000, 70), (33, 40, 2, 700, 4), (200, 20, 4, 130, 16), (767, 2, 1, 0, 2), (769, 4, 1, 300, 5), (1023, 4, 2, 300, 2),
                                            (17, 16, 1, 5000, 24), (17, 8, 1, 9000, 70), (18, 36, 3, 9000, 130), (32, 16, 1, 3000, 130),
                                            (270, 12, 3, 9000, 70)])
def test_minimaxm3_block_lists_row_kernel(ops, T, H, G, pos0, K):
    """Where the row kernel can go wrong: rows that see part of one block, head groups short of a matrix tile and one past it
    (20 heads: the other kernel), key heads that do not divide the XCDs, lists longer than a wave's 64 entries with holes,
    repeats and blocks wholly past the row, both sides of the rule between a work-group and a wave a (row, head), and of the one
    that leaves few pairs of long lists to the decode kernel's splits."""
    g = ops.gpu
    n = pos0 + T
    q = orc.randn(61, (T, H * 128))
    kc, _ = orc.randn_f16(62, (n, G, 128)); vc, _ = orc.randn_f16(63, (n, G, 128))
    rng = np.random.default_rng(T)
    sel = rng.integers(-1, (n + 127) // 128, (T, G, K)).astype(np.int32)          # holes, repeats, blocks past early rows
    sel[:, :, 0] = (pos0 + np.arange(T))[:, None] // 128                          # and the row's own block
    sel[T // 3] = -1                                                              # a row with nothing listed
    out = DevBuf(g, T * H * 128 * 4); out.fill(0xFF)
    ops.minimaxm3_attend(DevBuf.of(g, q), DevBuf.of(g, kc), DevBuf.of(g, vc), out, T, H, G, pos0, 0.0884, sel=DevBuf.of(g, sel), K=K)
    got = out.read(np.float32).reshape(T, H * 128)
    assert not got[T // 3].any()
    for t in sorted({0, 1, 3, T // 3 + 1, T // 2, T - 2, T - 1} | {int(t) for t in rng.integers(0, T, 8)}):
        want = orc.mm3_attend(q[t:t + 1], kc[:pos0 + t + 1], vc[:pos0 + t + 1], 1, H, G, pos0 + t, 0.0884, sel=sel[t:t + 1], K=K)
        close(got[t:t + 1], want)


@pytest.mark.parametrize("T,H,G,pos0,K", [(40, 32, 2, 2000, 9), (260, 24, 3, 900, 5)])
def test_minimaxm3_block_lists_row_kernel_keeps_float32_weights(ops, T, H, G, pos0, K):
    """With queries that are halfs as they are, the row kernel (a work-group a (row, head), a wave) has no rounding to half
    left: its weights carry 22 bits. What remains is float32: a score's error is at most 130 2^-24 of the sum of its
    products' sizes - 7.2 after the scale for standard normal rows of 128 -, and moves its weight by that share: 6e-5. One
    half a weight gives 2e-4."""
    g = ops.gpu
    n = pos0 + T
    qh, q = orc.randn_f16(81, (T, H * 128))
    kc, kf = orc.randn_f16(82, (n, G, 128)); vc, vf = orc.randn_f16(83, (n, G, 128))
    q, kf, vf = (np.asarray(a, np.float64) for a in (q, kf, vf))
    rng = np.random.default_rng(T)
    sel = np.stack([np.stack([rng.permutation((pos0 + t) // 128 + 1)[:K] for _ in range(G)]) for t in range(T)]).astype(np.int32)
    out = DevBuf(g, T * H * 128 * 4); out.fill(0xFF)
    ops.minimaxm3_attend(DevBuf.of(g, q.astype(np.float32)), DevBuf.of(g, kc), DevBuf.of(g, vc), out, T, H, G, pos0, 0.0884, sel=DevBuf.of(g, sel), K=K)
    got = out.read(np.float32).reshape(T, G, H // G, 128)
    q, kf, vf = q.reshape(T, G, H // G, 128), kf.reshape(n, G, 128), vf.reshape(n, G, 128)
    for t in range(0, T, 13):
        for gi in range(G):
            keys = (sel[t, gi][:, None] * 128 + np.arange(128)).ravel()
            keys = keys[keys <= pos0 + t]
            s = q[t, gi] @ kf[keys, gi].T * float(np.float32(0.0884))
            w = np.exp(s - s.max(1, keepdims=True))
            want = w @ vf[keys, gi] / w.sum(1, keepdims=True)
            rel = np.linalg.norm(got[t, gi] - want) / np.linalg.norm(want)
            assert rel <= 6e-5, (t, gi, rel)


@pytest.mark.parametrize("T,H,G", [(17, 8, 2), (40, 4, 1), (800, 4, 1)])
def test_minimaxm3_block_lists_row_kernel_of_infinite_values(ops, T, H, G):
    """An infinite value gives its feature the infinity of its sign, two of opposite signs and a NaN give NaN, in every row
    that lists them - in a work-group a (row, head), a wave -, and the other features stay what they are: float32's rules. (All
    weights lie within e^3 of each other, so none rounds to a half of 0.)"""
    g = ops.gpu
    pos0 = 512
    n = pos0 + T
    q = orc.randn(67, (T, H * 128), 0.3)
    kc, _ = orc.randn_f16(68, (n, G, 128), 0.3); vc, _ = orc.randn_f16(69, (n, G, 128))
    vc[5, :, 3], vc[130, :, 40], vc[131, :, 41], vc[300, :, 41], vc[301, :, 127] = 0x7C00, 0xFC00, 0x7C00, 0xFC00, 0x7E00
    sel = np.broadcast_to(np.array([2, 0, 1], np.int32), (T, G, 3)).copy()
    sel[1::2] = [3, 1, -1]                                                        # every other row: not the first and third block
    out = DevBuf(g, T * H * 128 * 4); out.fill(0xFF)
    ops.minimaxm3_attend(DevBuf.of(g, q), DevBuf.of(g, kc), DevBuf.of(g, vc), out, T, H, G, pos0, 0.0884, sel=DevBuf.of(g, sel), K=3)
    got = out.read(np.float32).reshape(T, H, 128)
    zeroed = np.where((vc & 0x7C00) == 0x7C00, 0, vc).astype(np.uint16)
    want = orc.mm3_attend(q, kc, zeroed, T, H, G, pos0, 0.0884, sel=sel, K=3).reshape(T, H, 128)
    want[::2, :, 3], want[::2, :, 127], want[::2, :, 41] = np.inf, np.nan, np.nan
    want[:, :, 40] = -np.inf
    want[1::2, :, 41] = np.inf
    fin = np.isfinite(want)
    assert np.array_equal(got[~fin], want[~fin], equal_nan=True)
    close(got[fin], want[fin])


@pytest.mark.parametrize("T,H,G", [(17, 8, 2), (40, 4, 1), (800, 4, 1)])
def test_minimaxm3_block_lists_row_kernel_of_infinite_and_nan_scores(ops, T, H, G):
    """A score of +inf or NaN leaves a (row, head) no sum of weights: zeros, as in the reference. One of -inf is a weight of 0."""
    g = ops.gpu
    pos0 = 512
    n = pos0 + T
    q = orc.randn(67, (T, H * 128), 0.3)
    kc, _ = orc.randn_f16(68, (n, G, 128), 0.3); vc, _ = orc.randn_f16(69, (n, G, 128))
    kc[5, :, 2], kc[300, :, 7] = 0x7C00, 0x7E00                                    # blocks 0 and 2
    sel = np.broadcast_to(np.array([1, 0, 3], np.int32), (T, G, 3)).copy()
    sel[1::3] = [3, 2, 1]
    sel[2::3] = [3, 1, -1]
    out = DevBuf(g, T * H * 128 * 4); out.fill(0xFF)
    ops.minimaxm3_attend(DevBuf.of(g, q), DevBuf.of(g, kc), DevBuf.of(g, vc), out, T, H, G, pos0, 0.0884, sel=DevBuf.of(g, sel), K=3)
    got = out.read(np.float32).reshape(T * H, 128)
    want = orc.mm3_attend(q, kc, vc, T, H, G, pos0, 0.0884, sel=sel, K=3).reshape(T * H, 128)
    none = ~want.any(1)
    assert none.reshape(T, H)[1::3].all() and not none.reshape(T, H)[2::3].any() and 0 < none.reshape(T, H)[::3].mean() < 1
    assert not got[none].any()
    close(got[~none], want[~none])


@pytest.mark.parametrize("T,H,G", [(17, 8, 2), (800, 4, 1)])
def test_minimaxm3_block_lists_row_kernel_output_at_any_float(ops, T, H, G):
    """Output rows at an address that is a float's and no more: the rows of an aligned output, bit for bit, and nothing beside."""
    g = ops.gpu
    q = DevBuf.of(g, orc.randn(64, (T, H * 128)))
    kc, vc = DevBuf.of(g, orc.randn_f16(65, (T, G, 128))[0]), DevBuf.of(g, orc.randn_f16(66, (T, G, 128))[0])
    sel = DevBuf.of(g, np.broadcast_to(np.arange(3, dtype=np.int32), (T, G, 3)).copy())
    n = T * H * 128
    want, room = DevBuf(g, n * 4), DevBuf(g, (n + 4) * 4)
    ops.minimaxm3_attend(q, kc, vc, want, T, H, G, 0, 0.0884, sel=sel, K=3)
    for at in (1, 2, 3):
        room.fill(0xFF)
        ops.minimaxm3_attend(q, kc, vc, room.view(4 * at, n * 4), T, H, G, 0, 0.0884, sel=sel, K=3)
        got = room.read(np.uint32)
        assert np.array_equal(got[at:at + n], want.read(np.uint32))
        assert (got[:at] == 0xFFFFFFFF).all() and (got[at + n:] == 0xFFFFFFFF).all()


def test_minimaxm3_block_lists_refuse_more_key_heads_than_a_launch_holds(ops):
    """Key heads past 65535 are refused whatever the rows (a position's row then spans 16 MiB, the limit of the row kernel's offsets)."""
    g = ops.gpu
    T, G = 17, 65536
    q, out, kc, vc = DevBuf(g, T * G * 512), DevBuf(g, T * G * 512), DevBuf(g, T * G * 256), DevBuf(g, T * G * 256)
    sel = DevBuf.of(g, np.zeros((T, G, 1), np.int32))
    with pytest.raises(Error, match="too many key heads|more scratch"):
        ops.minimaxm3_attend(q, kc, vc, out, T, G, G, 0, 0.0884, sel=sel, K=1)


def test_minimaxm3_indexer(ops):
    g = ops.gpu
    T, G, pos0, local, K = 3, 2, 3000, 2, 8
    n = pos0 + T
    nblk = (n + 127) // 128 + 1                         # one block wholly past the rows
    iq = orc.randn(44, (T, G, 128)); ik, _ = orc.randn_f16(45, (n, 128))
    bs = DevBuf(g, T * G * nblk * 4)
    ops.minimaxm3_idx_scores(DevBuf.of(g, iq), DevBuf.of(g, ik), bs, T, G, nblk, pos0, local)
    got = bs.read(np.float32).reshape(T, G, nblk)
    want = orc.mm3_idx_scores(iq, ik, T, G, nblk, pos0, local)
    fin = np.isfinite(want) & (want < 1e29)
    assert np.array_equal(np.isneginf(got), np.isneginf(want)) and np.array_equal(got > 1e29, want > 1e29)
    assert np.abs(got[fin] - want[fin]).max() < 1e-4
    # selection on the GPU's own scores against the oracle's selection on the same scores: bit for bit
    sel = DevBuf(g, T * G * K * 4)
    ops.minimaxm3_idx_topk(bs, sel, T, G, nblk, K)
    want_sel, want_left = orc.mm3_idx_topk(got, K)
    assert np.array_equal(sel.read(np.int32).reshape(T, G, K), want_sel)
    assert np.array_equal(bs.read(np.float32).reshape(T, G, nblk).view(np.uint32), want_left.view(np.uint32))
    # ties and exhaustion
    sc = np.array([[[1.0, 7.0, 7.0, -np.inf, 3.0, 7.0]]], np.float32)
    b2, s2 = DevBuf.of(g, sc), DevBuf(g, 6 * 4)
    ops.minimaxm3_idx_topk(b2, s2, 1, 1, 6, 6)
    assert s2.read(np.int32).tolist() == [1, 2, 5, 4, 0, -1]


@pytest.mark.parametrize("T,G,pos0,extra,local", [(1, 1, 0, 0, 1), (1, 2, 255, 1, 0), (2, 1, 127, 2, 1), (2, 1, 3000, 0, 0), (3, 1, 700, 0, 1), (1, 4, 127, 1, 0), (4, 4, 126, 2, 1), (5, 4, 640, 0, 2), (17, 3, 1000, 1, 1), (33, 4, 5000, 3, 1), (300, 2, 90, 0, 1)])
def test_minimaxm3_index_scores_keep_float32_queries(ops, T, G, pos0, extra, local):
    """Block scores against the float64 product of the same operands, for queries whose features span ten orders of magnitude:
    within a float32 sum's own rounding, 130 2^-24 of the sum of the products' sizes (128 additions, the scale, the query's
    last bit). Edges of the query tiles, the blocks and the slices."""
    g = ops.gpu
    n = pos0 + T
    nblk = (n + 127) // 128 + extra
    rng = np.random.default_rng(pos0 + T)
    iq = (orc.randn(71, (T, G, 128)) * 10.0 ** rng.uniform(-6, 4, (T, G, 128))).astype(np.float32)
    ik, _ = orc.randn_f16(72, (n, 128))
    bs = DevBuf(g, T * G * nblk * 4); bs.fill(0xFF)
    ops.minimaxm3_idx_scores(DevBuf.of(g, iq), DevBuf.of(g, ik), bs, T, G, nblk, pos0, local)
    got = bs.read(np.float32).reshape(T, G, nblk)
    k64 = np.asarray(orc.h2f(ik), np.float64).reshape(n, 128)
    for t in range(T):
        pos = pos0 + t
        own = pos // 128
        s = iq[t].astype(np.float64) @ k64[:pos + 1].T                            # [G][pos + 1]
        size = np.abs(iq[t].astype(np.float64)) @ np.abs(k64[:pos + 1]).T
        assert np.isneginf(got[t, :, own + 1:]).all()
        assert (got[t, :, max(0, own + 1 - local):own + 1] > 1e29).all()
        for b in range(0, own + 1 - local):
            lo, hi = 128 * b, min(pos + 1, 128 * b + 128)
            assert (np.abs(got[t, :, b] - s[:, lo:hi].max(1)) <= 130 * 2.0 ** -24 * size[:, lo:hi].max(1)).all(), (t, b)


@pytest.mark.parametrize("T,G,pos0,local", [(200, 4, 16000, 1), (130, 4, 30000, 0)])
def test_minimaxm3_index_scores_of_slices_of_many_tiles(ops, T, G, pos0, local):
    """Passes whose slices hold several query tiles (50 tiles of 32 block groups: 4 a slice; 33 of 59: 5, the last slice shorter)
    against the same rows five at a time, a tile or two of one tile a slice: bit for bit, also behind keys with an infinity and a
    NaN, whose tiles take the float32 products."""
    g = ops.gpu
    n = pos0 + T
    nblk = (n + 127) // 128
    iq, kf = orc.randn(73, (T, G, 128)), orc.randn(74, (n, 128))
    kf[700, 3], kf[9000, 5], kf[pos0 + T // 2, 7] = np.nan, np.inf, -np.inf
    q, k = DevBuf.of(g, iq), DevBuf.of(g, orc.f2h(kf))
    bs = DevBuf(g, T * G * nblk * 4); bs.fill(0xFF)
    ops.minimaxm3_idx_scores(q, k, bs, T, G, nblk, pos0, local)
    got = bs.read(np.float32)
    want = DevBuf(g, T * G * nblk * 4); want.fill(0xFF)
    for t in range(0, T, 5):
        ops.minimaxm3_idx_scores(q.view(t * G * 512, 5 * G * 512), k, want.view(t * G * nblk * 4, 5 * G * nblk * 4), 5, G, nblk, pos0 + t, local)
    assert np.array_equal(got.view(np.uint32), want.read(np.uint32))


def _score_bounds(iq, k64, pos0, nblk):
    """[T][G][nblk]: the float64 block maxima (-inf past the row) and the largest sum of a block's products' sizes."""
    T, G, _ = iq.shape
    q = iq.astype(np.float64).reshape(T * G, 128)
    n = len(k64)
    s, size = np.full((T * G, nblk * 128), -np.inf), np.zeros((T * G, nblk * 128))
    s[:, :n], size[:, :n] = q @ k64.T, np.abs(q) @ np.abs(k64).T
    past = np.arange(nblk * 128)[None] > (pos0 + np.arange(T * G) // G)[:, None]
    s[past], size[past] = -np.inf, 0.0
    return s.reshape(T, G, nblk, 128).max(3), size.reshape(T, G, nblk, 128).max(3)


@pytest.mark.parametrize("T,G,pos0", [(1, 4, 700), (40, 2, 900)])
@pytest.mark.parametrize("up", [0, 10, 13, 16, 20, 24, 27, 28, 30, 40, 80, 126])
def test_minimaxm3_index_scores_keep_small_features(ops, T, G, pos0, up):
    """Features far below their row's largest, behind keys that are zero there: the scores are the small features', within a
    float32 sum's rounding of them (130 2^-24 of the sum of the products' sizes, which has no part of the large one). Rows of
    ordinary features share the tiles with such rows."""
    g = ops.gpu
    n = pos0 + T
    nblk = (n + 127) // 128
    iq = orc.randn(75, (T, G, 128))
    iq[::2, 0, 11] = 2.0 ** up
    iq[:, 1, 11] = -1.5 * 2.0 ** up
    iq[:, G - 1] *= np.float32(2.0 ** -20)                                        # (and rows of another size)
    kf = orc.randn(76, (n, 128))
    kf[:, 11] = 0.0
    ik = orc.f2h(kf)
    bs = DevBuf(g, T * G * nblk * 4); bs.fill(0xFF)
    ops.minimaxm3_idx_scores(DevBuf.of(g, iq), DevBuf.of(g, ik), bs, T, G, nblk, pos0, 0)
    got = bs.read(np.float32).reshape(T, G, nblk)
    want, size = _score_bounds(iq, np.asarray(orc.h2f(ik), np.float64).reshape(n, 128), pos0, nblk)
    fin = np.isfinite(want)
    assert np.array_equal(np.isneginf(got), ~fin)
    assert (np.abs(got[fin] - want[fin]) <= 130 * 2.0 ** -24 * size[fin]).all(), (np.abs(got[fin] - want[fin]) / size[fin]).max()


@pytest.mark.parametrize("G", [1, 2])
@pytest.mark.parametrize("q,big", [(2.0 ** -100, 2.0 ** 127), (2.0 ** -149, 2.0 ** 127), (2.0 ** -30, 2.0 ** 127), (1.7e38, 0.0)])
def test_minimaxm3_index_scores_of_one_feature(ops, q, big, G):
    """The smallest and largest float32 features, alone in their row and under a large feature that every key is zero in: the
    one product there is, as float32 gives it."""
    g = ops.gpu
    n = 256
    iq = np.zeros((2, G, 128), np.float32)
    iq[:, :, 5] = q
    iq[1, :, 90] = big
    kf = np.zeros((n, 128), np.float32)
    kf[:, 5] = np.arange(n) % 100 / 64.0
    bs = DevBuf(g, 2 * G * 2 * 4)
    ops.minimaxm3_idx_scores(DevBuf.of(g, iq), DevBuf.of(g, orc.f2h(kf)), bs, 2, G, 2, n - 2, 0)
    want = np.full((2 * G, 2), np.float32(q) * np.float32(99 / 64.0), np.float32)
    assert np.array_equal(bs.read(np.float32).reshape(2 * G, 2), want)


@pytest.mark.parametrize("T,G,pos0", [(1, 2, 1000), (1, 4, 1000), (40, 2, 900)])
def test_minimaxm3_index_scores_of_infinities_and_nans(ops, T, G, pos0):
    """An infinite feature of a key or a query gives the float32 product's score - also where the query's feature is far
    below its row's largest -, a NaN is no key's best, and finite queries and blocks beside them keep their scores."""
    g = ops.gpu
    n = pos0 + T
    nblk = (n + 127) // 128
    iq = orc.randn(73, (T, G, 128))
    iq[:, 0, 7] = 1e-12
    ik, _ = orc.randn_f16(74, (n, 128))
    ik[130, 7], ik[300, 7], ik[500, 3] = 0x7C00, 0xFC00, 0x7E00                   # blocks 1, 2, 3: inf, -inf, NaN
    if T > 1:
        iq[5, 1, 9], iq[21, 1, 9] = np.inf, np.nan
    bs = DevBuf(g, T * G * nblk * 4); bs.fill(0xFF)
    ops.minimaxm3_idx_scores(DevBuf.of(g, iq), DevBuf.of(g, ik), bs, T, G, nblk, pos0, 0)
    got = bs.read(np.float32).reshape(T, G, nblk)
    k64 = np.asarray(orc.h2f(ik), np.float64).reshape(n, 128)
    with np.errstate(invalid="ignore"):
        for t in range(T):
            s = np.stack([(r.astype(np.float64) * k64[:pos0 + t + 1]).sum(1) for r in iq[t]])
            size = np.stack([np.abs(r.astype(np.float64) * k64[:pos0 + t + 1]).sum(1) for r in iq[t]])
            for b in range((pos0 + t) // 128 + 1):
                sl = s[:, 128 * b:128 * b + 128]
                want = np.where(np.isnan(sl), -np.inf, sl).max(1)
                fin = np.isfinite(want)
                assert np.array_equal(got[t, ~fin, b], want[~fin].astype(np.float32)), (t, b)
                bound = 130 * 2.0 ** -24 * np.where(np.isfinite(size[:, 128 * b:128 * b + 128]), size[:, 128 * b:128 * b + 128], 0).max(1)
                assert (np.abs(got[t, fin, b] - want[fin]) <= bound[fin]).all(), (t, b)


def test_minimaxm3_index_scores_of_many_query_tiles(ops):
    """A work-group that walks several query tiles - two buffers, the next tile split while this one is multiplied -, a slice of
    them shorter than the others and a ragged last tile, with an infinity and a query the halfs do not hold in later tiles
    of a slice: the float64 product within a float32 sum's rounding (130 2^-24 of the sum of the products' sizes)."""
    g = ops.gpu
    T, G, pos0 = 701, 4, 9000
    n, tiles = pos0 + T, (T * G + 15) // 16
    nblk = (n + 127) // 128
    up = lambda a, b: -(-a // b)
    lens = [up(tiles, s) for s in range(1, 65)]                                   # the library's rule for a slice's length
    per = min(lens, key=lambda x: up(up(nblk, 4) * up(tiles, x), 512) * (x + 4))
    assert per >= 3 and tiles % per and T * G % 16
    iq, kf = orc.randn(79, (T * G, 128)), orc.randn(80, (n, 128))
    kf[:, 7] = 0.0
    iq[(2 * per + 2) * 16 + 5, 9] = np.inf
    iq[(3 * per + 1) * 16 + 3, 7] = 2.0 ** 40
    ik = orc.f2h(kf)
    bs = DevBuf(g, T * G * nblk * 4); bs.fill(0xFF)
    ops.minimaxm3_idx_scores(DevBuf.of(g, iq.reshape(T, G, 128)), DevBuf.of(g, ik), bs, T, G, nblk, pos0, 0)
    got = bs.read(np.float32).reshape(T * G, nblk)
    k64 = np.asarray(orc.h2f(ik), np.float64).reshape(n, 128)
    odd = (2 * per + 2) * 16 + 5
    want, size = (a.reshape(T * G, nblk) for a in _score_bounds(np.where(np.isinf(iq), 0.0, iq).reshape(T, G, 128), k64, pos0, nblk))
    with np.errstate(invalid="ignore"):
        row = np.full(nblk * 128, -np.inf)
        row[:pos0 + odd // G + 1] = np.nan_to_num(iq[odd].astype(np.float64) * k64[:pos0 + odd // G + 1], nan=-np.inf, posinf=np.inf, neginf=-np.inf).sum(1)
    assert np.array_equal(got[odd], row.reshape(nblk, 128).max(1).astype(np.float32))
    fin = np.isfinite(want)
    fin[odd] = False
    assert np.array_equal(np.isneginf(got)[want == -np.inf], np.ones((want == -np.inf).sum(), bool))
    assert (np.abs(got[fin] - want[fin]) <= 130 * 2.0 ** -24 * size[fin]).all(), (np.abs(got[fin] - want[fin]) / size[fin]).max()


def test_minimaxm3_index_scores_of_odd_values_take_no_longer_than_float32(ops):
    """A pass whose queries are all NaNs, or with an infinity in every block, is a float32 product where an ordinary one is three
    products of halfs: 3 and 1.5 times its time. 12 times leaves room for a busy machine; a key feature at a time took 120."""
    g = ops.gpu
    T, G, n = 64, 4, 16384
    iq, (ik, _) = orc.randn(77, (T, G, 128)), orc.randn_f16(78, (n, 128))
    nan, inf = np.full_like(iq, np.nan), ik.copy()
    inf[64::128, 3] = 0x7C00
    bs = DevBuf(g, T * G * (n // 128) * 4)

    def took(q, k):
        qb, kb = DevBuf.of(g, q), DevBuf.of(g, k)
        best = None
        for _ in range(6):
            g.sync()
            t0 = time.perf_counter()
            for _ in range(20):
                ops.minimaxm3_idx_scores(qb, kb, bs, T, G, n // 128, n - T, 1)
            g.sync()
            t = time.perf_counter() - t0
            best = t if best is None else min(best, t)
        return best

    plain = took(iq, ik)
    assert took(nan, ik) <= 12 * plain and took(iq, inf) <= 12 * plain


@pytest.mark.parametrize("nblk,K", [(5, 8), (512, 16), (513, 16), (2048, 40), (2049, 3), (8192, 16), (8193, 5), (70, 70)])
def test_minimaxm3_topk_row_lengths(ops, nblk, K):
    """Every row length the selection has a kernel for (scores in 8, 32 or 128 registers a lane, or left in memory),
    on scores with ties, holes and boosted blocks: the lists and the scores left behind, bit for bit."""
    g = ops.gpu
    T, G = 2, 3
    rng = np.random.default_rng(nblk * 31 + K)
    sc = rng.integers(-50, 50, (T, G, nblk)).astype(np.float32) / 4            # many equal scores
    sc[rng.random((T, G, nblk)) < 0.2] = -np.inf
    sc[0, 0, : min(3, nblk)] += 1e30
    sc[1, 2] = -np.inf                                                         # a row with nothing to choose
    bs, sel = DevBuf.of(g, sc), DevBuf(g, T * G * K * 4)
    ops.minimaxm3_idx_topk(bs, sel, T, G, nblk, K)
    want_sel, want_left = orc.mm3_idx_topk(sc, K)
    assert np.array_equal(sel.read(np.int32).reshape(T, G, K), want_sel)
    assert np.array_equal(bs.read(np.float32).reshape(T, G, nblk).view(np.uint32), want_left.view(np.uint32))


@pytest.mark.parametrize("nblk,K", [(1, 1), (64, 64), (65, 64), (136, 16), (136, 65), (512, 17), (1024, 16), (2049, 64), (8192, 1)])
def test_minimaxm3_topk_candidates(ops, nblk, K):
    """The selection's bound at the rows that strain it: scores without ties, ascending and descending, the large ones all in
    one lane's share (every 64th block), more equal scores than lanes at the bound, fewer scores than K, the two zeros,
    infinities, and NaNs, which are never chosen and stay. The oracle's lists and the scores left behind, bit for bit."""
    g = ops.gpu
    rng = np.random.default_rng(nblk * 7 + K)
    base = rng.standard_normal(nblk).astype(np.float32)
    share = base.copy()
    share[5::64] += 100.0
    tied = np.where(np.arange(nblk) % 3 == 0, np.float32(2.0), base)
    few = np.full(nblk, -np.inf, np.float32)
    few[rng.permutation(nblk)[:K // 2 + 1]] = base[:min(nblk, K // 2 + 1)]
    zeros = np.where(rng.random(nblk) < 0.5, np.float32(-0.0), np.float32(0.0))
    odd = base.copy()
    odd[::7] = np.inf
    nan = base.copy()
    nan[rng.random(nblk) < 0.3] = np.nan
    sc = np.stack([base, np.sort(base), np.sort(base)[::-1], share, tied, few, zeros, odd, nan]).astype(np.float32)[None]
    bs, sel = DevBuf.of(g, sc), DevBuf(g, sc.shape[1] * K * 4)
    ops.minimaxm3_idx_topk(bs, sel, 1, sc.shape[1], nblk, K)
    want_sel, want_left = orc.mm3_idx_topk(np.where(np.isnan(sc), np.float32(-np.inf), sc), K)
    want_left = np.where(np.isnan(sc), sc, want_left)
    assert np.array_equal(sel.read(np.int32).reshape(1, -1, K), want_sel)
    assert np.array_equal(bs.read(np.float32).reshape(sc.shape).view(np.uint32), want_left.view(np.uint32))


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("T,H,pos0,K", [(1, 128, 5000, 64), (3, 64, 2500, 512), (2, 160, 900, 16), (2, 1, 900, 16), (2, 16, 5000, 300), (2, 17, 2500, 64)])
def test_glm_cell_pools(ops, q8, T, H, pos0, K):
    g = ops.gpu
    L, scale = 512, 0.044
    n = pos0 + T
    qa = orc.randn(46, (T, H * L), 0.3)
    x = orc.randn(47, (n, L))
    if q8:
        rows = orc.glm_to_q8row(x, L)
    else:
        rows = orc.f2h(x).view(np.uint8).reshape(n, 2 * L)
    rng = np.random.default_rng(7)
    npool = (pos0 + 1) // 4
    sel = np.stack([rng.permutation(npool)[:K] if K <= npool else np.r_[rng.permutation(npool), [0] * (K - npool)] for _ in range(T)]).astype(np.int32)
    cnt = np.array([min(K, npool)] + [K // 3, -1][:T - 1], np.int32)          # a full list, a short one, a dense row
    u = DevBuf(g, T * H * L * 4); u.fill(0xFF)
    ops.mla_attend(DevBuf.of(g, qa), DevBuf.of(g, rows), u, T, H, L, pos0, scale, q8=q8, sel=DevBuf.of(g, sel), sel_cnt=DevBuf.of(g, cnt), K=K)
    want = orc.glm_mla_attend_sel(qa, rows, q8, T, H, L, pos0, scale, sel, cnt, K)
    close(u.read(np.float32).reshape(T, H * L), want)
    # no counts: the dense pass, as before
    ops.mla_attend(DevBuf.of(g, qa), DevBuf.of(g, rows), u, T, H, L, pos0, scale, q8=q8)
    close(u.read(np.float32).reshape(T, H * L), orc.glm_mla_attend(qa, rows, q8, T, H, L, pos0, scale).reshape(T, H * L))


def test_glm_dense_row_past_the_selection_bound_is_marked(ops):
    """A selection pass is sized for its lists and for dense rows of up to 2,560 cells (the reference's bound: its kernel
    keeps a row's scores in that many floats). A longer dense row must not come out as a plausible answer: NaNs."""
    g = ops.gpu
    T, H, L, pos0, K = 2, 16, 512, 2999, 16
    n = pos0 + T
    qa = orc.randn(1, (T, H * L), 0.3)
    rows = orc.f2h(orc.randn(2, (n, L))).view(np.uint8).reshape(n, 2 * L)
    sel = np.tile(np.arange(K, dtype=np.int32), (T, 1))
    cnt = np.array([K, -1], np.int32)                     # row 0 listed, row 1 dense over 3001 cells
    u = DevBuf(g, T * H * L * 4); u.fill(0)
    ops.mla_attend(DevBuf.of(g, qa), DevBuf.of(g, rows), u, T, H, L, pos0, 0.05, sel=DevBuf.of(g, sel), sel_cnt=DevBuf.of(g, cnt), K=K)
    got = u.read(np.float32).reshape(T, H * L)
    want = orc.glm_mla_attend_sel(qa, rows, False, T, H, L, pos0, 0.05, sel, cnt, K)
    close(got[:1], want.reshape(T, H * L)[:1])
    assert np.isnan(got[1]).all()


def test_glm_indexer_pools(ops):
    """ns_idx_pool over the engine's sequence of passes (a prompt chunk, then decode and verify passes whose pools reach
    back into the ring): pooled keys within float32 rounding of the oracle's (the exponential comes from another library),
    the ring byte for byte."""
    g = ops.gpu
    D, n_tok = 128, 213
    ik, ig, ape = orc.randn(5, (n_tok, D)), orc.randn(6, (n_tok, D)), orc.randn(7, (4, D), 0.5)
    ring = np.zeros((8, 2 * D), np.float32)
    pooled = np.zeros((n_tok // 4 + 1, D), np.float32)
    rb, pb, ab = DevBuf.of(g, ring), DevBuf.of(g, pooled), DevBuf.of(g, ape)
    pos = 0
    for T in (150, 1, 1, 3, 5, 1, 2, 4, 9, 16, 1, 20):
        orc.glm_idx_pool(ring, ik[pos:pos + T], ig[pos:pos + T], ape, pooled, pos, T, D)
        kb, gb = DevBuf.of(g, ik[pos:pos + T]), DevBuf.of(g, ig[pos:pos + T])
        ops.ok(ops.k.idx_pool(ops.raw(), rb.ptr, kb.ptr, gb.ptr, ab.ptr, pb.ptr, pos, T, D), "ns_idx_pool")
        pos += T
        assert np.array_equal(rb.read(np.float32).reshape(ring.shape), ring)
    assert pos == n_tok
    got = pb.read(np.float32).reshape(pooled.shape)
    assert np.abs(got - pooled).max() <= 4e-6 * np.abs(pooled).max()
    assert (got[n_tok // 4] == 0).all()


@pytest.mark.parametrize("T,H,j0,n,ld,pos0", [(1, 32, 0, 2500, 2500, 9999), (5, 32, 128, 300, 700, 1700), (40, 8, 0, 64, 80, 100)])
def test_glm_indexer_scores(ops, T, H, j0, n, ld, pos0):
    g = ops.gpu
    S, w = orc.randn(9, (T * H, n)), orc.randn(10, (T, H))
    score = np.full((T, ld), 3.0, np.float32)
    sb = DevBuf.of(g, score)
    orc.glm_idx_score(S, w, score, T, H, j0, n, pos0)
    Sb, wb = DevBuf.of(g, S), DevBuf.of(g, w)
    ops.ok(ops.k.idx_score(ops.raw(), Sb.ptr, wb.ptr, sb.ptr, T, H, j0, n, ld, pos0), "ns_idx_score")
    got = sb.read(np.float32).reshape(score.shape)
    fin = np.isfinite(score)
    assert np.array_equal(np.isneginf(got), np.isneginf(score))
    # (a head's product may be fused into the sum on one side and not on the other)
    assert np.abs(got[fin] - score[fin]).max() <= 1e-5 * max(1.0, float(np.abs(score[fin]).max()))
    with pytest.raises(Error, match="a pool range inside a score row"):
        ops.ok(ops.k.idx_score(ops.raw(), Sb.ptr, wb.ptr, sb.ptr, T, H, j0, n, j0 + n - 1, pos0), "ns_idx_score")


@pytest.mark.parametrize("T,n,K", [(1, 1, 1), (3, 7, 3), (2, 300, 40), (4, 5000, 512), (1, 5000, 4999), (2, 37, 37), (2, 20, 50), (1, 33000, 2048),
                                   (8, 1024, 1024), (3, 1025, 1), (2, 8192, 100), (2, 8193, 2048), (1, 32768, 2048), (2, 32769, 700), (1, 65536, 2048), (1, 65537, 300),
                                   (3, 8194, 1024), (3, 12291, 1), (3, 25003, 512), (3, 65533, 1000),
                                   (2, 12288, 1025), (2, 12289, 1025), (257, 8193, 1025), (3, 8193, 900), (3, 65536, 860), (2, 25003, 25001)])
def test_glm_top_k(ops, T, n, K):
    """ns_topk: the oracle's list bit for bit - on rows with many equal scores (the ties at the K-th value go to the lowest
    positions), -inf tails, fewer scores than K (the list's rest is left as it was) - and the same list on a second run."""
    g = ops.gpu
    rng = np.random.default_rng(n + K)
    ld = n + 6
    sc = rng.choice((np.round(rng.standard_normal(max(n // 3, 2)), 1) + 0.05).astype(np.float32), size=(T, ld)).astype(np.float32)
    if T > 1:
        sc[1, n // 2:n] = -np.inf
    if T > 2:
        sc[2, :n] = rng.standard_normal(n).astype(np.float32)    # all different
    want = orc.glm_topk(sc, n, K)
    scb = DevBuf.of(g, sc)
    for _ in range(2):
        sb = DevBuf.of(g, np.full((T, K), -1, np.int32))
        ops.ok(ops.k.topk(ops.raw(), scb.ptr, sb.ptr, T, n, ld, K), "ns_topk")
        assert np.array_equal(sb.read(np.int32).reshape(T, K), want)


@pytest.mark.parametrize("n,K", [(1025, 1024), (1025, 1025), (2049, 512), (8193, 512), (12290, 1024), (16384, 1), (16385, 1024), (25000, 512), (25003, 1025), (65536, 1024)])
def test_glm_top_k_where_the_candidates_are_many_or_few(ops, n, K):
    """ns_topk's bound on the candidates at the rows that strain it: ascending and descending scores, all equal, the large
    ones all in one thread's share (every 1024th position), more equal scores at the bound than its list holds, rows of
    -inf but for a few, negative ones, a few equal ones at the K-th place, mostly zeros with fewer and with more above them
    than the list holds, whole numbers. The oracle's list bit for bit."""
    g = ops.gpu
    rng = np.random.default_rng(n + K)
    base = rng.standard_normal(n).astype(np.float32)
    few = np.full(n, -np.inf, np.float32)
    few[rng.permutation(n)[:K // 2 + 1]] = 1.5
    share = base.copy()
    share[5::1024] += 100.0
    tied = np.maximum(base - 1.0, 0.0).astype(np.float32)
    tied[n // 3:n // 3 + min(n // 3, 3000)] = 2.0
    low = -1.0 - np.abs(base)                                     # none from 0 up
    low[-3:] = -0.0
    edge = base.copy()                                            # equal scores at the K-th place, among few candidates
    edge[np.argsort(base)[-K - 1:][:3 if K > 2 else 1]] = np.sort(base)[-K]
    edge[-1] = np.inf
    zeros = [np.maximum(base - np.sort(base)[-k - 1], 0.0) for k in (min(K // 2 + 1, n - 1), min(K + 3, n - 1))]
    sc = np.stack([np.sort(base), np.sort(base)[::-1], np.full(n, -3.25, np.float32), share, tied, few, low, edge] + zeros + [np.rint(base)]).astype(np.float32)
    sb = DevBuf.of(g, np.full((len(sc), K), -1, np.int32))
    ops.ok(ops.k.topk(ops.raw(), DevBuf.of(g, sc).ptr, sb.ptr, len(sc), n, n, K), "ns_topk")
    assert np.array_equal(sb.read(np.int32).reshape(len(sc), K), orc.glm_topk(sc, n, K))


def test_glm_indexer_feeds_the_latent_attention(ops):
    """The engine's sequence for a layer (llm/glm5next/src/engine.rs:1965-2013): pooled keys pass by pass, then for a verify
    pass the pool scores (the iq . pooled^T product is the engine's GEMM: taken here in numpy), the top pools a row, the
    counts - and ns_mla_attend_sel over those lists. The lists are the oracle's select of the scores the GPU produced, bit
    for bit; the attention is the oracle's over the same lists."""
    g = ops.gpu
    D, hh, kp, H, L = 128, 4, 16, 16, 512
    n_tok, T = 301, 3
    pos0 = n_tok - T
    ik, ig, ape = orc.randn(21, (n_tok, D)), orc.randn(22, (n_tok, D)), orc.randn(23, (4, D), 0.5)
    rb, pb, ab = DevBuf(g, 8 * 2 * D * 4), DevBuf(g, (n_tok // 4 + 1) * D * 4), DevBuf.of(g, ape)
    rb.fill(0)
    pb.fill(0)
    pos = 0
    for t in (200, 60, 38, T):
        kb, gb = DevBuf.of(g, ik[pos:pos + t]), DevBuf.of(g, ig[pos:pos + t])
        ops.ok(ops.k.idx_pool(ops.raw(), rb.ptr, kb.ptr, gb.ptr, ab.ptr, pb.ptr, pos, t, D), "ns_idx_pool")
        pos += t
    n = (pos0 + T) // 4
    assert n > kp
    pooled = pb.read(np.float32).reshape(-1, D)[:n]
    iq, w = orc.randn(24, (T * hh, D)), orc.randn(25, (T, hh))
    S = (iq @ pooled.T).astype(np.float32)                                   # [T hh][n]
    Sb, wb, scb, selb = DevBuf.of(g, S), DevBuf.of(g, w), DevBuf(g, T * n * 4), DevBuf.of(g, np.full((T, kp), -1, np.int32))
    ops.ok(ops.k.idx_score(ops.raw(), Sb.ptr, wb.ptr, scb.ptr, T, hh, 0, n, n, pos0), "ns_idx_score")
    ops.ok(ops.k.topk(ops.raw(), scb.ptr, selb.ptr, T, n, n, kp), "ns_topk")
    score = scb.read(np.float32).reshape(T, n)
    sel = selb.read(np.int32).reshape(T, kp)
    assert np.array_equal(sel, orc.glm_topk(score, n, kp))
    for r in range(T):
        assert (sel[r] < (pos0 + r + 1) // 4).all() and (np.diff(sel[r]) > 0).all()      # pools the row sees, in position order
    cnt = np.array([kp if (pos0 + r + 1) // 4 > kp else -1 for r in range(T)], np.int32)
    qa = orc.randn(26, (T, H * L), 0.3)
    rows = orc.f2h(orc.randn(27, (n_tok, L))).view(np.uint8).reshape(n_tok, 2 * L)
    u = DevBuf(g, T * H * L * 4)
    u.fill(0xFF)
    ops.mla_attend(DevBuf.of(g, qa), DevBuf.of(g, rows), u, T, H, L, pos0, 0.044, sel=selb, sel_cnt=DevBuf.of(g, cnt), K=kp)
    close(u.read(np.float32).reshape(T, H * L), orc.glm_mla_attend_sel(qa, rows, False, T, H, L, pos0, 0.044, sel, cnt, kp))


@pytest.mark.gpu
def test_glm_prompt_path_pieces(ops):
    """ns_mla_cells bit for bit and ns_softmax_masked within float32 rounding of the oracle: lists with room to spare and
    cut short, rows without lists, and score rows of every kernel form (kept in registers, and re-read)."""
    g = ops.gpu
    T, K, pos0 = 7, 9, 1234
    rng = np.random.default_rng(5)
    sel = rng.integers(0, (pos0 + 1) // 4, (T, K)).astype(np.int32)
    cnt = np.array([9, 0, -1, 4, 1, -1, 9], np.int32)
    for NC, lists in ((64, True), (17, True), (1280, True), (1280, False), (300, False)):
        ib, nb = DevBuf(g, T * NC * 4), DevBuf(g, T * 4)
        ib.fill(0xFF)
        nb.fill(0xFF)
        ops.mla_cells(T, K if lists else 0, pos0, ib, nb, NC, DevBuf.of(g, sel) if lists else None, DevBuf.of(g, cnt) if lists else None)
        want_i, want_n = orc.glm_mla_cells(T, K if lists else 0, pos0, NC, sel if lists else None, cnt if lists else None)
        assert np.array_equal(nb.read(np.int32), want_n), (NC, lists)
        assert np.array_equal(ib.read(np.int32).reshape(T, NC), want_i), (NC, lists)
    for R, H, NC, counts in ((3, 4, 64, (64, 0, 13)), (2, 3, 1024, (1000, 1)), (2, 2, 2112, (2051, 2112)), (2, 2, 5000, (4999, 300)), (1, 5, 257, (200,)),
                             (2, 1, 9000, (8999, 5)), (1, 2, 20000, (19998,)), (1, 2, 32768, (32768,)), (1, 2, 40000, (39990,)), (1, 2, 5001, (4000,)),
                             (1, 1, 17001, (17001,))):
        S = orc.randn(R + NC, (R * H, NC), 3.0)
        n = np.array(counts, np.int32)
        sb = DevBuf.of(g, S)
        ops.softmax_masked(sb, R, H, NC, DevBuf.of(g, n), 0.29)
        got = sb.read(np.float32).reshape(R * H, NC)
        want = orc.glm_softmax_masked(S, R, H, NC, n, 0.29)
        assert np.array_equal(got == 0.0, want == 0.0) or np.abs(got - want).max() < 1e-7
        # (the oracle, as the reference's work-item does, adds a row's exponentials one after another in float32: over
        # thousands of cells its own sum drifts, so long rows are also held to the float64 closed form of the same
        # float32 scaled scores)
        assert np.abs(got - want).max() <= 2e-6 * max(1.0, (NC / 1024.0) ** 0.5) * max(want.max(), 1e-30) + 1e-9, (R, H, NC)
        x = (S * np.float32(0.29)).astype(np.float64)
        for rh in range(R * H):
            m = n[rh // H]
            if m:
                e = np.exp(x[rh, :m] - x[rh, :m].max())
                assert np.abs(got[rh, :m] - e / e.sum()).max() <= 2e-6 * (e / e.sum()).max() + 1e-12, (R, H, NC, rh)
        for rh in range(R * H):
            assert not got[rh, n[rh // H]:].any()
            if n[rh // H]:
                assert abs(got[rh].sum() - 1.0) < 1e-5
