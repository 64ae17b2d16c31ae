"""Parity of the causal flash-attention prefill kernel (ns_attn_prompt_t and the reference-named entry points over it)
against the oracle's float64 closed form, through the C ABI, on seeded inputs."""
import numpy as np
import pytest

from helpers import check_close, gpu_decode, gpu_prompt, make_kv, make_q
from nextsycl_amd import DevBuf
from nextsycl_amd.attn import BF16, F16, F32, TUNE_PREFILL_BF16, TUNE_PREFILL_SPLITS, TUNE_PREFILL_WAVES
from oracle import orc

pytestmark = pytest.mark.gpu

SMALL = [
    # T, Hq, Hkv, p0, win, kt, qt
    (17, 4, 1, 0, 0, 0, F32),        # the shortest prompt pass
    (128, 4, 2, 0, 0, 0, F32),       # one row block exactly
    (129, 4, 2, 0, 0, 0, F16),       # one row into the second
    (300, 10, 2, 0, 0, 3, BF16),     # G 5, bfloat16 cache and rows (BASELINE config 2's types)
    (200, 8, 2, 1000, 0, 0, F32),    # a later chunk of a prompt: p0 > 0
    (333, 16, 1, 77, 0, 0, F16),     # G 16 (museglimmer's ratio)
    (260, 4, 1, 500, 256, 0, F32),   # a window
    (96, 6, 6, 31, 0, 3, F32),       # G 1
]


@pytest.mark.parametrize("T,Hq,Hkv,p0,win,kt,qt", SMALL)
def test_prefill_small(ops, T, Hq, Hkv, p0, win, kt, qt):
    D = 128
    cap = p0 + T + 5
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T)
    qd, qf = make_q(qt, T, Hq, D)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got, ref, qt, "prefill vs float64 closed form", kt=kt)


def _random_cases(n, seed):
    """Seeded shapes over what the kernel branches on: rows around the block sizes, groups, head size, every cache form
    (q8_0 / q4_0 rows of 128 values are 136 / 72 bytes: 8-byte aligned chunks), a context before the pass, windows shorter
    and longer than a tile and than the pass."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        D = int(rng.choice([128, 128, 256]))
        kt = int(rng.choice([0, 3, 1, 2]))
        Hkv = int(rng.integers(1, 3))
        G = int(rng.choice([1, 2, 4, 5, 8]))
        T = int(rng.choice([rng.integers(17, 70), rng.integers(70, 300), rng.integers(300, 600)]))
        p0 = int(rng.choice([0, rng.integers(1, 100), rng.integers(100, 900)]))
        win = int(rng.choice([0, 0, rng.integers(1, 64), rng.integers(64, 700)]))
        qt = BF16 if kt == 3 else int(rng.choice([F32, F16]))
        out.append((T, Hkv * G, Hkv, D, p0, win, kt, qt))
    return out


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,kt,qt", _random_cases(32, 20240608))
def test_prefill_seeded_shapes(ops, T, Hq, Hkv, D, p0, win, kt, qt):
    cap = p0 + T + 5
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T, cfg=T % 5)
    qd, qf = make_q(qt, T, Hq, D, cfg=p0 % 3)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got, ref, qt, "prefill vs float64 closed form", kt=kt)


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,kt,qt", [(700, 10, 2, 128, 300, 0, 3, BF16), (513, 4, 1, 128, 0, 400, 0, F32),
                                                     (300, 8, 2, 256, 100, 0, 3, BF16), (260, 4, 1, 256, 0, 200, 0, F32),
                                                     (200, 4, 2, 256, 60, 0, 1, F16), (140, 4, 1, 256, 0, 0, 2, F32)])
def test_prefill_work_groups_of_8_waves(ops, tune, T, Hq, Hkv, D, p0, win, kt, qt):
    """Long passes run work-groups of 8 waves (blocks of 256 rows; 128 at head size 256), short ones of 4: the same rows,
    keys and order of a wave's arithmetic, so the two agree bit for bit; forced here on shapes the oracle finishes in
    seconds."""
    cap = p0 + T + 5
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T)
    qd, qf = make_q(qt, T, Hq, D)
    tune(TUNE_PREFILL_WAVES, 8)
    got8, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    tune(TUNE_PREFILL_WAVES, 4)
    got4, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got8, ref, qt, "prefill (8 waves) vs float64 closed form", kt=kt)
    assert np.array_equal(got8, got4)


QROWS128 = [
    # T, Hq, Hkv, p0, win, kt, qt        q8_0 / q4_0 rows of 128 values: both work-group sizes, a window, key splits
    (17, 4, 1, 0, 0, 1, F32),
    (700, 16, 2, 300, 0, 1, F16),        # blocks of 256 rows (8 waves)
    (700, 16, 2, 300, 0, 2, F16),        # q4_0: 4 waves always
    (260, 8, 2, 1000, 200, 1, F32),
    (150, 4, 1, 64, 0, 2, F32),
    (64, 8, 1, 9000, 0, 1, F16),         # key splits
    (64, 8, 1, 9000, 0, 2, F32),
]


@pytest.mark.parametrize("T,Hq,Hkv,p0,win,kt,qt", QROWS128)
def test_prefill_quantized_rows_of_128(ops, T, Hq, Hkv, p0, win, kt, qt):
    D = 128
    cap = p0 + T + 1                     # (an odd row count: the second cache starts 8 bytes off a 16-byte boundary)
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T)
    qd, qf = make_q(qt, T, Hq, D)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got, ref, qt, "prefill, q8_0 / q4_0 rows of 128", kt=kt)


SPLIT = [
    # T, Hq, Hkv, D, p0, win, kt, qt: few row blocks over many keys - the pass is cut into key splits and merged
    (64, 8, 2, 128, 5000, 0, 0, F16),
    (33, 4, 4, 128, 12000, 0, 3, BF16),
    (300, 4, 1, 128, 9000, 3000, 0, F32),       # a window: the splits start at its first key
    (40, 4, 2, 256, 4000, 0, 0, F32),
    (130, 6, 2, 256, 2500, 0, 1, F16),          # quantized rows at head size 256
    (17, 2, 1, 128, 40000, 0, 0, F32),
    # a key head's rows all in one work-group behind 32768 keys and more: the tiles' transfers stream
    (20, 4, 1, 128, 33000, 0, 3, BF16),         # ... bfloat16 rows kept as they are
    (24, 4, 1, 128, 33000, 0, 3, F32),          # ... float32 query rows over them, in two parts
    (17, 5, 1, 128, 33000, 0, 0, F16),          # ... rows end to end
    # rows end to end in splits over one block and several, one of them behind a window's first key
    (37, 32, 8, 128, 11000, 0, 3, BF16),
    (33, 32, 2, 128, 18400, 0, 0, F16),
    (100, 16, 4, 128, 12000, 10500, 1, F32),
    (50, 24, 4, 128, 8000, 0, 0, F16),          # one head's rows a work-group, one a CU
    (64, 20, 4, 128, 20011, 0, 3, BF16),
]


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,kt,qt", SPLIT)
def test_prefill_key_splits(ops, T, Hq, Hkv, D, p0, win, kt, qt):
    cap = p0 + T + 9
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T, cfg=3)
    qd, qf = make_q(qt, T, Hq, D, cfg=5)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got, ref, qt, "prefill with key splits vs float64 closed form", kt=kt)


@pytest.mark.parametrize("T,Hq,Hkv,p0,kt,qt,ns", [
    (49, 5, 1, 9230, 0, F32, 73),               # 52 splits, 35 work-groups on the fullest XCD: 64 places, splits no shorter than two tiles
    (33, 7, 1, 2585, 3, BF16, 21),              # ... behind fewer keys 32
    (119, 30, 6, 9675, 0, F16, 16),             # 17 splits, 65 on the fullest XCD: one fewer
])
def test_prefill_key_splits_in_whole_rounds(ops, T, Hq, Hkv, p0, kt, qt, ns):
    """Few pairs of one head's rows a work-group whose count would leave an XCD's places unevenly filled: whole rounds of them."""
    D = 128
    plan = ops.prompt_plan(qt, kt, T, Hq, Hkv, D, p0)
    assert not plan["flat"] and plan["splits"] == ns, plan
    kc, vc = make_kv(kt, Hkv, D, p0 + T, p0 + T, cfg=3)
    qd, qf = make_q(qt, T, Hq, D, cfg=5)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, p0 + T, p0)
    check_close(got, orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, p0 + T, p0), qt, "prefill, splits in whole rounds", kt=kt)


def test_prefill_streamed_in_8_waves_of_one_heads_rows(ops, tune):
    """Five heads to an 8-wave work-group behind 33000 keys, each read once (the rule lays these rows end to end)."""
    T, Hq, Hkv, D, p0 = 17, 5, 1, 128, 33000
    tune(TUNE_PREFILL_WAVES, 8)
    plan = ops.prompt_plan(F16, 0, T, Hq, Hkv, D, p0)
    assert not plan["flat"] and plan["waves"] == 8 and plan["pack"] == 5 and plan["stream"], plan
    kc, vc = make_kv(0, Hkv, D, p0 + T, p0 + T, cfg=3)
    qd, qf = make_q(F16, T, Hq, D, cfg=5)
    got, _ = gpu_prompt(ops, F16, 0, qd, kc, vc, T, Hq, Hkv, D, p0 + T, p0)
    check_close(got, orc.attn_f64(qf, kc, vc, 0, T, Hq, Hkv, D, p0 + T, p0), F16, "prefill, five heads to 8 waves, streamed")


@pytest.mark.parametrize("ns", [2, 5, 16])
@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win", [(200, 4, 2, 128, 0, 0), (150, 2, 1, 128, 700, 90), (70, 4, 2, 256, 333, 0)])
def test_prefill_forced_splits(ops, tune, ns, T, Hq, Hkv, D, p0, win):
    """Splits forced onto short passes: splits wholly past a row block's last key, splits a window leaves empty, a last
    split of a few keys - the same result as the unsplit pass within the path's bar, and the same whatever the
    work-group size (bit for bit)."""
    cap = p0 + T + 1
    kc, vc = make_kv(0, Hkv, D, cap, p0 + T, cfg=1)
    qd, qf = make_q(F32, T, Hq, D, cfg=2)
    ref = orc.attn_f64(qf, kc, vc, 0, T, Hq, Hkv, D, cap, p0, win=win)
    tune(TUNE_PREFILL_SPLITS, ns)
    tune(TUNE_PREFILL_WAVES, 8)
    got8, _ = gpu_prompt(ops, F32, 0, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    tune(TUNE_PREFILL_WAVES, 4)
    got4, _ = gpu_prompt(ops, F32, 0, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got8, ref, F32, "prefill with %d forced splits" % ns)
    assert np.array_equal(got8, got4)


FLAT = [
    # T, Hq, Hkv, D, p0, win, kt, qt, ns: a pass's (row, head) pairs end to end, 16 a row tile, up to 16 (D = 256: 8) tiles a block
    (17, 1, 1, 128, 60, 0, 0, F16, 0),           # G 1: a tile and one pair of the next
    (17, 4, 1, 128, 300, 0, 0, F32, 3),          # 5 tiles: waves without one
    (32, 8, 2, 128, 500, 0, 3, BF16, 2),         # 8: every wave one
    (33, 4, 1, 128, 500, 0, 3, F32, 2),          # 9 (the last of 4 pairs): the first wave two; float32 rows in two parts
    (64, 4, 1, 128, 700, 0, 0, F32, 4),          # 16: every wave two
    (65, 4, 1, 128, 700, 0, 1, F16, 4),          # 17: two blocks of 9 and 8
    (50, 10, 2, 128, 900, 0, 2, F32, 3),         # q4_0 rows of 128: two threads a block of 32; G 5
    (45, 3, 1, 128, 41, 33, 2, F16, 0),          # ... a window's edge inside a tile, no splits
    (64, 16, 1, 128, 900, 0, 0, F16, 5),         # G 16: four blocks
    (21, 6, 1, 256, 400, 0, 0, F32, 3),          # D 256: 126 pairs, 8 tiles
    (22, 6, 1, 256, 400, 0, 1, F16, 3),          # ... 9: two blocks of 5 and 4
    (37, 12, 2, 256, 700, 0, 2, F32, 4),
    (40, 8, 2, 256, 500, 100, 3, BF16, 2),
    (40, 8, 2, 256, 500, 0, 3, F32, 9),          # ... more splits than key tiles
    (300, 8, 2, 128, 0, 0, 0, F16, 1),           # a prompt's start, unsplit: blocks of unequal keys
    (150, 8, 1, 256, 0, 0, 0, F32, 1),
    (333, 6, 2, 128, 200, 70, 3, BF16, 1),       # a window shorter than the pass; G 3: a row's heads in two blocks
]


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,kt,qt,ns", FLAT)
def test_prefill_rows_end_to_end(ops, tune, T, Hq, Hkv, D, p0, win, kt, qt, ns):
    """Forced onto short contexts, over rows as they are cached and widened, in work-groups of 8 waves and of 4 (half rows of 128)."""
    cap = p0 + T + 1
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T, cfg=4)
    qd, qf = make_q(qt, T, Hq, D, cfg=6)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    tune(TUNE_PREFILL_SPLITS, ns)
    for waves, form in [(16, 1), (16, 2), (12, 2)][0 if kt else 1:3 if D == 128 else 2]:
        tune(TUNE_PREFILL_WAVES, waves)
        tune(TUNE_PREFILL_BF16, form)
        plan = ops.prompt_plan(qt, kt, T, Hq, Hkv, D, p0, win)
        assert plan["flat"] and plan["waves"] == (4 if waves == 12 else 8) and plan["widen"] == (kt != 0 and form == 2), plan
        got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
        check_close(got, ref, qt, "prefill, rows end to end (%d, form %d)" % (waves, form), kt=kt)


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,cap,win,kt,qt", [
    (37, 32, 8, 128, 20011, 0, 0, 3, BF16), (37, 24, 4, 256, 5000, 0, 0, 0, F32), (100, 24, 4, 256, 6000, 0, 0, 1, F16), (33, 8, 8, 128, 900, 0, 0, 1, F32),
    (300, 16, 2, 128, 5000, 0, 0, 2, F32),       # q4_0 rows: ten blocks over two keys' groups
    (17, 5, 1, 128, 33000, 0, 0, 0, F32),        # one block behind 32768 keys: streamed
    (40, 10, 2, 128, 9000, 5039, 5000, 0, F32),  # a wrapped ring
    (700, 16, 2, 128, 1000, 900, 200, 0, F32),   # ... under a short window: work-groups of 4 waves
    (700, 16, 2, 128, 1500, 0, 0, 3, BF16),      # behind twice its own length
])
def test_prefill_rows_end_to_end_by_the_rule(ops, T, Hq, Hkv, D, p0, cap, win, kt, qt):
    """Passes the rule gives to that kernel, position-major too."""
    n = p0 + T
    plan = ops.prompt_plan(qt, kt, T, Hq, Hkv, D, p0, win)
    assert plan["flat"] and plan["waves"] == (4 if win == 200 else 8) and plan["stream"] == (p0 == 33000), plan
    kc, vc = make_kv(kt, Hkv, D, n, n, cfg=5)
    qd, qf = make_q(qt, T, Hq, D, cfg=7)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, n, p0, win=win)
    if cap:
        slot = np.arange(n - cap, n) % cap
        rings = [np.zeros((Hkv, cap, kc.shape[2]), np.uint8) for _ in range(2)]
        for ring, c in zip(rings, (kc, vc)):
            ring[:, slot] = c[:, n - cap:]
        kc, vc = rings
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap or n, p0, win=win)
    check_close(got, ref, qt, "prefill, rows end to end", kt=kt)
    if not cap:
        pm, _ = gpu_prompt(ops, qt, kt, qd, *(np.ascontiguousarray(c.transpose(1, 0, 2)) for c in (kc, vc)), T, Hq, Hkv, D, n, p0, win=win, pm=True)
        assert np.array_equal(pm.view(np.uint32), got.view(np.uint32))


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,qt", [(700, 16, 2, 128, 1000, 200, F32), (900, 32, 4, 128, 0, 300, F16), (500, 24, 4, 256, 1500, 256, F32)])
def test_prefill_windowed_rows_end_to_end_lose_no_bits(ops, tune, T, Hq, Hkv, D, p0, win, qt):
    """Rows end to end under a window lie no further from the float64 closed form than whole waves of one head's rows."""
    n = p0 + T
    kc, vc = make_kv(0, Hkv, D, n, n, cfg=4)
    qd, qf = make_q(qt, T, Hq, D, cfg=6)
    ref = orc.attn_f64(qf, kc, vc, 0, T, Hq, Hkv, D, n, p0, win=win)
    rel = []
    tune(TUNE_PREFILL_SPLITS, 1)
    for waves in (8, 16, 12)[:3 if D == 128 else 2]:
        tune(TUNE_PREFILL_WAVES, waves)
        got, _ = gpu_prompt(ops, qt, 0, qd, kc, vc, T, Hq, Hkv, D, n, p0, win=win)
        rel.append(check_close(got, ref, qt, "prefill under a window (%d)" % waves)[1])
    assert max(rel[1:]) <= rel[0], rel


@pytest.mark.parametrize("T,Hq,Hkv,D,p0", [(76, 64, 16, 128, 4300), (102, 8, 1, 256, 38000)])
@pytest.mark.parametrize("size", [2.0 ** 18, 2.0 ** -20])
def test_prefill_rows_end_to_end_keep_bfloat16_values(ops, T, Hq, Hkv, D, p0, size):
    """Values that are no halfs - over 65504, under half's normal range - through passes whose rows lie end to end and which the other form makes over
    the rows as they are cached: widened, the first saturate and the second are rounded to a few bits."""
    n = p0 + T
    kc, _ = make_kv(3, Hkv, D, n, n, cfg=1)
    _, vc = make_kv(3, Hkv, D, n, n, cfg=1, sigma=size)
    qd, qf = make_q(BF16, T, Hq, D, cfg=5)
    assert ops.prompt_plan(BF16, 3, T, Hq, Hkv, D, p0)["flat"]
    got, _ = gpu_prompt(ops, BF16, 3, qd, kc, vc, T, Hq, Hkv, D, n, p0)
    for r in (0, T // 2, T - 3):
        ref = orc.attn_f64(qf[r:r + 3], kc, vc, 3, 3, Hq, Hkv, D, n, p0 + r)
        check_close(got[r:r + 3], ref, BF16, "prefill, bfloat16 values of %g, rows %d" % (size, r), kt=3)


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,kt,qt", [(1100, 64, 4, 128, 1000, 0, F32), (1403, 48, 8, 128, 1500, 3, BF16), (2100, 16, 2, 256, 2200, 1, F16),
                                                   (2100, 64, 4, 128, 1700, 0, F16)])
def test_prefill_whole_blocks_beside_split_ones(ops, tune, T, Hq, Hkv, D, p0, kt, qt):
    """More row blocks than a round of the CUs holds: the last rows' run over all their keys, the first ones' in splits that are merged. Every
    row against the form that takes one head's rows a work-group, rows all over the pass against the float64 closed form."""
    n = p0 + T
    kc, vc = make_kv(kt, Hkv, D, n, n, cfg=2)
    qd, qf = make_q(qt, T, Hq, D, cfg=3)
    plan = ops.prompt_plan(qt, kt, T, Hq, Hkv, D, p0)
    assert plan["flat"] and plan["splits"] > 1 and 0 < plan["whole"] < plan["blocks"], plan
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, n, p0)
    tune(TUNE_PREFILL_WAVES, 8)
    other, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, n, p0)
    # (two results within the path's bar of one reference, whose largest value no row outgrows)
    assert np.abs(got - other).max() <= 4e-3 and np.linalg.norm(got - other) <= (4e-3 if qt == BF16 else 2e-3) * np.linalg.norm(other)
    for r in range(0, T - 3, T // 23):
        ref = orc.attn_f64(qf[r:r + 4], kc, vc, kt, 4, Hq, Hkv, D, n, p0 + r)
        check_close(got[r:r + 4], ref, qt, "prefill, whole and split blocks, rows %d" % r, kt=kt)


@pytest.mark.parametrize("kt,qt", [(3, BF16), (1, F32), (2, F16)])
def test_prefill_splits_leave_room_to_widen(ops, tune, kt, qt):
    """Rows end to end in 32 MiB of scratch, where six splits' partials would fit, or three and the widened rows (5 MB a split, 17.6 MB): the pass
    is within the oracle's bar and is the widened one - it rounds otherwise than the one over the rows' own form."""
    T, Hq, Hkv, D, p0 = 300, 32, 8, 128, 4000
    n = p0 + T
    kc, vc = make_kv(kt, Hkv, D, n, n, cfg=2)
    qd, qf = make_q(qt, T, Hq, D, cfg=3)
    tune(6, 32)
    tune(TUNE_PREFILL_WAVES, 16)
    tune(TUNE_PREFILL_BF16, 2)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, n, p0)
    tune(TUNE_PREFILL_BF16, 1)
    own, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, n, p0)
    for r in (0, 150, T - 4):
        ref = orc.attn_f64(qf[r:r + 4], kc, vc, kt, 4, Hq, Hkv, D, n, p0 + r)
        check_close(got[r:r + 4], ref, qt, "prefill, rows end to end in little scratch, rows %d" % r, kt=kt)
    if kt == 3:       # (quantized rows are staged as the very halfs that widening writes)
        assert not np.array_equal(got, own)


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("T,Hq,Hkv,win,cap,p0,ns", [(200, 4, 2, 300, 512, 900, 0), (200, 4, 2, 300, 512, 1024 - 200, 0), (130, 2, 1, 500, 640, 640 * 3 - 64, 0),
                                                    (300, 2, 1, 100, 401, 3000, 0), (129, 4, 1, 700, 829, 829 * 2 - 1, 0), (70, 4, 2, 1000, 1069, 2500, 3)])
def test_prefill_ring_is_the_unwrapped_pass(ops, tune, waves, T, Hq, Hkv, win, cap, p0, ns):
    """A ring whose end falls inside a tile, between two, in a split's first or last one: bit for bit the pass over a cache that
    holds the same rows in position order."""
    n, D = p0 + T, 128
    kc, vc = make_kv(0, Hkv, D, n, n, cfg=cap)
    slot = np.arange(n - cap, n) % cap
    rings = [np.zeros((Hkv, cap, 2 * D), np.uint8) for _ in range(2)]
    for ring, c in zip(rings, (kc, vc)):
        ring[:, slot] = c[:, n - cap:]
    qd, _ = make_q(F32, T, Hq, D, cfg=p0)
    tune(TUNE_PREFILL_WAVES, waves)
    tune(TUNE_PREFILL_SPLITS, ns)
    want, _ = gpu_prompt(ops, F32, 0, qd, kc, vc, T, Hq, Hkv, D, n, p0, win=win)
    got, _ = gpu_prompt(ops, F32, 0, qd, rings[0], rings[1], T, Hq, Hkv, D, cap, p0, win=win)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_prefill_ring(ops):
    T, Hq, Hkv, D, cap, win, p0 = 150, 4, 2, 128, 512, 300, 900
    k = orc.randn(11, (p0 + T, Hkv * D))
    v = orc.randn(12, (p0 + T, Hkv * D))
    kc = np.zeros((Hkv, cap, 2 * D), np.uint8)
    vc = np.zeros((Hkv, cap, 2 * D), np.uint8)
    for s in range(0, p0 + T, 128):
        e = min(p0 + T, s + 128)
        orc.kv_store(0, k[s:e], v[s:e], Hkv, D, cap, s, kc, vc, ring=True)
    qd, qf = make_q(F32, T, Hq, D)
    got, _ = gpu_prompt(ops, F32, 0, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, 0, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got, ref, F32, "ring prefill")


@pytest.mark.parametrize("T,Hq,Hkv,cap,win,p0,kt,qt", [
    (150, 4, 2, 512, 300, 900, 0, F32),          # a wrapped ring under a window
    (260, 2, 1, 640, 350, 1500, 3, BF16),        # the window's first key mid-tile, the ring's seam inside the pass's keys
    (40, 2, 2, 0, 0, 0, 0, F16),                 # one tile
    (100, 2, 1, 0, 0, 28, 3, BF16),              # two tiles
    (130, 2, 1, 0, 0, 62, 0, F32),               # three
    (200, 2, 1, 0, 0, 56, 0, F16),               # four, a pass that starts mid-tile
    (256, 2, 1, 0, 0, 1024, 3, F32),             # whole tiles only
    (257, 2, 1, 0, 100, 777, 0, BF16),           # a row block of one row
])
def test_prefill_tiles_sent_straight_to_lds(ops, tune, T, Hq, Hkv, cap, win, p0, kt, qt):
    """Over 16-bit rows of 128 both forms move their tiles global -> LDS without registers, the 8-wave form into three
    buffers a stream, the 4-wave form into two: passes of one to many tiles (every buffer rotation of either), rings
    with their seam among the pass's keys, windows whose edge falls inside a tile - against the float64 closed form, and
    the two forms bit for bit against each other."""
    D = 128
    n = p0 + T
    if cap:
        k = orc.randn(31, (n, Hkv * D))
        v = orc.randn(32, (n, Hkv * D))
        kc = np.zeros((Hkv, cap, 2 * D), np.uint8)
        vc = np.zeros((Hkv, cap, 2 * D), np.uint8)
        for s0 in range(0, n, 128):
            e = min(n, s0 + 128)
            orc.kv_store(kt, k[s0:e], v[s0:e], Hkv, D, cap, s0, kc, vc, ring=True)
    else:
        cap = n + 3
        kc, vc = make_kv(kt, Hkv, D, cap, n, cfg=2)
    qd, qf = make_q(qt, T, Hq, D, cfg=1)
    tune(TUNE_PREFILL_WAVES, 8)
    got8, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    tune(TUNE_PREFILL_WAVES, 4)
    got4, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got8, ref, qt, "prefill, tiles straight to LDS", kt=kt)
    assert np.array_equal(got8, got4)


def test_prompt_rows_agree_with_decode_rows(ops):
    """The reference's --prompt-decode check (cli/nextsycl/src/main.rs:869-917): a prompt pass's row t against the
    decode pass at position p0 + t - two kernels, one result within the path's tolerance."""
    T, Hq, Hkv, D, p0 = 64, 8, 2, 128, 200
    cap = p0 + T
    kc, vc = make_kv(0, Hkv, D, cap, cap)
    qd, qf = make_q(F32, T, Hq, D)
    g = ops.gpu
    bufs = (DevBuf.of(g, kc), DevBuf.of(g, vc))
    pr, _ = gpu_prompt(ops, F32, 0, qd, kc, vc, T, Hq, Hkv, D, cap, p0, bufs=bufs)
    for t in (0, 1, 31, 63):
        de, _ = gpu_decode(ops, F32, 0, qd[t:t + 1], kc, vc, 1, Hq, Hkv, D, cap, p0 + t, bufs=bufs)
        mx, rel, _ = orc.compare(pr[t:t + 1], de.astype(np.float64))
        assert mx <= 2e-3 and rel <= 1e-3, (t, mx, rel)


def test_softmax_weights_sum_to_one(ops):
    """V = 1 everywhere -> every output is 1: a row's weights sum to one (to the rounding of the weights to half)."""
    T, Hq, Hkv, D = 400, 4, 1, 128
    kc, vc = make_kv(0, Hkv, D, T, T)
    vc = np.ascontiguousarray(np.broadcast_to(np.array([0x3C00], np.uint16).view(np.uint8), (Hkv, T, D, 2)).reshape(Hkv, T, 2 * D))
    qd, _ = make_q(F32, T, Hq, D)
    got, _ = gpu_prompt(ops, F32, 0, qd, kc, vc, T, Hq, Hkv, D, T, 0)
    assert np.abs(got - 1.0).max() < 5e-4


def test_reference_named_prompt_entry_points(ops):
    T, Hq, Hkv, D, p0 = 70, 8, 2, 128, 10
    cap = p0 + T
    kc, vc = make_kv(0, Hkv, D, cap, cap)
    qd, _ = make_q(F32, T, Hq, D)
    g = ops.gpu
    bufs = (DevBuf.of(g, kc), DevBuf.of(g, vc))
    want, _ = gpu_prompt(ops, F32, 0, qd, kc, vc, T, Hq, Hkv, D, cap, p0, bufs=bufs)
    qb, ob = DevBuf.of(g, qd), DevBuf(g, T * Hq * D * 4)
    k = ops.k
    assert k.mg_attn_prompt_supported(T, Hq, Hkv, D) == 1 and k.mg_attn_prompt_supported(16, Hq, Hkv, D) == 0
    ops.mg_attn_prompt(qb, bufs[0], bufs[1], T, Hq, Hkv, D, cap, p0, 0, ob)
    assert np.array_equal(ob.read(np.float32).reshape(T, -1), want)
    ob.fill(0)
    ops.mg_attn(qb, bufs[0], bufs[1], T, Hq, Hkv, D, cap, p0, 0, True, ob, None)
    assert np.array_equal(ob.read(np.float32).reshape(T, -1), want)
    ob.fill(0)
    ops.q35_attn(qb, Hq * D, bufs[0], bufs[1], T, Hq, Hkv, D, cap, p0, ob, None)
    assert np.array_equal(ob.read(np.float32).reshape(T, -1), want)
    assert k.attn_prompt_t(g.raw, 0, 0, 0, qb.ptr, Hq * D, bufs[0].ptr, bufs[1].ptr, T, Hq, Hkv, 64, cap, p0, 0, 0.0, ob.ptr) == -1
    assert "heads of 128 or 256" in k.api.error()


WIDE = [
    # T, Hq, Hkv, p0, win, kt, qt        heads of 256 (Qwen3.5's), every cache form of the reference's prompt kernel
    (17, 6, 1, 0, 0, 0, F32),
    (200, 12, 2, 333, 0, 0, F32),        # G 6, a later chunk
    (130, 4, 2, 0, 0, 3, BF16),
    (190, 12, 2, 100, 0, 1, F32),        # q8_0 rows (272 bytes)
    (150, 6, 1, 60, 0, 2, F16),          # q4_0 rows (144 bytes)
    (100, 4, 1, 700, 128, 1, F32),       # q8_0 under a window
]


@pytest.mark.parametrize("T,Hq,Hkv,p0,win,kt,qt", WIDE)
def test_prefill_heads_of_256_and_quantized_rows(ops, T, Hq, Hkv, p0, win, kt, qt):
    D = 256
    cap = p0 + T + 3
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T)
    qd, qf = make_q(qt, T, Hq, D)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got, ref, qt, "prefill, heads of 256", kt=kt)


@pytest.mark.parametrize("T,Hq,Hkv,D,p0", [(90, 12, 2, 256, 40), (300, 16, 2, 128, 500), (1100, 16, 1, 128, 0)])
def test_q35_prompt_kv_entry_point(ops, T, Hq, Hkv, D, p0):
    """ns_q35_attn_prompt_kv as the engine calls it (llm/qwen35/src/engine.rs:1598-1617): float32 rows, D = 256, Hq = 6 Hkv;
    and over heads of 128 (136- / 72-byte rows: the cache form of the 128K q8_0 decode configuration taking a prompt)."""
    cap = p0 + T
    g = ops.gpu
    qd, qf = make_q(F32, T, Hq, D)
    for kt in (0, 1, 2):
        kc, vc = make_kv(kt, Hkv, D, cap, cap)
        ob = DevBuf(g, T * Hq * D * 4); ob.fill(0xFF)
        qb, kb, vb = DevBuf.of(g, qd), DevBuf.of(g, kc), DevBuf.of(g, vc)        # held: a buffer is freed with its object
        rc = ops.k.q35_attn_prompt_kv(g.raw, kt, qb.ptr, Hq * D, kb.ptr, vb.ptr, T, Hq, Hkv, D, cap, p0, ob.ptr)
        assert rc == 0, ops.k.api.error()
        check_close(ob.read(np.float32).reshape(T, -1), orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0), F32, "ns_q35_attn_prompt_kv kt %d" % kt)


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,kt,qt", [
    (200, 8, 2, 128, 300, 0, 0, F32),
    (200, 8, 2, 128, 300, 0, 3, BF16),           # the bfloat16 rows are widened out of a position-major cache
    (333, 10, 2, 128, 1000, 150, 3, F32),        # under a window: the widened copy starts at the window's first key
    (90, 4, 4, 256, 40, 0, 3, F16),
    (300, 6, 2, 128, 200, 0, 1, F16),
])
def test_prompt_over_a_position_major_cache(ops, T, Hq, Hkv, D, p0, win, kt, qt):
    """Prompt passes over caches laid out [position][key head][row] (MiniMax-M3's layout: kernels/llm/minimaxm3/mm3.h:33-37),
    every cache form the typed entry point takes - a bfloat16 cache's rows are widened to half from that layout too."""
    n = p0 + T
    cap = n + 5
    kc, vc = make_kv(kt, Hkv, D, cap, n, cfg=1, pm=True)
    qd, qf = make_q(qt, T, Hq, D, cfg=2)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win, pm=True)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win, pm=True)
    check_close(got, ref, qt, "prompt over a position-major cache", kt=kt)


PACKED = [
    # T, Hq, Hkv, D, p0, win, kt, qt: passes of so few rows that a work-group holds 2 or 4 query heads of its key head
    (17, 8, 2, 128, 5000, 0, 0, F16),           # 4 heads a work-group, key splits
    (32, 16, 2, 128, 300, 0, 0, F32),           # G 8: two work-groups of 4 heads a key head
    (33, 8, 2, 128, 9000, 0, 3, BF16),          # 2 heads a work-group; bfloat16 operands (few rows: not widened)
    (20, 12, 2, 128, 700, 256, 1, F16),         # G 6: 2 heads; a window; q8_0 rows widened
    (64, 6, 1, 128, 2000, 0, 2, F32),           # q4_0 rows of 128 in the kernel's own staging, 2 heads
    (17, 12, 2, 256, 4000, 0, 0, F32),          # heads of 256: 17 rows fill two of four waves
    (5, 8, 2, 256, 1000, 0, 1, F16),            # ... 5 rows: 4 heads a work-group
    (16, 10, 2, 128, 100, 0, 0, F32),           # G 5: five heads to an 8-wave work-group, three waves without rows
    (30, 20, 4, 128, 6000, 0, 3, BF16),         # ... behind key splits, bfloat16
    (40, 14, 2, 128, 900, 0, 0, F16),           # G 7, two waves a head: no divisor fits - one head a work-group
    (9, 14, 2, 256, 900, 0, 0, F16),            # G 7 at heads of 256: seven heads to 8 waves
    (20, 6, 2, 128, 3000, 0, 1, F32),           # G 3: three heads to 4 waves
    (33, 20, 2, 128, 2000, 100, 0, F32),        # G 10, two waves a head: 2 heads (4 waves); a window
    (40, 4, 1, 128, 0, 0, 0, F16),              # no context: the last rows' blocks see few keys
]


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,kt,qt", PACKED)
def test_prefill_work_groups_holding_several_heads(ops, T, Hq, Hkv, D, p0, win, kt, qt):
    cap = p0 + T + 3
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T, cfg=4)
    qd, qf = make_q(qt, T, Hq, D, cfg=2)
    got, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(got, ref, qt, "prefill, several heads a work-group", kt=kt)


@pytest.mark.parametrize("T,Hq,Hkv,D,p0", [(20, 16, 2, 128, 3000), (64, 8, 2, 128, 500), (100, 4, 2, 128, 9000), (10, 8, 1, 256, 700), (30, 8, 2, 256, 0)])
def test_prefill_8_wave_work_groups_holding_several_heads(ops, tune, T, Hq, Hkv, D, p0):
    """The 8-wave form (knob 2) over passes of few rows: 8, 4 or 2 heads a work-group; the same results as the 4-wave
    form's to the bound (their key splits differ with the heads a work-group holds)."""
    cap = p0 + T + 1
    kc, vc = make_kv(0, Hkv, D, cap, p0 + T, cfg=1)
    qd, qf = make_q(F16, T, Hq, D, cfg=3)
    ref = orc.attn_f64(qf, kc, vc, 0, T, Hq, Hkv, D, cap, p0)
    for waves in (8, 4):
        tune(TUNE_PREFILL_WAVES, waves)
        got, _ = gpu_prompt(ops, F16, 0, qd, kc, vc, T, Hq, Hkv, D, cap, p0)
        check_close(got, ref, F16, "prefill, %d waves, several heads a work-group" % waves)


def _own_form_cases():
    """Every case of the tables above over a cache that is not half, as (T, Hq, Hkv, D, p0, win, kt, qt)."""
    out = [(T, Hq, Hkv, 128, p0, win, kt, qt) for T, Hq, Hkv, p0, win, kt, qt in SMALL + QROWS128]
    out += [(T, Hq, Hkv, 256, p0, win, kt, qt) for T, Hq, Hkv, p0, win, kt, qt in WIDE]
    out += SPLIT + _random_cases(32, 20240608)
    return [c for c in out if c[6] != 0]


@pytest.mark.parametrize("T,Hq,Hkv", [(257, 4, 1), (350, 4, 1), (351, 4, 1), (1400, 1, 1), (1401, 1, 1)])
def test_prefill_over_q4_rows_at_the_own_forms_edge(ops, tune, T, Hq, Hkv):
    """q4_0 rows of 128 keep their form up to 1400 rows a key head: below, at and past that, the form taken and both forced ones
    agree bit for bit."""
    p0 = 200
    cap = p0 + T
    kc, vc = make_kv(2, Hkv, 128, cap, cap, cfg=2)
    qd, _ = make_q(F32, T, Hq, 128, cfg=1)
    bits = []
    for form in (0, 1, 2):
        tune(5, form)
        bits.append(gpu_prompt(ops, F32, 2, qd, kc, vc, T, Hq, Hkv, 128, cap, p0)[1])
    assert all(np.array_equal(b, bits[0]) for b in bits)


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,kt,qt", _own_form_cases())
def test_prefill_over_the_caches_own_form(ops, tune, T, Hq, Hkv, D, p0, win, kt, qt):
    """A pass over bfloat16, q8_0 or q4_0 rows first widens them to half rows in the library's scratch and runs as a
    pass over a half cache (knob 5 = 2 here: always); a pass of few rows, or one whose context is too long for the scratch
    (knob 5 = 1 here), keeps the rows' own form in the kernel. Both meet the bound; over quantized rows both stage the same halfs (half(q x d), one rounding) and walk the
    keys in the same order, so they agree bit for bit."""
    cap = p0 + T + 7
    kc, vc = make_kv(kt, Hkv, D, cap, p0 + T, cfg=2)
    qd, qf = make_q(qt, T, Hq, D, cfg=1)
    tune(5, 2)
    wide, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    tune(5, 1)
    own, _ = gpu_prompt(ops, qt, kt, qd, kc, vc, T, Hq, Hkv, D, cap, p0, win=win)
    ref = orc.attn_f64(qf, kc, vc, kt, T, Hq, Hkv, D, cap, p0, win=win)
    check_close(wide, ref, qt, "prefill, rows widened first", kt=kt)
    # (bfloat16 operands: query rows of another type enter the first product as two bfloat16 numbers - the same bound)
    check_close(own, ref, qt, "prefill, the cache's own form in the kernel", kt=kt)
    if kt in (1, 2) and not (kt == 2 and D == 128):
        assert np.array_equal(np.asarray(wide).view(np.uint8), np.asarray(own).view(np.uint8))
