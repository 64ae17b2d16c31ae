"""What a prompt pass's sizes decide about how it runs (ns_attn_prompt_plan: host arithmetic, no GPU), on both sides of the lines
that measurement drew."""
import ctypes as C
import os

import pytest

from nextsycl_amd import Error, library_path
from nextsycl_amd.attn import BF16, F16, F32, KV_BF16, KV_F16, KV_Q4_0, KV_Q8_0, TUNE_PREFILL_BF16, TUNE_PREFILL_SPLITS, TUNE_PREFILL_WAVES, TUNE_SCRATCH_MIB, Ops


@pytest.fixture(scope="module")
def ops():
    if not os.path.exists(library_path()):
        from nextsycl_amd.build import build
        build()
    return Ops(None)


@pytest.fixture
def tune(ops):
    touched = set()

    def set_knob(knob, value):
        touched.add(knob)
        ops.tune(knob, value)

    yield set_knob
    for k in touched:
        ops.tune(k, 0)


PLANS = [
    # T, Hq, Hkv, D, p0, win, kt, qt, what of the plan
    (37, 32, 8, 128, 20011, 0, KV_BF16, BF16, dict(flat=1, waves=8, splits=32, widen=0, blocks=1)),
    (37, 32, 8, 128, 1000, 0, KV_BF16, BF16, dict(flat=0)),
    (8192, 40, 8, 128, 0, 0, KV_BF16, BF16, dict(flat=1, splits=1, widen=1)),
    (1024, 32, 8, 128, 0, 0, KV_F16, F16, dict(flat=0)),
    # a window: 4 waves, 8 for a round of the CUs nearly or quite full
    (3000, 32, 8, 128, 8000, 512, KV_F16, F32, dict(flat=1, waves=4, splits=1)),
    (2001, 32, 2, 128, 10007, 1024, KV_F16, F32, dict(flat=1, waves=8, blocks=126)),
    (2048, 32, 2, 128, 10007, 1024, KV_F16, F32, dict(flat=1, waves=8, blocks=128)),
    (2064, 32, 2, 128, 10007, 1024, KV_F16, F32, dict(flat=1, waves=4, blocks=258)),
    (2001, 32, 2, 128, 0, 1024, KV_F16, F32, dict(flat=0)),
    # bfloat16 rows end to end are read as they are cached wherever the other form would
    (83, 32, 8, 128, 7100, 0, KV_BF16, BF16, dict(flat=1, widen=0)),
    (366, 32, 32, 128, 3870, 0, KV_BF16, BF16, dict(flat=1, widen=0)),
    (512, 32, 32, 128, 3768, 0, KV_BF16, BF16, dict(flat=1, widen=0)),
    (96, 16, 2, 256, 53771, 0, KV_BF16, BF16, dict(flat=1, widen=0)),
    (117, 24, 4, 256, 47165, 0, KV_BF16, BF16, dict(flat=1, widen=0)),
    (210, 8, 2, 256, 22395, 0, KV_BF16, BF16, dict(flat=1, widen=0)),
    (513, 32, 32, 128, 3768, 0, KV_BF16, BF16, dict(widen=1)),
    # q8_0 rows of 128: few key heads, or several blocks behind few keys, stay with the other form
    (36, 16, 8, 128, 2041, 0, KV_Q8_0, F32, dict(flat=1, widen=0, blocks=1)),
    (17, 64, 64, 128, 1649, 0, KV_Q8_0, F32, dict(flat=1, widen=0)),
    (61, 64, 8, 128, 1160, 0, KV_Q8_0, F32, dict(flat=0)),
    (61, 64, 8, 128, 1500, 0, KV_Q8_0, F32, dict(flat=1, blocks=2)),
    (39, 24, 2, 128, 690, 0, KV_Q8_0, F32, dict(flat=0)),
    (88, 24, 2, 128, 1849, 0, KV_Q8_0, F32, dict(flat=0)),
    (364, 24, 2, 128, 7055, 0, KV_Q8_0, F16, dict(flat=1)),
    # whole blocks in whole rounds, what is left over in splits
    (1403, 48, 8, 128, 9568, 0, KV_BF16, BF16, dict(flat=1, blocks=33, whole=30)),
    (2048, 24, 4, 256, 8192, 0, KV_Q8_0, F32, dict(flat=0, widen=1)),
    (17, 5, 1, 128, 33000, 0, KV_F16, F16, dict(flat=1, stream=1)),
    (20, 4, 1, 128, 33000, 0, KV_F16, F16, dict(flat=0, stream=1, pack=4)),
    (20, 4, 1, 128, 32700, 0, KV_F16, F16, dict(stream=0)),
    (64, 8, 1, 128, 9000, 0, KV_Q4_0, F32, dict(widen=0)),
    # q4_0 rows read once in either form, half a block of them behind a long context
    (105, 32, 32, 128, 84857, 0, KV_Q4_0, F16, dict(flat=0)),
    (49, 64, 32, 128, 60339, 0, KV_Q4_0, F32, dict(flat=0)),
    (142, 16, 16, 128, 60339, 0, KV_Q4_0, F32, dict(flat=1)),
    (34, 48, 16, 128, 34883, 0, KV_Q4_0, F32, dict(flat=1)),
]


@pytest.mark.parametrize("T,Hq,Hkv,D,p0,win,kt,qt,want", PLANS)
def test_plan(ops, T, Hq, Hkv, D, p0, win, kt, qt, want):
    plan = ops.prompt_plan(qt, kt, T, Hq, Hkv, D, p0, win)
    assert {k: plan[k] for k in want} == want


def test_plan_of_blocks_that_are_not_causal(ops):
    """Behind a long context they lie end to end as causal passes do; a first key of their own keeps long ones whole waves of a head."""
    assert ops.prompt_plan(F32, KV_F16, 37, 32, 8, 128, 20011, causal=False)["flat"]
    assert ops.prompt_plan(F32, KV_F16, 40, 8, 2, 128, 700, causal=False)["flat"] == 0
    assert ops.prompt_plan(F32, KV_F16, 3000, 32, 8, 128, 9000)["flat"] and not ops.prompt_plan(F32, KV_F16, 3000, 32, 8, 128, 9000, causal=False, kfirst=100)["flat"]


@pytest.mark.parametrize("kt", [KV_BF16, KV_Q8_0, KV_Q4_0])
def test_splits_leave_room_for_the_widened_rows(ops, tune, kt):
    """32 MiB of scratch hold six splits' partials (5 MB each), or three and the widened rows (17.6 MB)."""
    tune(TUNE_SCRATCH_MIB, 32)
    tune(TUNE_PREFILL_WAVES, 16)
    tune(TUNE_PREFILL_BF16, 2)
    plan = ops.prompt_plan(F16, kt, 300, 32, 8, 128, 4000)
    assert plan["flat"] and plan["splits"] <= 3 and plan["widen"], plan


def test_forced_forms(ops, tune):
    for waves, flat, got in ((4, 0, 4), (8, 0, 8), (16, 1, 8), (12, 1, 4)):
        tune(TUNE_PREFILL_WAVES, waves)
        plan = ops.prompt_plan(F16, KV_F16, 90, 16, 2, 128, 700)
        assert (plan["flat"], plan["waves"]) == (flat, got)
    tune(TUNE_PREFILL_WAVES, 12)
    assert ops.prompt_plan(F16, KV_Q8_0, 90, 16, 2, 128, 700)["waves"] == 8          # (4 waves hold half rows only)
    tune(TUNE_PREFILL_WAVES, 0)
    tune(TUNE_PREFILL_SPLITS, 3)
    assert ops.prompt_plan(F16, KV_F16, 40, 16, 2, 128, 700)["splits"] == 3


@pytest.mark.parametrize("bad", [(F32, KV_F16, 0, 8, 2, 128, 0), (F32, KV_F16, 20, 7, 2, 128, 0), (F32, KV_F16, 20, 8, 2, 64, 0), (3, KV_F16, 20, 8, 2, 128, 0),
                                 (F32, 4, 20, 8, 2, 128, 0), (F32, KV_F16, 20, 8, 2, 128, -1), (F32, KV_F16, 20, 8, 0, 128, 0)])
def test_refused(ops, bad):
    with pytest.raises(Error, match="ns_attn_prompt_plan"):
        ops.prompt_plan(*bad)
    assert ops.k.attn_prompt_plan(F32, KV_F16, 20, 8, 2, 128, 0, 0, 1, 5, (C.c_int64 * 8)()) == -1      # a first key past the first row
    assert ops.k.attn_prompt_plan(F32, KV_F16, 20, 8, 2, 128, 0, 0, 1, -1, None) == -1
