"""The native step behind Ops.decode / prompt / pre_store (csrc/ops_fast.c): on the CPU against entry points that record what they
are given - the same arguments as through ctypes, no call where a buffer is a byte short or an argument is not the plain kind -
and on the GPU against the general way, results and refusals."""
import ctypes as C
import types

import numpy as np
import pytest

from nextsycl_amd import DevBuf, Error
from nextsycl_amd import attn
from nextsycl_amd.attn import ATTN_H, F16, F32, PRE_H, Ops, kv_row_bytes
from oracle import orc

fast = pytest.importorskip("nextsycl_amd._ops_fast")


class Buf:
    def __init__(self, ptr, n):
        self.ptr, self.len = ptr, n


def recorded(rc=0, scratch=100):
    """An Ops over entry points that note their arguments, and the notes."""
    notes, keep = [], []

    def entry(name, table):
        res, args = table[name]
        def f(*a):
            if name == "ns_attn_decode_scratch":
                return scratch
            notes.append((name, a))
            return rc
        keep.append(C.CFUNCTYPE(res, *args)(f))
        return keep[-1]

    k = types.SimpleNamespace(keep=keep, api=types.SimpleNamespace(error=lambda: "refused"))
    for name, table in (("ns_attn_decode_scratch", ATTN_H), ("ns_attn_decode_t", ATTN_H), ("ns_attn_prompt_t", ATTN_H), ("ns_attn_pre_store", PRE_H)):
        setattr(k, name[3:], entry(name, table))
    return Ops(types.SimpleNamespace(raw=C.c_void_p(4096), handle=4096), k), notes


def calls(kt=1, qt=F16, T=3, Hq=8, Hkv=2, D=128, cap=50, p0=7):
    """name -> (arguments by name, the buffers' least sizes)."""
    e, c = {0: 4, 1: 2, 2: 2}[qt], Hkv * cap * kv_row_bytes(kt, D)
    rows = dict(qt=qt, kt=kt, q=0, qs=Hq * D + 8, kc=0, vc=0, T=T, Hq=Hq, Hkv=Hkv, D=D, cap=cap, p0=p0, out=0)
    need = dict(q=((T - 1) * (Hq * D + 8) + Hq * D) * e, out=T * Hq * D * e, kc=c, vc=c)
    pre = dict(rope=1, qt=qt, kt=kt, ring=True, q=0, qss=Hq * (D + 4), qhs=D + 4, qo=0, qos=Hq * D, k=0, kss=Hkv * D, khs=D, v=0, vss=Hkv * D + 4, qw=0, kw=0,
               eps=1e-6, n_rot=64, theta=1e6, T=T, Hq=Hq, Hkv=Hkv, D=D, cap=cap, p0=p0, kc=0, vc=0)
    pneed = dict(q=((T - 1) * Hq * (D + 4) + (Hq - 1) * (D + 4) + D) * 4, qo=T * Hq * D * e, k=T * Hkv * D * 4, v=((T - 1) * (Hkv * D + 4) + Hkv * D) * 4, qw=D * 4,
                 kw=D * 4, kc=c, vc=c)
    return {"decode": (dict(rows, scratch=0, win=5, pm=False, scale=0.25), dict(need, scratch=400)), "prompt": (dict(rows, win=0, pm=True, scale=0.0), need),
            "pre_store": (pre, pneed)}


@pytest.mark.parametrize("name", ["decode", "prompt", "pre_store"])
@pytest.mark.parametrize("kt,qt", [(0, 0), (1, 1), (2, 0), (3, 2)])
def test_the_same_call_as_the_general_way(name, kt, qt):
    args, need = calls(kt, qt)[name]
    bufs = {b: Buf(1 << 20 | i << 12, n) for i, (b, n) in enumerate(need.items())}
    got = []
    for general in (False, True):
        ops, notes = recorded()
        if general:
            ops._at = None
        getattr(ops, name)(**dict(args, **bufs))
        assert len(notes) == 1
        got.append(notes[0])
    assert got[0] == got[1]
    # a byte short, one buffer after another: refused with the general way's words, and nothing is called
    for b in need:
        short = dict(args, **bufs)
        short[b] = Buf(bufs[b].ptr, need[b] - 1)
        words = []
        for general in (False, True):
            ops, notes = recorded()
            if general:
                ops._at = None
            with pytest.raises(Error) as err:
                getattr(ops, name)(**short)
            words.append(str(err.value))
            assert not notes
        assert words[0] == words[1]


def test_unplain_arguments_go_the_general_way(monkeypatch):
    """No buffer, no address, numbers of another type, sizes out of range: the native step calls nothing."""
    args, need = calls()["prompt"]
    bufs = {b: Buf(1 << 20, n) for b, n in need.items()}
    order = list(attn.Ops.prompt.__code__.co_varnames[1:attn.Ops.prompt.__code__.co_argcount])
    ops, notes = recorded()
    good = [dict(args, **bufs)[k] for k in order]
    assert fast.prompt(ops._at[2], 4096, *good) is True and len(notes) == 1
    for i, bad in [(2, None), (2, Buf(None, 1 << 30)), (2, Buf(1 << 20, None)), (6, 3.0), (6, -1), (6, 0), (6, 1 << 40), (7, 1 << 80), (0, 7), (1, 9), (15, "x"), (14, 1)]:
        other = list(good)
        other[i] = bad
        assert fast.prompt(ops._at[2], 4096, *other) is False, (i, bad)
    assert fast.prompt(ops._at[2], None, *good) is False and fast.prompt(ops._at[2], 4096, *good[:-1]) is False
    assert len(notes) == 1
    ops, notes = recorded(rc=-1)
    with pytest.raises(Error, match="refused"):
        ops.prompt(**dict(args, **bufs))


@pytest.mark.parametrize("name", ["decode", "prompt", "pre_store"])
def test_any_kernels_and_gpu_do(name):
    """Entries replaced on the kernels after the fact, or that are no library functions, are the ones called; a gpu needs no handle
    and kernels no entry but those that are called."""
    args, need = calls()[name]
    bufs = {b: Buf(1 << 20, n) for b, n in need.items()}
    entry, before = {"decode": "attn_decode_t", "prompt": "attn_prompt_t", "pre_store": "attn_pre_store"}[name], []
    ops, notes = recorded()
    setattr(ops.k, entry, lambda *a: before.append(a) or 0)
    getattr(ops, name)(**dict(args, **bufs))
    assert len(before) == 1 and not notes
    bare = types.SimpleNamespace(api=ops.k.api, attn_decode_scratch=lambda *a: 100, **{entry: getattr(ops.k, entry)})
    getattr(Ops(types.SimpleNamespace(raw=C.c_void_p(4096)), bare), name)(**dict(args, **bufs))
    assert len(before) == 2
    ops, notes = recorded()
    del ops.gpu.handle
    getattr(ops, name)(**dict(args, **bufs))
    assert len(notes) == 1


@pytest.mark.parametrize("name", ["decode", "prompt", "pre_store"])
def test_a_call_the_library_fails_is_made_once(name):
    """A failure may come behind launches that were made: the error is raised, and nothing is called a second time."""
    args, need = calls()[name]
    bufs = {b: Buf(1 << 20, n) for b, n in need.items()}
    words = []
    for general in (False, True):
        ops, notes = recorded(rc=-7)
        if general:
            ops._at = None
        with pytest.raises(Error, match="refused") as err:
            getattr(ops, name)(**dict(args, **bufs))
        words.append(str(err.value))
        assert len(notes) == 1
    assert words[0] == words[1]


@pytest.mark.gpu
@pytest.mark.parametrize("T,kt", [(1, 0), (4, 1), (40, 2)])
def test_the_general_way_gives_the_same(ops, T, kt):
    Hq, Hkv, D, p0 = 8, 2, 128, 300
    n, g = p0 + T, ops.gpu
    k, v = orc.randn(1, (n, Hkv * D)), orc.randn(2, (n, Hkv * D))
    kc, vc = orc.kv_store(kt, k, v, Hkv, D, n, 0)
    raw = [orc.randn(3 + i, (T, h * D)) for i, h in enumerate((Hq, Hkv, Hkv))] + [1.0 + 0.1 * orc.randn(9, (D,)) for _ in range(2)]
    out = []
    for general in (False, True):
        o = Ops(g)
        if general:
            o._at = None
        cb, q, r = [DevBuf.of(g, c) for c in (kc, vc)], DevBuf(g, T * Hq * D * 4), [DevBuf.of(g, x.astype(np.float32)) for x in raw]
        o.pre_store(1, F32, kt, False, r[0], Hq * D, D, q, Hq * D, r[1], Hkv * D, D, r[2], Hkv * D, r[3], r[4], 1e-6, D // 2, 1e6, T, Hq, Hkv, D, n, p0, cb[0], cb[1])
        y = DevBuf(g, T * Hq * D * 4)
        if T <= 16:
            o.decode(F32, kt, q, Hq * D, cb[0], cb[1], T, Hq, Hkv, D, n, p0, y, DevBuf(g, 4 * o.decode_scratch(T, Hq, Hkv, D, p0)))
        else:
            o.prompt(F32, kt, q, Hq * D, cb[0], cb[1], T, Hq, Hkv, D, n, p0, y)
        out.append((y.read(np.uint32), cb[0].read(np.uint8), cb[1].read(np.uint8)))
        with pytest.raises(Error, match="past the cache's capacity"):
            (o.decode(F32, kt, q, Hq * D, cb[0], cb[1], T, Hq, Hkv, D, n, n, y, DevBuf(g, 1 << 20)) if T <= 16 else
             o.prompt(F32, kt, q, Hq * D, cb[0], cb[1], T, Hq, Hkv, D, n, n, y))
    assert all(np.array_equal(a, b) for a, b in zip(*out))
