"""The host side of include/rwkv_decode.h: what a decode step's entry points
refuse, before any HIP call."""

import ctypes

import pytest

from conftest import load_pkg

F32, BF16 = 0, 1
NULL, SHAPE, ALIGNMENT, OVERLAP = 1, 2, 6, 7
HIP = 9            # past the checks: the launch, where there is no GPU
GIB = 1 << 30      # spacing of addresses that are never dereferenced


@pytest.fixture(scope="module")
def native():
    torch = pytest.importorskip("torch")
    if torch.cuda.is_available():
        pytest.skip("an accepted call would launch on addresses that are not memory")
    return load_pkg()._native


def _params(native, first):
    p = native.DecodeCellParams()
    at = 1000 * GIB
    for name, kind in p._fields_:
        if kind is ctypes.c_void_p:
            at += GIB
            if not (first and name.startswith("residual")):
                setattr(p, name, at)
    for i in range(6):
        at += GIB
        p.mix[i] = at
    p.decay_rank = p.rate_rank = p.gate_rank = 32
    p.residual_rank = 0 if first else 32
    return p


def _cell(native, p, **over):
    a = dict(x=GIB, ids=2 * GIB, state=3 * GIB, ti=4 * GIB, to=5 * GIB, ci=6 * GIB, co=7 * GIB, et=8 * GIB,
             rows=3, heads=2, slots=4, dtype=BF16, dither=1, ws=9 * GIB, nbytes=None)
    a.update(over)
    if a["nbytes"] is None:
        a["nbytes"] = max(0, native.lib().rwkv_decode_workspace_bytes(a["rows"], a["heads"]))
    return native.lib().rwkv_decode_cell(
        ctypes.addressof(p), a["x"], a["ids"], a["state"], a["ti"], a["to"], a["ci"], a["co"], a["et"],
        a["rows"], a["heads"], a["slots"], a["dtype"], a["dither"], a["ws"], a["nbytes"], None)


@pytest.mark.parametrize("first", [True, False])
def test_a_cell_refuses_what_the_recurrence_refuses(native, first):
    p = _params(native, first)
    assert _cell(native, p) == HIP                              # nothing to refuse
    assert _cell(native, p, rows=4) == HIP
    assert _cell(native, p, rows=5) == SHAPE                    # more rows than slots
    assert _cell(native, p, rows=1, slots=0) == SHAPE
    assert _cell(native, p, rows=0, slots=0) == 0
    assert _cell(native, p, ids=2 * GIB + 2) == ALIGNMENT
    assert _cell(native, p, et=8 * GIB + 1) == ALIGNMENT
    assert _cell(native, p, et=None) == NULL
    assert _cell(native, p, dtype=F32, dither=0, et=None) == HIP
    assert _cell(native, p, nbytes=16) == SHAPE


@pytest.mark.parametrize("first", [True, False])
def test_a_cell_refuses_overlap(native, first):
    p = _params(native, first)
    row, shift, state = 128 * 4, 4 * 128 * 4, 4 * 2 * 64 * 64 * 2
    ends = dict(x=3 * row, state=state, to=shift, co=shift,
                ws=native.lib().rwkv_decode_workspace_bytes(3, 2))
    ins = dict(ids=2 * GIB, ti=4 * GIB, ci=6 * GIB, et=8 * GIB)
    for name, size in ends.items():
        for other, at in ins.items():           # over the input's first bytes, and just before it
            assert _cell(native, p, **{name: at}) == OVERLAP, (name, other)
            assert _cell(native, p, **{name: at - size + 16}) == OVERLAP, (name, other)
            assert _cell(native, p, **{name: at - size}) == HIP, (name, other)
        at = p.channel_value
        assert _cell(native, p, **{name: at + 4 * 128 * 128 * 4 - 16}) == OVERLAP, name
        assert _cell(native, p, **{name: at + 4 * 128 * 128 * 4}) == HIP, name
        if not first:
            assert _cell(native, p, **{name: p.residual_b}) == OVERLAP, name
    assert _cell(native, p, x=3 * GIB + state - 16) == OVERLAP  # two that are written
    assert _cell(native, p, to=7 * GIB) == OVERLAP
    assert _cell(native, p, ws=5 * GIB) == OVERLAP


def test_a_head_refuses_overlap(native):
    lib = native.lib()
    need = lib.rwkv_decode_workspace_bytes(3, 2)

    def head(x=GIB, w=2 * GIB, b=3 * GIB, un=4 * GIB, logits=5 * GIB, ws=6 * GIB):
        return lib.rwkv_decode_head(x, w, b, 1e-5, un, 3, 2, 50, logits, ws, need, None)
    assert head() == HIP
    assert head(logits=GIB + 3 * 128 * 4 - 16) == OVERLAP
    assert head(logits=2 * GIB) == OVERLAP and head(ws=4 * GIB + 50 * 128 * 4 - 16) == OVERLAP
    assert head(ws=5 * GIB) == OVERLAP and head(ws=5 * GIB + 304) == HIP   # 3 x 50 logits end at 300
