"""One decode step of the model on the fused kernels (include/rwkv_decode.h)
against the modules it stands in for, at the sizes where its row tiles, column
tiles and slots begin and end. Both round every intermediate to bf16 at the same
places and differ only in the order of sums, so a value near a tie comes out one
bf16 ulp off and travels on: per layer about 3e-3 relative, held to 1e-2 on a
two-cell model's logits and shifts."""

import pytest
import torch

from conftest import announce, load_pkg
from model_helpers import tiny_model

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _err(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm())


def _model(heads=2, vocab=97, cells=2, seed=1):
    return tiny_model(seed=seed, cells=cells, heads=heads, vocab=vocab, std=0.2,
                      wkv7_dtype=torch.bfloat16, neighbor_ops="hip").to(DEV)


def _state(model, slots, state_dtype, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    st = model.new_infer_state(slots, state_dtype=state_dtype)
    for t in st.shift_time + st.state + st.shift_channel:
        t.copy_(torch.randn(t.shape, generator=g, device=DEV) * 0.5)
    st.elapsed_t.copy_(torch.randint(0, 99, (slots,), generator=g, device=DEV))
    return st


def _infer(model, toks, ids, st, mode="last"):
    with torch.autocast("cuda", dtype=torch.bfloat16):
        return model.infer(toks, ids, st, unembed_mode=mode)


@pytest.mark.parametrize("rows,slots,heads,vocab,state_dtype", [
    (1, 1, 1, 1, torch.bfloat16), (3, 5, 2, 97, torch.bfloat16), (16, 16, 2, 16, torch.float32),
    (17, 20, 3, 33, torch.bfloat16), (33, 33, 2, 97, torch.float32), (64, 70, 2, 130, torch.bfloat16),
])
def test_a_fused_step_matches_the_modules(monkeypatch, rows, slots, heads, vocab, state_dtype):
    announce("decode step", rows, slots, heads, vocab, str(state_dtype))
    decode = load_pkg().decode
    model = _model(heads, vocab)
    ids = torch.randperm(slots, generator=torch.Generator().manual_seed(rows))[:rows].to(DEV)
    toks = torch.randint(0, vocab, (rows, 1), generator=torch.Generator().manual_seed(3)).to(DEV)
    a, b = _state(model, slots, state_dtype, 7), _state(model, slots, state_dtype, 7)
    before = [t.clone() for t in a.state + a.shift_time + a.shift_channel]
    taken = []
    real = decode.step
    monkeypatch.setattr(decode, "step", lambda *x: taken.append(real(*x)) or taken[-1])
    got = _infer(model, toks, ids, a)
    monkeypatch.setattr(decode, "step", lambda *x: None)
    want = _infer(model, toks, ids, b)
    torch.cuda.synchronize()
    assert taken[0] is not None and got.dtype == want.dtype and got.shape == want.shape
    assert _err(got, want) < 1e-2
    idle = [s for s in range(slots) if s not in ids.tolist()]
    for x, y, z in zip(a.state + a.shift_time + a.shift_channel,
                       b.state + b.shift_time + b.shift_channel, before):
        assert x.dtype == y.dtype and _err(x, y) < 1e-2
        assert torch.equal(x[idle], z[idle])
    monkeypatch.setattr(decode, "step", real)
    c = _state(model, slots, state_dtype, 7)
    assert _infer(model, toks, ids, c, "skip") is None
    assert all(torch.equal(x, y) for x, y in zip(c.state + c.shift_time, a.state + a.shift_time))


def test_what_the_kernels_do_not_take_goes_through_the_modules():
    announce("decode step, calls that stay with the modules")
    decode = load_pkg().decode
    model = _model()
    st = _state(model, 4, torch.bfloat16, 1)
    ids, toks = torch.arange(3, device=DEV), torch.zeros(3, 1, dtype=torch.long, device=DEV)

    def taken(m=model, t=toks, i=ids, s=st, mask=None):
        with torch.autocast("cuda", dtype=torch.bfloat16), torch.no_grad():
            return decode.step(m, t, i, s, mask, "last") is not None
    assert taken()
    assert not taken(t=toks.expand(3, 2)) and not taken(mask=torch.ones(3, 1, device=DEV))
    with torch.no_grad():
        assert decode.step(model, toks, ids, st, None, "last") is None      # no autocast
    seen = []
    hook = model.cells.cells[1].channel_mixer.key.register_forward_hook(lambda *x: seen.append(1))
    assert not taken()
    _infer(model, toks, ids, st)
    assert seen == [1]
    hook.remove()
    assert taken()

    class Other(torch.nn.Linear):
        pass
    old = model.cells.cells[0].time_mixer.gated_readout.projection_output
    model.cells.cells[0].time_mixer.gated_readout.projection_output = Other(128, 128, bias=False).to(DEV)
    assert not taken()
    model.cells.cells[0].time_mixer.gated_readout.projection_output = old
    w = model.cells.cells[0].channel_mixer.key.weight
    w.data = w.data.t().contiguous().t()
    assert not taken()
    w.data = w.data.contiguous().to(torch.bfloat16)
    assert not taken()


def test_an_id_out_of_range_touches_no_slot():
    announce("decode step, a slot out of range")
    model = _model()
    st, ref = _state(model, 4, torch.bfloat16, 2), _state(model, 4, torch.bfloat16, 2)
    toks = torch.arange(2, device=DEV).reshape(2, 1)
    _infer(model, toks, torch.tensor([9, 2], device=DEV), st)
    torch.cuda.synchronize()
    for x, y in zip(st.state + st.shift_time + st.shift_channel,
                    ref.state + ref.shift_time + ref.shift_channel):
        assert torch.equal(x[[0, 1, 3]], y[[0, 1, 3]]) and not torch.equal(x[2], y[2])


def test_more_rows_than_slots_are_refused():
    announce("decode step, more rows than slots")
    model = _model()
    st, ref = _state(model, 2, torch.bfloat16, 2), _state(model, 2, torch.bfloat16, 2)
    toks = torch.arange(3, device=DEV).reshape(3, 1)
    with pytest.raises(load_pkg()._native.Wkv7Error, match="WKV7_ERR_SHAPE"):
        _infer(model, toks, torch.tensor([0, 1, 1], device=DEV), st)
    torch.cuda.synchronize()
    for x, y in zip(st.state + st.shift_time + st.shift_channel,
                    ref.state + ref.shift_time + ref.shift_channel):
        assert torch.equal(x, y)


def test_the_first_norms_output_is_not_written():
    # what a hook on it keeps (activation capture), or the norm itself
    announce("decode step, the first norm's output kept by others")
    model = _model()
    ids, toks = torch.arange(3, device=DEV), torch.arange(3, device=DEV).reshape(3, 1)
    plain = _infer(model, toks, ids, _state(model, 4, torch.bfloat16, 1))
    kept = []
    hook = model.layer_norm_for_first_cell.register_forward_hook(lambda m, i, out: kept.append(out))
    hooked = _infer(model, toks, ids, _state(model, 4, torch.bfloat16, 1))
    hook.remove()
    want = model.layer_norm_for_first_cell(model.embed(toks))
    assert len(kept) == 1 and torch.equal(kept[0], want) and torch.equal(hooked, plain)

    class Kept(torch.nn.Module):
        def forward(self, x):
            return want
    model.layer_norm_for_first_cell = Kept()
    before = want.clone()
    for _ in range(2):
        assert torch.equal(_infer(model, toks, ids, _state(model, 4, torch.bfloat16, 1)), plain)
    assert torch.equal(want, before)


def test_the_embedding_and_the_first_norm_run_once(monkeypatch):
    # a first norm whose result the kernels do not take: the modules go on from it
    announce("decode step, a first norm in bf16")
    decode = load_pkg().decode
    model = _model()
    ids, toks = torch.arange(3, device=DEV), torch.arange(3, device=DEV).reshape(3, 1)
    calls = []

    class Norm(torch.nn.Module):
        def forward(self, x):
            calls.append("norm")
            return x.bfloat16()
    model.layer_norm_for_first_cell = Norm()
    model.embed.register_forward_hook(lambda *x: calls.append("embed"))
    a, b = _state(model, 4, torch.bfloat16, 1), _state(model, 4, torch.bfloat16, 1)
    got = _infer(model, toks, ids, a)
    assert calls == ["embed", "norm"]
    assert _infer(model, toks, ids, _state(model, 4, torch.bfloat16, 1), "skip") is None
    monkeypatch.setattr(decode, "step", lambda *x: None)
    assert torch.equal(got, _infer(model, toks, ids, b))
    for x, y in zip(a.state + a.shift_time + a.shift_channel, b.state + b.shift_time + b.shift_channel):
        assert x.dtype == y.dtype and torch.equal(x, y)


class _Wrap(torch.nn.Module):
    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, *args, **kwargs):
        return self.inner(*args, **kwargs)


class _Table(torch.nn.Module):
    def __init__(self, table):
        super().__init__()
        self.register_buffer("table", table)

    def forward(self, ids):
        return self.table[ids]


def _as_attribute(module, name):
    value = getattr(module, name).detach()
    delattr(module, name)
    setattr(module, name, value)


def _wrap(module, name):
    setattr(module, name, _Wrap(getattr(module, name)))


def _list_of_cells(model):
    cells = list(model.cells.cells)
    del model.cells.cells
    model.cells.cells = cells


@pytest.mark.parametrize("change", [
    lambda m: m.cells.cells.__setitem__(1, _Wrap(m.cells.cells[1])),
    lambda m: _wrap(m.cells.cells[0], "time_mixer"),
    lambda m: _wrap(m.cells.cells[0].time_mixer, "weight_prepare"),
    lambda m: _wrap(m, "cells"),
    _list_of_cells,
    lambda m: _as_attribute(m.cells.cells[1].channel_mixer.value, "weight"),
    lambda m: _as_attribute(m.cells.cells[1].pre_layer_norm_for_time_mix, "bias"),
    lambda m: _as_attribute(m.cells.cells[0].time_mixer.weight_prepare, "param_key"),
    lambda m: _as_attribute(m.cells.cells[0].time_mixer.weight_prepare.param_weight_decay_lora, "w_a"),
    lambda m: _as_attribute(m.cells.cells[0].time_mixer.weight_prepare.param_weight_decay_lora, "bias"),
    lambda m: _as_attribute(m.layer_norm_for_unembed, "weight"),
    lambda m: setattr(m.cells.cells[0].time_mixer.weight_prepare.param_weight_decay_lora, "product",
                      lambda x: x * 0.0),
    lambda m: setattr(m, "embed", _Table(m.embed.weight.detach())),
], ids=["cell", "time_mixer", "weight_prepare", "cells", "list", "linear", "norm", "scale", "lora", "lora_bias",
        "head_norm", "product", "embed"])
def test_a_changed_model_still_runs(monkeypatch, request, change):
    announce("decode step, a changed model", request.node.name)
    decode = load_pkg().decode
    model = _model()
    ids, toks = torch.arange(3, device=DEV), torch.arange(3, device=DEV).reshape(3, 1)
    plain = _infer(model, toks, ids, _state(model, 4, torch.bfloat16, 1))
    st = [_state(model, 4, torch.bfloat16, 1) for _ in range(2)]
    change(model)
    got = _infer(model, toks, ids, st[0])
    if "embed" in request.node.callspec.id:      # the kernels do not look at it
        assert torch.equal(got, plain)
        return
    monkeypatch.setattr(decode, "step", lambda *x: None)
    assert torch.equal(got, _infer(model, toks, ids, st[1]))
    assert all(torch.equal(x, y) for x, y in zip(st[0].state + st[0].shift_time, st[1].state + st[1].shift_time))


def test_a_residual_stream_off_the_states_device_stays_with_the_modules(monkeypatch):
    # here on the host: the modules refuse it; no kernel may see its address
    announce("decode step, an embedding on the host")
    native = load_pkg()._native

    def no_library():
        raise AssertionError("the fused step took it")
    model = _model()
    st = _state(model, 4, torch.float32, 1)
    model.embed = model.embed.cpu()
    model.layer_norm_for_first_cell = torch.nn.Identity()
    monkeypatch.setattr(native, "lib", no_library)
    with pytest.raises(RuntimeError, match="device"):
        _infer(model, torch.zeros(2, 1, dtype=torch.long), torch.arange(2, device=DEV), st)


def test_a_state_without_elapsed_t_is_refused_as_by_the_modules():
    announce("decode step, no elapsed_t")
    model = _model()
    st = _state(model, 4, torch.float32, 1)
    st.elapsed_t = None
    with pytest.raises(ValueError, match="elapsed_t required"):
        _infer(model, torch.zeros(2, 1, dtype=torch.long, device=DEV), torch.arange(2, device=DEV), st)


def _wide_model(heads, cells=1, vocab=33):
    m = load_pkg().model
    with torch.device(DEV):
        model = m.AutoRegressiveModel(vocab, cells, heads * 64, heads, 64, wkv7_dtype=torch.bfloat16,
                                      neighbor_ops="hip")
    # products of the size that std 0.2 gives at two heads
    return model.init_random(0.2 * (2 / heads) ** 0.5, torch.Generator(DEV).manual_seed(1))


@pytest.mark.parametrize("heads,fused", [(64, True), (65, False)])
def test_the_widest_model_of_the_fused_step(monkeypatch, heads, fused):
    announce("decode step, where the widths end", heads)
    decode = load_pkg().decode
    model = _wide_model(heads)
    taken = []
    real = decode.step
    monkeypatch.setattr(decode, "step", lambda *x: taken.append(real(*x)) or taken[-1])
    ids, toks = torch.arange(2, device=DEV), torch.arange(2, device=DEV).reshape(2, 1)
    _infer(model, toks, ids, _state(model, 2, torch.bfloat16, 1))
    assert (taken[0] is not None) == fused


@pytest.mark.parametrize("heads,rows,state_dtype", [
    (16, 5, torch.bfloat16),                              # C = 1024: the last of four channels a thread
    (17, 3, torch.bfloat16), (31, 18, torch.float32), (32, 33, torch.bfloat16),     # eight: 1088 .. 2048
    (33, 2, torch.float32), (64, 17, torch.bfloat16), (128, 3, torch.bfloat16),     # 32: 2112 .. 8192
])
def test_a_fused_step_of_a_wide_model_matches_the_modules(monkeypatch, heads, rows, state_dtype):
    # each instance of the norms, and the products' rounds over K = C and 4 C;
    # the kernels' widest is wider than what infer sends to them
    announce("decode step, wide", heads, rows, str(state_dtype))
    decode = load_pkg().decode
    monkeypatch.setattr(decode, "MAX_DIM", 8192)
    model = _wide_model(heads)
    ids, toks = torch.arange(rows, device=DEV), torch.arange(rows, device=DEV).reshape(rows, 1) % 33
    a, b = _state(model, rows, state_dtype, 7), _state(model, rows, state_dtype, 7)
    taken = []
    real = decode.step
    monkeypatch.setattr(decode, "step", lambda *x: taken.append(real(*x)) or taken[-1])
    got = _infer(model, toks, ids, a)
    monkeypatch.setattr(decode, "step", lambda *x: None)
    want = _infer(model, toks, ids, b)
    assert taken[0] is not None and _err(got, want) < 1e-2
    for x, y in zip(a.state + a.shift_time + a.shift_channel, b.state + b.shift_time + b.shift_channel):
        assert _err(x, y) < 1e-2


def test_a_captured_step_replays_and_streams_do_not_share():
    # the workspace and the residual stream come from the capture's pool; eager
    # steps of another size between the replays, and two streams at once
    announce("decode step in a graph and on two streams")
    model = _model(3)
    ids, toks = torch.arange(5, device=DEV), torch.arange(5, device=DEV).reshape(5, 1)
    start = _state(model, 6, torch.bfloat16, 1)
    st = _state(model, 6, torch.bfloat16, 1)
    lists = ("state", "shift_time", "shift_channel")

    def reset(s, to=start):
        for n in lists:
            for x, y in zip(getattr(s, n), getattr(to, n)):
                x.copy_(y)
    eager = _state(model, 6, torch.bfloat16, 1)
    want = _infer(model, toks, ids, eager).clone()
    # the shifts' next buffers replace those of infer_state, so a captured step
    # starts from the tensors that it was captured with
    held = {n: list(getattr(st, n)) for n in lists}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _infer(model, toks, ids, _state(model, 6, torch.bfloat16, 1))
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = _infer(model, toks, ids, st)
    out = {n: list(getattr(st, n)) for n in lists}
    for _ in range(3):
        got.zero_()
        for n in lists:
            for x, y in zip(held[n], getattr(start, n)):
                x.copy_(y)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        for n in lists:
            assert all(torch.equal(x, y) for x, y in zip(out[n], getattr(eager, n)))
        _infer(model, toks[:2], ids[:2], _state(model, 6, torch.float32, 2))
    streams, got = [torch.cuda.Stream() for _ in range(2)], [[], []]
    sts = [_state(model, 6, torch.bfloat16, 1) for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(4):
        for i, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                reset(sts[i])
                got[i].append(_infer(model, toks, ids, sts[i]))
    torch.cuda.synchronize()
    assert all(torch.equal(x, want) for g in got for x in g)
