"""Calls with few (batch, head) pairs, whose sequences run cut into segments
(wkv7_forward_ws / wkv7_backward_ws, include/wkv7_segments.h; the Python calls pass the
workspace by themselves), against the same calls in one piece
(wkv7_forward_ex / wkv7_backward_ex, no workspace). The two differ only in how
a segment's start state is formed, by products of the same precision, so they
are held to twice the deviation that the kernels in one piece have from fp32
arithmetic: bf16 operands 2 x 6e-6 on the fp32 tensors, and on bf16 tensors
the rounding of values that close (2e-4 measured between the families); fp32
operands 2 x 1e-6 on outputs and states and 2 x 1e-5 on the gradients (the
bar between their families, set by the reversal between checkpoints)."""

import pytest
import torch

from conftest import GRAD_NAMES, NAMES, announce, load_pkg, rel_l2, to_dev, to_np

F32, BF16 = 0, 1


@pytest.fixture(scope="module")
def wk():
    return load_pkg().wkv7


def _bytes(which, B, T, H, chunk, dtype):
    lib = load_pkg()._native.lib()
    return getattr(lib, f"wkv7_{which}_workspace_bytes")(B, T, H, 64, chunk, dtype, None)


def _segments(which, B, T, H, chunk, dtype):
    # two 64 x 64 fp32 matrices and a 4-byte word per pair and segment
    return _bytes(which, B, T, H, chunk, dtype) // (B * H * (2 * 4096 * 4 + 4))


def _in_one_piece(name, args):
    """A *_ws call's arguments (workspace, bytes, stream last) without the workspace."""
    load_pkg()._native.call(name, *args[:-3], args[-1])


CASES = [
    # B, T, H, chunk, dtype: one pair; an uneven last segment; a prime chunk
    # count; the most pairs that still get three forward segments; two
    # backward segments only; longer checkpoint intervals (backward)
    (1, 1024, 1, 16, BF16),
    (1, 2048 + 16 * 5, 3, 16, BF16),
    (2, 16 * 131, 5, 16, BF16),
    (5, 1536, 17, 16, BF16),
    (8, 1024, 16, 16, BF16),
    (1, 32 * 40, 4, 32, BF16),
    (1, 48 * 31, 2, 48, BF16),
    # fp32 products: fp32 operands, and bf16 ones at a longer interval above
    (1, 1024, 1, 16, F32),
    (1, 2048 + 16 * 5, 3, 16, F32),
    (2, 16 * 131, 5, 16, F32),
    (4, 512, 8, 16, F32),
    (1, 32 * 41, 4, 32, F32),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("edges", [True, False], ids=["states", "no_states"])
def test_segments_match_one_piece(wk, monkeypatch, case, edges):
    B, T, H, chunk, dtype = case
    announce("segments", case, edges)
    pkg = load_pkg()
    bf16 = dtype == BF16
    td = torch.bfloat16 if bf16 else torch.float32
    d = pkg.synthetic.make_inputs(B, T, H, 64, seed=T + H, s0_std=0.5, bf16=bf16)
    if chunk > 32:     # decays near one: the reversal between checkpoints amplifies nothing
        d["w"] = d["w"] - 6.0
    ins = [to_dev(d[n], td) for n in NAMES]
    s0, dy = to_dev(d["s0"]), to_dev(d["dy"], td)
    dsT = 0.3 * torch.randn(B, H, 64, 64, device="cuda", generator=torch.Generator("cuda").manual_seed(T))
    nf, nb = (_segments(w, B, T, H, chunk, dtype) for w in ("forward", "backward"))
    print(f"segments: forward {nf}, backward {nb}", flush=True)
    assert nb > 1

    def both():
        f = wk.wkv7_forward_ex(*ins, s0, chunk, edges, True)
        g = wk.wkv7_backward_ex(*ins, base.state, base.removal_state, dy, dsT, chunk, edges, True)
        return f, g
    native = wk._native

    class OnePiece:
        def __getattr__(self, name):
            return getattr(native, name)

        @staticmethod
        def call(name, *args):
            _in_one_piece(name.replace("_ws", "_ex"), args)
    with monkeypatch.context() as m:
        m.setattr(wk, "_native", OnePiece())
        base = wk.wkv7_forward_ex(*ins, s0, chunk, edges, True)
        f1, g1 = both()
    f2, g2 = both()
    torch.cuda.synchronize()
    assert wk.take_faults() == 0
    state_tol = 1.2e-5 if bf16 else 2e-6
    out_tol, grad_tol = (4e-4, 4e-4) if bf16 else (2e-6, 2e-5)
    for name, tol in (("output", out_tol), ("state", state_tol), ("removal_state", state_tol),
                      ("final_state", state_tol)):
        err = rel_l2(to_np(getattr(f2, name)), to_np(getattr(f1, name)))
        assert err <= tol, (name, err)
    for name in GRAD_NAMES + ("initial_state_grad",):
        tol = state_tol if name == "initial_state_grad" else grad_tol
        err = rel_l2(to_np(getattr(g2, name)), to_np(getattr(g1, name)))
        assert err <= tol, (name, err)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
def test_segments_replay_in_a_graph(wk, dtype):
    # workspace from the capture's pool; eager calls of another shape between
    announce("segments in a graph", dtype)
    pkg = load_pkg()
    td = torch.bfloat16 if dtype == BF16 else torch.float32
    B, T, H = 1, 1536, 4
    d = pkg.synthetic.make_inputs(B, T, H, 64, seed=5, s0_std=0.1, bf16=dtype == BF16)
    ins = [to_dev(d[n], td) for n in NAMES]
    s0, dy, z = to_dev(d["s0"]), to_dev(d["dy"], td), torch.zeros(B, H, 64, 64, device="cuda")

    def step(k=1):
        part = [x[:, :T // k].contiguous() for x in ins]
        f = wk.wkv7_statepass_forward(*part, s0, 16)
        g = wk.wkv7_statepass_backward(*part, f.state, f.removal_state,
                                       dy[:, :T // k].contiguous(), z, 16)
        return [f.output, f.final_state, f.state, g.key_grad, g.weight_decay_grad, g.initial_state_grad]
    want = [t.clone() for t in step()]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step()
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)
        step(2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
def test_a_given_up_wait_poisons_the_whole_pair(wk, dtype):
    # every wait limited to one poll (a run that ends normally): a pair any of
    # whose segments gave up comes back all NaN and is counted once, the others
    # are those of a normal run
    announce("segments, hand-over fault path (forced from the host)", dtype)
    pkg = load_pkg()
    td = torch.bfloat16 if dtype == BF16 else torch.float32
    B, T, H = 2, 1024, 4
    d = pkg.synthetic.make_inputs(B, T, H, 64, seed=52, s0_std=0.1, bf16=dtype == BF16)
    ins = [to_dev(d[n], td) for n in NAMES]
    s0, dy, z = to_dev(d["s0"]), to_dev(d["dy"], td), torch.zeros(B, H, 64, 64, device="cuda")
    assert _segments("forward", B, T, H, 16, dtype) > 1 and wk.take_faults() == 0
    good = wk.wkv7_statepass_forward(*ins, s0, 16)
    good_g = wk.wkv7_statepass_backward(*ins, good.state, good.removal_state, dy, z, 16)
    bad = wk.wkv7_forward_ex(*ins, s0, 16, handover_spin_limit=1)
    fwd_faults = wk.take_faults()
    options = wk._options("auto", 1)
    bg, bds0 = wk._backward(*ins, good.state, good.removal_state, dy, z, 16, True, True, options)
    bwd_faults = wk.take_faults()
    hit = [0, 0]
    for b in range(B):
        for h in range(H):
            fwd = [(getattr(bad, n), getattr(good, n)) for n in ("output", "removal_state")]
            fwd = [(x[b, :, h], y[b, :, h]) for x, y in fwd]
            fwd += [(getattr(bad, n)[b, h], getattr(good, n)[b, h]) for n in ("state", "final_state")]
            bwd = [(x[b, :, h], getattr(good_g, n)[b, :, h]) for x, n in zip(bg, GRAD_NAMES)]
            bwd += [(bds0[b, h], good_g.initial_state_grad[b, h])]
            for i, parts in enumerate((fwd, bwd)):
                if any(torch.isnan(x.float()).any() for x, _ in parts):
                    assert all(torch.isnan(x.float()).all() for x, _ in parts), (b, h)
                    hit[i] += 1
                else:
                    assert all(torch.equal(x, y) for x, y in parts), (b, h)
    print("forced hand-over faults:", fwd_faults, bwd_faults, "poisoned pairs:", hit, flush=True)
    assert [fwd_faults, bwd_faults] == hit and hit[0] > 0
    again = wk.wkv7_statepass_forward(*ins, s0, 16)
    assert wk.take_faults() == 0 and torch.equal(again.output, good.output)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [(1, 32 * 40, 4, 32, BF16), (2, 32 * 20, 8, 32, BF16), (1, 32 * 41, 4, 32, F32),
                                  (1, 2048 + 16 * 5, 3, 16, F32), (1, 2048 + 16 * 5, 3, 16, BF16)])
def test_backward_from_the_segmented_forwards_checkpoints(wk, monkeypatch, case):
    # at chunk_len 32 the backward rebuilds states from the checkpoints, which
    # multiplies their deviation by about 1.35 a step (120 over the 16 between
    # them); the two forwards' checkpoints are 1e-8 apart at fp32 products, so
    # their 1e-6 stays inside the gradients' bar
    B, T, H, chunk, dtype = case
    announce("segments, forward's checkpoints into the backward", case)
    bf16 = dtype == BF16
    td = torch.bfloat16 if bf16 else torch.float32
    d = load_pkg().synthetic.make_inputs(B, T, H, 64, seed=T + H, s0_std=0.5, bf16=bf16)
    ins = [to_dev(d[n], td) for n in NAMES]
    s0, dy = to_dev(d["s0"]), to_dev(d["dy"], td)
    dsT = 0.3 * torch.randn(B, H, 64, 64, device="cuda", generator=torch.Generator("cuda").manual_seed(T))
    assert _segments("forward", B, T, H, chunk, dtype) > 1 and _segments("backward", B, T, H, chunk, dtype) > 1

    def chain():
        f = wk.wkv7_statepass_forward(*ins, s0, chunk)
        return wk.wkv7_statepass_backward(*ins, f.state, f.removal_state, dy, dsT, chunk)
    cut = chain()
    native = wk._native

    class OnePiece:
        def __getattr__(self, name):
            return getattr(native, name)

        @staticmethod
        def call(name, *args):
            _in_one_piece(name.replace("_ws", "_ex"), args)
    with monkeypatch.context() as m:
        m.setattr(wk, "_native", OnePiece())
        one = chain()
    torch.cuda.synchronize()
    for name in GRAD_NAMES + ("initial_state_grad",):
        err = rel_l2(to_np(getattr(cut, name)), to_np(getattr(one, name)))
        print(name, err, flush=True)
        assert err <= ((1.2e-5 if name == "initial_state_grad" else 4e-4) if bf16 else 2e-5), (name, err)
