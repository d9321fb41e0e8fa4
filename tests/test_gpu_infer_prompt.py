"""Prompts on few (row, head) pairs. bf16 state (wkv7_infer_prompt.hip) against
the bf16 oracle, whose operations round in the same order; fp32 state
(wkv7_infer_rows_kernel) against the same rows in a call that is too large for
it. Both equal bit for bit, outputs and states, at the sizes where the staged
steps and tiles begin and end."""

import numpy as np
import pytest
import torch

from conftest import NAMES, announce, load_pkg, to_dev, to_np

pytestmark = pytest.mark.gpu


def _mask(kind, rows, T, rng):
    m = np.ones((rows, T), np.float32)
    if kind == "left":                       # padding of unequal length
        for i in range(rows):
            m[i, :(i * 7 + 3) % T] = 0
    elif kind == "holes":
        m = (rng.random((rows, T)) < 0.6).astype(np.float32)
    elif kind == "edges":                    # first row dead, then one live step each
        m[:] = 0
        for i in range(1, rows):
            m[i, (T - 1) * (i % 2)] = 1
    return m


@pytest.mark.parametrize("rows,T,H,mask", [
    (1, 2, 1, None), (2, 3, 2, None), (1, 4, 3, "holes"), (3, 5, 2, "edges"), (2, 8, 1, "left"),
    (3, 63, 2, "holes"), (2, 64, 3, "left"), (3, 65, 1, "edges"), (2, 130, 2, "left"),
    (3, 200, 2, "holes"),
    # 128 and 129 pairs (rows of a pair over two workgroups, over one); up to four
    # steps 256 and 257 (the last that run here, the first that do not), from
    # five on 512 and 513
    (32, 4, 4, "holes"), (43, 4, 3, None), (43, 9, 3, "left"), (128, 4, 4, "left"), (171, 3, 3, "holes"),
    (64, 4, 4, "left"), (257, 4, 1, None), (128, 5, 4, "left"), (171, 5, 3, "holes"),
])
def test_prompts_equal_the_oracle(oracle, rows, T, H, mask):
    announce("bf16 prompt", rows, T, H, mask)
    pkg = load_pkg()
    wk = pkg.wkv7
    rng = np.random.default_rng(rows * 1000 + T)
    d = pkg.synthetic.make_inputs(rows, T, H, 64, seed=T, bf16=True, with_grad=False)
    slots = rows + 2
    state = pkg.synthetic.bf16_round(rng.standard_normal((slots, H, 64, 64)).astype(np.float32))
    ids = rng.permutation(slots)[:rows].astype(np.int32)
    elapsed = rng.integers(0, 5000, slots).astype(np.int32)
    m = _mask(mask, rows, T, rng) if mask else None
    st_gpu = to_dev(state, torch.bfloat16)
    y = wk.wkv7_infer_forward(*(to_dev(d[n], torch.bfloat16) for n in NAMES),
                              torch.from_numpy(ids).cuda(), st_gpu,
                              None if m is None else to_dev(m, torch.bfloat16),
                              torch.from_numpy(elapsed).cuda()).output
    torch.cuda.synchronize()
    want = state.copy()
    y_want = oracle.infer_bf16(*(d[n] for n in NAMES), ids, want, m, elapsed.view(np.uint32))
    assert np.array_equal(to_np(y), y_want)
    assert np.array_equal(to_np(st_gpu), want)


def test_a_refused_slot_touches_nothing(oracle):
    announce("bf16 prompt, a slot out of range")
    pkg = load_pkg()
    d = pkg.synthetic.make_inputs(2, 6, 2, 64, seed=3, bf16=True, with_grad=False)
    st = torch.randn(2, 2, 64, 64, device="cuda").to(torch.bfloat16)
    before = st.clone()
    out = pkg.wkv7.wkv7_infer_forward(*(to_dev(d[n], torch.bfloat16) for n in NAMES),
                                      torch.tensor([7, 1], dtype=torch.int32, device="cuda"), st,
                                      None, torch.zeros(2, dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    assert not out.output[0].any() and out.output[1].any()
    assert torch.equal(st[0], before[0]) and not torch.equal(st[1], before[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("rows,T,H,mask", [
    (1, 2, 1, None), (2, 15, 3, "holes"), (3, 16, 2, "left"), (2, 17, 2, None), (3, 33, 2, "edges"),
    (32, 18, 4, "holes"), (64, 18, 4, "holes"),             # 128 pairs: the last that run here; 256
])
def test_fp32_state_prompts_equal_a_larger_call(dtype, rows, T, H, mask):
    announce("fp32-state prompt", rows, T, H, mask, str(dtype))
    pkg = load_pkg()
    all_rows = max(rows, 256 // H) + 1                      # over 256 pairs (128 would do)
    rng = np.random.default_rng(T)
    d = pkg.synthetic.make_inputs(all_rows, T, H, 64, seed=T + rows, bf16=dtype == torch.bfloat16,
                                  with_grad=False)
    ops = [to_dev(d[n], dtype) for n in NAMES]
    m = torch.from_numpy(_mask(mask, all_rows, T, rng)).cuda().to(dtype) if mask else None
    ids = torch.from_numpy(rng.permutation(all_rows).astype(np.int32)).cuda()
    state = torch.from_numpy(rng.standard_normal((all_rows, H, 64, 64)).astype(np.float32)).cuda()
    big, small = state.clone(), state.clone()
    want = pkg.wkv7.wkv7_infer_forward(*ops, ids, big, m, None).output
    got = pkg.wkv7.wkv7_infer_forward(*(x[:rows].contiguous() for x in ops), ids[:rows].contiguous(),
                                      small, None if m is None else m[:rows].contiguous(), None).output
    torch.cuda.synchronize()
    assert torch.equal(got, want[:rows])
    used = ids[:rows].long()
    assert torch.equal(small[used], big[used])
    rest = ids[rows:].long()
    assert torch.equal(small[rest], state[rest])


@pytest.mark.parametrize("rows", [2, 130])                  # below and above 256 pairs
@pytest.mark.parametrize("dtype,state_dtype", [
    (torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16)])
def test_a_call_without_tokens_leaves_the_states(rows, dtype, state_dtype):
    announce("prompt of no tokens", rows, str(dtype), str(state_dtype))
    wk = load_pkg().wkv7
    ops = [torch.empty(rows, 0, 2, 64, dtype=dtype, device="cuda") for _ in range(6)]
    st = torch.randn(rows, 2, 64, 64, device="cuda").to(state_dtype)
    before = st.clone()
    out = wk.wkv7_infer_forward(*ops, torch.arange(rows, dtype=torch.int32, device="cuda"), st, None,
                                torch.zeros(rows, dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    assert out.output.shape == (rows, 0, 2, 64) and torch.equal(st, before)
