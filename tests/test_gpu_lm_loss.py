"""GPU parity of the fused loss (include/rwkv_lm_loss.h) against float64
PyTorch on the CPU: l2wrap as the model's torch Function (kernels/l2wrap/
mod.rs:38-66) followed by ``F.cross_entropy`` (the mean over rows, as
examples/rwkv-lm/src/model.rs:161-169), forward and backward.

Every row gets a unique maximum, so the argmax that l2wrap's term lands on
is the same in both. Bars: the loss and the per-row statistics within 1e-5
relative (both read the same logits and compute in fp32 / fp64); the
logits' gradient within 1e-5 relative L2 in fp32 and 8e-3 in bf16 (its
rounding).
"""

import pytest
import torch
import torch.nn.functional as F

from conftest import announce, load_pkg, rel_l2
from model_helpers import _model_mod

pytestmark = pytest.mark.gpu

CASES = [
    dict(rows=6, V=97, dt="f32"),          # element path (vocab not a multiple of 8)
    dict(rows=33, V=512, dt="f32"),        # vector path
    dict(rows=17, V=50, dt="bf16"),
    dict(rows=40, V=1000, dt="bf16"),
    dict(rows=64, V=65536, dt="bf16"),     # config[4]'s vocabulary
    dict(rows=3, V=8, dt="f32"),           # fewer logits than threads
]
DT = {"f32": torch.float32, "bf16": torch.bfloat16}


def _case_id(c):
    return "rows{rows}_V{V}_{dt}".format(**c)


def _inputs(rows, V, dt, seed):
    g = torch.Generator().manual_seed(seed)
    logits = 3.0 * torch.randn(rows, V, generator=g)
    peak = torch.randint(0, V, (rows,), generator=g)
    logits[torch.arange(rows), peak] = logits.max(dim=1).values + 1.0   # unique maximum
    logits = logits.to(DT[dt])
    targets = torch.randint(0, V, (rows,), generator=g)
    return logits, targets, peak


@pytest.mark.parametrize("case", CASES, ids=_case_id)
def test_cross_entropy_l2wrap_matches_torch(case):
    ll = load_pkg().lm_loss
    m = _model_mod()
    rows, V, dt = case["rows"], case["V"], case["dt"]
    logits, targets, peak = _inputs(rows, V, dt, rows * 7 + V)

    x64 = logits.double().requires_grad_(True)
    want = F.cross_entropy(m.l2wrap(x64, rows), targets)
    want.backward()

    dev = torch.device("cuda:0")
    x = logits.to(dev).requires_grad_(True)
    announce("cross_entropy_l2wrap", _case_id(case))
    got = ll.cross_entropy_l2wrap(x, targets.to(dev))
    got.backward()
    torch.cuda.synchronize()
    assert abs(got.item() - want.item()) <= 1e-5 * abs(want.item()), (got.item(), want.item())
    tol = 8e-3 if dt == "bf16" else 1e-5
    assert x.grad.dtype == logits.dtype
    assert rel_l2(x.grad.double().cpu().numpy(), x64.grad.numpy()) <= tol


def test_row_statistics_and_out_of_range_target():
    ll = load_pkg().lm_loss
    rows, V = 5, 300
    logits, targets, peak = _inputs(rows, V, "f32", 11)
    targets[2] = V + 4                          # out of range: NaN loss, no target term
    dev = torch.device("cuda:0")
    x = logits.to(dev).requires_grad_(True)
    announce("cross_entropy_l2wrap", "rows5_V300_bad_target")
    per_row = ll.cross_entropy_l2wrap_rows(x, targets.to(dev), rows)
    w = torch.arange(1, rows + 1, dtype=torch.float32, device=dev)   # uneven row weights
    per_row.backward(w)
    torch.cuda.synchronize()
    got = per_row.double().cpu()
    lse = torch.logsumexp(logits.double(), dim=1)
    ok = torch.arange(rows) != 2
    want = lse - logits.double()[torch.arange(rows), targets.clamp(max=V - 1)]
    assert torch.isnan(got[2])
    assert torch.allclose(got[ok], want[ok], rtol=1e-5, atol=0)
    # gradient: w_r (softmax - onehot) + 1e-4 / rows * max at the argmax
    sm = torch.softmax(logits.double(), dim=1)
    onehot = torch.zeros(rows, V, dtype=torch.float64)
    onehot[ok, targets[ok]] = 1.0
    ref = w.double().cpu()[:, None] * (sm - onehot)
    ref[torch.arange(rows), peak] += 1e-4 / rows * logits.double().max(dim=1).values
    assert rel_l2(x.grad.double().cpu().numpy(), ref.numpy()) <= 1e-5


@pytest.mark.parametrize("rows,V,dt,offset", [
    (1, 1, "bf16", 0), (3, 7, "bf16", 0), (9, 8201, "bf16", 0), (513, 2051, "bf16", 0),
    (5, 4099, "f32", 0), (520, 2057, "f32", 0), (16, 65529, "bf16", 0),
    (256, 16384, "bf16", 0), (257, 16387, "bf16", 0), (4, 16383, "f32", 0), (6, 16391, "f32", 1),
    (9, 333, "bf16", 1), (7, 2051, "f32", 3),
    # both widths of the forward at rows of whole pieces and not, rows taken one by
    # one (up to 512) and in pieces, each with and without blocks that share a row
    (3, 24568, "f32", 0), (3, 24576, "bf16", 0), (2, 24576, "f32", 0), (3, 24577, "bf16", 0),
    (5, 511, "bf16", 0), (5, 513, "f32", 0), (300, 64, "f32", 0), (2100, 48, "bf16", 0),
    (2100, 509, "bf16", 0), (2100, 523, "bf16", 0), (300, 523, "f32", 0),
])
def test_rows_that_begin_anywhere(rows, V, dt, offset):
    """Heads, pieces and tails of rows at every alignment, on both widths of the
    forward and with rows shared by blocks in the backward; ``offset`` elements
    put the logits, not their gradient, off a 16-byte boundary. Some logits are
    -inf, a masked vocabulary's, over whole pieces. The module's bars."""
    ll = load_pkg().lm_loss
    logits, targets, peak = _inputs(rows, V, dt, rows + V)
    col = torch.arange(V)
    masked = ((col < 40) | (col >= V - 3)) & (col[None, :] != peak[:, None]) & (
        col[None, :] != targets[:, None])
    logits[masked] = float("-inf")
    dev = torch.device("cuda:0")
    flat = torch.empty(rows * V + offset, dtype=DT[dt], device=dev)
    x = flat[offset:].view(rows, V)
    x.copy_(logits)
    x = x.detach().requires_grad_(True)
    announce("cross_entropy_l2wrap", f"rows{rows}_V{V}_{dt}_offset{offset}")
    got = ll.cross_entropy_l2wrap_rows(x, targets.to(dev), rows)
    w = torch.linspace(0.5, 2.0, rows, device=dev)
    got.backward(w)
    torch.cuda.synchronize()
    z = logits.double()
    at = torch.arange(rows)
    lse = torch.logsumexp(z, dim=1)
    want = lse - z[at, targets]
    # loss = lse - x_t in fp32: an error of 1e-5 of the larger term
    assert bool(((got.double().cpu() - want).abs() <= 1e-5 * (lse.abs() + z[at, targets].abs())).all())
    ref = torch.softmax(z, dim=1)
    ref[at, targets] -= 1.0
    ref *= w.double().cpu()[:, None]
    ref[at, peak] += 1e-4 / rows * z.max(dim=1).values
    grad = x.grad.double().cpu()
    assert rel_l2(grad.numpy(), ref.numpy()) <= (8e-3 if dt == "bf16" else 1e-5)
    assert bool((grad[masked] == 0).all())
