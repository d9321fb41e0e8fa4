"""One decode step of the model on the kernels of include/rwkv_decode.h.

``AutoRegressiveModel.infer`` uses it for a step of up to 64 sequences under
bf16 autocast with fp32 parameters (``step`` says when), in place of the
modules' forwards one after another: nine launches a cell issued by one native
call, against about sixty from Python. Everything is read from the modules on
every call, and nothing is kept between calls.

The embedding and the first layer norm run as the modules they are. The cells
and the head are passed by, so anything attached to one of their modules (a
hook, a replaced or subclassed module, a parameter that is no longer one, a
forward set on the instance) sends the whole step back to the modules.
"""

from __future__ import annotations

import ctypes
from typing import Optional

import torch
import torch.nn as nn

from . import _native

MAX_ROWS = 64        # RWKV_DECODE_MAX_ROWS
# The kernels take C up to RWKV_DECODE_MAX_DIM (8192), but they read the fp32
# weights on every step, and a loop inside one autocast context has the modules
# cast them once and read half as much. us a step, such a loop through the
# modules and here, 1 / 17 / 64 sequences: C = 2560, 4 cells 2643 / 535, 2684 / 674,
# 2653 / 1075; C = 4096, 3 cells 1937 / 632, 1952 / 772, 1953 / 1268; C = 6400, 2
# cells 1337 / 1067, 1363 / 1308, 1355 / 2168; C = 8192, 2 cells 1369 / 1437, 1468 /
# 1738, 1601 / 2878. (Replayed from a graph that holds no casts the modules take
# 1124 at C = 4096 and 64 sequences against 1252, elsewhere up to 4096 they are
# slower; with a context a step, 2157 and more at C = 4096.)
MAX_DIM = 4096


def _plain(module, cls) -> bool:
    """Exactly ``cls`` (a missing module, None, is not), calling nothing but
    its own forward."""
    if type(module) is not cls:
        return False
    d = module.__dict__
    return not d["_forward_hooks"] and not d["_forward_pre_hooks"] and "forward" not in d


class _Unsupported(LookupError):
    """Also what a parameter or submodule that is not there raises (KeyError is
    a LookupError, too): both are caught where the modules are read."""


class _Reader:
    """Addresses of parameters and buffers, each checked to be what the kernels
    read: a plain contiguous fp32 tensor of the expected shape on the device."""

    def __init__(self, device):
        self.index = device.index

    def tensor(self, t, shape, dtype=torch.float32) -> int:
        if (type(t) not in (nn.Parameter, torch.Tensor) or t.dtype is not dtype
                or t.shape != shape or t.get_device() != self.index or not t.is_contiguous()):
            raise _Unsupported
        p = t.data_ptr()
        if p & 15:
            raise _Unsupported
        return p

    def param(self, module, name, shape) -> int:
        """A parameter; one replaced by another kind of attribute is not taken."""
        return self.tensor(module._parameters[name], shape)

    def linear(self, module, d_in, d_out) -> int:
        if not _plain(module, nn.Linear) or module._parameters["bias"] is not None:
            raise _Unsupported
        return self.param(module, "weight", (d_out, d_in))

    def norm(self, module, dim):
        if (not _plain(module, nn.LayerNorm) or module.normalized_shape != (dim,)
                or not 0.0 <= module.eps < float("inf")):
            raise _Unsupported
        return (self.param(module, "weight", (dim,)), self.param(module, "bias", (dim,)),
                float(module.eps))


def _cell_params(m, cell, rd: _Reader, C: int, H: int):
    """The rwkv_decode_cell_params of one CausalCell."""
    if not _plain(cell, m.CausalCell):
        raise _Unsupported
    sub = cell._modules
    tm, cm = sub["time_mixer"], sub["channel_mixer"]
    if not (_plain(tm, m.TimeMixer) and _plain(cm, m.ChannelMixer)):
        raise _Unsupported
    wp, gr = tm._modules["weight_prepare"], tm._modules["gated_readout"]
    if not (_plain(wp, m.WeightPrepare) and _plain(gr, m.GatedReadout)):
        raise _Unsupported
    if (not tm.neighbor_ops == wp.neighbor_ops == gr.neighbor_ops == cm.neighbor_ops == "hip"
            or tm.wkv7_dtype != torch.bfloat16 or tm.num_heads != H or tm.head_size != 64
            or wp.num_heads != H):
        raise _Unsupported
    p = _native.DecodeCellParams()
    p.norm_time_weight, p.norm_time_bias, p.norm_time_eps = rd.norm(
        sub["pre_layer_norm_for_time_mix"], C)
    p.norm_channel_weight, p.norm_channel_bias, p.norm_channel_eps = rd.norm(
        sub["pre_layer_norm_for_channel_mix"], C)
    row = (1, 1, C)
    for i, name in enumerate(("receptance", "weight_decay", "key", "value", "learning_rate")):
        p.mix[i] = rd.param(wp, "param_" + name, row)
    p.mix[5] = rd.param(gr, "param_gate", row)
    wsub, gsub = wp._modules, gr._modules
    p.receptance = rd.linear(wsub["projection_receptance"], C, C)
    p.key = rd.linear(wsub["projection_key"], C, C)
    p.value = rd.linear(wsub["projection_value"], C, C)
    p.output = rd.linear(gsub["projection_output"], C, C)

    def lora(module, activation, bias):
        # the modules call the LoRA's product, or its forward, which does
        if (not _plain(module, m.LoRA) or module.activation != activation
                or "product" in module.__dict__):
            raise _Unsupported
        a = module._parameters["w_a"]
        if a is None or a.dim() != 2:
            raise _Unsupported
        rank = a.shape[1]
        out = [rd.tensor(a, (C, rank)), rd.param(module, "w_b", (rank, C)), rank]
        if bias:
            out.append(rd.param(module, "bias", row))
        elif module.__dict__["bias"] is not None:
            raise _Unsupported
        return out
    p.decay_a, p.decay_b, p.decay_rank, p.decay_bias = lora(
        wsub["param_weight_decay_lora"], "tanh", True)
    p.rate_a, p.rate_b, p.rate_rank, p.rate_bias = lora(
        wsub["param_learning_rate_lora"], "none", True)
    p.gate_a, p.gate_b, p.gate_rank = lora(gsub["param_output_gate_lora"], "sigmoid", False)
    residual = wsub["param_value_residual_lora"] if wp.cell_id != 0 else None
    if residual is not None:
        p.residual_a, p.residual_b, p.residual_rank, p.residual_bias = lora(residual, "none", True)
    elif wp.cell_id != 0:
        raise _Unsupported
    p.key_removal = rd.param(wp, "param_key_removal", row)
    p.key_replacement = rd.param(wp, "param_key_replacement", row)
    p.bonus = rd.param(gr, "param_receptance_key_bonus", (H, 64))
    gn = gsub["group_norm"]
    if type(gn) is not nn.GroupNorm:
        raise _Unsupported
    p.group_norm_weight = rd.param(gn, "weight", (C,))
    p.group_norm_bias = rd.param(gn, "bias", (C,))
    p.group_norm_eps = m.GROUP_NORM_EPS
    p.channel_mix = rd.param(cm, "token_shift_diff_scale", row)
    p.channel_key = rd.linear(cm._modules["key"], C, 4 * C)
    p.channel_value = rd.linear(cm._modules["value"], 4 * C, C)
    for rank in (p.decay_rank, p.rate_rank, p.gate_rank, p.residual_rank or 32):
        if rank % 32 or not 0 < rank <= C:
            raise _Unsupported
    if p.decay_rank + p.rate_rank + p.gate_rank + (p.residual_rank or 0) > 4 * C:
        raise _Unsupported
    return p


def step(model, contexts, batch_ids, infer_state, context_mask,
         unembed_mode: str) -> Optional[tuple]:
    """``(logits or None,)`` of one decode step, its slots of ``infer_state``
    updated, or None where the step is not one these kernels take: one token of
    at most 64 sequences, no mask, bf16 autocast over fp32 parameters on the
    GPU, and a model made of the framework's own modules."""
    from . import model as m
    rows, T = contexts.shape
    if not infer_state.state or infer_state.elapsed_t is None:
        return None
    dev = infer_state.state[0].device
    if (T != 1 or not 0 < rows <= MAX_ROWS or context_mask is not None or dev.type != "cuda"
            or model.neighbor_ops != "hip" or not torch.is_autocast_enabled("cuda")
            or torch.get_autocast_dtype("cuda") is not torch.bfloat16
            or nn.modules.module._global_forward_hooks
            or nn.modules.module._global_forward_pre_hooks):
        return None
    stack = model._modules.get("cells")
    if not _plain(stack, m.MultiCausalCells) or type(stack._modules.get("cells")) is not nn.ModuleList:
        return None
    cells = list(stack._modules["cells"])
    slots, H = infer_state.state[0].shape[:2]
    C = 64 * H
    if (not 0 < C <= MAX_DIM or batch_ids.shape != (rows,) or infer_state.elapsed_t.shape != (slots,)
            or not len(infer_state.state) == len(infer_state.shift_time)
            == len(infer_state.shift_channel) == len(cells)):
        return None
    state_dtype = infer_state.state[0].dtype
    if state_dtype not in (torch.float32, torch.bfloat16):
        return None
    rd = _Reader(dev)
    try:
        calls = [(_cell_params(m, c, rd, C, H), rd.tensor(s, (slots, H, 64, 64), state_dtype),
                  rd.tensor(t, (slots, C)), rd.tensor(ch, (slots, C)))
                 for c, s, t, ch in zip(cells, infer_state.state, infer_state.shift_time,
                                        infer_state.shift_channel)]
        if calls[0][0].residual_a or not all(c[0].residual_a for c in calls[1:]):
            return None   # the first cell is the one without a value residual
        head = None
        if unembed_mode != "skip":
            head = (rd.norm(model._modules["layer_norm_for_unembed"], C),
                    rd.linear(model._modules["unembed"], C, model.vocab_size))
    except LookupError:
        return None
    ids = batch_ids.to(device=dev, dtype=torch.int32).contiguous()
    elapsed = infer_state.elapsed_t.to(device=dev, dtype=torch.int32).contiguous()
    x = model.layer_norm_for_first_cell(model.embed(contexts))
    if x.dtype != torch.float32 or x.shape != (rows, 1, C) or x.device != dev:
        # the embedding and the norm have run, and run once a step
        return (model._infer_cells(x, T, batch_ids, infer_state, context_mask, unembed_mode),)
    # the cells add to it in place, and a hook or the norm itself may hold x
    x = x.clone(memory_format=torch.contiguous_format)
    lib = _native.lib()
    nbytes = lib.rwkv_decode_workspace_bytes(rows, H)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    stream = torch.cuda.current_stream(dev).cuda_stream
    bf16_state = state_dtype is torch.bfloat16
    code = _native.DTYPE_BF16 if bf16_state else _native.DTYPE_F32
    next_time = [torch.empty_like(t) for t in infer_state.shift_time]
    next_channel = [torch.empty_like(t) for t in infer_state.shift_channel]
    for (p, state, time_in, channel_in), time_out, channel_out in zip(calls, next_time, next_channel):
        _native.check(lib.rwkv_decode_cell(
            ctypes.addressof(p), x.data_ptr(), ids.data_ptr(), state, time_in, time_out.data_ptr(),
            channel_in, channel_out.data_ptr(), elapsed.data_ptr(), rows, H, slots, code,
            int(bf16_state), ws.data_ptr(), nbytes, stream))
    infer_state.shift_time[:] = next_time
    infer_state.shift_channel[:] = next_channel
    if head is None:
        return (None,)
    (weight, bias, eps), unembed = head
    logits = torch.empty((rows, 1, model.vocab_size), dtype=torch.bfloat16, device=dev)
    _native.check(lib.rwkv_decode_head(x.data_ptr(), weight, bias, eps, unembed, rows, H,
                                       model.vocab_size, logits.data_ptr(), ws.data_ptr(), nbytes,
                                       stream))
    return (logits,)
