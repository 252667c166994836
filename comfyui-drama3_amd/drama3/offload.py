"""A layer's routed experts in the reference's own formats on an MI355X: every name drama3/model.py, loader.py and
generate.py import from drama3/offload.py (FP8Experts, experts_decode, gather_experts, kernel_bank, resident_decode,
resident_prefill; ExpertStore, HostEmbedding, OffloadedExperts), with the reference's signatures and results, running
the gfx950 kernels of kernels.py.

Storage. An MI355X holds 288 GB, many times a converted model's experts (every layer's banks of the reference model
in int8: about 13 GB), so an ExpertStore's session first tries to make the banks resident: every layer copied to
the device once, expert e of layer l in slot l * E + e, and a decode row or a prompt then runs the resident kernels
(the plan is the identity: no lookup, no host copy, nothing waits on the host). Only when the banks do not fit the
budget (a small `cache_bytes`, or other models in the way) does the session keep the reference's host-offload scheme:
banks in page-locked host memory, a slot cache in HBM kept by kernels.resolve (decayed use counts), the GEMVs reading
missed experts from host memory and filling their slots, and, for int8 banks and a small cache, the CPU running part
of the missed experts beside the GPU.

The cache's state (table, owners, use counts, pending copies) stays on the device throughout: the decode kernels keep
it there, and the host-side lookups (a prompt's pass, formats without kernels) are torch operations on the same
tensors, so nothing moves it between host and device between passes.

Banks are field dicts of flat tensors, as the kernels read them (offload.py:72-90, 264-273):
  int8   {"_qdata": int8 [E * N, K], "scale": float32 [E * N]}                 ConvRot basis (H256 per 256 columns)
  fp8    {"weight": uint8 e4m3 [E * N, K], "scale": float32 [E * N / 128, K / 128]}
  w4/w6  {"_qdata": uint8 [E * N, K * bits / 8], "scale": uint8 e4m3 [E * N, K / 16], "s_channel": float32 [E * N]},
         plus a float32 [16] codebook per bank at 4 bits                       ConvRot basis

ComfyUI (comfy.quant_ops, comfy.model_management) is used when it is importable; without it a quantized weight is any
object with QuantizedTensor's `_qdata`, `_params` and `_layout_cls`, and the memory budget comes from torch.
"""
import collections
import concurrent.futures
import contextlib
import dataclasses
import functools
import logging
import time

import torch
import torch.nn as nn

from . import kernels

# The reference's policy constants (offload.py:30-51), with its names and values.
RESERVE_BASE = 512 * 1024 ** 2           # device memory a generation needs besides the model and the cache
RESERVE_PER_ROW = 0.3 * 1024 ** 2        # ... and per row of prompt and frames
EVICTION_PAUSE = 2.0                     # seconds for comfy's memory reading to catch up after it evicted weights
FP8_BLOCK = 128
CPU_EXPERT_US, CPU_ROW_US = 60, 13       # first guess of the CPU's cost of one int8 expert, and per row through it
PCIE_BYTES_PER_US = 12e3                 # host -> device rate the split assumes for a missed expert
HALF_LIFE = 128                          # passes over which a use count halves
MAX_EXPERTS_PER_ROW = 8
RESERVE_START, RESERVE_MIN, RESERVE_MAX = 32, 8, 256  # slots a decode step may reserve for the CPU's experts
ADMIT = 6.0                              # ... only for experts used this many times (decayed)
AWAIT_US = 5000                          # a decode layer's wait for the host's experts before running them itself

try:  # optional: ComfyUI
    from comfy.quant_ops import QuantizedTensor
    import comfy.model_management as _mm
except ImportError:  # pragma: no cover - comfy is not part of this package
    QuantizedTensor = None
    _mm = None


# ----------------------------------------------------------------------------------------------- format contract
def _quantized(weight):
    if QuantizedTensor is not None:
        return isinstance(weight, QuantizedTensor)
    return all(hasattr(weight, a) for a in ("_qdata", "_params", "_layout_cls"))


def pinned(tensor, pin):
    """A contiguous copy of `tensor`, in page-locked host memory when `pin` (offload.py:54-58)."""
    if not pin:
        return tensor.contiguous()
    host = torch.empty(tensor.shape, dtype=tensor.dtype, pin_memory=True)
    host.copy_(tensor)
    return host


def tensor_fields(weight):
    """{name: tensor} of a quantized weight's parameters that are tensors (offload.py:61-63)."""
    params = weight._params
    found = ((f.name, getattr(params, f.name)) for f in dataclasses.fields(params))
    return {name: value for name, value in found if torch.is_tensor(value)}


def per_row_fields(weight):
    """The bank's tensors with one entry per weight row, which move with the rows (offload.py:66-69): the packed rows
    under "_qdata" and every parameter tensor with as many rows."""
    rows = weight._qdata.shape[0]
    fields = {"_qdata": weight._qdata}
    fields.update((name, t) for name, t in tensor_fields(weight).items() if t.ndim >= 1 and t.shape[0] == rows)
    return fields


def kernel_bank(weight):
    """(kind, fields) of a flat quantized bank [E * out, ...] the kernels read, or None (offload.py:72-90): "int8"
    (ConvRot groups of 256) with {"_qdata", "scale"}; "w4" (with a codebook) or "w6" (without) with {"_qdata",
    "scale", "s_channel"}, scale groups of 16, ConvRot 256. In-features above 2048 are not taken."""
    if not _quantized(weight) or weight._qdata.ndim != 2:
        return None
    params, fields = weight._params, per_row_fields(weight)
    if params.orig_shape[-1] > 2048:
        return None
    names = set(fields)
    if weight._layout_cls == "TensorWiseINT8Layout":
        ok = getattr(params, "convrot", False) and params.convrot_groupsize == 256 and names == {"_qdata", "scale"}
        return ("int8", fields) if ok else None
    if weight._layout_cls != "AsymW4A8Int8Layout":
        return None
    if (params.group_size, params.convrot_groupsize, params.correction, params.transposed) != (16, 256, None, False):
        return None
    if names != {"_qdata", "scale", "s_channel"}:
        return None
    bits = weight._qdata.shape[1] * 8 // params.orig_shape[-1]
    with_codebook = params.codebook is not None
    return (f"w{bits}", fields) if (bits, with_codebook) in ((4, True), (6, False)) else None


def swiglu(y):
    """SiLU(gate) * up of rows [..., 2I], the gate half first (the split comfy.ops._swiglu_eager makes)."""
    half = y.shape[-1] // 2
    return nn.functional.silu(y[..., :half]) * y[..., half:]


@functools.lru_cache(maxsize=4)
def _rotation(size):
    h4 = torch.tensor([[1.0, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]])
    levels = max(1, (size.bit_length() - 1) // 2)
    if 4 ** levels != size:
        raise ValueError(f"ConvRot sizes are powers of 4, not {size}")
    return functools.reduce(torch.kron, [h4] * levels) / size ** 0.5


def hadamard(size):
    """ConvRot's rotation of order `size` (a power of 4): the Kronecker power of h4 = [[1,1,1,-1], [1,1,-1,1],
    [1,-1,1,1], [-1,1,1,1]], normalized to be orthogonal; symmetric, so it is its own inverse (offload.py:170-176)."""
    return _rotation(size).clone()


def dequantize_fp8(weight, scale, dtype):
    """Float8 rows [R, C] with one float32 scale per 128 x 128 block [R / 128, C / 128] -> dtype (offload.py:163-167):
    each block's scale is spread over its rows and columns, then multiplied in float32."""
    rows, cols = weight.shape
    full = scale.repeat_interleave(FP8_BLOCK, 0)[:rows].repeat_interleave(FP8_BLOCK, 1)[:, :cols]
    return (weight.float() * full).to(dtype)


def gather_experts(weight, ids, num_experts):
    """Experts `ids` [k] of a flat [E * out, in] bank as one [k * out, in] weight, on the bank's device
    (offload.py:152-160). A quantized bank keeps its type with its per-row fields gathered; a field dict is gathered
    field by field (block-scale grids by their own rows per expert)."""
    def pick(t):
        return t.unflatten(0, (num_experts, t.shape[0] // num_experts)).index_select(0, ids).flatten(0, 1)
    if isinstance(weight, dict):
        return {name: pick(t) for name, t in weight.items()}
    if not _quantized(weight):
        return pick(weight)
    picked = {name: pick(t) for name, t in per_row_fields(weight).items()}
    qdata = picked.pop("_qdata")
    params = dataclasses.replace(weight._params, orig_shape=(qdata.shape[0], weight._params.orig_shape[-1]), **picked)
    return type(weight)(qdata, weight._layout_cls, params)


def experts_decode(x, gate_up, down, weights):
    """One row x [1, H] through k experts (gate_up [k * 2I, H] and down [k * H, I], dense) summed by `weights` [k]
    (offload.py:192-199): gate_up as one product for all k, then each expert's down projection of its own hidden row
    as one batched product, [1, H] in x's dtype."""
    k = weights.shape[0]
    hidden = swiglu(nn.functional.linear(x, gate_up).view(k, -1))               # [k, I]
    per_expert = down.view(k, -1, hidden.shape[-1])                             # [k, H, I]
    out = torch.bmm(per_expert, hidden.unsqueeze(-1).contiguous()).squeeze(-1)  # [k, H]
    return (weights.to(out.dtype).unsqueeze(-1) * out).sum(0, keepdim=True)


def experts_on_cpu(banks, experts, counts, x, rotation):
    """Rows x [rows, H] (bf16, already in the ConvRot basis; counts[i] rows for experts[i], in turn) through their
    int8 ConvRot experts on the CPU (offload.py:179-189): [rows, H] float32. The matmuls run expert by expert on each
    expert's run of rows; SwiGLU and the rotation of the hidden rows run on all the rows at once."""
    gate_up, down = banks
    ends = torch.tensor(counts).cumsum(0).tolist()
    runs = [(e, end - n, end) for e, n, end in zip(experts, counts, ends)]
    hidden = swiglu(torch.cat([gate_up.cpu_linear(x[a:b], e) for e, a, b in runs]).float())
    group = rotation.shape[0]
    hidden = torch.matmul(hidden.unflatten(-1, (-1, group)), rotation).flatten(-2).to(torch.bfloat16)
    return torch.cat([down.cpu_linear(hidden[a:b], e) for e, a, b in runs]).float()


def timed(function, *args):
    """(function(*args), the seconds it took)."""
    t0 = time.perf_counter()
    result = function(*args)
    return result, time.perf_counter() - t0


# ------------------------------------------------------------------------------------------------ kernel dispatch
def quantized_gemv(kind, x, ids, plan, took_over, late, slot_fields, host_fields, rows, codebook):
    """[k, rows] of a decode row's experts in an int8, W4A8 or W6A8 bank against x (float32, rotated)
    (offload.py:93-98)."""
    if kind == "int8":
        return kernels.gemv_int8(x, ids, plan, took_over, late, slot_fields, host_fields, rows)
    return kernels.gemv_codes(x, ids, plan, slot_fields, host_fields, codebook, int(kind[1]), rows)


def quantized_grouped(kind, x, groups, slot_fields, host_fields, rows, codebook):
    """quantized_gemv for a prompt's rows grouped by expert (offload.py:101-105)."""
    if kind == "int8":
        return kernels.grouped_int8(x, groups, slot_fields, host_fields, rows)
    return kernels.grouped_codes(x, groups, slot_fields, host_fields, codebook, int(kind[1]), rows)


_consts = {}


def _constants(device):
    """Per device: int32 [0] (took_over: no expert left to the CPU) and [1] (the rotation always runs)."""
    key = (device.type, device.index)
    if key not in _consts:
        if torch.cuda.is_available() and torch.cuda.is_current_stream_capturing():
            raise RuntimeError("drama3.offload: run one call before capturing a graph (constants must exist)")
        _consts[key] = torch.arange(2, dtype=torch.int32, device=device).split(1)
    return _consts[key]


def _rows(kind, fields, num_experts):
    return fields["weight" if kind == "fp8" else "_qdata"].shape[0] // num_experts


# Launches of the resident decode where the layer's shape allows: 2 (kernels.resident_decode / resident_decode_routed)
# or 1 (kernels.resident_decode_fused, the hidden rows handed between workgroups of one launch). Both give the same
# output, ids and weights, bit for bit. Two is the default: measured on MI355X (us per routed layer, hidden 2048,
# FFN 768, top-8, layers chained in HIP graphs; two launches / one): int8 17.2 / 17.4, fp8 17.0 / 17.6, W4A8 18.1 /
# 18.4, W6A8 21.3 / 21.1. The one launch saves the second launch's gap but its down workgroups wait for the hidden
# rows through device-coherent memory, which costs about as much.
RESIDENT_LAUNCHES = 2


def resident_decode(x, ids, weights, banks, rows, kind, codebooks):
    """One row x [1, H] through experts `ids` [k] of banks held whole on the GPU (expert e in slot e, `rows` per
    expert) (offload.py:108-123): bf16 [1, H]. One launch (kernels.resident_decode_fused) or two (gate_up with x
    rotated in its prologue; down with SwiGLU, the rotation and the weighted sum) where the shapes allow, else the
    reference's five. Nothing waits on the host."""
    gate_up_rows, down_rows = rows
    H, I = down_rows, gate_up_rows // 2
    if H in (1024, 2048) and I in (512, 768, 1024) and ids.shape[0] <= 8 and x.dtype == torch.bfloat16:
        if RESIDENT_LAUNCHES == 1 and kernels.resident_fused_fits(kind, H, I, ids.shape[0]):
            return kernels.resident_decode_fused(x, banks, kind, codebooks, H, I, ids=ids, weights=weights.float())
        return kernels.resident_decode(x, ids, weights.float(), banks, kind, codebooks, H, I)
    return resident_decode_unfused(x, ids, weights, banks, rows, kind, codebooks)


def routed_decode(x, logits, k, banks, rows, kind, codebooks):
    """kernels.route(logits, k), then resident_decode (model.py:116-118, then offload.py:108-123), for one row:
    (out [1, H] bf16, ids [1, k], weights [1, k]). The routing runs inside the (gate_up) launch where the shapes
    allow."""
    gate_up_rows, down_rows = rows
    H, I = down_rows, gate_up_rows // 2
    experts = _rows(kind, banks[0], 1) // gate_up_rows
    if logits.numel() != experts:
        raise ValueError(f"{logits.numel()} logits for banks of {experts} experts: a routed id past the banks would be "
                         f"read out of bounds")
    if (H in (1024, 2048) and I in (512, 768, 1024) and k <= 8 and k <= logits.numel() <= 256
            and x.dtype == torch.bfloat16 and logits.dtype == torch.bfloat16):
        if RESIDENT_LAUNCHES == 1 and kernels.resident_fused_fits(kind, H, I, k):
            return kernels.resident_decode_fused(x, banks, kind, codebooks, H, I, logits=logits, k=k)
        return kernels.resident_decode_routed(x, logits, k, banks, kind, codebooks, H, I)
    ids, weights = kernels.route(logits.reshape(1, -1), k)
    return resident_decode(x, ids[0], weights[0], banks, rows, kind, codebooks), ids, weights


def resident_decode_unfused(x, ids, weights, banks, rows, kind, codebooks):
    """resident_decode as the reference launches it: rotate, gemv, rotate (SwiGLU), gemv, weighted_sum (fp8: gemv,
    SiLU(gate) * up, gemv, weighted_sum)."""
    plan = torch.stack((ids.to(torch.int32), torch.zeros_like(ids, dtype=torch.int32)), dim=-1)
    return _slot_decode(x, ids, weights.float(), plan, banks, banks, rows, kind, codebooks, _constants(x.device))


def _slot_decode(x, ids, weights, plan, slot_banks, host_banks, rows, kind, codebooks, flags, cpu_side=None):
    """The GEMV chain of a decode row under a resolved `plan`: [1, H]. flags = (took_over, always) on the device.
    With `cpu_side` = (CpuSide, layer, step) the experts the plan leaves to the CPU come back through its mailbox, or
    run here if the host is late."""
    took_over, always = flags
    if kind == "fp8":
        hidden = swiglu(kernels.gemv_fp8(x.float(), ids, plan, slot_banks[0], host_banks[0], rows[0]))
        return kernels.weighted_sum(kernels.gemv_fp8(hidden, ids, plan, slot_banks[1], host_banks[1], rows[1]), weights)
    rotated = kernels.rotate(x, always)

    def chain(late):
        """Each expert's output [k, H], unweighted; with `late`, only the CPU's experts, once the GPU took them."""
        hidden = quantized_gemv(kind, rotated, ids, plan, took_over, late, slot_banks[0], host_banks[0], rows[0],
                                codebooks[0])
        hidden = kernels.rotate(hidden, took_over if late else always, swiglu=True)
        return quantized_gemv(kind, hidden, ids, plan, took_over, late, slot_banks[1], host_banks[1], rows[1],
                              codebooks[1])

    if cpu_side is None:
        return kernels.weighted_sum(chain(False), weights)
    side, layer, step = cpu_side
    side.post(layer, plan, ids, weights, rotated.to(torch.bfloat16), step)
    total = weights @ chain(False) + side.wait(layer, plan, step, took_over)
    return (total + weights @ chain(True)).to(x.dtype)


def grouped_experts(sorted_x, groups, slot_banks, host_banks, rows, kind, codebooks, always):
    """[rows, H] float32: sorted_x's rows through their experts, one grouped kernel per bank (offload.py:126-136);
    `always` is an int32 1 on the GPU."""
    return _grouped_pairs(sorted_x, None, groups, slot_banks, host_banks, rows, kind, codebooks, always)


def _grouped_pairs(x, gather, groups, slot_banks, host_banks, rows, kind, codebooks, always, fills_first=False,
                   work=None, planes=None):
    """grouped_experts over the pairs' rows: x's rows sorted by expert (gather None), or with gather = (order, top_k)
    row order[p] // top_k of x for pair p. On the matrix cores (bank widths multiples of 64, 128 for fp8) x's rows are
    rotated and split into planes once each (int8 planes for the int8 cores: int8 and the codes; bf16 rows are fp8's
    one plane as they are), the products read pair p's row through `order`, and the second bank's planes come from
    the hidden rows by one kernel (SwiGLU, rotation, split); `fills_first` as for kernels.grouped_fp8_planes, `work` the
    groups' plan and `planes` x's int8 planes and scales when the grouping's launch made them."""
    step = 128 if kind == "fp8" else 64
    if x.is_cuda and rows[0] % step == 0 and rows[1] % step == 0:
        order, top_k = gather if gather is not None else (None, 1)
        P = order.shape[0] if order is not None else x.shape[0]
        if work is None:
            work = kernels.grouped_plan(groups, P)
        if kind != "fp8":
            planes, scales = planes if planes is not None else kernels.prep_planes_i8(x, True)
            hidden = kernels.grouped_i8(kind, planes, scales, P, x.shape[1], groups, work, slot_banks[0],
                                        host_banks[0], codebooks[0], rows[0], fills_first, order, top_k)
            planes, scales = kernels.prep_planes_i8(hidden, True, swiglu=True)
            return kernels.grouped_i8(kind, planes, scales, P, rows[0] // 2, groups, work, slot_banks[1],
                                      host_banks[1], codebooks[1], rows[1], fills_first)
        if x.dtype == torch.bfloat16:   # bf16 rows are their own one plane
            planes = x.contiguous().view(1, -1)
        else:
            planes = kernels.prep_planes(x, False)
        hidden = kernels.grouped_fp8_planes(planes, P, x.shape[1], groups, work, slot_banks[0], host_banks[0],
                                            rows[0], fills_first, order, top_k)
        planes = kernels.prep_planes(hidden, False, swiglu=True)
        return kernels.grouped_fp8_planes(planes, P, rows[0] // 2, groups, work, slot_banks[1], host_banks[1],
                                          rows[1], fills_first)
    sorted_x = x if gather is None else x[gather[0] // gather[1]]
    if kind == "fp8":
        hidden = swiglu(kernels.grouped_fp8(sorted_x.float(), groups, slot_banks[0], host_banks[0], rows[0]))
        return kernels.grouped_fp8(hidden, groups, slot_banks[1], host_banks[1], rows[1])
    hidden = quantized_grouped(kind, kernels.rotate(sorted_x.float(), always), groups, slot_banks[0], host_banks[0],
                               rows[0], codebooks[0])
    return quantized_grouped(kind, kernels.rotate(hidden, always, swiglu=True), groups, slot_banks[1], host_banks[1],
                             rows[1], codebooks[1])


def expert_groups(topk_idx, num_experts):
    """A prompt's (token, k) pairs grouped by expert, without a host sync: (order [T * k] int64, inverse [T * k]
    int32 = each pair's place in order, groups [num_experts, 5] int32 = (expert, expert, 0, first, rows)). Experts
    without rows keep a group of 0 rows, which the grouped kernels skip without reading anything. In place of
    offload.py:140-143's sort and bincount().tolist(), so a prompt's pass can be captured in a graph. On the GPU one
    counting-sort kernel (the order within a group is not fixed; no result depends on it); on the CPU a stable sort."""
    if topk_idx.is_cuda:
        return kernels.expert_groups(topk_idx, num_experts)
    return _groups_on_host(topk_idx, num_experts)


def _groups_on_host(topk_idx, num_experts):
    flat = topk_idx.reshape(-1)
    order = torch.sort(flat, stable=True).indices
    inverse = torch.empty_like(order)
    inverse[order] = torch.arange(order.shape[0], device=order.device)
    counts = torch.zeros(num_experts, dtype=torch.int64, device=flat.device).scatter_add_(0, flat, torch.ones_like(flat))
    first = torch.cumsum(counts, 0) - counts
    experts = torch.arange(num_experts, dtype=torch.int64, device=flat.device)
    groups = torch.stack((experts, experts, torch.zeros_like(experts), first, counts), dim=1).to(torch.int32)
    return order, inverse.to(torch.int32), groups


def _combine(sorted_out, inverse, topk_weight, dtype):
    """The pairs' rows of sorted_out ([T * k, H], pair p at inverse[p]) weighted and summed over k in k's order:
    [T, H] of `dtype`, summed in float32 (offload.py:144-149)."""
    if sorted_out.is_cuda:
        return kernels.combine_rows(sorted_out, inverse, topk_weight, dtype)
    num_tokens, top_k = topk_weight.shape
    pairs = sorted_out.float().index_select(0, inverse.long()) * topk_weight.reshape(-1, 1).float()
    return pairs.view(num_tokens, top_k, -1).sum(dim=1).to(dtype)


def _wide_pairs(x, topk_idx, banks, rows, kind, codebooks, num_experts):
    """(the pairs' rows through their experts [T * k, H] float32, inverse): resident_prefill's products in wide passes,
    SiLU(gate) * up formed with the first bank's."""
    top_k, width, inner = topk_idx.shape[1], x.shape[1], rows[0] // 2
    if kind == "fp8":
        order, inverse, passes = kernels.prompt_groups(topk_idx, num_experts)
        if x.dtype == torch.bfloat16:   # bf16 rows are their own one plane, which the copies to LDS want 16-byte aligned
            x = x.contiguous()
            planes = (x if x.data_ptr() % 16 == 0 else x.clone()).view(1, -1)
        else:
            planes = kernels.prep_planes(x, False)
        P = order.shape[0]
        hidden = kernels.prompt_fp8(planes, P, width, passes, num_experts, banks[0], rows[0], order, top_k, swiglu=True)
        planes = kernels.prep_planes(hidden, False)
        return kernels.prompt_fp8(planes, P, inner, passes, num_experts, banks[1], rows[1]), inverse
    order, inverse, passes, planes, scales = kernels.prompt_prep_i8(topk_idx, num_experts, x, True)
    P = order.shape[0]
    hidden = kernels.prompt_i8(kind, planes, scales, P, width, passes, num_experts, banks[0], codebooks[0], rows[0],
                               order, top_k, swiglu=True)
    planes, scales = kernels.prep_planes_i8(hidden, True)
    return kernels.prompt_i8(kind, planes, scales, P, inner, passes, num_experts, banks[1], codebooks[1],
                             rows[1]), inverse


def resident_prefill(x, topk_idx, topk_weight, banks, rows, kind, codebooks, num_experts):
    """Many rows x [T, H] through banks held whole on the GPU (offload.py:138-149): one grouped kernel per bank over
    the pairs grouped by expert on the device, each product weighted and summed over k; x's dtype."""
    top_k = topk_idx.shape[1]
    planes = None
    if topk_idx.is_cuda and kernels.prompt_wide_fits(kind, banks, rows, topk_idx.numel(), num_experts, x.shape[1]):
        sorted_out, inverse = _wide_pairs(x, topk_idx, banks, rows, kind, codebooks, num_experts)
        return _combine(sorted_out, inverse, topk_weight, x.dtype)
    if topk_idx.is_cuda and kind != "fp8" and rows[0] % 64 == 0 and rows[1] % 64 == 0:
        # one launch: the grouping, its plan of the grouped products' passes, and x's rows as int8 planes
        order, inverse, groups, work, *planes = kernels.expert_groups_prep_i8(topk_idx, num_experts, x, True)
    elif topk_idx.is_cuda:   # the grouping's launch also plans the grouped products' passes
        order, inverse, groups, work = kernels.expert_groups(topk_idx, num_experts, plan=True)
    else:
        (order, inverse, groups), work = _groups_on_host(topk_idx, num_experts), None
    _, always = _constants(x.device)
    sorted_out = _grouped_pairs(x, (order, top_k), groups, banks, banks, rows, kind, codebooks, always, work=work,
                                planes=planes)
    return _combine(sorted_out, inverse, topk_weight, x.dtype)


# ----------------------------------------------------------------------------------------------------- host banks
class HostBank:
    """One bank of a layer's experts: field tensors whose first dimension holds expert e's rows at [e * rows,
    (e + 1) * rows), page-locked in host memory when `pin` so the kernels can read them in place (offload.py:202-219).
    `kernel` names the kernel family that reads the bank, or None."""

    kernel = None

    def __init__(self, num_experts, fields, pin):
        self.num_experts = num_experts
        self.fields = {name: pinned(t, pin) for name, t in fields.items()}
        self._per_expert = {name: t.shape[0] // num_experts for name, t in self.fields.items()}

    def rows(self, name):
        """Rows of field `name` per expert."""
        return self._per_expert[name]

    def take(self, fields, first, last):
        """Experts [first, last) of `fields` (this bank's, or a slot pool's: host or device), as views."""
        return {name: t.narrow(0, first * self.rows(name), (last - first) * self.rows(name)) for name, t in fields.items()}

    def to_device(self, first, last, device):
        return {name: t.to(device, non_blocking=True) for name, t in self.take(self.fields, first, last).items()}

    def pick(self, experts):
        """This bank's fields of `experts` (a sequence of ints), one expert after another, in host memory."""
        index = torch.tensor(list(experts), dtype=torch.long)
        return {name: t.view(self.num_experts, self.rows(name), *t.shape[1:]).index_select(0, index).flatten(0, 1)
                for name, t in self.fields.items()}

    def codebook(self, device):
        """The bank's 4-bit codebook on `device` (W4A8 banks), else None."""
        return None

    def weight(self, fields, device):
        """The experts of `fields` as one dense bf16 weight on `device`, in the model's own basis: what
        nn.functional.linear takes on the paths without kernels."""
        raise NotImplementedError


class QuantHostBank(HostBank):
    """A flat quantized bank (int8 ConvRot, W4A8, W6A8) taken from a `comfy.ops.MoEExperts`-like module: `module.weight`
    a QuantizedTensor (or an object with its `_qdata`, `_params`, `_layout_cls`), `module.num_experts`
    (offload.py:223-261). The CPU's int8 matmul reads it in place."""

    def __init__(self, module, pin):
        weight = module.weight
        if not _quantized(weight) or weight._qdata.ndim != 2:
            raise ValueError("Drama 3 keeps only flat quantized or FP8 expert banks in host memory")
        fields = per_row_fields(weight)
        found = kernel_bank(weight)
        self._setup(module.num_experts, None if found is None else found[0], fields, pin,
                    {name: t for name, t in tensor_fields(weight).items() if name not in fields},
                    weight._params.orig_shape[-1])
        self.layout, self.params = weight._layout_cls, weight._params

    @classmethod
    def from_fields(cls, num_experts, kind, fields, pin, codebook=None):
        """A bank given as its kernel kind and field dict (a converted file's tensors, drama3/loader.py)."""
        self = cls.__new__(cls)
        in_features = fields["_qdata"].shape[1] * 8 // (8 if kind == "int8" else int(kind[1]))
        self._setup(num_experts, kind, fields, pin, {} if codebook is None else {"codebook": codebook}, in_features)
        self.layout = self.params = None
        return self

    def _setup(self, num_experts, kind, fields, pin, shared, in_features):
        HostBank.__init__(self, num_experts, fields, pin)
        self.kernel, self.shared, self.in_features = kind, shared, in_features
        self._shared_on = {}
        if kind == "int8":
            self.scale_bf16 = self.fields["scale"].reshape(-1).to(torch.bfloat16)  # the CPU matmul's scale dtype

    def _shared(self, device):
        if device not in self._shared_on:
            self._shared_on[device] = {name: t.to(device) for name, t in self.shared.items()}
        return self._shared_on[device]

    def codebook(self, device):
        return self._shared(torch.device(device)).get("codebook")

    def cpu_linear(self, x, expert):
        """Rows x [M, K] (bf16, rotated) through int8 expert `expert` on the CPU, from host memory: [M, N]."""
        rows = self.rows("_qdata")
        return torch._weight_int8pack_mm(x, self.fields["_qdata"].narrow(0, expert * rows, rows),
                                         self.scale_bf16.narrow(0, expert * rows, rows))

    def weight(self, fields, device):
        """Dequantized (int8 * scale, or the decoded code grid * s_channel) and rotated out of the ConvRot basis."""
        fields = {name: t.to(device) for name, t in fields.items()}
        if self.kernel == "int8":
            w = fields["_qdata"].float() * fields["scale"].float().reshape(-1, 1)
        elif self.kernel in ("w4", "w6"):
            grid = kernels.decode_codes(fields["_qdata"], fields["scale"], self.codebook(device), int(self.kernel[1]))
            w = grid.float() * fields["s_channel"].float().reshape(-1, 1)
        else:
            raise ValueError(f"no dense form for a {self.layout} bank outside the kernels' formats")
        rot = hadamard(256).to(device)
        return torch.matmul(w.unflatten(-1, (-1, 256)), rot).flatten(-2).to(torch.bfloat16)


class FP8HostBank(HostBank):
    """Experts as Fish ships them: float8 rows [E, N, K] and 128 x 128 block scales [E, N / 128, K / 128]
    (offload.py:264-273)."""

    kernel = "fp8"

    def __init__(self, weight, scale, pin):
        fields = {"weight": weight.view(torch.uint8).flatten(0, 1), "scale": scale.flatten(0, 1)}
        super().__init__(weight.shape[0], fields, pin)

    @classmethod
    def from_fields(cls, num_experts, fields, pin):
        """A bank given as its field dict ({"weight" uint8, "scale"}, flat), as drama3/loader.py reads it."""
        self = cls.__new__(cls)
        HostBank.__init__(self, num_experts, fields, pin)
        return self

    def weight(self, fields, device):
        w = fields["weight"].to(device).view(torch.float8_e4m3fn)
        return dequantize_fp8(w, fields["scale"].to(device), torch.bfloat16)


# ------------------------------------------------------------------------------------------------------ slot cache
def _next_reserve(reserve, lagging):
    """The reservations the next decode step may make (the reference's rule, offload.py:646): a quarter fewer
    (rounded down, at least RESERVE_MIN) while the copies lag, a quarter and one more (at most RESERVE_MAX) while they
    keep up."""
    if lagging:
        return max(RESERVE_MIN, reserve * 3 // 4)
    return min(RESERVE_MAX, reserve * 5 // 4 + 1)


def _put(target, index, values, mask):
    """target[index[i]] = values[i] where mask[i], in place on target's device, with no host sync: the entries left
    out write to a spare element past the end, which is dropped. The masked-in positions must be distinct."""
    n = target.shape[0]
    pos = torch.where(mask, index.long(), n)
    written = torch.zeros(n + 1, dtype=torch.bool, device=target.device).index_fill_(0, pos, True)
    staged = target.new_empty(n + 1).index_copy_(0, pos, values.to(target.dtype).expand(pos.shape[0]))
    target.copy_(torch.where(written[:n], staged[:n], target))


class _CopyQueue:
    """Host -> slot copies of reserved experts on a side stream, in batches that run behind the work already launched;
    a batch's (key, slot) pairs are mapped once its event has passed."""

    def __init__(self, device):
        self.device = device
        self.stream = None
        self.batches = collections.deque()   # (event, [(key, slot)])

    def busy(self):
        return bool(self.batches)

    def submit(self, writes, pairs):
        """Run `writes` (a callable issuing the copies) on the side stream after the current stream's work."""
        if self.stream is None:
            self.stream = torch.cuda.Stream(self.device)
        self.stream.wait_stream(torch.cuda.current_stream(self.device))
        with torch.cuda.stream(self.stream):
            writes()
            event = torch.cuda.Event()
            event.record(self.stream)
        self.batches.append((event, pairs))

    def landed(self):
        """The pairs of the batches whose copies have completed, oldest first."""
        done = []
        while self.batches and self.batches[0][0].query():
            done.extend(self.batches.popleft()[1])
        return done

    def drain(self):
        """Every batch's pairs, once all copies have completed."""
        if self.stream is not None:
            self.stream.synchronize()
        done = [pair for _, pairs in self.batches for pair in pairs]
        self.batches.clear()
        return done


class SlotPool:
    """`count` expert slots in HBM over host banks, filled on demand, the least used expert out first
    (offload.py:560-753's policy).

    The state lives on the device for the pool's whole life: table [L * E] maps a key (layer * E + expert) to its slot,
    -1 (not cached) or -2 - slot (pending: the host is copying it in); owner [count] maps a slot to its key (-1: free);
    score / at [L * E] hold each key's use count as of step `at` (pass * layers + layer; -1: never), halving every
    HALF_LIFE passes; clock counts passes; reads counts decode rows' (hits, fills, CPU experts). `fields` holds the
    slots in the banks' row layout. kernels.resolve keeps it during decode; the host-side passes work on the same
    tensors.

    Every host-side pass is a batch over the experts it touches: their counts decay and grow together, and the slots a
    batch of misses takes are the smallest (decayed count, slot) keys in one stable sort over the pool (free slots
    first, value -1; never a slot holding an expert the layer used in this pass), handed out in the batch's order: the
    order in which one claim after another would take them, and the order kernels.resolve's selection rounds take.
    Nothing is read back to the host unless the caller needs it there."""

    def __init__(self, banks, budget, device):
        self.banks = banks
        self.device = torch.device(device)
        self.layers, self.num_experts = len(banks), banks[0][0].num_experts
        self.rows = [{name: bank.rows(name) for name in bank.fields} for bank in banks[0]]
        self.expert_bytes = sum(t[:1].nbytes * bank.rows(name) for bank in banks[0] for name, t in bank.fields.items())
        keys = self.layers * self.num_experts
        self.count = int(max(8, min(keys, budget // self.expert_bytes)))
        self.fields = [{name: torch.empty((self.count * bank.rows(name), *t.shape[1:]), dtype=t.dtype,
                                          device=self.device) for name, t in bank.fields.items()}
                       for bank in banks[0]]
        on = dict(device=self.device)
        self.table = torch.full((keys,), -1, dtype=torch.int32, **on)
        self.owner = torch.full((self.count,), -1, dtype=torch.int32, **on)
        self.score = torch.zeros((keys,), dtype=torch.float32, **on)
        self.at = torch.full((keys,), -1, dtype=torch.int32, **on)
        self.pending = torch.zeros((self.count,), dtype=torch.int32, **on)
        self.clock = torch.zeros((1,), dtype=torch.int32, **on)
        self.reads = torch.zeros((3,), dtype=torch.int32, **on)
        # log2 of a use count's decay per step, in float32 as kernels.resolve computes it
        half_life = torch.tensor(float(HALF_LIFE), dtype=torch.float32) * torch.tensor(float(self.layers))
        self.log2_decay = (torch.tensor(-1.0, dtype=torch.float32) / half_life).to(self.device)
        self.reserve = RESERVE_START
        self.budget = torch.tensor(self._reservations(), dtype=torch.int32, **on)
        # a layer's step, whether the GPU took the CPU's experts over, a set flag; the GPU's share of missed experts
        self.step, self.took_over, self.always = torch.tensor([[0], [0], [1]], dtype=torch.int32, **on)
        self.share = torch.zeros((1,), dtype=torch.float32, **on)
        self.reserved = []   # (layer, expert, slot) the CPU's experts reserved in this decode phase, not yet copying
        self._copies = _CopyQueue(self.device)
        self._decoding = False

    # -- the decode kernels' view
    def device_state(self):
        """(table, owner, score, at, pending, clock, budget, reads, step, share) for kernels.resolve. From here until
        the next host-side pass the pool is in a decode phase, whose reservations `promote` copies in."""
        self._decoding = True
        return (self.table, self.owner, self.score, self.at, self.pending, self.clock, self.budget, self.reads,
                self.step, self.share)

    def host(self):
        """Ready for a host-side pass, which ends a decode phase: its copies land and are mapped first (the state itself
        never leaves the device)."""
        if self._decoding:
            self.settle()
            self._decoding = False

    def _reservations(self):
        """[slots a decode step may reserve, at most per layer]: the step's budget spread over the layers, twice over
        so that a busy layer can take more than its share."""
        return [self.reserve, max(1, (2 * self.reserve + self.layers - 1) // self.layers)]

    def _map(self, pairs):
        """Copies landed: their keys now map to their slots, which are no longer pending."""
        if pairs:
            keys, slots = torch.tensor(pairs, dtype=torch.long).to(self.device).unbind(1)
            self.table.index_copy_(0, keys, slots.to(torch.int32))
            self.pending.index_fill_(0, slots, 0)

    def promote(self):
        """Between decode steps: map what the copy queue has landed, queue copies of the experts reserved since the last
        call, and size the next step's reservations by whether the queue kept up. Outside a decode phase nothing was
        reserved and the budget stays."""
        if not self._decoding:
            return
        self._map(self._copies.landed())
        lagging = self._copies.busy()
        if self.reserved:
            batch, self.reserved = self.reserved, []

            def writes():
                for layer, expert, slot in batch:
                    self.write([slot], [bank.take(bank.fields, expert, expert + 1) for bank in self.banks[layer]])

            self._copies.submit(writes, [(layer * self.num_experts + e, s) for layer, e, s in batch])
        self.reserve = _next_reserve(self.reserve, lagging)
        self.budget.copy_(torch.tensor(self._reservations(), dtype=torch.int32), non_blocking=True)

    def settle(self):
        """Every reserved expert copied into its slot and mapped."""
        self.promote()
        self._map(self._copies.drain())

    # -- slots and their contents
    def write(self, slots, sources):
        """Copy experts into `slots` (ints): sources[b] holds bank b's fields of those experts, one after another, in
        host memory. One slot is copied straight from its source (without waiting, from page-locked memory); several
        go over together and are scattered on the device."""
        slots = list(slots)
        for fields, rows, source in zip(self.fields, self.rows, sources):
            for name, target in fields.items():
                rows_in = source[name]
                if len(slots) == 1:
                    target.narrow(0, slots[0] * rows[name], rows[name]).copy_(rows_in, non_blocking=True)
                    continue
                per_slot = target.view(self.count, rows[name], *target.shape[1:])
                index = torch.tensor(slots, dtype=torch.long).to(self.device)
                per_slot.index_copy_(0, index, rows_in.to(self.device).view(len(slots), rows[name], *target.shape[1:]))

    def slot_fields(self, index, slot):
        """Bank `index`'s fields of the expert in `slot`, laid out like a host bank's expert."""
        rows = self.rows[index]
        return {name: t.narrow(0, slot * rows[name], rows[name]) for name, t in self.fields[index].items()}

    def gather(self, index, slots):
        """Bank `index`'s fields of the experts in `slots`, one after another: the slots' row ranges picked from each
        field at once."""
        out = {}
        for name, t in self.fields[index].items():
            n = self.rows[index][name]
            picked = (slots.reshape(-1, 1) * n + torch.arange(n, device=t.device)).reshape(-1)
            out[name] = t.index_select(0, picked)
        return out

    # -- the host-side passes, batched on the device
    def _step(self, layer, advance):
        """`layer`'s step in the current pass, a device int32 [1]; with `advance`, layer 0 starts a new pass."""
        if advance and layer == 0:
            self.clock += 1
        return self.clock * self.layers + layer

    def _decayed(self, keys, now):
        """Use counts of `keys` as of step `now` (0 for keys never used)."""
        at = self.at[keys]
        counts = self.score[keys] * torch.exp2(self.log2_decay * (now - at).float())
        return torch.where(at < 0, torch.zeros_like(counts), counts)

    def _touch(self, layer, experts, mask=None):
        """A pass's use of `experts` (int64, distinct) of `layer`, those with `mask` if given: each counts a use now.
        Returns (keys, their slots, -1 where not cached; now)."""
        now = self._step(layer, True)
        keys = experts + layer * self.num_experts
        counts = self._decayed(keys, now) + 1.0
        if mask is None:
            self.score.index_copy_(0, keys, counts)
            self.at.index_copy_(0, keys, now.expand(keys.shape[0]))
        else:
            _put(self.score, keys, counts, mask)
            _put(self.at, keys, now.expand(keys.shape[0]), mask)
        return keys, self.table[keys].long(), now

    def _blocked(self, now):
        """Per slot: whether a claim at step `now` must pass it by (it holds an expert used at `now`, i.e. by this layer
        in this pass, or one being copied in)."""
        held = self.owner.long()
        return (held >= 0) & (self.at[held.clamp(min=0)] == now) | (self.pending != 0)

    def _claim_order(self, now):
        """The slots in the order claims at step `now` take them, and how many may be taken: free slots first (value
        -1), then by decayed use count, the lower slot first among equals; blocked slots last."""
        held = self.owner.long()
        value = torch.where(held >= 0, self._decayed(held.clamp(min=0), now), torch.full_like(self.score[:1], -1.0))
        blocked = self._blocked(now)
        order = torch.sort(value.masked_fill(blocked, float("inf")), stable=True).indices
        return order, (~blocked).sum()

    def _bind(self, slots, keys, mask):
        """Slots[i] now holds keys[i] where mask[i]; the experts they held leave the table."""
        before = self.owner[slots].long()
        _put(self.table, before.clamp(min=0), torch.full((), -1, dtype=torch.int32, device=self.device),
             mask & (before >= 0))
        _put(self.owner, slots, keys, mask)
        _put(self.table, keys, slots, mask)

    def use(self, layer, experts):
        """{expert: slot} of the cached ones among `experts`; each of them counts a use in this pass."""
        self.host()
        _, slots, _ = self._touch(layer, torch.tensor(list(experts), dtype=torch.long).to(self.device))
        return {e: s for e, s in zip(experts, slots.tolist()) if s >= 0}

    def free_slots(self):
        return torch.where(self.owner < 0)[0].tolist()

    def assign(self, slot, layer, expert):
        """Give `slot` to an expert of `layer`; its previous expert leaves the table. The caller fills the slot."""
        one = torch.ones(1, dtype=torch.bool, device=self.device)
        self._bind(torch.tensor([slot], device=self.device), torch.tensor([layer * self.num_experts + expert],
                                                                           device=self.device), one)
        return slot

    def claim(self, layer, expert):
        """The slot of the least used cached expert (a free one first) that `layer` has not used in this pass."""
        order, free = self._claim_order(self._step(layer, False))
        if int(free) == 0:
            raise RuntimeError(f"drama3: every slot holds an expert layer {layer} uses in this pass")
        return self.assign(int(order[0]), layer, expert)

    def room(self, layer):
        """How many slots `layer` may still claim in this pass: those not holding an expert it used."""
        return int((~self._blocked(self._step(layer, False))).sum())

    def insert(self, layer, expert, sources):
        """A slot for an expert `layer` uses in this pass, filled from `sources` (host memory)."""
        slot = self.claim(layer, expert)
        self.write([slot], sources)
        return slot

    def slots(self, layer, experts, banks):
        """The host-lookup decode: slots of the row's `experts` [k], the missed ones claimed in routing order and copied
        in from `banks`; int64 on the device. One read-back: which experts were copied."""
        self.host()
        keys, found, now = self._touch(layer, torch.tensor(list(experts), dtype=torch.long).to(self.device))
        missed = found < 0
        order, _ = self._claim_order(now)
        placed = torch.where(missed, order[(missed.cumsum(0) - 1).clamp(min=0)], found)
        self._bind(placed, keys, missed)
        self.reads[:2] += torch.stack(((~missed).sum(), missed.sum())).to(torch.int32)
        for e, s, m in zip(experts, placed.tolist(), missed.tolist()):
            if m:
                self.write([s], [bank.take(bank.fields, e, e + 1) for bank in banks])
        return placed

    def _prompt_counts(self, layer, counts):
        """A prompt pass's use of `layer`'s experts with counts [E] rows (int64, device): (keys, cached slot or -1,
        uncached-and-used mask, the experts most rows first with the uncached ones ahead, each expert's place in that
        order, now)."""
        experts = torch.arange(self.num_experts, device=self.device)
        used = counts > 0
        keys, found, now = self._touch(layer, experts, used)
        uncached = used & (found < 0)
        order = torch.sort(torch.where(uncached, -counts, torch.ones_like(counts)), stable=True).indices
        place = torch.empty_like(order).index_copy_(0, order, experts)
        return keys, found, uncached, order, place, now

    def prompt_fills(self, layer, counts):
        """The kernels' prompt pass over `layer` (offload.py:468-484's policy): counts [E] rows per expert on the device.
        The uncached experts with most rows take the free slots, in ascending slot order, up to count // layers of
        them; the grouped kernels fill those slots as they read the experts. Returns (slot [E] int64: cached, or filled
        this pass, else -1 (and -1 for experts without rows); fill [E] bool; the experts most rows first, uncached ones ahead; uncached [E] bool), all on
        the device: nothing waits on the host."""
        self.host()
        keys, found, uncached, order, place, _ = self._prompt_counts(layer, counts)
        free = self.owner < 0
        free_first = torch.sort((~free).to(torch.int8), stable=True).indices
        fills = torch.minimum(free.sum(), uncached.sum()).clamp(max=self.count // self.layers)
        fill = uncached & (place < fills)
        target = free_first[place.clamp(max=self.count - 1)]
        self._bind(target, keys, fill)
        return torch.where(fill, target, torch.where(counts > 0, found, -1)), fill, order, uncached

    def prompt_keep(self, layer, counts):
        """The prompt pass without kernels (offload.py:528-545's policy): the uncached experts with most rows, up to
        min(count // layers, the slots this layer may claim), claim slots in ascending expert order. Returns (slot [E]
        int64: cached or claimed, else -1 (and for experts without rows); claimed [E] bool) on the device; the caller copies the claimed experts in."""
        self.host()
        keys, found, uncached, order, place, now = self._prompt_counts(layer, counts)
        claims, room = self._claim_order(now)
        keep = uncached & (place < room.clamp(max=self.count // self.layers))
        target = claims[(keep.cumsum(0) - 1).clamp(min=0)]
        self._bind(target, keys, keep)
        return torch.where(keep, target, torch.where(counts > 0, found, -1)), keep

    def report(self):
        self.host()
        hits, fills, on_cpu = self.reads.tolist()
        reads = hits + fills + on_cpu
        if reads:
            gib = sum(t.nbytes for f in self.fields for t in f.values()) / 1024 ** 3
            logging.info("drama3: %d cached expert slots (%.1f GiB) served %d decode reads: %d hits (%.0f%%), %d read "
                         "from host memory, %d run on the CPU", self.count, gib, reads, hits, 100 * hits / reads, fills,
                         on_cpu)


# -------------------------------------------------------------------------------------------------------- CPU side
class CpuSide:
    """Mailboxes between a decode step's layers and the host, one per layer in page-locked memory, so that the host
    serves one layer while the next is already launched (offload.py:276-299's protocol). The layer posts its plan,
    routing, rotated row and step (`post`) and then waits on the device, at most AWAIT_US, for the flag to reach its
    step (`wait`); the host takes the experts the plan left to it (`collect`), runs them and hands back their weighted
    sum, result first, then the flag (`deliver`)."""

    def __init__(self, layers, k, hidden):
        box = functools.partial(torch.zeros, pin_memory=True)
        self.plan = box((layers, k, 2), dtype=torch.int32)
        self.ids = box((layers, k), dtype=torch.long)
        self.weights = box((layers, k), dtype=torch.float32)
        self.rows = box((layers, 1, hidden), dtype=torch.bfloat16)
        self.step = box((layers,), dtype=torch.int32)
        self.flag = box((layers,), dtype=torch.int32)
        self.result = box((layers, hidden), dtype=torch.bfloat16)
        self.posted = [torch.cuda.Event() for _ in range(layers)]

    def post(self, layer, plan, ids, weights, rows, step):
        for box, value in ((self.plan, plan), (self.ids, ids), (self.weights, weights), (self.rows, rows)):
            box[layer].copy_(value, non_blocking=True)
        self.step.narrow(0, layer, 1).copy_(step, non_blocking=True)
        self.posted[layer].record()

    def wait(self, layer, plan, step, took_over):
        return kernels.await_cpu(plan, self.flag.narrow(0, layer, 1), step, self.result[layer], AWAIT_US, took_over)

    def collect(self, layer):
        """Once `layer` has posted: (experts the plan left to the CPU, their reserved slots or -1, their routing
        weights [n] float32, the rotated row [1, H] bf16), or None when it left none."""
        self.posted[layer].synchronize()
        plan = self.plan[layer]
        mine = (plan[:, 1] == 2).nonzero().flatten()
        if mine.numel() == 0:
            return None
        return (self.ids[layer, mine].tolist(), plan[mine, 0].tolist(), self.weights[layer, mine], self.rows[layer])

    def deliver(self, layer, value):
        """The host's result for `layer`'s posted step: written before the flag that releases the layer's wait."""
        self.result[layer].copy_(value)
        self.flag[layer] = self.step[layer]


# ----------------------------------------------------------------------------------------------------- the store
def _blend(old, measured, keep):
    """A running estimate: `keep` of the old one, the rest from the new measurement."""
    return keep * old + (1.0 - keep) * measured


DECODE_COST_KEEP = 0.9   # a decode step's CPU cost per expert: slow-moving average over the steps
PROMPT_SCALE_KEEP = 0.5  # measured / modelled cost of a prompt pass's CPU and GPU shares: half from each new pass


class ExpertStore:
    """Every layer's experts, added one layer at a time (`add`), held for generations (`session`) (offload.py:302-552's
    surface).

    In a session the store is either resident (every bank copied to the device: an MI355X holds them many times over)
    or a slot cache over page-locked host banks. `forward` runs a decode row or a prompt's rows through a layer's
    experts; `sync_free` says whether a decode row runs without waiting on the host."""

    def __init__(self, cache_bytes, pin):
        """`cache_bytes` 0: as much device memory as is free when a session starts. `pin` keeps the banks in
        page-locked host memory, which the kernels need to read them in place."""
        self.banks = []
        self.cache = None
        self.cache_bytes = cache_bytes
        self.pin = pin
        self.sync_free = False   # per session: decode rows run the kernels, never waiting on the host
        self.resident = None     # per resident session: each layer's banks on the device, expert e in slot e
        self.codebooks = []      # per session: each layer's (gate_up, down) codebooks on the device
        self.cpu = concurrent.futures.ThreadPoolExecutor(1, thread_name_prefix="drama3-experts")
        self.cpu_scale = self.gpu_scale = 1.0   # measured / modelled cost of the CPU's and the GPU's share of a prompt
        self.rotation = hadamard(256)
        self.cpu_experts = False  # per session: the CPU may run part of the missed int8 experts
        self.cpu_side = None      # per session with cpu_decode: the decode steps' mailboxes
        self.cpu_expert_us = CPU_EXPERT_US + CPU_ROW_US   # a decode step's expert on the CPU, as measured

    # -- building
    def add(self, experts):
        """Take a layer's experts (an FP8Experts, or a module with MoEExperts-like gate_up_proj / down_proj) into host
        memory; returns the module that stands in for them in the model."""
        if isinstance(experts, FP8Experts):
            banks = (FP8HostBank(experts.gate_up_weight, experts.gate_up_scale, self.pin),
                     FP8HostBank(experts.down_weight, experts.down_scale, self.pin))
        else:
            banks = (QuantHostBank(experts.gate_up_proj, self.pin), QuantHostBank(experts.down_proj, self.pin))
        return self._add(banks)

    def add_fields(self, kind, gate_up, down, num_experts, codebooks=(None, None)):
        """add() for a layer given as field dicts and codebooks (drama3/loader.py's form of a converted file)."""
        if kind == "fp8":
            banks = tuple(FP8HostBank.from_fields(num_experts, f, self.pin) for f in (gate_up, down))
        else:
            banks = tuple(QuantHostBank.from_fields(num_experts, kind, f, self.pin, cb)
                          for f, cb in zip((gate_up, down), codebooks))
        return self._add(banks)

    def _add(self, banks):
        if self.banks:
            first = self.banks[0][0]
            if (banks[0].kernel, banks[0].num_experts) != (first.kernel, first.num_experts):
                raise ValueError("every layer of a store holds the same format and expert count")
        self.banks.append(banks)
        return OffloadedExperts(self, len(self.banks) - 1)

    @property
    def bank_bytes(self):
        """Bytes of every layer's banks."""
        return sum(t.nbytes for banks in self.banks for bank in banks for t in bank.fields.values())

    # -- sessions
    def _device_budget(self, device, patchers, rows):
        """Device memory a session's cache may take: what is free less what the patchers' weights still need on this
        device and what the longest take needs for `rows` rows, within `cache_bytes` when that is set. With ComfyUI,
        other models are asked to make room first; if that evicted weights of the patchers themselves, they are loaded
        again before the free memory is read, so the cache is never sized into memory they are about to take."""
        reserve = RESERVE_BASE + int(RESERVE_PER_ROW * rows)

        def still_needed():
            return sum(p.model_size() - p.loaded_size() for p in patchers if p.load_device == device)

        if _mm is None:
            free = torch.cuda.mem_get_info(device)[0]
        else:
            loaded = sum(p.loaded_size() for p in patchers)
            _mm.free_memory((self.cache_bytes or self.bank_bytes) + still_needed() + reserve, device,
                            [m for m in _mm.current_loaded_models if m.model in patchers])
            if sum(p.loaded_size() for p in patchers) < loaded:
                # comfy made that room partly out of these patchers' own weights (its reading of free memory lags
                # what was just unloaded): let the reading catch up, load them back, then read
                time.sleep(EVICTION_PAUSE)
                _mm.load_models_gpu(patchers)
            free = _mm.get_free_memory(device)
        budget = max(0, free - still_needed() - reserve)
        return min(budget, self.cache_bytes) if self.cache_bytes else budget

    def _make_resident(self):
        """Every layer's banks copied into the slot pool, expert e of layer l in slot l * E + e, all mapped: each
        layer's slots are then its banks, read in place by the resident kernels."""
        cache, E = self.cache, self.banks[0][0].num_experts
        for layer, banks in enumerate(self.banks):
            for fields, rows, bank in zip(cache.fields, cache.rows, banks):
                for name, target in fields.items():
                    target.narrow(0, layer * E * rows[name], E * rows[name]).copy_(bank.fields[name], non_blocking=True)
        keys = torch.arange(len(self.banks) * E, dtype=torch.int32, device=cache.device)
        cache.table.copy_(keys)
        cache.owner.copy_(keys)
        self.resident = [[{name: t.narrow(0, layer * E * rows[name], E * rows[name]) for name, t in fields.items()}
                          for fields, rows in zip(cache.fields, cache.rows)] for layer in range(len(self.banks))]

    def _open(self, device, patchers, cpu_decode, rows, cpu_experts):
        budget = self._device_budget(device, patchers, rows)
        self.cache = SlotPool(self.banks, budget, device)
        first, keys = self.banks[0][0], len(self.banks) * self.banks[0][0].num_experts
        if self.cache.count == keys and budget >= self.bank_bytes:
            self._make_resident()
        # on the device before any decode step is captured in a graph, which cannot copy them
        self.codebooks = [tuple(bank.codebook(device) for bank in banks) for banks in self.banks]
        self.sync_free = (first.kernel is not None and kernels.available(device)
                          and (self.pin or self.resident is not None))
        # the CPU runs part of the missed int8 experts while the cache holds under half of them (offload.py:374-378)
        self.cpu_experts = (cpu_experts and self.sync_free and self.resident is None and first.kernel == "int8"
                            and 2 * self.cache.count < keys)
        if cpu_decode and self.cpu_experts:
            self.cpu_side = CpuSide(len(self.banks), MAX_EXPERTS_PER_ROW, first.in_features)

    def _close(self):
        self.cache.report()
        self.cache = self.resident = self.cpu_side = None
        self.sync_free = self.cpu_experts = False
        if _mm is not None:
            _mm.soft_empty_cache()

    @contextlib.contextmanager
    def session(self, device, patchers, cpu_decode, rows, cpu_experts=True):
        """One generation's hold on the experts (offload.py:334-384): resident when every bank fits the budget, else
        a slot cache of what fits. A session opened inside another shares its state. `cpu_decode`: every decode step
        calls `after_layer` after each layer; `cpu_experts`: the CPU may run part of the missed int8 experts."""
        if self.cache is not None:
            yield
            return
        self._open(torch.device(device), patchers, cpu_decode, rows, cpu_experts)
        try:
            yield
        finally:
            self._close()

    def between_steps(self):
        """Between decode steps with the CPU side: start copying the experts it ran into the slots they reserved, and
        set the GPU's share of a layer's missed experts so that both sides finish together: the CPU's measured cost per
        expert over that plus the expert's PCIe time."""
        self.cache.promote()
        pcie_us = self.cache.expert_bytes / PCIE_BYTES_PER_US
        self.cache.share.fill_(self.cpu_expert_us / (self.cpu_expert_us + pcie_us))

    # -- running a layer
    def _bank_rows(self, layer):
        return [bank.rows("weight" if bank.kernel == "fp8" else "_qdata") for bank in self.banks[layer]]

    def forward(self, layer, x, topk_idx, topk_weight):
        """A layer's experts for rows x [M, H] routed by topk_idx / topk_weight [M, k]: [M, H] in x's dtype."""
        banks = self.banks[layer]
        here = self.cache is not None and x.device == self.cache.device
        one_row = x.shape[0] == 1
        if self.resident is not None and self.sync_free and here:
            kind, rows, cbs = banks[0].kernel, self._bank_rows(layer), self.codebooks[layer]
            if one_row:
                return resident_decode(x, topk_idx[0], topk_weight[0], self.resident[layer], rows, kind, cbs)
            return resident_prefill(x, topk_idx, topk_weight, self.resident[layer], rows, kind, cbs,
                                    banks[0].num_experts)
        if one_row and self.sync_free and here:
            return self.decode(layer, banks, x, topk_idx[0], topk_weight[0])
        if one_row and self.cache is not None:
            slots = self.cache.slots(layer, topk_idx[0].tolist(), banks)
            dense = [bank.weight(self.cache.gather(i, slots), x.device).to(x.dtype) for i, bank in enumerate(banks)]
            return experts_decode(x, *dense, topk_weight[0])
        return self.prefill(layer, banks, x, topk_idx, topk_weight)

    def decode(self, layer, banks, x, ids, weights):
        """One row x [1, H] through its experts `ids` [k] from the slot cache and the host banks: the cache resolved on
        the device, then the GEMVs (cached experts from their slots, missed ones from host memory, filling their
        slots). With the CPU side the experts left to the CPU go to the host (`after_layer`) and come back through
        kernels.await_cpu; if the host is late, the GEMVs run them too."""
        cache, side = self.cache, self.cpu_side
        plan = kernels.resolve(ids, layer, len(self.banks), banks[0].num_experts, HALF_LIFE, side is not None, ADMIT,
                               *cache.device_state())
        return _slot_decode(x, ids, weights.float(), plan, cache.fields, [bank.fields for bank in banks],
                            self._bank_rows(layer), banks[0].kernel, self.codebooks[layer],
                            (cache.took_over, cache.always), None if side is None else (side, layer, cache.step))

    def after_layer(self, layer):
        """The host's part of decode layer `layer`, already launched (offload.py:434-452's protocol): take the experts
        its plan left to the CPU, reserve the slots the plan gave them for copying in between steps, run them, and hand
        the weighted sum back. Their measured cost steers the next steps' share."""
        task = self.cpu_side.collect(layer)
        if task is None:
            return
        experts, slots, weights, row = task
        self.cache.reserved.extend((layer, e, s) for e, s in zip(experts, slots) if s >= 0)
        out, seconds = timed(experts_on_cpu, self.banks[layer], experts, [1] * len(experts),
                             row.expand(len(experts), -1), self.rotation)
        self.cpu_side.deliver(layer, weights @ out)
        self.cpu_expert_us = _blend(self.cpu_expert_us, 1e6 * seconds / len(experts), DECODE_COST_KEEP)

    def prefill(self, layer, banks, x, topk_idx, topk_weight):
        """Many rows: each expert the rows use runs once on its rows (offload.py:454-466). The rows are grouped by
        expert on the device (expert_groups); through the kernels nothing is read back unless the CPU takes a share."""
        top_k = topk_idx.shape[1]
        order, inverse, groups = expert_groups(topk_idx, banks[0].num_experts)
        if self.sync_free:
            sorted_out = self._prefill_pairs(layer, banks, x, (order, top_k), groups[:, 4].long())
        else:
            sorted_out = self.prefill_host(layer, banks, x[order // top_k], groups[:, 4].tolist())
        return _combine(sorted_out, inverse, topk_weight, x.dtype)

    def split(self, experts, counts, expert_bytes):
        """(experts for the CPU, the CPU's modelled us, the GPU's modelled us) of `experts` (most rows first)
        (offload.py:514-526's rule): each goes to the side that would be done with it first, the CPU on a tie; the
        GPU's cost is reading the expert over PCIe, the CPU's CPU_EXPERT_US + CPU_ROW_US per row; both scaled by what
        earlier passes measured, the modelled times returned without the scales."""
        per_read = self.gpu_scale * expert_bytes / PCIE_BYTES_PER_US
        done = [0.0, 0.0]   # scaled us of work given to the CPU, the GPU
        on_cpu = []
        for e in experts:
            on_cpu_cost = self.cpu_scale * (CPU_EXPERT_US + CPU_ROW_US * counts[e])
            to_cpu = done[0] + on_cpu_cost <= done[1] + per_read
            done[0 if to_cpu else 1] += on_cpu_cost if to_cpu else per_read
            if to_cpu:
                on_cpu.append(e)
        return on_cpu, done[0] / self.cpu_scale, done[1] / self.gpu_scale

    def _cpu_share(self, layer, banks, rows_of, counts, first, fill, order, uncached):
        """The prompt's CPU share, when the CPU side is on: the uncached experts that fill no slot, most rows first,
        split by the cost model; their rows (rows_of(positions in the pairs' sorted order)) rotated into the ConvRot
        basis and handed to the CPU worker. Returns (experts, their rows' positions in the sorted order, the job, the
        modelled CPU and GPU us) or None. Reads the pass's plan back to the host once."""
        counts_h, first_h = counts.tolist(), first.tolist()
        rest = (uncached & ~fill)[order].tolist()
        candidates = [e for e, r in zip(order.tolist(), rest) if r]
        on_cpu, cpu_us, gpu_us = self.split(candidates, counts_h, self.cache.expert_bytes)
        if not on_cpu:
            return None
        picked = torch.cat([torch.arange(first_h[e], first_h[e] + counts_h[e]) for e in on_cpu]).to(counts.device)
        rows = torch.matmul(rows_of(picked).float().unflatten(-1, (-1, 256)),
                            self.rotation.to(counts.device)).flatten(-2)
        job = self.cpu.submit(timed, experts_on_cpu, banks, on_cpu, [counts_h[e] for e in on_cpu],
                              rows.to(torch.bfloat16).cpu(), self.rotation)
        return on_cpu, picked, job, cpu_us, gpu_us

    def prefill_kernels(self, layer, banks, sorted_x, counts):
        """The rows `sorted_x` (sorted by expert, counts[e] rows each: a list or a device tensor) through their
        experts, unweighted, float32 (offload.py:468-512's policy): cached experts from their slots, the uncached ones
        with most rows filling free slots as the grouped kernels read them (a filled expert crosses the bus once: its
        first pass fills the slot, the later ones read it there), the rest from host memory; with the CPU side, part
        of the rest on the CPU meanwhile. Without the CPU side nothing here waits on the host."""
        return self._prefill_pairs(layer, banks, sorted_x, None, counts)

    def _prefill_pairs(self, layer, banks, x, gather, counts):
        """prefill_kernels over the pairs' rows: x's rows sorted by expert (gather None), or with gather = (order,
        top_k) row order[p] // top_k of x for pair p."""
        cache, device = self.cache, x.device
        counts = torch.as_tensor(counts, dtype=torch.long).to(device)
        slot, fill, by_rows, uncached = cache.prompt_fills(layer, counts)
        first = counts.cumsum(0) - counts
        rows = counts
        share = None
        if self.cpu_experts:
            if gather is None:
                rows_of = functools.partial(torch.index_select, x, 0)
            else:
                rows_of = lambda at: x.index_select(0, gather[0].index_select(0, at) // gather[1])  # noqa: E731
            share = self._cpu_share(layer, banks, rows_of, counts, first, fill, by_rows, uncached)
            if share is not None:
                rows = counts.index_fill(0, torch.tensor(share[0], device=device), 0)   # the kernels skip them
        experts = torch.arange(counts.shape[0], device=device)
        groups = torch.stack((experts, slot, fill.long(), first, rows), dim=1).to(torch.int32)
        if share is not None:   # the GPU's part is timed for the cost model
            started, ended = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            started.record()
        out = _grouped_pairs(x, gather, groups, cache.fields, [bank.fields for bank in banks], self._bank_rows(layer),
                              banks[0].kernel, self.codebooks[layer], cache.always, fills_first=True)
        if share is not None:
            ended.record()
            _, picked, job, cpu_us, gpu_us = share
            result, cpu_seconds = job.result()
            out.index_copy_(0, picked, result.to(device, torch.float32))
            self.cpu_scale = _blend(self.cpu_scale, 1e6 * cpu_seconds / cpu_us, PROMPT_SCALE_KEEP)
            if gpu_us:
                ended.synchronize()
                self.gpu_scale = _blend(self.gpu_scale, 1e3 * started.elapsed_time(ended) / gpu_us, PROMPT_SCALE_KEEP)
        return out

    def prefill_host(self, layer, banks, sorted_x, counts):
        """prefill_kernels without the kernels (unpinned banks, formats without kernels) (offload.py:528-552's policy):
        the uncached experts with most rows take slots (up to the layer's share of the cache, never a slot this layer
        reads) and are copied in at once; then expert by expert, dense bf16 products from its slot or straight from
        host memory."""
        cache, device = self.cache, sorted_x.device
        slot, keep = cache.prompt_keep(layer, torch.as_tensor(counts, dtype=torch.long).to(cache.device))
        slot, keep = slot.tolist(), keep.tolist()
        kept = [e for e, k in enumerate(keep) if k]
        if kept:
            cache.write([slot[e] for e in kept], [bank.pick(kept) for bank in banks])
        out = torch.empty_like(sorted_x)
        start = 0
        for e, n in enumerate(counts):
            if not n:
                continue
            if slot[e] >= 0:
                sources = [cache.slot_fields(i, slot[e]) for i in range(len(banks))]
            else:
                sources = [bank.to_device(e, e + 1, device) for bank in banks]
            gate_up, down = (bank.weight(src, device).to(sorted_x.dtype) for bank, src in zip(banks, sources))
            out[start:start + n] = nn.functional.linear(swiglu(nn.functional.linear(sorted_x[start:start + n],
                                                                                    gate_up)), down)
            start += n
        return out


class ExpertTable:
    """Banks placed whole in HBM, layer by layer (`place`), read in place by the resident kernels (expert e in slot e):
    a converted checkpoint's experts on an MI355X without a store (drama3/loader.py). `bytes` is what it holds."""

    def __init__(self, device):
        self.device = torch.device(device)
        self.layers = {}

    def place(self, layer, kind, gate_up, down, codebooks=(None, None)):
        banks = tuple({name: t.to(self.device, non_blocking=True).contiguous() for name, t in f.items()}
                      for f in (gate_up, down))
        cbs = tuple(None if c is None else c.to(self.device) for c in codebooks)
        self.layers[layer] = (kind, banks, cbs)
        return self.layers[layer]

    @property
    def bytes(self):
        return sum(t.nbytes for _, banks, _ in self.layers.values() for f in banks for t in f.values())

    def fits(self, extra=0):
        """Whether `extra` more bytes fit in the device's free memory."""
        free, _ = torch.cuda.mem_get_info(self.device)
        return extra <= free

    def decode(self, layer, x, ids, weights, num_experts):
        kind, banks, cbs = self.layers[layer]
        return resident_decode(x, ids, weights, banks, [_rows(kind, b, num_experts) for b in banks], kind, cbs)

    def prefill(self, layer, x, topk_idx, topk_weight, num_experts):
        kind, banks, cbs = self.layers[layer]
        return resident_prefill(x, topk_idx, topk_weight, banks, [_rows(kind, b, num_experts) for b in banks], kind,
                                cbs, num_experts)


# ------------------------------------------------------------------------------------------------- model modules
class FP8Experts(nn.Module):
    """Routed experts as Fish ships them: float8 e4m3 weights with a float32 scale per 128 x 128 block
    (offload.py:755-802). A decode row runs resident_decode, a prompt resident_prefill, on the gfx950 kernels; there is
    no torch path here: on any other device the call raises."""

    def __init__(self, num_experts, hidden, intermediate, device=None, dtype=None):
        super().__init__()
        self.num_experts = num_experts
        self.dtype = dtype
        for name, rows, cols in (("gate_up", 2 * intermediate, hidden), ("down", hidden, intermediate)):
            weight = torch.empty((num_experts, rows, cols), dtype=torch.float8_e4m3fn, device=device)
            scale = torch.empty((num_experts, rows // FP8_BLOCK, cols // FP8_BLOCK), dtype=torch.float32, device=device)
            self.register_parameter(f"{name}_weight", nn.Parameter(weight, requires_grad=False))
            self.register_parameter(f"{name}_scale", nn.Parameter(scale, requires_grad=False))

    def sync_free(self, device):
        """Whether a decode row on `device` runs without waiting on the host: the kernels run there."""
        return kernels.available(torch.device(device))

    def experts(self, name, ids):
        """Experts `ids` of bank `name` ("gate_up" or "down"), dequantized to the module's dtype, one after another."""
        weight = getattr(self, f"{name}_weight")
        picked = weight.view(torch.uint8).index_select(0, ids).flatten(0, 1).view(torch.float8_e4m3fn)
        return dequantize_fp8(picked, getattr(self, f"{name}_scale").index_select(0, ids).flatten(0, 1), self.dtype)

    def _banks(self):
        names = ("gate_up", "down")
        banks = [{"weight": getattr(self, f"{n}_weight").view(torch.uint8).flatten(0, 1),
                  "scale": getattr(self, f"{n}_scale").flatten(0, 1)} for n in names]
        return banks, [getattr(self, f"{n}_weight").shape[1] for n in names]

    def forward(self, x, topk_idx, topk_weight):
        if not kernels.available(x.device):
            raise RuntimeError(f"drama3.offload.FP8Experts: the gfx950 kernels do not run on {x.device}")
        banks, rows = self._banks()
        if x.shape[0] == 1:
            return resident_decode(x, topk_idx[0], topk_weight[0], banks, rows, "fp8", (None, None))
        return resident_prefill(x, topk_idx, topk_weight, banks, rows, "fp8", (None, None), self.num_experts)


class HostEmbedding(nn.Module):
    """The token embedding table left in host memory beside the experts (offload.py:805-815): a prompt or a frame
    reads a few of its rows, and the device memory goes to the experts instead."""

    def __init__(self, embedding):
        super().__init__()
        self.table = embedding.weight.detach()

    def forward(self, ids, out_dtype=None):
        rows = self.table.index_select(0, ids.reshape(-1).to(self.table.device))
        return rows.unflatten(0, ids.shape).to(ids.device, out_dtype)


class OffloadedExperts(nn.Module):
    """Stands in for a layer's experts kept by an ExpertStore (offload.py:817-830)."""

    def __init__(self, store, layer):
        super().__init__()
        self.store = store
        self.layer = layer

    def sync_free(self, device):
        """Whether a decode row on `device` runs without waiting on the host, in the current session."""
        store = self.store
        return bool(store.sync_free and store.cache is not None and torch.device(device) == store.cache.device)

    def forward(self, x, topk_idx, topk_weight):
        return self.store.forward(self.layer, x, topk_idx, topk_weight)
