"""What this framework is measured on: calls of its public entry points over the sizes, formats and routings that a
program with this model runs. A case is one call (or one token's calls through several layers) and names its path:

  linear      kernels.fp8_linear: one FP8 weight with row scales against a few bf16 rows
  lines       moe.moe_layer on A8 banks: a decode step of `rows` lines through `layers` layers, captured in a HIP graph
              as a serving loop captures its step
  block       moe.moe_block, one line: router, routed experts and shared expert, through `layers` layers in a graph
  ref_line    offload.routed_decode on banks in the reference's layouts: one line's step through `layers` layers in a
              graph
  prompt      moe.moe_prefill on A8 banks: a prompt's rows through one layer
  ref_prompt  offload.resident_prefill on banks in the reference's layouts: a prompt's rows through one layer

Hidden size 2048, top-8 of 128 experts with FFN 768 (the benchmark's layer) or of 256 with FFN 512 (the model's).
Prompts go up to 8192 rows, the longest one the model takes. Weights are N(0, 0.02) quantized (the ConvRot formats in
their rotated basis, where N(0, 0.02) weights have the same distribution), activations N(0, 1) in bf16, router logits
N(0, 1) or drawn so that the top-8 follow Zipf(1.1) over a random order of the experts.
"""
import math
import pathlib
import sys

import torch

_PACKAGE = str(pathlib.Path(__file__).resolve().parents[1] / "comfyui-drama3_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from drama3 import formats, kernels, moe, offload  # noqa: E402

H, TOPK = 2048, 8
SHAPES = {128: 768, 256: 512}     # experts -> FFN size
LAYERS = 8                        # of a token's step: more routed bytes than the memory-side cache holds
MAX_PROMPT = 8192
DEV = "cuda:0"
A8 = {"int8": formats.FMT_I8, "w4": formats.FMT_W4, "w6": formats.FMT_W6, "fp8": formats.FMT_F8}


def listed():
    return [
        # the smallest call: one expert's FP8 weight against one row, launched on its own
        {"name": "linear_fp8", "path": "linear", "rows": 1, "n": 1536, "k": 2048},
        # one voice, frame by frame: the decode step that a take spends its time in
        {"name": "line1_int8", "path": "lines", "format": "int8", "rows": 1, "experts": 128, "routing": "normal"},
        # the same frame with the router and the shared expert in the layer's launch
        {"name": "block1_int8", "path": "block", "format": "int8", "rows": 1, "experts": 128, "routing": "normal"},
        # four lines of a story decoded together
        {"name": "lines4_w4", "path": "lines", "format": "w4", "rows": 4, "experts": 128, "routing": "normal"},
        # the most lines a step takes
        {"name": "lines16_fp8", "path": "lines", "format": "fp8", "rows": 16, "experts": 128, "routing": "normal"},
        # a converted checkpoint at the model's shape, one voice
        {"name": "ref1_w4", "path": "ref_line", "format": "w4", "rows": 1, "experts": 256, "routing": "normal"},
        # a short text chunk before its frames, in the original FP8 weights
        {"name": "ref_fp8_77", "path": "ref_prompt", "format": "fp8", "rows": 77, "experts": 256,
         "routing": "normal"},
        # the benchmark's prompt on a converted checkpoint
        {"name": "ref_int8_256", "path": "ref_prompt", "format": "int8", "rows": 256, "experts": 128,
         "routing": "zipf"},
        # a reference voice's frames as the prompt (odd length), at the model's shape
        {"name": "ref_w4_2391", "path": "ref_prompt", "format": "w4", "rows": 2391, "experts": 256,
         "routing": "normal"},
        # the longest prompt a take accepts
        {"name": "ref_w6_8192", "path": "ref_prompt", "format": "w6", "rows": 8192, "experts": 128,
         "routing": "zipf"},
        # the benchmark's prompt on A8 banks, and a long one
        {"name": "a8_fp8_256", "path": "prompt", "format": "fp8", "rows": 256, "experts": 128, "routing": "zipf"},
        {"name": "a8_int8_4096", "path": "prompt", "format": "int8", "rows": 4096, "experts": 128,
         "routing": "normal"},
    ]


def draw(rng):
    path = rng.choices(("linear", "lines", "block", "ref_line", "prompt", "ref_prompt"), (1, 3, 1, 2, 4, 6))[0]
    if path == "linear":
        return {"path": path, "rows": rng.randint(1, 4), "n": 64 * rng.randint(4, 64), "k": 512 * rng.randint(1, 4)}
    case = {"path": path, "format": rng.choice(("int8", "fp8", "w4", "w6")), "rows": 1,
            "experts": rng.choice((128, 256)), "routing": rng.choice(("normal", "zipf"))}
    if path == "lines":
        case["rows"] = rng.randint(1, moe.MAX_ROWS)
    elif path in ("prompt", "ref_prompt"):
        case["rows"] = round(math.exp(rng.uniform(math.log(17), math.log(MAX_PROMPT))))
    return case


def _layers(case):
    return LAYERS if case["path"] in ("lines", "block", "ref_line") else 1


# ------------------------------------------------------------------------------------------------------- inputs
def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV)


def _logits(gen, case):
    T, E = case["rows"], case["experts"]
    if case["routing"] == "normal":
        return _normal(gen, T, E).to(torch.bfloat16)
    logp = -1.1 * torch.log(torch.arange(1, E + 1, device=DEV, dtype=torch.float32))
    base = torch.empty(E, device=DEV)
    base[torch.randperm(E, generator=gen, device=DEV)] = logp
    u = torch.rand((T, E), generator=gen, device=DEV).clamp_(1e-12, 1 - 1e-7)
    return (base - torch.log(-torch.log(u))).to(torch.bfloat16)


def _a8_banks(gen, case, experts):
    I, fmt = SHAPES[case["experts"]], A8[case["format"]]
    return tuple(formats.quantize(_normal(gen, experts, n, k) * 0.02, fmt) for n, k in ((2 * I, H), (H, I)))


# a fixed ascending codebook of the 4-bit rows: normal quantiles spread over +-8
_CODEBOOK = [8.0 * math.sqrt(2) * float(torch.erfinv(torch.tensor((2 * i + 1) / 16 - 1))) / (
    math.sqrt(2) * float(torch.erfinv(torch.tensor(15 / 16)))) for i in range(16)]


def _ref_bank(gen, kind, experts, n, k):
    """One bank in the reference's layout: the fields that its loader hands out."""
    w = _normal(gen, experts * n, k) * 0.02
    if kind == "fp8":
        blocks = w.view(experts * n // 128, 128, k // 128, 128)
        scale = blocks.abs().amax(dim=(1, 3)) / 448.0
        q = (blocks / scale[:, None, :, None]).to(torch.float8_e4m3fn)
        return {"weight": q.view(torch.uint8).view(experts * n, k), "scale": scale}
    channel = w.abs().amax(dim=1) / 127.0
    w /= channel[:, None]
    if kind == "int8":
        return {"_qdata": w.round_().clamp_(-127, 127).to(torch.int8), "scale": channel}
    groups = w.view(experts * n, k // 16, 16)
    top = 8.0 if kind == "w4" else 31.0
    scale = (groups.abs().amax(dim=2) / top).to(torch.float8_e4m3fn)
    groups /= scale.float().clamp_min_(2.0 ** -9)[..., None]
    if kind == "w4":
        book = torch.tensor(_CODEBOOK, device=DEV)
        code = torch.bucketize(w, (book[1:] + book[:-1]) / 2, out_int32=True).to(torch.uint8)
        rows = code[:, 0::2] | (code[:, 1::2] << 4)
    else:
        code = (w.round_().clamp_(-32, 31) + 32).to(torch.uint8)
        low, two = code & 15, (code >> 4).view(experts * n, k // 4, 4)
        high = two[..., 0] | (two[..., 1] << 2) | (two[..., 2] << 4) | (two[..., 3] << 6)
        rows = torch.cat((low[:, 0::2] | (low[:, 1::2] << 4), high), dim=1)
    return {"_qdata": rows.contiguous(), "scale": scale.view(torch.uint8), "s_channel": channel}


def _ref_banks(gen, case):
    E, I, kind = case["experts"], SHAPES[case["experts"]], case["format"]
    book = torch.tensor(_CODEBOOK, device=DEV) if kind == "w4" else None
    return (_ref_bank(gen, kind, E, 2 * I, H), _ref_bank(gen, kind, E, H, I)), (book, book)


def _softmax_topk(logits):
    """The router's softmax, top-k and renormalization of a prompt's rows, as the model computes them."""
    w, ids = torch.softmax(logits.float(), dim=-1).topk(TOPK, dim=-1)
    return ids, (w / w.sum(dim=-1, keepdim=True)).to(torch.bfloat16)


def _inputs(case, seed):
    """Everything a case's call reads, from the seed alone: a dict of tensors and banks, one per layer."""
    gen = torch.Generator(device=DEV).manual_seed(1000003 * seed + 17)
    path = case["path"]
    if path == "linear":
        w = _normal(gen, case["n"], case["k"]) * 0.02
        scale = (w.abs().amax(dim=1) / 448.0).to(torch.bfloat16)
        return [{"x": _normal(gen, case["rows"], case["k"]).to(torch.bfloat16), "scale": scale,
                 "weight": (w / scale.float()[:, None]).to(torch.float8_e4m3fn)}]
    layers = []
    for _ in range(_layers(case)):
        d = {"x": _normal(gen, case["rows"], H).to(torch.bfloat16)}
        if path in ("ref_line", "ref_prompt"):
            d["banks"], d["books"] = _ref_banks(gen, case)
        else:
            d["banks"] = _a8_banks(gen, case, case["experts"])
        if path == "block":
            d["router"] = (_normal(gen, case["experts"], H) / math.sqrt(H)).to(torch.bfloat16)
            d["shared"] = _a8_banks(gen, case, 1)
            d["shared_gate"] = (_normal(gen, H) / math.sqrt(H)).to(torch.bfloat16)
        else:
            d["logits"] = _logits(gen, case)
        if path == "ref_prompt":
            d["ids"], d["weights"] = _softmax_topk(d["logits"])
        layers.append(d)
    return layers


# ---------------------------------------------------------------------------------------------------- the calls
def _call(case, d):
    path, I = case["path"], SHAPES.get(case.get("experts"))
    if path == "linear":
        return kernels.fp8_linear(d["x"], d["weight"], d["scale"])
    if path == "lines":
        return moe.moe_layer(d["x"], d["logits"], *d["banks"], TOPK)
    if path == "block":
        return moe.moe_block(d["x"], *d["banks"], TOPK, router=d["router"], shared=d["shared"],
                             shared_gate=d["shared_gate"])
    if path == "ref_line":
        return offload.routed_decode(d["x"], d["logits"], TOPK, d["banks"], (2 * I, H), case["format"], d["books"])
    if path == "prompt":
        return moe.moe_prefill(d["x"], *d["banks"], TOPK, logits=d["logits"], routing=True)
    return offload.resident_prefill(d["x"], d["ids"], d["weights"], d["banks"], (2 * I, H), case["format"],
                                    d["books"], case["experts"])


_stream = None


def _capture_stream():
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream(DEV)
    return _stream


def prepare(case, seed):
    layers = _inputs(case, seed)
    state = {"case": case, "layers": layers, "graph": None}
    if _layers(case) > 1:  # a decode step: captured once, replayed per token
        stream = _capture_stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            moe.prepare(DEV, H, SHAPES[case["experts"]], stream)
            _call(case, layers[0])  # what the first call makes exists before the capture
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                state["out"] = [_call(case, d) for d in layers]
        torch.cuda.current_stream().wait_stream(stream)
        state["graph"] = graph
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return _call(state["case"], state["layers"][0])


# ------------------------------------------------------------------------------------------- work and tolerance
_ROW_BYTES = {"int8": 1.0, "fp8": 1.0, "w4": 0.5, "w6": 0.75}


def _expected_experts(case):
    """The experts that the rows' routes are expected to touch."""
    E, T = case["experts"], case["rows"]
    if case["routing"] == "normal":
        return E * (1 - (1 - TOPK / E) ** T)
    p = [r ** -1.1 for r in range(1, E + 1)]
    total = sum(p)
    return max(TOPK, sum(1 - (1 - min(1.0, TOPK * v / total)) ** T for v in p))


def work(case):
    if case["path"] == "linear":
        n, k, rows = case["n"], case["k"], case["rows"]
        return {"bytes": n * k + 2 * n + 2 * rows * (n + k), "flops": 2 * rows * n * k}
    T, I, f = case["rows"], SHAPES[case["experts"]], case["format"]
    weights = 3 * H * I * _ROW_BYTES[f]
    if case["path"] in ("ref_line", "ref_prompt"):
        rows = 2 * I + H
        weights += 3 * H * I / 16384 * 4 if f == "fp8" else rows * 4 if f == "int8" else rows * 4 + 3 * H * I / 16
    else:
        weights += 3 * H * I / 128 * 2 if f in ("w4", "w6") else (2 * I + H) * 2
    per_layer = _expected_experts(case) * weights + T * (2 * H * 2 + case["experts"] * 2)
    pairs = T * TOPK
    if case["path"] == "block":
        per_layer += weights + case["experts"] * H * 2 + H * 2
        pairs += T
    n = _layers(case)
    return {"bytes": n * per_layer, "flops": n * 2 * pairs * 3 * H * I}


def tolerance(case):
    # outputs are bf16: one rounding each is 1.7e-3 of the result, and what is off from the 64-bit results. The A8
    # layers also round their activations to 8 bits: a value on a rounding boundary flips a code when a sum's order
    # or the scale's last bit changes, and a line's output moves by up to 9e-3 (FP8 5e-3 to 7e-3)
    if case["path"] in ("prompt", "lines", "block"):
        return {"rel": 1e-2, "max": 1e-1, "differ": 1e-3}
    return {"rel": 7e-3, "max": 5e-2, "differ": 1e-3}


# ------------------------------------------------------------------------------------------------ 64-bit results
def _silu_up(gu):
    half = gu.shape[-1] // 2
    return torch.nn.functional.silu(gu[..., :half]) * gu[..., half:]


def _a8_weight(bank, e):
    """Expert e's rows of an A8 bank in 64 bits, from the layout's definition."""
    rows = slice(e * bank.rows, (e + 1) * bank.rows)
    b, s = bank.weight[rows], bank.scale[rows].double()
    if bank.fmt == formats.FMT_F8:
        return b.view(torch.float8_e4m3fn).double() * s[:, None]
    if bank.fmt == formats.FMT_I8:
        return b.view(torch.int8).double() * s[:, None]
    if bank.fmt == formats.FMT_W4:
        q = torch.stack((b & 15, b >> 4), dim=-1).flatten(-2).double()
        q = torch.where(q >= 8, q - 16, q)
    else:
        u = b.view(bank.rows, -1, 12)
        t = (u >> 6).view(bank.rows, -1, 3, 4)
        last = t[:, :, 0] | (t[:, :, 1] << 2) | (t[:, :, 2] << 4)
        q = torch.cat((u & 63, last), dim=-1).flatten(-2).double()
        q = torch.where(q >= 32, q - 64, q)
    return (q.view(bank.rows, -1, 128) * s[..., None]).view(bank.rows, bank.cols)


def _a8_act(v, fmt):
    """Rows as the format's activations hold them: int8 at absmax / 127, or e4m3 at absmax / 448."""
    qmax = 448.0 if fmt == formats.FMT_F8 else 127.0
    amax = v.abs().amax(dim=-1, keepdim=True).clamp_min(1e-300)
    q = v * (qmax / amax)
    q = q.float().to(torch.float8_e4m3fn).double() if fmt == formats.FMT_F8 else q.round()
    return q * (amax / qmax)


def _rotation():
    h4 = torch.tensor([[1.0, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device=DEV)
    m = h4
    for _ in range(3):
        m = torch.kron(m, h4)
    return m / 16.0


def _ref_weight(kind, fields, book, e, n):
    rows = slice(e * n, (e + 1) * n)
    if kind == "fp8":
        s = fields["scale"][e * n // 128:(e + 1) * n // 128].double()
        w = fields["weight"][rows].view(torch.float8_e4m3fn).double()
        return (w.view(n // 128, 128, -1, 128) * s[:, None, :, None]).view(n, -1)
    if kind == "int8":
        return fields["_qdata"][rows].double() * fields["scale"][rows].double()[:, None]
    q = fields["_qdata"][rows]
    k = q.shape[1] * 8 // int(kind[1])
    low = q[:, :k // 2]
    code = torch.stack((low & 15, low >> 4), dim=-1).flatten(-2).long()
    if kind == "w4":
        value = book.double()[code]
    else:
        high = torch.stack([(q[:, k // 2:] >> s) & 3 for s in (0, 2, 4, 6)], dim=-1).flatten(-2).long()
        value = (code + 16 * high - 32).double()
    scale = fields["scale"][rows].view(torch.float8_e4m3fn).double().repeat_interleave(16, dim=1)
    grid = (value * scale).round().clamp(-127, 127)
    return grid * fields["s_channel"][rows].double()[:, None]


def _experts(x, ids, weights, weight_of, between):
    """sum over k of weights * down(between(gate_up(x))) in 64 bits, expert by expert."""
    parts = torch.zeros((*ids.shape, H), dtype=torch.float64, device=DEV)
    for e in ids.unique().tolist():
        t, j = (ids == e).nonzero(as_tuple=True)
        parts[t, j] = between(_silu_up(x[t] @ weight_of(0, e).T)) @ weight_of(1, e).T
    return (weights.double()[..., None] * parts).sum(dim=1)


def _exact_layer(case, d):
    path, x = case["path"], d["x"].double()
    if path == "linear":
        w = (d["weight"].float() * d["scale"].float()[:, None]).to(torch.bfloat16).double()
        return x @ w.T
    lg = (x @ d["router"].double().T).to(torch.bfloat16) if path == "block" else d["logits"]
    if "ids" in d:
        ids, w = d["ids"], d["weights"].double()
    else:  # ties go to the lower index
        top, ids = torch.sort(lg.double(), dim=-1, descending=True, stable=True)
        ids, w = ids[:, :TOPK], torch.softmax(top[:, :TOPK], dim=-1).to(torch.bfloat16).double()
    if path in ("ref_line", "ref_prompt"):
        kind = case["format"]
        rot = (lambda v: v) if kind == "fp8" else (
            lambda v, m=_rotation(): (v.unflatten(-1, (-1, 256)) @ m).flatten(-2))
        n = (2 * SHAPES[case["experts"]], H)
        out = _experts(rot(x), ids, w, lambda b, e: _ref_weight(kind, d["banks"][b], d["books"][b], e, n[b]), rot)
        return out if path == "ref_prompt" else [out, None, w]
    fmt = A8[case["format"]]
    act = lambda v: _a8_act(v, fmt)  # noqa: E731
    out = _experts(act(x), ids, w, lambda b, e: _a8_weight(d["banks"][b], e), act)
    if path == "block":
        one = torch.zeros((1, 1), dtype=torch.int64, device=DEV)
        shared = _experts(act(x), one, one + 1.0, lambda b, e: _a8_weight(d["shared"][b], e), act)
        return out + torch.sigmoid(x @ d["shared_gate"].double())[:, None] * shared
    return out if path == "lines" else [out, None, w]


def exact(case, seed):
    got = [_exact_layer(case, d) for d in _inputs(case, seed)]
    return got if len(got) > 1 else got[0]
