"""The workloads by which the speed of the MoE path is followed.

Each case is one pass of work that a program using the library asks of it, through the pointer-level entry
points such a program calls (device tensors in, device tensors out, no host synchronisation):

  decode   one MoE layer over a decode batch of 1 to 16 tokens (MoELayer.decode_device): router, top-k,
           routed and shared MXFP4 experts, ordered combine
  prefill  one MoE layer over a prompt (MoELayer.prefill_device), routed by the layer's own router or by
           given routing with Zipf skew
  proj128  the FP8 attention projections with FP32 128 x 128 block scales: q_a and kv_a stacked (they read
           the same input), q_b and o, one call each (fp8_projection)
  attn32   the reference model's FP8 projections with E8M0 32 x 32 block scales: wq_a, wq_b, wkv, wo_b, and
           the grouped output projection wo_a on its rounded input (fp8_projection, kv_round32,
           fp8_grouped_projection)
  shared   the FP8 block-32 shared expert of four consecutive layers (fp8_expert_forward)
  bf16     the MXFP4 expert with BF16 activations, of eight consecutive layers (expert_forward_bf16)

`model` picks the shapes: "base" is vesper_amd.config.BASELINE (7168 x 2048, 256 experts, 8 per token) and
"ref" is vesper_amd.config.REFERENCE (5120 x 2304, 384 experts, 6 per token, clamped, biased selection).
Weights, inputs and routing are drawn on the device from the seed alone. The three states a measurement goes
through in turn hold more weights than the 256 MB Infinity Cache, as the layers of a model do.
"""

import ctypes as C
import math

import torch

from vesper_amd import _lib
from vesper_amd.config import BASELINE, REFERENCE
from vesper_amd.layer import TENSORS, ExpertBank, MoELayer

MODELS = {"base": BASELINE, "ref": REFERENCE}
# rows x width; q_a (1536) and kv_a (576) read one input and run as one projection of their stacked rows
PROJ128 = {"q_kv_a": (2112, 7168), "q_b": (24576, 1536), "o": (7168, 16384)}
ATTN32 = {"wq_a": (1280, 5120), "wq_b": (32768, 1280), "wkv": (512, 5120), "wo_b": (5120, 8192)}
WO_A_GROUPS, WO_A_ROWS, WO_A_WIDTH = 8, 1024, 4096
SHARED_LAYERS, BF16_LAYERS = 4, 8
ZIPF = 1.1
SCALE_CODES = (118, 121)   # E8M0 codes [118, 120] of the MXFP4 experts: gate and up values of order 1

DEVICE = "cuda"


def listed():
    return [
        # one user's next token through one layer: the latency that an interactive session sees
        {"name": "decode-1", "kind": "decode", "model": "base", "tokens": 1},
        # a small batch of sessions
        {"name": "decode-4", "kind": "decode", "model": "base", "tokens": 4},
        # the largest decode batch
        {"name": "decode-16", "kind": "decode", "model": "base", "tokens": 16},
        # the reference model's layer at an odd batch: clamp, selection bias, sqrtsoftplus scores, 384 experts
        {"name": "decode-ref-7", "kind": "decode", "model": "ref", "tokens": 7},
        # a prompt of ordinary length, routed by the layer itself: few rows per expert
        {"name": "prefill-ref-1000", "kind": "prefill", "model": "ref", "tokens": 1000, "routing": "layer"},
        # a long prompt with skewed routing: from no rows to thousands per expert
        {"name": "prefill-4096", "kind": "prefill", "model": "base", "tokens": 4096, "routing": "zipf"},
        # the attention projections of one token
        {"name": "proj128-1", "kind": "proj128", "tokens": 1},
        # and of the largest decode batch
        {"name": "proj128-16", "kind": "proj128", "tokens": 16},
        # and of a prompt
        {"name": "proj128-2048", "kind": "proj128", "tokens": 2048},
        # the reference model's projections at the most rows that its own calls take
        {"name": "attn32-8", "kind": "attn32", "tokens": 8},
        # the reference model's shared experts for one token
        {"name": "shared-1", "kind": "shared", "tokens": 1},
        # one expert after another without activation quantization, for one token
        {"name": "bf16-1", "kind": "bf16", "tokens": 1},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "proj128", "proj128", "attn32", "shared",
                       "bf16"])
    if kind == "decode":
        return {"kind": kind, "model": rng.choice(["base", "ref"]), "tokens": rng.randint(1, 16)}
    if kind == "prefill":
        return {"kind": kind, "model": rng.choice(["base", "ref"]), "tokens": _log_int(rng, 17, 3500),
                "routing": rng.choice(["layer", "zipf"])}
    if kind == "proj128":
        return {"kind": kind, "tokens": _log_int(rng, 1, 2048)}
    if kind == "attn32":
        return {"kind": kind, "tokens": rng.randint(1, 32)}
    return {"kind": kind, "tokens": rng.randint(1, 16)}


# -- seeded inputs -------------------------------------------------------------------------------------

def _gen(seed, *tag):
    g = torch.Generator(device=DEVICE)
    value = seed & 0xFFFFFFFF
    for t in tag:
        value = (value * 1000003 + t + 1) & 0x7FFFFFFFFFFF
    g.manual_seed(value)
    return g


def _normal_bf16(g, *shape):
    return torch.randn(shape, generator=g, device=DEVICE).to(torch.bfloat16)


def _mxfp4_layout(hidden, intermediate):
    rows = {"w1": (intermediate, hidden), "w3": (intermediate, hidden), "w2": (hidden, intermediate)}
    return {f"{n}_{part}": (r, k // (2 if part == "weight" else 32)) for n, (r, k) in rows.items()
            for part in ("weight", "scale")}


def _mxfp4_expert(seed, expert, hidden, intermediate):
    """The six tensors of one expert: packed E2M1 codes and E8M0 scales, uniform over their ranges."""
    g = _gen(seed, 1, expert)
    return {name: torch.randint(0, 256, shape, generator=g, device=DEVICE, dtype=torch.uint8)
            if name.endswith("weight") else
            torch.randint(*SCALE_CODES, shape, generator=g, device=DEVICE, dtype=torch.uint8)
            for name, shape in _mxfp4_layout(hidden, intermediate).items()}


def _fp8_weight(seed, tag, rows, width, block):
    """N(0, 0.02) weights as E4M3 codes [rows, width] and their block scales, FP32 (block 128: amax / 448) or
    E8M0 codes (block 32: the smallest power of two that keeps amax / scale within 448)."""
    w = torch.randn((rows, width), generator=_gen(seed, 2, tag), device=DEVICE) * 0.02
    rb, wb = -(-rows // block), width // block
    padded = torch.nn.functional.pad(w, (0, 0, 0, rb * block - rows)).view(rb, block, wb, block)
    amax = padded.abs().amax(dim=(1, 3)).clamp_min(1e-12)
    if block == 128:
        scales = amax / 448.0
        value = scales
    else:
        e = torch.ceil(torch.log2(amax.double() / 448.0)).to(torch.int32)
        scales = (e + 127).to(torch.uint8)
        value = torch.exp2(e.float())
    codes = (padded / value[:, None, :, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return codes.view(torch.uint8).reshape(rb * block, width)[:rows].contiguous(), scales.contiguous()


def _router(seed, cfg):
    g = _gen(seed, 3)
    w = torch.randn((cfg.experts, cfg.hidden), generator=g, device=DEVICE) * 0.02
    bias = torch.randn(cfg.experts, generator=g, device=DEVICE) * 0.05 if cfg is REFERENCE else None
    return w, bias


def _zipf_routing(seed, cfg, tokens):
    """Experts drawn without replacement with probability falling as 1 / rank^ZIPF over a random order of the
    experts (the largest of log p + Gumbel noise), weights positive and normalized to the route scale."""
    g = _gen(seed, 4)
    rank = torch.randperm(cfg.experts, generator=g, device=DEVICE).double() + 1
    noise = -torch.log(-torch.log(torch.rand((tokens, cfg.experts), generator=g, device=DEVICE,
                                             dtype=torch.float64).clamp(1e-300, 1 - 1e-16)))
    ids = torch.topk(noise - ZIPF * torch.log(rank), cfg.top_k, dim=1).indices.to(torch.int32).contiguous()
    raw = torch.rand((tokens, cfg.top_k), generator=g, device=DEVICE) * 0.95 + 0.05
    return ids, (raw / raw.sum(1, keepdim=True) * cfg.route_scale).contiguous()


# -- states --------------------------------------------------------------------------------------------

_context = None


def _ctx():
    """The program's one device context."""
    global _context
    if _context is None:
        _context = _lib.Context(0)
    return _context


class _State:
    """What the program keeps; its device memory goes back when it is dropped."""

    def __init__(self, case):
        self.case, self.ctx, self.kind, self.tokens = case, _ctx(), case["kind"], case["tokens"]
        self.closers = []

    def __del__(self):
        while self.closers:
            self.closers.pop()()


def _p(t):
    return C.c_void_p(t.data_ptr())


def _tile_expert(ctx, arrays, hidden, intermediate, dst):
    ptrs = _lib.MxExpertPtrs(*[arrays[n].data_ptr() for n in TENSORS])
    ctx.lib.tile_expert(ctx._h(), C.byref(ptrs), hidden, intermediate, C.c_void_p(int(dst)), None)


def _bank(state, cfg, seed, count):
    bank = ExpertBank(state.ctx, cfg, count)
    state.closers.append(bank.free)
    for e in range(count):
        _tile_expert(state.ctx, _mxfp4_expert(seed, e, cfg.hidden, cfg.intermediate), cfg.hidden, cfg.intermediate,
                     bank.tiled_ptr(e))
    return bank


def _layer(state, cfg, seed):
    bank = _bank(state, cfg, seed, cfg.experts + 1)
    state.router = _router(seed, cfg)
    w, bias = (t if t is None else _lib.DeviceArray(state.ctx, tuple(t.shape), "float32", t.data_ptr())
               for t in state.router)
    state.layer = MoELayer(state.ctx, cfg, w, bank, bias)
    state.closers.append(state.layer.close)


def _fp8_tiled(state, codes, scales, block):
    rows, width = codes.shape
    blob = state.ctx.malloc(int(state.ctx.lib.cdll.mx_fp8_tiled_bytes(rows, width, block)))
    state.closers.append(lambda: state.ctx.free(blob))
    state.ctx.lib.fp8_tile(state.ctx._h(), _p(codes), _p(scales), rows, width, block, C.c_void_p(blob), None)
    return C.c_void_p(blob)


def prepare(case, seed):
    s = _State(case)
    t = s.tokens
    empty = lambda *shape, dtype=torch.bfloat16: torch.empty(shape, dtype=dtype, device=DEVICE)  # noqa: E731
    if s.kind in ("decode", "prefill"):
        cfg = MODELS[case["model"]]
        _layer(s, cfg, seed)
        s.x, s.y = _normal_bf16(_gen(seed, 5), t, cfg.hidden), empty(t, cfg.hidden)
        if s.kind == "prefill":
            s.workspace = empty(s.layer.workspace_bytes(t), dtype=torch.uint8)
            s.routing = _zipf_routing(seed, cfg, t) if case["routing"] == "zipf" else None
    elif s.kind == "proj128":
        s.weights = [_fp8_tiled(s, *_fp8_weight(seed, i, n, k, 128), 128) for i, (n, k) in enumerate(PROJ128.values())]
        s.x = [_normal_bf16(_gen(seed, 5, i), t, k) for i, (_, k) in enumerate(PROJ128.values())]
        s.y = [empty(t, n) for n, _ in PROJ128.values()]
    elif s.kind == "attn32":
        s.weights = [_fp8_tiled(s, *_fp8_weight(seed, i, n, k, 32), 32) for i, (n, k) in enumerate(ATTN32.values())]
        s.x = [_normal_bf16(_gen(seed, 5, i), t, k) for i, (_, k) in enumerate(ATTN32.values())]
        s.y = [empty(t, n) for n, _ in ATTN32.values()]
        s.wo_a = _fp8_tiled(s, *_fp8_weight(seed, 9, WO_A_GROUPS * WO_A_ROWS, WO_A_WIDTH, 32), 32)
        s.heads = _normal_bf16(_gen(seed, 5, 9), t, WO_A_GROUPS, WO_A_WIDTH)
        s.rounded, s.grouped = torch.empty_like(s.heads), empty(t, WO_A_GROUPS * WO_A_ROWS)
        s.codes = empty(t, WO_A_GROUPS, WO_A_WIDTH, dtype=torch.uint8)
        s.scales = empty(t, WO_A_GROUPS, WO_A_WIDTH // 32, dtype=torch.uint8)
    elif s.kind == "shared":
        h, i = REFERENCE.hidden, REFERENCE.intermediate
        s.weights = [[_fp8_tiled(s, *_fp8_weight(seed, 3 * n + j, *shape, 32), 32)
                      for j, shape in enumerate(((i, h), (i, h), (h, i)))] for n in range(SHARED_LAYERS)]
        s.x = [_normal_bf16(_gen(seed, 5, n), t, h) for n in range(SHARED_LAYERS)]
        s.y = [empty(t, h) for _ in range(SHARED_LAYERS)]
    else:
        cfg = BASELINE
        s.bank = _bank(s, cfg, seed, BF16_LAYERS)
        s.x = [_normal_bf16(_gen(seed, 5, n), t, cfg.hidden) for n in range(BF16_LAYERS)]
        s.y = [empty(t, cfg.hidden) for _ in range(BF16_LAYERS)]
    return s


def run(s):
    lib, h, t = s.ctx.lib, s.ctx._h(), s.tokens
    if s.kind == "decode":
        s.layer.decode_device(s.x.data_ptr(), t, s.y.data_ptr())
        return s.y
    if s.kind == "prefill":
        ids, weights = (r.data_ptr() for r in s.routing) if s.routing else (None, None)
        s.layer.prefill_device(s.x.data_ptr(), t, s.y.data_ptr(), s.workspace.data_ptr(), s.workspace.numel(), ids,
                               weights)
        return s.y
    if s.kind in ("proj128", "attn32"):
        block, layout = (128, PROJ128) if s.kind == "proj128" else (32, ATTN32)
        for w, (n, k), x, y in zip(s.weights, layout.values(), s.x, s.y):
            lib.fp8_projection(h, w, n, k, block, _p(x), t, _p(y), None, None, None, None)
        if s.kind == "proj128":
            return s.y
        lib.kv_round32(h, _p(s.heads), s.heads.numel(), _p(s.rounded), _p(s.codes), _p(s.scales), None)
        lib.fp8_grouped_projection(h, s.wo_a, WO_A_GROUPS, WO_A_ROWS, WO_A_WIDTH, _p(s.codes), _p(s.scales), t,
                                   _p(s.grouped), None, None)
        return s.y + [s.rounded, s.codes, s.scales, s.grouped]
    if s.kind == "shared":
        for w, x, y in zip(s.weights, s.x, s.y):
            lib.fp8_expert_forward(h, *w, REFERENCE.hidden, REFERENCE.intermediate, _p(x), t, REFERENCE.swiglu_limit,
                                   None, _p(y), None, None)
        return s.y
    for n, (x, y) in enumerate(zip(s.x, s.y)):
        lib.expert_forward_bf16(h, C.c_void_p(s.bank.tiled_ptr(n)), BASELINE.hidden, BASELINE.intermediate, _p(x), t,
                                None, None, None, _p(y), None)
    return s.y


# -- work and tolerance --------------------------------------------------------------------------------

def _proj_work(layout, t, block):
    scale = (lambda n, k: -(-n // 128) * (k // 128) * 4) if block == 128 else (lambda n, k: n * k // 1024)
    return (sum(n * k + scale(n, k) + 2 * t * (n + k) for n, k in layout.values()),
            sum(2 * t * n * k for n, k in layout.values()))


def work(case):
    kind, t = case["kind"], case["tokens"]
    if kind in ("decode", "prefill"):
        cfg = MODELS[case["model"]]
        if case.get("routing") == "zipf":
            p = [1.0 / r ** ZIPF for r in range(1, cfg.experts + 1)]
            distinct = sum(1 - (1 - min(1.0, cfg.top_k * q / sum(p))) ** t for q in p)
        else:
            distinct = cfg.experts * (1 - (1 - cfg.top_k / cfg.experts) ** t)
        read = (distinct + 1) * cfg.expert_bytes + 4 * t * cfg.hidden
        flops = 2 * t * (cfg.top_k + 1) * 3 * cfg.hidden * cfg.intermediate
        if case.get("routing") != "zipf":
            read, flops = read + 4 * cfg.experts * cfg.hidden, flops + 2 * t * cfg.experts * cfg.hidden
        return {"bytes": read, "flops": flops}
    if kind == "proj128":
        nbytes, flops = _proj_work(PROJ128, t, 128)
    elif kind == "attn32":
        nbytes, flops = _proj_work(ATTN32, t, 32)
        rows, width, groups = WO_A_ROWS, WO_A_WIDTH, WO_A_GROUPS
        nbytes += groups * (rows * width * 33 // 32 + t * (2 * rows + 5 * width + width // 32))
        flops += 2 * t * groups * rows * width
    elif kind == "shared":
        h, i = REFERENCE.hidden, REFERENCE.intermediate
        nbytes = SHARED_LAYERS * (3 * h * i * 1025 // 1024 + 4 * t * h)
        flops = SHARED_LAYERS * 6 * t * h * i
    else:
        nbytes = BF16_LAYERS * (BASELINE.expert_bytes + 4 * t * BASELINE.hidden)
        flops = BF16_LAYERS * 6 * t * BASELINE.hidden * BASELINE.intermediate
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # BF16 outputs of FP32 sums over exactly converted codes, 1.6e-3 to 2.4e-3 from exact() (the rounding of the
    # result, and a down-input code that moves with a rounding of W1 or W3): three to four times that. The codes
    # and scales of the rounding (attn32) stay the same.
    return {"rel": 7e-3, "max": 0.1}


# -- the same results in 64 bits -----------------------------------------------------------------------

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _e8m0(codes):
    return torch.exp2(codes.double() - 127.0)


def _mxfp4_values(packed, scales):
    table = torch.tensor(_E2M1, dtype=torch.float64, device=DEVICE)
    v = torch.stack((table[(packed & 15).long()], table[(packed >> 4).long()]), dim=-1)
    return (v.view(packed.shape[0], -1, 32) * _e8m0(scales)[..., None]).view(packed.shape[0], -1)


def _fp8_values(codes, scales, block):
    rows, width = codes.shape
    s = scales.double() if block == 128 else _e8m0(scales)
    v = codes.view(torch.float8_e4m3fn).double()
    return (v.view(rows, width // block, block)
            * s.repeat_interleave(block, 0)[:rows, :, None]).view(rows, width)


def _quantized(x, block):
    """(values, E4M3 codes, E8M0 codes or FP32 scales) of BF16-valued x quantized per `block` along the last axis:
    the formats' own definition, in FP32 (amax floored at 1e-4; block 32: the power of two at or above
    amax / 448 as FP32 forms it; block 128: amax / 448)."""
    v = x.float().view(*x.shape[:-1], -1, block)
    amax = v.abs().amax(-1).clamp_min(torch.tensor(1e-4, device=DEVICE))
    if block == 128:
        scale = amax / torch.full_like(amax, 448.0)   # by a tensor: a division, not a product with 1 / 448
        code = scale
    else:
        bits = (amax * torch.tensor(1.0 / 448.0, dtype=torch.float32, device=DEVICE)).view(torch.int32)
        code = ((bits >> 23) & 255) + ((bits & 0x7FFFFF) != 0).int()
        scale = torch.exp2(code.float() - 127.0)
        code = code.to(torch.uint8)
    q = (v / scale[..., None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return (q.double() * scale.double()[..., None]).view(x.shape), q.view(torch.uint8).view(x.shape), code


def _swiglu(gate, up, limit):
    if limit > 0:
        gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
    return gate / (1 + torch.exp(-gate)) * up


def _w4a8_rows(xq, w1, w3, w2, limit, route=None):
    """The quantized expert's output rows: W1 and W3 rounded to BF16, SwiGLU, route weight, BF16, quantized, W2."""
    gate, up = ((xq @ w.T).to(torch.bfloat16).double() for w in (w1, w3))
    h = _swiglu(gate, up, limit)
    if route is not None:
        h = h * route[:, None]
    return _quantized(h.to(torch.bfloat16), 32)[0] @ w2.T


def _exact_layer(case, seed):
    cfg, t = MODELS[case["model"]], case["tokens"]
    x = _normal_bf16(_gen(seed, 5), t, cfg.hidden)
    if case.get("routing") == "zipf":
        ids, weights = _zipf_routing(seed, cfg, t)
    else:
        w, bias = _router(seed, cfg)
        z = x.double() @ w.double().T
        score = torch.sigmoid(z) if cfg.score_func == "sigmoid" else torch.sqrt(torch.nn.functional.softplus(z))
        ids = torch.topk(score if bias is None else score + bias.double(), cfg.top_k, dim=1).indices
        raw = score.gather(1, ids)
        weights = raw / raw.sum(1, keepdim=True) * cfg.route_scale
    xq = _quantized(x, 32)[0]
    y = torch.zeros((t, cfg.hidden), dtype=torch.float64, device=DEVICE)
    for e in range(cfg.experts + 1):
        rows, rank = (torch.arange(t, device=DEVICE), None) if e == cfg.experts else torch.where(ids == e)
        if not rows.numel():
            continue
        a = _mxfp4_expert(seed, e, cfg.hidden, cfg.intermediate)
        w1, w3, w2 = (_mxfp4_values(a[f"{n}_weight"], a[f"{n}_scale"]) for n in ("w1", "w3", "w2"))
        route = None if rank is None else weights[rows, rank].double()
        y.index_add_(0, rows, _w4a8_rows(xq[rows], w1, w3, w2, cfg.swiglu_limit, route))
    return y


def exact(case, seed):
    kind, t = case["kind"], case["tokens"]
    if kind in ("decode", "prefill"):
        return _exact_layer(case, seed)
    if kind in ("proj128", "attn32"):
        block, layout = (128, PROJ128) if kind == "proj128" else (32, ATTN32)
        out = []
        for i, (n, k) in enumerate(layout.values()):
            xq = _quantized(_normal_bf16(_gen(seed, 5, i), t, k), block)[0]
            out.append(xq @ _fp8_values(*_fp8_weight(seed, i, n, k, block), block).T)
        if kind == "proj128":
            return out
        heads = _normal_bf16(_gen(seed, 5, 9), t, WO_A_GROUPS, WO_A_WIDTH)
        xq = _quantized(heads, 32)[0]
        w = _fp8_values(*_fp8_weight(seed, 9, WO_A_GROUPS * WO_A_ROWS, WO_A_WIDTH, 32), 32)
        w = w.view(WO_A_GROUPS, WO_A_ROWS, WO_A_WIDTH)
        return out + [xq, None, None, torch.cat([xq[:, g] @ w[g].T for g in range(WO_A_GROUPS)], dim=1)]
    if kind == "shared":
        h, i = REFERENCE.hidden, REFERENCE.intermediate
        out = []
        for n in range(SHARED_LAYERS):
            xq = _quantized(_normal_bf16(_gen(seed, 5, n), t, h), 32)[0]
            w = [_fp8_values(*_fp8_weight(seed, 3 * n + j, *shape, 32), 32)
                 for j, shape in enumerate(((i, h), (i, h), (h, i)))]
            out.append(_w4a8_rows(xq, *w, REFERENCE.swiglu_limit))
        return out
    out = []
    for n in range(BF16_LAYERS):
        a = _mxfp4_expert(seed, n, BASELINE.hidden, BASELINE.intermediate)
        w1, w3, w2 = (_mxfp4_values(a[f"{p}_weight"], a[f"{p}_scale"]) for p in ("w1", "w3", "w2"))
        x = _normal_bf16(_gen(seed, 5, n), t, BASELINE.hidden).double()
        out.append(_swiglu(x @ w1.T, x @ w3.T, 0.0) @ w2.T)
    return out
