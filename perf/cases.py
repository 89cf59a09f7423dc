"""The work this library is timed on: matrix products over quantized and float weights, as a model's
host program issues them through the C API (one op, a fused op, or a recorded plan).

A case is one of four kinds:

  product   one MUL_MAT (one weight) or MUL_MAT_MULTI (several weights sharing x) through op_execute:
            dtype, rows ("12288" or "4096+1024+1024"), K, tokens
  layers    a plan over the products of `layers` transformer layers: q/k/v, o, gate/up in Q4_K and
            down in Q6_K (hidden, kv, ffn), tokens
  experts   a plan over the MUL_MAT_IDs of `layers` mixture-of-experts layers: gate and up in Q4_K,
            down in Q6_K (experts, used, hidden, ffn), tokens
  slices    one MUL_MAT over several slices of float weights, each read by `share` slices of x:
            dtype, rows, K, tokens, count, share

The inputs are drawn on the GPU from the seed: weights ~ N(0, 0.02) rounded to the block formats,
activations ~ N(0, 1) with one channel in 64 eight times larger (the outlier channels of real
activations), expert choices distinct per token.
"""
import ctypes
import math

import numpy as np
import torch

import scrapgpulibrary_amd as sg

DTYPES = {"q4_0": sg.Q4_0, "q8_0": sg.Q8_0, "q4_k": sg.Q4_K, "q6_k": sg.Q6_K, "f16": sg.F16, "bf16": sg.BF16, "f32": sg.F32}
BYTES_PER_WEIGHT = {"q4_0": 18 / 32, "q8_0": 34 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256, "f16": 2.0, "bf16": 2.0, "f32": 4.0}
QUANT = ("q4_0", "q8_0", "q4_k", "q6_k")


# ---- the cases ----------------------------------------------------------------------------------


def listed():
    return [
        # one small product issued by itself: the standalone matmul example (latency and launch cost)
        {"name": "single_q4_0", "kind": "product", "dtype": "q4_0", "rows": "4096", "K": 4096, "tokens": 1},
        # generation at batch 1: the products of 8 of the 36 layers of a Qwen3-8B Q4_K_M token
        {"name": "decode_layers", "kind": "layers", "layers": 8, "hidden": 4096, "kv": 1024, "ffn": 12288, "tokens": 1},
        # generation at batch 1: the output head
        {"name": "lm_head_decode", "kind": "product", "dtype": "q6_k", "rows": "151936", "K": 4096, "tokens": 1},
        # serving 8 sequences at once: the Llama-7B MLP's down projection
        {"name": "batch8_q8_0", "kind": "product", "dtype": "q8_0", "rows": "4096", "K": 11008, "tokens": 8},
        # a short prompt of odd length
        {"name": "prompt37_q4_k", "kind": "product", "dtype": "q4_k", "rows": "12288", "K": 4096, "tokens": 37},
        # one layer of a prompt processed 512 tokens at a time
        {"name": "prefill_layer", "kind": "layers", "layers": 1, "hidden": 4096, "kv": 1024, "ffn": 12288, "tokens": 512},
        # a long prompt in one call (the largest amount of arithmetic)
        {"name": "prefill2048_q4_k", "kind": "product", "dtype": "q4_k", "rows": "12288", "K": 4096, "tokens": 2048},
        # mixture of experts, generation at batch 1: 8 layers of Qwen3-30B-A3B-shaped experts
        {"name": "moe_decode", "kind": "experts", "layers": 8, "experts": 128, "used": 8, "hidden": 2048, "ffn": 768, "tokens": 1},
        # mixture of experts, a 512-token prompt through one layer
        {"name": "moe_prefill", "kind": "experts", "layers": 1, "experts": 128, "used": 8, "hidden": 2048, "ffn": 768, "tokens": 512},
        # an unquantized model serving 8 sequences: gate of the MLP
        {"name": "batch8_f16", "kind": "product", "dtype": "f16", "rows": "12288", "K": 4096, "tokens": 8},
        # an unquantized model's prompt
        {"name": "prefill512_bf16", "kind": "product", "dtype": "bf16", "rows": "12288", "K": 4096, "tokens": 512},
        # the expert router of a prompt: float32 weights, few rows
        {"name": "router512_f32", "kind": "product", "dtype": "f32", "rows": "128", "K": 2048, "tokens": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes spread over the range (logarithmically), odd ones among them."""
    while True:
        kind = rng.choice(["product"] * 8 + ["layers", "layers", "experts", "experts", "slices"])
        if kind == "product":
            dtype = rng.choice(["q4_0", "q8_0", "q4_k", "q4_k", "q6_k", "f16", "bf16", "f32"])
            tokens = rng.choice([1, rng.randint(2, 8), _log_int(rng, 9, 128), _log_int(rng, 129, 2048)])
            if dtype == "f32":  # float32 rows are small tensors: routers and the like
                c = {"rows": str(_log_int(rng, 8, 512)), "K": 8 * _log_int(rng, 64, 1024)}
            else:
                step = 256 if dtype in ("q4_k", "q6_k") else 32 if dtype in QUANT else rng.choice([128, 128, 8])
                count = rng.choice([1, 1, 1, 2, 3])
                c = {"rows": "+".join(str(_log_int(rng, 64, 28672)) for _ in range(count)), "K": step * max(1, _log_int(rng, 512, 14336) // step)}
            c = {"kind": kind, "dtype": dtype, **c, "tokens": tokens}
        elif kind == "layers":
            c = {"kind": kind, "layers": rng.randint(1, 8), "hidden": 256 * rng.randint(4, 20), "kv": 128 * rng.randint(2, 16), "ffn": 256 * rng.randint(8, 56),
                 "tokens": rng.choice([1, 1, rng.randint(2, 8), _log_int(rng, 9, 512)])}
        elif kind == "experts":
            experts = rng.choice([8, 16, 32, 64, 128])
            c = {"kind": kind, "layers": rng.randint(1, 8), "experts": experts, "used": rng.randint(2, min(8, experts)), "hidden": 256 * rng.randint(4, 16),
                 "ffn": 256 * rng.randint(2, 12), "tokens": rng.choice([1, rng.randint(2, 8), _log_int(rng, 9, 512)])}
        else:
            share = rng.choice([1, 2, 4, 8])
            c = {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "rows": _log_int(rng, 64, 8192), "K": rng.choice([64, 128, 256]), "tokens": rng.choice([1, rng.randint(2, 8), _log_int(rng, 9, 256)]),
                 "count": rng.randint(1, 8), "share": share}
        big = _weights(c) * 4  # (rounding weights to blocks takes a few float copies of them)
        w, most = work(c), work(listed()[6])
        plain = c.get("dtype") == "f32" or (c.get("dtype") in ("f16", "bf16") and c["K"] % 128 != 0)  # no 16-bit matrix units
        if w["flops"] * (20 if plain else 1) <= most["flops"] and w["bytes"] <= 5.2e8 and big <= 1.2e10:
            return c


def _weights(c):
    """The number of weights that preparing the case makes."""
    if c["kind"] == "product":
        return sum(_rows(c)) * c["K"]
    if c["kind"] == "layers":
        return c["layers"] * sum(m * k for _, m, k in _layer(c))
    if c["kind"] == "experts":
        return 3 * c["layers"] * c["experts"] * c["hidden"] * c["ffn"]
    return c["count"] * c["rows"] * c["K"]


def _rows(c):
    return [int(m) for m in c["rows"].split("+")]


def _layer(c):
    """(dtype, rows, K) of a layer's products: q, k, v; o; gate, up; down."""
    h, kv, f = c["hidden"], c["kv"], c["ffn"]
    return [("q4_k", h, h), ("q4_k", kv, h), ("q4_k", kv, h), ("q4_k", h, h), ("q4_k", f, h), ("q4_k", f, h), ("q6_k", h, f)]


def work(case):
    """Bytes (each weight that the call reads, x and y once) and operations of one pass."""
    n = case["tokens"]
    if case["kind"] == "product":
        m, k = sum(_rows(case)), case["K"]
        return {"bytes": m * k * BYTES_PER_WEIGHT[case["dtype"]] + 4 * n * (k + m), "flops": 2 * m * k * n}
    if case["kind"] == "layers":
        h, f, L = case["hidden"], case["ffn"], case["layers"]
        mats = _layer(case)
        byts = sum(m * k * BYTES_PER_WEIGHT[d] + 4 * n * m for d, m, k in mats) + 4 * n * (3 * h + f)
        return {"bytes": L * byts, "flops": L * 2 * n * sum(m * k for _, m, k in mats)}
    if case["kind"] == "experts":
        e, u, h, f, L = (case[k] for k in ("experts", "used", "hidden", "ffn", "layers"))
        hit = e * (1 - (1 - u / e) ** n)  # experts that some token chose, on average
        byts = hit * h * f * (2 * BYTES_PER_WEIGHT["q4_k"] + BYTES_PER_WEIGHT["q6_k"]) + 4 * n * (h + 3 * u * f + u * h + u)
        return {"bytes": L * byts, "flops": L * 2 * n * u * 3 * h * f}
    m, k, s = case["rows"], case["K"], case["count"]
    return {"bytes": s * m * k * BYTES_PER_WEIGHT[case["dtype"]] + 4 * n * s * case["share"] * (k + m), "flops": 2 * m * k * n * s * case["share"]}


def tolerance(case):
    """About four times the largest error of the path against 64-bit products of the same inputs:
    float32-level sums up to 8 tokens and for float32 weights (9e-7 and less), 16-bit operands above
    (Q4_K weights rounded to f16 with their offsets 1.1e-3, bf16 operands 1.8e-3, the others 4e-4)."""
    if case["tokens"] <= 8 or case.get("dtype") == "f32":
        return {"rel": 4e-6, "max": 4e-5}
    if case["kind"] == "experts" and case["tokens"] * case["used"] < 4 * case["experts"]:
        return {"rel": 4e-6, "max": 4e-5}
    return {"rel": 8e-3 if case.get("dtype") == "bf16" else 4e-3}


# ---- weights and activations --------------------------------------------------------------------


def _gen(seed, part):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + part * 7919 + 17) & 0x7FFFFFFFFFFF)


def _halves(v):
    """float16 little-endian bytes, a trailing axis of 2."""
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(*v.shape, 2)


def _round_to(dtype, w):
    """Rounds float32 weights [n, K] to `dtype`: (natural bytes [n, row bytes] as uint8, a function
    giving the float64 values that those bytes hold)."""
    n, K = w.shape
    if dtype in ("f16", "bf16", "f32"):
        v = w.to({"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dtype])
        return v.contiguous().view(torch.uint8).reshape(n, -1), lambda: v.double()
    if dtype == "q4_0":
        b = w.reshape(n, K // 32, 32)
        top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        d = (top / -8).half().float()
        q = torch.where(d == 0, torch.zeros_like(b), b / torch.where(d == 0, torch.ones_like(d), d)).round().add_(8).clamp_(0, 15).to(torch.uint8)
        raw = torch.cat([_halves(d[..., 0]), q[..., :16] | (q[..., 16:] << 4)], -1)
        return raw.reshape(n, -1), lambda: (d.double() * (q.double() - 8)).reshape(n, K)
    if dtype == "q8_0":
        b = w.reshape(n, K // 32, 32)
        d = (b.abs().amax(-1, keepdim=True) / 127).half().float()
        q = torch.where(d == 0, torch.zeros_like(b), b / torch.where(d == 0, torch.ones_like(d), d)).round().clamp_(-127, 127).to(torch.int8)
        raw = torch.cat([_halves(d[..., 0]), q.view(torch.uint8)], -1)
        return raw.reshape(n, -1), lambda: (d.double() * q.double()).reshape(n, K)
    if dtype == "q4_k":  # per 256: d, dmin, 8 six-bit (scale, min) pairs, 8 x 32 four-bit codes
        b = w.reshape(n, K // 256, 8, 32)
        low = (-b.amin(-1)).clamp_(min=0)
        span = (b.amax(-1) + low) / 15
        d = (span.amax(-1, keepdim=True) / 63).half().float()
        dm = (low.amax(-1, keepdim=True) / 63).half().float()
        one = torch.ones_like(d)
        sc = (span / torch.where(d == 0, one, d)).round().clamp_(0, 63)
        mn = (low / torch.where(dm == 0, one, dm)).round().clamp_(0, 63)
        s, o = (d * sc)[..., None], (dm * mn)[..., None]
        q = torch.where(s == 0, torch.zeros_like(b), (b + o) / torch.where(s == 0, torch.ones_like(s), s)).round().clamp_(0, 15).to(torch.uint8)
        si, mi = sc.to(torch.uint8), mn.to(torch.uint8)
        heads = torch.cat([si[..., :4] | ((si[..., 4:] >> 4) << 6), mi[..., :4] | ((mi[..., 4:] >> 4) << 6), (si[..., 4:] & 15) | ((mi[..., 4:] & 15) << 4)], -1)
        codes = (q[..., 0::2, :] | (q[..., 1::2, :] << 4)).reshape(n, K // 256, 128)
        raw = torch.cat([_halves(d[..., 0]), _halves(dm[..., 0]), heads, codes], -1)
        return raw.reshape(n, -1), lambda: ((d.double() * sc.double())[..., None] * q.double() - (dm.double() * mn.double())[..., None]).reshape(n, K)
    # q6_k: per 256: 128 bytes of low nibbles, 64 bytes of high bit pairs, 16 int8 scales, d
    b = w.reshape(n, K // 256, 16, 16)
    span = b.abs().amax(-1) / 31
    d = (span.amax(-1, keepdim=True) / 127).half().float()
    sc = (span / torch.where(d == 0, torch.ones_like(d), d)).round().clamp_(0, 127)
    s = (d * sc)[..., None]
    q = torch.where(s == 0, torch.zeros_like(b), b / torch.where(s == 0, torch.ones_like(s), s)).round().clamp_(-32, 31).add_(32).to(torch.uint8)
    c = q.reshape(n, K // 256, 2, 4, 32)
    lo, hi = c & 15, c >> 4
    ql = torch.cat([lo[..., 0, :] | (lo[..., 2, :] << 4), lo[..., 1, :] | (lo[..., 3, :] << 4)], -1).reshape(n, K // 256, 128)
    qh = (hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)).reshape(n, K // 256, 64)
    raw = torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _halves(d[..., 0])], -1)
    return raw.reshape(n, -1), lambda: ((d.double() * sc.double())[..., None] * (q.double() - 32)).reshape(n, K)


def _weight(dtype, n, K, seed, part):
    return _round_to(dtype, torch.randn(n, K, generator=_gen(seed, part), device="cuda").mul_(0.02))


def _acts(n, K, seed, part):
    x = torch.randn(n, K, generator=_gen(seed, part), device="cuda")
    x[:, 5::64] *= 8
    return x


def _choices(tokens, experts, used, seed, part):
    """`used` distinct experts per token, int32 [tokens, used]."""
    return torch.rand(tokens, experts, generator=_gen(seed, part), device="cuda").topk(used, -1).indices.to(torch.int32)


# ---- the host program's objects -----------------------------------------------------------------

_gpu = None


def _device():
    """The one device and stream of the program."""
    global _gpu
    if _gpu is None:
        dev = sg.Device(0)
        _gpu = (dev, dev.stream())
    return _gpu


class _Mem:
    """A device buffer that is freed with its last user, and its memory as a torch tensor (a view)."""

    def __init__(self, size):
        self.buf = _device()[0].alloc(size)

    def __del__(self):
        self.buf.free()

    def tensor(self, *shape):
        # a buffer object holds its vtable, its device, its address and its size, in this order
        _, _, at, size = (ctypes.c_uint64 * 4).from_address(self.buf.handle)
        if size != self.buf.size:
            raise RuntimeError("buffer objects are laid out in another way")

        class View:
            __cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (at, False), "version": 2}
            mem = self

        return torch.as_tensor(View(), device="cuda")


class _Plan:
    def __init__(self, ops):
        nodes = (sg.PlanNode * len(ops))(*[sg.PlanNode(ctypes.sizeof(sg.PlanNode), op, 1) for op, _ in ops])
        desc = sg.PlanDesc(ctypes.sizeof(sg.PlanDesc), nodes, len(ops))
        self.handle = ctypes.c_void_p()
        sg.check(sg.lib().scrapgpu_plan_build(_device()[0].handle, ctypes.byref(desc), ctypes.byref(self.handle)), "plan_build")

    def __del__(self):
        sg.lib().scrapgpu_plan_free(self.handle)


class _State:
    """What the program keeps: tensors in device memory, the op or plan, the outputs."""

    def __init__(self):
        self.plan, self.op, self.outs, self.keep = None, None, [], []

    def put(self, dtype, ne, host, layout=sg.NATURAL):
        mem = _Mem(host.nbytes)
        self.keep.append(mem)
        t = sg.tdesc(dtype, ne, mem.buf, layout=layout)
        _device()[1].upload(t, host)
        return t

    def weight(self, dtype, n, K, slices, seed, part):
        raw = _weight(dtype, n * slices, K, seed, part)[0].cpu().numpy().reshape(-1)
        return self.put(DTYPES[dtype], (K, n, slices), raw, sg.R32 if dtype in QUANT else sg.NATURAL)

    def acts(self, x, ne):
        return self.put(sg.F32, ne, x.cpu().numpy())

    def out(self, *ne):
        mem = _Mem(4 * int(np.prod(ne)))
        self.keep.append(mem)
        self.outs.append(mem.tensor(*reversed(ne)))
        return sg.tdesc(sg.F32, ne, mem.buf)


def prepare(case, seed):
    s, n = _State(), case["tokens"]
    if case["kind"] == "product":
        K, dtype = case["K"], case["dtype"]
        ws = [s.weight(dtype, m, K, 1, seed, j) for j, m in enumerate(_rows(case))]
        x = s.acts(_acts(n, K, seed, 100), (K, n))
        ys = [s.out(m, n) for m in _rows(case)]
        s.op, keep = sg.mul_mat_op(ws[0], x, ys[0]) if len(ws) == 1 else sg.multi_op(ws, x, ys)
        s.keep.append(keep)
    elif case["kind"] == "layers":
        ops = []
        for j in range(case["layers"]):
            w = [s.weight(d, m, k, 1, seed, 10 * j + i) for i, (d, m, k) in enumerate(_layer(case))]
            xs = [s.acts(_acts(n, k, seed, 1000 + 10 * j + i), (k, n)) for i, k in enumerate((case["hidden"], case["hidden"], case["hidden"], case["ffn"]))]
            y = [s.out(m, n) for _, m, _ in _layer(case)]
            ops += [sg.multi_op(w[:3], xs[0], y[:3]), sg.mul_mat_op(w[3], xs[1], y[3]), sg.multi_op(w[4:6], xs[2], y[4:6]), sg.mul_mat_op(w[6], xs[3], y[6])]
        s.keep.append(ops)
        s.plan = _Plan(ops)
    elif case["kind"] == "experts":
        e, u, h, f = (case[k] for k in ("experts", "used", "hidden", "ffn"))
        ops = []
        for j in range(case["layers"]):
            gate, up = (s.weight("q4_k", f, h, e, seed, 10 * j + i) for i in (0, 1))
            down = s.weight("q6_k", h, f, e, seed, 10 * j + 2)
            x, hid = s.acts(_acts(n, h, seed, 1000 + 10 * j), (h, 1, n)), s.acts(_acts(n * u, f, seed, 1001 + 10 * j), (f, u, n))
            ids = s.put(sg.I32, (u, n), _choices(n, e, u, seed, 2000 + j).cpu().numpy())
            ops += [sg.mul_mat_id_op(gate, x, ids, s.out(f, u, n), u), sg.mul_mat_id_op(up, x, ids, s.out(f, u, n), u), sg.mul_mat_id_op(down, hid, ids, s.out(h, u, n), u)]
        s.keep.append(ops)
        s.plan = _Plan(ops)
    else:
        K, m, c, r = case["K"], case["rows"], case["count"], case["share"]
        w = s.weight(case["dtype"], m, K, c, seed, 0)
        x = s.acts(_acts(n * c * r, K, seed, 100), (K, n, c * r))
        s.op, keep = sg.mul_mat_op(w, x, s.out(m, n, c * r), allow_broadcast=1)
        s.keep.append(keep)
    return s


def run(state):
    stream = _device()[1]
    if state.plan is not None:
        sg.check(sg.lib().scrapgpu_plan_execute(stream.handle, state.plan.handle), "plan_execute")
    else:
        stream.execute(state.op)
    return state.outs


# ---- the same in 64 bits ------------------------------------------------------------------------


def exact(case, seed):
    n = case["tokens"]

    def times(dtype, m, K, part, x):
        values = _weight(dtype, m, K, seed, part)[1]()
        return x.double() @ values.t()

    if case["kind"] == "product":
        x = _acts(n, case["K"], seed, 100)
        return [times(case["dtype"], m, case["K"], j, x) for j, m in enumerate(_rows(case))]
    if case["kind"] == "layers":
        outs = []
        for j in range(case["layers"]):
            xs = [_acts(n, k, seed, 1000 + 10 * j + i) for i, k in enumerate((case["hidden"], case["hidden"], case["hidden"], case["ffn"]))]
            outs += [times(d, m, k, 10 * j + i, xs[(0, 0, 0, 1, 2, 2, 3)[i]]) for i, (d, m, k) in enumerate(_layer(case))]
        return outs
    if case["kind"] == "experts":
        e, u, h, f = (case[k] for k in ("experts", "used", "hidden", "ffn"))
        outs = []
        for j in range(case["layers"]):
            x, hid = _acts(n, h, seed, 1000 + 10 * j), _acts(n * u, f, seed, 1001 + 10 * j)
            ids = _choices(n, e, u, seed, 2000 + j).reshape(-1).long()
            for i, (d, m, k) in enumerate((("q4_k", f, h), ("q4_k", f, h), ("q6_k", h, f))):
                values = _weight(d, m * e, k, seed, 10 * j + i)[1]().reshape(e, m, k)
                src = (x.repeat_interleave(u, 0) if i < 2 else hid).double()
                y = torch.empty(n * u, m, dtype=torch.float64, device="cuda")
                for ex in ids.unique().tolist():
                    at = (ids == ex).nonzero()[:, 0]
                    y[at] = src[at] @ values[ex].t()
                outs.append(y.reshape(n, u, m))
        return outs
    K, m, c, r = case["K"], case["rows"], case["count"], case["share"]
    values = _weight(case["dtype"], m * c, K, seed, 0)[1]().reshape(c, m, K)
    x = _acts(n * c * r, K, seed, 100).double().reshape(c * r, n, K)
    return [torch.stack([x[i] @ values[i // r].t() for i in range(c * r)])]
