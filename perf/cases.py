"""The MoE feed-forward work a program has this framework do: decode steps,
small batches, prompt chunks and whole prefills through the C ABI's forward
entry points.

A case is one call on a model that sits in HBM.  Its weights are GGUF blocks
of the formats that mixture-of-experts files use, drawn about zero-mean as
trained weights are (block scales |N|, sub-block scales and quants uniform,
mins that centre each sub-block); activations are N(0, 1) as after an
RMSNorm, or a residual stream for the calls that normalise themselves.
Layers are registered (tile-major copies) wherever a program that runs such
batches registers them: from three tokens on, except for the
no-allocation entry point, which takes none.

All calls go to one torch stream, as a program's steps do.
"""
import ctypes as C
import math

import numpy as np
import torch

from orome_amd import _lib
from orome_amd._lib import check, lib
from orome_amd.moe import Context

Q4_K, Q5_K, Q6_K, Q8_0 = "q4_k", "q5_k", "q6_k", "q8_0"
QFMT = {Q4_K: _lib.QFMT_GGUF_Q4_K, Q5_K: _lib.QFMT_GGUF_Q5_K, Q6_K: _lib.QFMT_GGUF_Q6_K, Q8_0: _lib.QFMT_GGUF_Q8_0}
# weights and bytes of one block
BLOCK = {Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), Q8_0: (32, 34)}
EPS = 1e-6
ZIPF_S = 1.1
ROUTER_STD = 0.02


def _case(name, call, T, layers=1, H=2048, E=256, K=8, M=512, down=Q4_K, shared=Q4_K, shared_down=Q4_K, q6k_every=0,
          zipf=False):
    c = dict(call=call, tokens=T, layers=layers, hidden=H, experts=E, top_k=K, intermediate=M, down=down, shared=shared,
             shared_down=shared_down, q6k_every=q6k_every, zipf=zipf)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one user's decode step through consecutive layers, every fourth with
        # a Q6_K down projection
        _case("decode 1, 8 layers", "stack", 1, layers=8, q6k_every=4),
        # the smallest call: one token, one layer, in the layout of Q4_K_M
        # files (Q5_K down, Q8_0 shared expert), with the combine's residual
        # copy and sums of squares that an engine's next norm takes
        _case("decode 1, one layer", "forward", 1, down=Q5_K, shared=Q8_0, shared_down=Q8_0),
        # a few sequences in a serving loop that may not allocate
        _case("decode 5, no allocation", "noalloc", 5),
        # eight sequences decoded together
        _case("decode 8", "layer", 8),
        # a short prompt, or the tokens of many sequences
        _case("prompt 37", "forward", 37),
        # a prompt chunk through consecutive layers (the next layer's norm is
        # computed with a layer's combine)
        _case("prefill 128, 3 layers", "stack", 128, layers=3, q6k_every=3),
        # another width and expert count
        _case("prefill 300, hidden 3072", "forward", 300, H=3072, E=128),
        # the usual prefill chunk, balanced routing
        _case("prefill 512", "forward", 512),
        # the same with skewed routing: a few experts take most tokens
        _case("prefill 512, skewed", "forward", 512, down=Q6_K, zipf=True),
        # a ragged chunk in the layout of Q4_K_M files
        _case("prefill 777, Q5_K and Q8_0", "forward", 777, down=Q5_K, shared=Q8_0, shared_down=Q8_0),
        # a long chunk
        _case("prefill 2048", "layer", 2048),
        # the longest chunk, Q6_K down
        _case("prefill 4096", "layer", 4096, down=Q6_K),
    ]


def draw(rng):
    T = int(round(math.exp(rng.uniform(0.0, math.log(4096.0)))))
    H, E, M = rng.choice([(2048, 256, 512)] * 5 + [(3072, 128, 512), (1024, 384, 256), (4096, 64, 512)])
    call = rng.choice(["forward", "layer", "stack"])
    if T <= 16 and rng.random() < 0.25:
        call = "noalloc"
    layers = rng.randint(2, 4) if call == "stack" and T <= 512 else 1
    K = rng.choice([8, 8, 8, 4, 6] + ([16] if T <= 512 else []))
    shared, shared_down = rng.choice([(Q4_K, Q4_K), (Q4_K, Q4_K), (Q8_0, Q8_0), (Q4_K, Q6_K)])
    return _case(None, call, T, layers=layers, H=H, E=E, K=K, M=M, down=rng.choice([Q4_K, Q4_K, Q5_K, Q6_K]),
                 shared=shared, shared_down=shared_down, q6k_every=rng.choice([0, 2]) if layers > 1 else 0,
                 zipf=rng.random() < 0.2)


# ---------------------------------------------------------------- inputs
def _halves(g, n, std):
    return (torch.randn(n, generator=g, device="cuda").abs_() * std).half()


def _put(blocks, at, h):
    blocks[:, at:at + 2] = h.view(torch.uint8).view(-1, 2)


def _quantised(g, fmt, weights):
    """`weights` weights of a format as blocks of bytes, about zero-mean."""
    per, size = BLOCK[fmt]
    n = weights // per
    # 256 bytes past the end, as the library's own allocator leaves
    buf = torch.randint(0, 256, (n * size + 256,), generator=g, device="cuda", dtype=torch.uint8)
    b = buf[:n * size].view(n, size)
    if fmt in (Q4_K, Q5_K):
        d = _halves(g, n, 2e-3 if fmt == Q4_K else 1e-3)
        _put(b, 0, d)
        _put(b, 2, (d.float() * (7.5 if fmt == Q4_K else 15.5)).half())
        b[:, 8:12] = b[:, 4:8]  # mins = scales
        b[:, 14:16] = b[:, 12:14]
    elif fmt == Q6_K:
        b[:, 192:208] = torch.randint(-64, 64, (n, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
        _put(b, 208, _halves(g, n, 2e-3))
    else:
        _put(b, 0, _halves(g, n, 4e-3))
        b[:, 2:][b[:, 2:] == 128] = 0  # int8 quants in -127..127
    return buf


def _layer_formats(c, l):
    down = Q6_K if c["q6k_every"] and l % c["q6k_every"] == c["q6k_every"] - 1 else c["down"]
    return {"gate": Q4_K, "up": Q4_K, "down": down, "shared_gate": c["shared"], "shared_up": c["shared"],
            "shared_down": c["shared_down"]}


def _layer_weights(c, g, l):
    H, E, M = c["hidden"], c["experts"], c["intermediate"]
    w = {}
    for name, fmt in _layer_formats(c, l).items():
        w[name] = _quantised(g, fmt, (1 if name.startswith("shared") else E) * M * H)
    w["router"] = torch.randn(E, H, generator=g, device="cuda") * ROUTER_STD
    w["shared_router"] = torch.randn(H, generator=g, device="cuda") * ROUTER_STD
    w["norm"] = torch.ones(H, device="cuda")
    w["bias"] = None
    if c["zipf"]:
        p = torch.arange(1, E + 1, device="cuda", dtype=torch.float64) ** -ZIPF_S
        order = torch.randperm(E, generator=g, device="cuda")
        w["bias"] = (p / p.sum()).log()[order].float()
    return w


def _inputs(c, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    T, H = c["tokens"], c["hidden"]
    layers = [_layer_weights(c, g, l) for l in range(c["layers"])]
    x = torch.randn(T, H, generator=g, device="cuda")
    h = torch.randn(T, H, generator=g, device="cuda")
    return layers, x, h


# ------------------------------------------------------------- the program
_STREAM = []


def _stream():
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


class Model:
    """A model in HBM, bound through the C ABI's references, with the context
    that runs it; freed with the object."""

    def __init__(self, c, layers):
        self.weights, self.stream = layers, _stream()
        cfg = _lib.ModelConfig()
        cfg.hidden_dim, cfg.num_layers, cfg.rms_norm_eps = c["hidden"], c["layers"], EPS
        cfg.num_experts, cfg.num_experts_per_tok = c["experts"], c["top_k"]
        cfg.moe_intermediate = cfg.shared_intermediate = c["intermediate"]
        self.cfg = cfg
        n = c["layers"]
        self.elrs, self.caches = (_lib.ExpertLayerRef * n)(), (_lib.LayerTensorCache * n)()
        for l, w in enumerate(layers):
            self._bind(c, l, w)
        self.ctx = None
        if c["call"] != "noalloc":
            self.ctx = Context(cfg, max(c["tokens"], 16))
            if c["tokens"] > 2:
                for l in range(n):
                    check(lib.orome_hip_pack_layer(self.ctx.handle, C.byref(cfg), C.byref(self.elrs[l]),
                                                   C.byref(self.caches[l])), "orome_hip_pack_layer")

    def _bind(self, c, l, w):
        H, E, M = c["hidden"], c["experts"], c["intermediate"]
        f = _layer_formats(c, l)
        # one base address, offsets from it, as in one resident file
        names = ("gate", "up", "down")
        base = min(w[k].data_ptr() for k in names)
        e = self.elrs[l]
        e.buffer = base
        for k in names:
            p = getattr(e, k)
            per, size = BLOCK[f[k]]
            p.offset, p.expert_stride, p.format = w[k].data_ptr() - base, M * H // per * size, QFMT[f[k]]
        t = self.caches[l]

        def ref(dst, tensor, fmt, rows, cols):
            if tensor is not None:
                dst.buffer, dst.offset, dst.format, dst.out_dim, dst.in_dim = tensor.data_ptr(), 0, fmt, rows, cols

        ref(t.post_norm, w["norm"], _lib.QFMT_F32, 1, H)
        ref(t.routing_gate, w["router"], _lib.QFMT_F32, E, H)
        ref(t.shared_gate, w["shared_gate"], QFMT[f["shared_gate"]], M, H)
        ref(t.shared_up, w["shared_up"], QFMT[f["shared_up"]], M, H)
        ref(t.shared_down, w["shared_down"], QFMT[f["shared_down"]], H, M)
        ref(t.shared_expert_gate, w["shared_router"], _lib.QFMT_F32, 1, H)
        ref(t.routing_bias, w["bias"], _lib.QFMT_F32, 1, E)

    def __del__(self):
        if getattr(self, "ctx", None) is not None:
            self.stream.synchronize()
            self.ctx.close()
            self.ctx = None


def prepare(case, seed):
    layers, x, h = _inputs(case, seed)
    torch.cuda.synchronize()
    T, H = case["tokens"], case["hidden"]
    s = {"case": case, "model": Model(case, layers)}
    if case["call"] in ("stack", "layer"):
        s["arrived"] = h  # the residual stream as attention leaves it
        s["h"] = torch.empty_like(h)
    else:
        s["x"], s["h"], s["out"] = x, h, torch.empty_like(h)
        s["residual"] = torch.empty_like(h)
        s["sumsq"] = torch.empty(T, H // 256, device="cuda")
    return s


def run(state):
    c, m = state["case"], state["model"]
    T, K, st = c["tokens"], c["top_k"], m.stream.cuda_stream
    cfg = C.byref(m.cfg)
    if c["call"] in ("stack", "layer"):
        h = state["h"]
        with torch.cuda.stream(m.stream):
            h.copy_(state["arrived"])
        if c["call"] == "stack":
            check(lib.orome_moe_stack_forward(m.ctx.handle, cfg, m.elrs, m.caches, c["layers"], h.data_ptr(), T, K, st))
        else:
            check(lib.orome_moe_layer_forward(m.ctx.handle, cfg, C.byref(m.elrs[0]), C.byref(m.caches[0]),
                                              h.data_ptr(), T, K, st))
        return h
    args = (cfg, C.byref(m.elrs[0]), C.byref(m.caches[0]), state["x"].data_ptr(), state["h"].data_ptr(),
            state["out"].data_ptr(), state["residual"].data_ptr(), state["sumsq"].data_ptr(), T, K, st)
    if c["call"] == "noalloc":
        check(lib.orome_moe_forward_noalloc(*args))
    else:
        check(lib.orome_moe_forward(m.ctx.handle, *args))
    return state["out"], state["residual"], state["sumsq"]


# -------------------------------------------------------------------- work
def _touched(c):
    """Experts that a layer's tokens select, over the router's distribution."""
    T, E, K = c["tokens"], c["experts"], c["top_k"]
    rng = np.random.default_rng(0)
    z = rng.standard_normal((T, E), dtype=np.float32) * np.float32(ROUTER_STD * math.sqrt(c["hidden"]))
    if c["zipf"]:
        p = np.arange(1, E + 1, dtype=np.float64) ** -ZIPF_S
        z += np.log(p / p.sum()).astype(np.float32)
    return int(np.unique(np.argpartition(-z, K - 1, axis=1)[:, :K]).size)


def work(case):
    T, H, E, K, M = (case[k] for k in ("tokens", "hidden", "experts", "top_k", "intermediate"))
    u = _touched(case)
    bytes_ = flops = 0
    for l in range(case["layers"]):
        for name, fmt in _layer_formats(case, l).items():
            per, size = BLOCK[fmt]
            bytes_ += (1 if name.startswith("shared") else u) * (M * H // per * size)
        bytes_ += (E + 1) * H * 4
        flops += 2 * T * (E + 1) * H + 6 * M * H * T * (K + 1)
    if case["call"] in ("stack", "layer"):
        bytes_ += 2 * T * H * 4
    else:
        bytes_ += 4 * T * H * 4 + T * H // 256 * 4
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Activations and weights reach the products as fp16, sums are fp32: one
    layer is 4e-4 to 8e-4 from 64 bits.  Through several layers a token whose
    K-th and next expert are nearly tied may take the other one."""
    return {"rel": 3e-3 if case["layers"] == 1 else 3e-2}


# ------------------------------------------------------------- in 64 bits
def _f64(halves):
    return halves.contiguous().view(torch.float16).double()


def _decoded(fmt, blocks):
    """Blocks of bytes [..., size] -> weights [..., per] in 64 bits.  Q4_K and
    Q5_K scales are packed as the engine packs them: sub-blocks 4..7 take
    their low four bits from byte 8 + j of the scale bytes (scales 4|5, 6|7),
    then 10 + j (mins), their high two from the bytes of sub-blocks 0..3."""
    b = blocks
    if fmt == Q8_0:
        return _f64(b[..., 0:2]) * b[..., 2:].contiguous().view(torch.int8).double()
    if fmt == Q6_K:
        d, sc = _f64(b[..., 208:210]), b[..., 192:208].contiguous().view(torch.int8).double()
        out = []
        for half in range(2):
            ql, qh = b[..., 64 * half:64 * half + 64], b[..., 128 + 32 * half:160 + 32 * half]
            for part in range(4):
                low = ql[..., 32 * (part & 1):32 * (part & 1) + 32]
                low = low >> 4 if part >= 2 else low & 15
                q = (low | (((qh >> (2 * part)) & 3) << 4)).double() - 32.0
                s = sc[..., 8 * half + 2 * part:8 * half + 2 * part + 2].repeat_interleave(16, -1)
                out.append(d * s * q)
        return torch.cat(out, -1)
    d, dmin, s = _f64(b[..., 0:2]), _f64(b[..., 2:4]), b[..., 4:16]
    sc = [s[..., j] & 63 for j in range(4)] + [(s[..., 8 + j // 2] >> (4 * (j & 1)) & 15) | (s[..., j] >> 6) << 4 for j in range(4)]
    mn = [s[..., 4 + j] & 63 for j in range(4)] + [(s[..., 10 + j // 2] >> (4 * (j & 1)) & 15) | (s[..., 4 + j] >> 6) << 4 for j in range(4)]
    out = []
    for j in range(8):
        g = j // 2
        at = (16 if fmt == Q4_K else 48) + 32 * g
        q = b[..., at:at + 32]
        q = q >> 4 if j & 1 else q & 15
        if fmt == Q5_K:
            q = q | ((b[..., 16:48] >> j) & 1) << 4
        out.append(d * sc[j].double()[..., None] * q.double() - dmin * mn[j].double()[..., None])
    return torch.cat(out, -1)


def _matrix(fmt, buf, e, rows, cols):
    per, size = BLOCK[fmt]
    n = rows * cols // per * size
    return _decoded(fmt, buf[e * n:(e + 1) * n].view(rows, cols // per, size)).reshape(rows, cols)


def _block(c, l, w, x):
    """The MoE block of normalised inputs, without the residual."""
    H, E, K, M = c["hidden"], c["experts"], c["top_k"], c["intermediate"]
    f = _layer_formats(c, l)

    def expert(xs, e, names):
        gate, up = (xs @ _matrix(f[k], w[k], e, M, H).T for k in names[:2])
        return (gate * torch.sigmoid(gate) * up) @ _matrix(f[names[2]], w[names[2]], e, H, M).T

    z = x @ w["router"].double().T
    if w["bias"] is not None:
        z = z + w["bias"].double()
    top, idx = z.topk(K, dim=1)
    p = torch.softmax(top, 1)
    out = torch.sigmoid(x @ w["shared_router"].double())[:, None] * expert(x, 0, ("shared_gate", "shared_up", "shared_down"))
    for e in idx.unique().tolist():
        t, k = (idx == e).nonzero(as_tuple=True)
        out[t] += p[t, k][:, None] * expert(x[t], e, ("gate", "up", "down"))
    return out


def exact(case, seed):
    layers, x, h = _inputs(case, seed)
    x, h = x.double(), h.double()
    if case["call"] in ("stack", "layer"):
        for l, w in enumerate(layers):
            n = h * torch.rsqrt((h * h).mean(1, keepdim=True) + EPS) * w["norm"].double()
            h = h + _block(case, l, w, n)
        return h
    out = h + _block(case, 0, layers[0], x)
    T, H = out.shape
    return out, out, (out * out).view(T, H // 256, 256).sum(2)
