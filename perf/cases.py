"""Performance cases of the quantized-weight matmul path, through the entry points a model calls.

A projection is a `PackedLinear` over GGUF blocks, an MLX affine pack (with or without the 128-point
Walsh-Hadamard rotation of its input) or an EXL3 trellis tensor; a MoE block is `moe.swiglu` /
`moe.swiglu_affine`. A case multiplies a bank of projections of one shape, each with weights and
activations of its own, as a model's layers do (so the weights of a decode step come from HBM, not
from a cache that still holds the last call's).

Calls of up to 16 rows (decode, and the verification of drafted tokens) are captured once in a HIP
graph that a pass replays, which is how a serving loop runs them; `graph` False and longer prompts
call the Python entry points directly.
"""
import math
import os
import re

import torch

from ishizuki_amd import exl3, ggml, gguf, moe
from ishizuki_amd.linear import PackedLinear

DEV = "cuda"
TYPES = {"q4_0": ggml.Q4_0, "q4_k": ggml.Q4_K, "q6_k": ggml.Q6_K, "iq2_xs": ggml.IQ2_XS}
BLOCK = {"q4_0": (32, 18), "q4_k": (256, 144), "q6_k": (256, 210), "iq2_xs": (256, 74)}
SCALES_AT = {"q4_0": (0,), "q4_k": (0, 2), "q6_k": (208,), "iq2_xs": (0,)}  # fp16 fields of a block
# super-scale of each format for weights of a trained layer's size (a few hundredths)
SIZE = {"q4_0": 0.01, "q4_k": 2e-4, "q6_k": 5e-5, "iq2_xs": 5e-4}
DTYPE = {"fp16": torch.float16, "bf16": torch.bfloat16}
GROUP = 64      # MLX affine group
HAD = 128       # Hadamard block


def _linear(name, fmt, n, k, rows, dtype="fp16", bank=1, graph=True, down=False):
    return {"name": name, "kind": "linear", "fmt": fmt, "n": n, "k": k, "rows": rows, "dtype": dtype, "bank": bank,
            "graph": graph, "down": down}


def _moe(name, fmt, tokens, e, h, i, topk, dtype="fp16", shared=False, graph=True):
    return {"name": name, "kind": "moe", "fmt": fmt, "tokens": tokens, "e": e, "h": h, "i": i, "topk": topk,
            "dtype": dtype, "shared": shared, "graph": graph}


def listed():
    return [
        # one small projection of one token, called from Python: launch and host latency
        _linear("q4_0_4096_decode_eager", "q4_0", 4096, 4096, 1, graph=False),
        # a decode step's 2-bit rotated projections (17408 x 5120, the 27B ternary model's MLP)
        _linear("affine2_rot_decode", "affine2_rot", 17408, 5120, 1, bank=8),
        # a decode step through a 27B MLP (gate / up 25600 x 5120, down 5120 x 25600), bf16 model
        _linear("q4_k_mlp_decode_bf16", "q4_k", 25600, 5120, 1, "bf16", bank=2, down=True),
        # a decode step's EXL3 2-bit projections
        _linear("exl3_2_decode", "exl3_4", 17408, 5120, 1, bank=8),
        # eight drafted tokens verified against i-quant MLP projections
        _linear("iq2_xs_mlp_verify8", "iq2_xs", 25600, 5120, 8, bank=3, down=True),
        # four drafted tokens against the 2-bit rotated pack
        _linear("affine2_rot_verify4", "affine2_rot", 17408, 5120, 4, bank=8),
        # sixteen rows (a batch of sequences) against 6-bit projections, bf16 model
        _linear("q6_k_batch16_bf16", "q6_k", 17408, 5120, 16, "bf16", bank=3),
        # a prompt of 512 tokens through a GGUF projection, bf16 model
        _linear("q4_k_prefill512_bf16", "q4_k", 17408, 5120, 512, "bf16", graph=False),
        # a ragged prompt through the 2-bit rotated pack
        _linear("affine2_rot_prefill300", "affine2_rot", 17408, 5120, 300, graph=False),
        # a short prompt through an EXL3 projection
        _linear("exl3_2_prefill128", "exl3_4", 17408, 5120, 128, graph=False),
        # eight tokens through a 128-expert MoE layer (Q4_K experts, top 8)
        _moe("moe_q4_k_verify8", "q4_k", 8, 128, 2048, 768, 8),
        # a prompt of 512 tokens through the MoE layer with 4-bit affine experts, bf16 model
        _moe("moe_affine4_prefill512_bf16", "affine4", 512, 128, 2048, 768, 8, "bf16", graph=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    dtype = rng.choice(["fp16", "bf16"])
    if rng.random() < 0.2:
        t = _log(rng, 1, 512)
        h, i = 256 * rng.randint(4, 10), 256 * rng.randint(2, 5)
        c = _moe("", rng.choice(["q4_k", "affine4"]), t, rng.choice([32, 64, 128]), h, i, rng.choice([4, 6, 8]),
                 dtype, rng.random() < 0.5, graph=t <= 16)
    else:
        fmt = rng.choice(["q4_0", "q4_k", "q6_k", "iq2_xs", "affine2_rot", "affine4", "exl3_4", "exl3_8"])
        rows = rng.choice([1, rng.randint(2, 16), _log(rng, 17, 512)])
        n, k = _log(rng, 1024, 17408), 256 * _log(rng, 4, 68)
        if fmt.startswith("exl3"):
            n = max(128, n // 128 * 128)
        if fmt == "q4_0":
            k += rng.choice([0, 64, 128])
        # the affine pack without a rotation takes bf16 through an allocation, which a graph does not hold
        graph = rows <= 16 and not (fmt == "affine4" and dtype == "bf16")
        while rows * n * k > 512 * 17408 * 5120:
            n = max(128, n // 256 * 128)
        bank = max(1, min(8, 45_000_000 // (n * k))) if graph else 1
        c = _linear("", fmt, n, k, rows, dtype, bank, graph)
    del c["name"]
    return c


# ------------------------------------------------------------------ weights
def _bytes_per_row(fmt, k):
    if fmt in BLOCK:
        return k // BLOCK[fmt][0] * BLOCK[fmt][1]
    if fmt.startswith("exl3"):
        return k * int(fmt[5:]) // 16
    return k * int(fmt[6]) // 8 + k // GROUP * 4


def _ggml(fmt, n, k, gen):
    bs, ts = BLOCK[fmt]
    nb = n * (k // bs)
    blk = torch.randint(0, 256, (nb, ts), dtype=torch.uint8, device=DEV, generator=gen)
    for o in SCALES_AT[fmt]:
        d = torch.randn(nb, device=DEV, generator=gen).abs().mul_(SIZE[fmt]).half()
        blk[:, o:o + 2] = d.view(torch.uint8).view(nb, 2)
    return blk.view(-1)


def _affine(bits, n, k, gen, rows=None):
    """Codes, scales and biases [*rows, n, ...] of an MLX pack; 2 bits: ternary codes 0, 1, 2."""
    shape = (rows or ()) + (n,)
    s = torch.randn(shape + (k // GROUP,), device=DEV, generator=gen).abs().mul_(0.05 if bits == 2 else 0.01).half()
    if bits == 2:
        u = torch.rand(shape + (k // 16, 16), device=DEV, generator=gen)
        q = (u > 0.3).int() + (u > 0.7).int()
        codes = torch.zeros(shape + (k // 16,), dtype=torch.int32, device=DEV)
        for i in range(16):
            codes |= q[..., i] << (2 * i)
        return codes, s, -s
    codes = torch.randint(-2**31, 2**31, shape + (k * bits // 32,), dtype=torch.int64, device=DEV,
                          generator=gen).to(torch.int32)
    return codes, s, -s * (1 << (bits - 1))


def _signs(n, gen):
    return torch.randint(0, 2, (n,), device=DEV, generator=gen).float() * 2 - 1


def _shapes(case):
    return [(case["n"], case["k"])] + ([(case["k"], case["n"])] if case["down"] else [])


def _packs(case, gen):
    """The raw weights of the bank: (n, k, tensors) of every projection."""
    fmt, out = case["fmt"], []
    for _ in range(case["bank"]):
        for n, k in _shapes(case):
            if fmt in BLOCK:
                w = (_ggml(fmt, n, k, gen),)
            elif fmt.startswith("exl3"):
                t = torch.randint(-32768, 32768, (k // 16, n // 16, 8 * int(fmt[5:])), dtype=torch.int16, device=DEV,
                                  generator=gen)
                suh = _signs(k, gen) * (0.5 + torch.rand(k, device=DEV, generator=gen))
                svh = _signs(n, gen) * (0.01 + 0.02 * torch.rand(n, device=DEV, generator=gen))
                w = (t, suh.half(), svh.half())
            else:
                w = _affine(int(fmt[6]), n, k, gen) + ((_signs(k, gen),) if fmt.endswith("rot") else (None,))
            out.append((n, k, w))
    return out


def _projection(fmt, n, k, w):
    if fmt in BLOCK:
        return PackedLinear.from_ggml(gguf.GGUFBlocks(w[0], TYPES[fmt], (n, k)))
    if fmt.startswith("exl3"):
        return PackedLinear.from_exl3(exl3.EXL3Tensor(*w))
    return PackedLinear(*w, block=HAD if w[3] is not None else 0, group_size=GROUP, bits=int(fmt[6]))


def _experts(case, gen):
    """gate, up [E, I, H] and down [E, H, I] of a MoE layer."""
    e, h, i, fmt = case["e"], case["h"], case["i"], case["fmt"]
    if fmt in BLOCK:
        return [_ggml(fmt, e * n, k, gen) for n, k in ((i, h), (i, h), (h, i))]
    return [_affine(int(fmt[6]), n, k, gen, (e,)) for n, k in ((i, h), (i, h), (h, i))]


def _moe_inputs(case, gen):
    t, dt = case["tokens"], DTYPE[case["dtype"]]
    x = torch.randn(t, case["h"], device=DEV, generator=gen).to(dt)
    logits = torch.randn(t, case["e"], device=DEV, generator=gen)
    if not case["shared"]:
        return x, logits, None, None
    return (x, logits, torch.randn(t, case["h"], device=DEV, generator=gen).to(dt),
            torch.randn(t, device=DEV, generator=gen).to(dt))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


# ------------------------------------------------------------------ the measured call
def prepare(case, seed):
    gen = _gen(seed)
    if case["kind"] == "moe":
        w = _experts(case, gen)
        x, logits, shared, gate = _moe_inputs(case, gen)
        if case["fmt"] in BLOCK:
            ex = moe.GGMLExperts(*w, TYPES[case["fmt"]], case["e"], case["h"], case["i"])
            f = moe.swiglu
        else:
            ex = moe.AffineExperts(*w, int(case["fmt"][6]), GROUP, case["e"], case["h"], case["i"])
            f = moe.swiglu_affine

        def call():
            return [f(x, logits, ex, top_k=case["topk"], shared=shared, shared_gate=gate)]
    else:
        bank = [_projection(case["fmt"], n, k, w) for n, k, w in _packs(case, gen)]
        xs = [torch.randn(case["rows"], p.input_dim, device=DEV, generator=gen).to(DTYPE[case["dtype"]]) for p in bank]

        def call():
            return [p(x) for p, x in zip(bank, xs)]
    if not case["graph"]:
        return {"call": call}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return {"call": call, "graph": graph, "out": out}


def run(state):
    if "graph" not in state:
        return state["call"]()
    state["graph"].replay()
    return state["out"]


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    if case["kind"] == "moe":
        t, e, h, i, k = (case[f] for f in ("tokens", "e", "h", "i", "topk"))
        routed = e * (1 - (1 - k / e) ** t)  # experts that get a token, for even routing
        per = 2 * i * _bytes_per_row(case["fmt"], h) + h * _bytes_per_row(case["fmt"], i)
        return {"bytes": routed * per + t * (4 * h + 4 * e + (2 * h + 2 if case["shared"] else 0)),
                "flops": 6 * t * k * h * i}
    m, b, f = case["rows"], 0, 0
    for n, k in _shapes(case):
        b += n * _bytes_per_row(case["fmt"], k) + 2 * m * (n + k)
        f += 2 * m * n * k
    return {"bytes": b * case["bank"], "flops": f * case["bank"]}


def tolerance(case):
    # outputs (and, in the MoE layer, the intermediates) are rounded to the activations' type; against
    # 64 bits this measures 2e-4 to 4e-4 in fp16, 1.7e-3 (2.4e-3 where the weights are expanded to
    # bf16) in bf16, and 4e-3 in the bf16 MoE layer
    if case["dtype"] == "fp16":
        return {"rel": 1e-3}
    return {"rel": 1.6e-2 if case["kind"] == "moe" else 8e-3}


# ------------------------------------------------------------------ the same in 64 bits
def _grid():
    """The IQ2_XS codebook (format data): 512 entries of eight bytes."""
    here = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    with open(os.path.join(here, "ishizuki_amd", "csrc", "ggml_grids.inc")) as f:
        body = re.search(r"ishz_iq2xs_grid\[512\]\s*=\s*\{([^}]*)\}", f.read()).group(1)
    v = [int(x, 16) for x in re.findall(r"0x[0-9a-fA-F]+", body)]
    return torch.tensor([[(e >> (8 * j)) & 255 for j in range(8)] for e in v], dtype=torch.float64, device=DEV)


def _half(b, o):
    return b[:, o:o + 2].contiguous().view(torch.float16).double()  # [blocks, 1]


def _dense_ggml(fmt, n, k, raw):
    b = raw.view(-1, BLOCK[fmt][1])
    nb = b.shape[0]
    if fmt == "q4_0":
        q = b[:, 2:].int()
        w = (torch.cat([q & 15, q >> 4], 1) - 8) * _half(b, 0)
    elif fmt == "q4_k":
        s, q = b[:, 4:16].int(), b[:, 16:].int().view(nb, 4, 32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6) << 4], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6) << 4], 1)
        q = torch.stack([q & 15, q >> 4], 2).view(nb, 8, 32)
        w = (_half(b, 0) * sc).unsqueeze(2) * q - (_half(b, 2) * mn).unsqueeze(2)
    elif fmt == "q6_k":
        ql, qh = b[:, :128].int().view(nb, 2, 2, 32), b[:, 128:192].int().view(nb, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)                       # [nb, half, quarter, 32]
        hi = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(nb, 2, 4, 2, 1)
        w = (_half(b, 208).view(nb, 1, 1, 1, 1) * sc) * ((lo | hi << 4) - 32).view(nb, 2, 4, 2, 16)
    else:
        q = b[:, 2:66].contiguous().view(torch.int16).int() & 0xffff  # [nb, 32]
        nib = torch.stack([b[:, 66:74] & 15, b[:, 66:74] >> 4], 2).view(nb, 16).double()
        db = (_half(b, 0) * (0.5 + nib) * 0.25).repeat_interleave(2, 1)
        s = q >> 9
        s = torch.stack([(s >> j) & 1 for j in range(7)], 2)
        s = torch.cat([s, s.sum(2, keepdim=True) & 1], 2)
        w = db.unsqueeze(2) * _grid()[(q & 511).long()] * (1 - 2 * s)
    return w.reshape(n, k)


def _dense_affine(bits, n, k, codes, s, b):
    per = 32 // bits
    q = torch.stack([(codes.view(n, -1) >> (bits * i)) & ((1 << bits) - 1) for i in range(per)], 2).view(n, k // GROUP, GROUP)
    return (q * s.view(n, -1, 1).double() + b.view(n, -1, 1).double()).view(n, k)


def _dense_exl3(bits2, n, k, t):
    """The trellis decoded with the 3INST codebook, [K, N]: position p of a tile is the image of the 16
    bits of its MSB-first ring that end at bit bits * (p + 1)."""
    bits = bits2 // 2
    w = t.view(torch.int32).view(-1, 8 * bits).long() & 0xffffffff
    words, ring = 8 * bits, 256 * bits
    out = torch.empty(w.shape[0], 16, 16, dtype=torch.float64, device=DEV)
    for p in range(256):
        b = ((p + 1) * bits - 16) % ring
        j, o = b // 32, b % 32
        state = ((w[:, j] << 16 | w[:, (j + 1) % words] >> 16) >> (32 - o) if o > 16
                 else w[:, j] >> (16 - o)) & 0xffff
        x = (state * 89226354 + 64248484) & 0xffffffff
        x = (x & 0x8fff8fff) ^ 0x3b603b60
        h = torch.stack([x & 0xffff, x >> 16], 1).to(torch.int32).to(torch.int16).view(torch.float16)
        lane, i = p // 8, p % 8
        out[:, lane % 4 * 2 + (0, 1, 8, 9)[i % 4], lane // 4 + 8 * (i // 4)] = (h[:, 0].float() + h[:, 1].float()).half().double()
    return out.view(k // 16, n // 16, 16, 16).transpose(1, 2).reshape(k, n)


def _wht(x):
    h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    while h.shape[0] < HAD:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, HAD) @ h / math.sqrt(HAD)).reshape(x.shape)


def exact(case, seed):
    gen = _gen(seed)
    if case["kind"] == "moe":
        return [_exact_moe(case, gen)]
    packs, out = _packs(case, gen), []
    xs = [torch.randn(case["rows"], k, device=DEV, generator=gen).to(DTYPE[case["dtype"]]) for _, k, _ in packs]
    for (n, k, w), x in zip(packs, xs):
        x, fmt = x.double(), case["fmt"]
        if fmt in BLOCK:
            out.append(x @ _dense_ggml(fmt, n, k, w[0]).T)
        elif fmt.startswith("exl3"):
            out.append(_wht(_wht(x * w[1].double()) @ _dense_exl3(int(fmt[5:]), n, k, w[0])) * w[2].double())
        else:
            x = x if w[3] is None else _wht(x * w[3].double())
            out.append(x @ _dense_affine(int(fmt[6]), n, k, *w[:3]).T)
    return out


def _exact_moe(case, gen):
    w = _experts(case, gen)
    x, logits, shared, gate = _moe_inputs(case, gen)
    e, h, i, fmt = case["e"], case["h"], case["i"], case["fmt"]
    val, ids = logits.double().softmax(1).topk(case["topk"], 1)
    val = val / val.sum(1, keepdim=True)
    x = x.double()
    y = torch.zeros_like(x)

    def dense(j, ex, n, k):
        if fmt in BLOCK:
            return _dense_ggml(fmt, n, k, w[j].view(e, -1)[ex].contiguous())
        return _dense_affine(int(fmt[6]), n, k, *(t[ex] for t in w[j]))
    for ex in range(e):
        tok, slot = (ids == ex).nonzero(as_tuple=True)
        if tok.numel():
            a = torch.nn.functional.silu(x[tok] @ dense(0, ex, i, h).T) * (x[tok] @ dense(1, ex, i, h).T)
            y.index_add_(0, tok, (a @ dense(2, ex, h, i).T) * val[tok, slot].unsqueeze(1))
    if shared is not None:
        y += torch.sigmoid(gate.double()).unsqueeze(1) * shared.double()
    return y
