"""The work that a program has this library do, as cases that can be timed and compared.

Each case is one block of a decoder's prefill, run through the package's calls on
device memory, as the ggml backend and the stack runner run it: the weights are
converted and the buffers allocated beforehand, the activations arrive in fp32.

    mul_mat    pack the activations, one matmul
    attn_in    norm, the q/k/v group, (per-head norms of q and k), rope of q and k
    attn_out   pack the attention output, the O projection with the residual added
    ffn        norm, the fused gate/up matmul, the down projection with the residual added
    ffn_parts  the same with gate and up of different types, which cannot be fused
    head       norm and the output projection, every row's logits
    layer      attn_in, attn_out (on q, as attention is not part of the path) and ffn
    convert    one GGUF weight, or a gate/up pair, into its cache entry

Sizes: hidden 1024 (16 layers, Q8_0), the Qwen3-4B shape (hidden 2560, Q4_K with
Q8_0 or Q6_K for O and down), the 27B-class shape (hidden 5120, Q4_K), and widths
between them; 32 to 4096 tokens at a time, whole chunks and ragged ones.
"""
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

F32, F16, Q4_0, Q4_1, Q5_0, Q5_1, Q8_0 = 0, 1, 2, 3, 6, 7, 8
Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, IQ4_NL, IQ4_XS, BF16 = 10, 11, 12, 13, 14, 20, 23, 30
GEGLU, SWIGLU = 1, 2  # the package's numbers
EPS = 1e-6

# hidden, q width, k/v width, head width, ffn: the three model shapes
SHAPES = {"small": dict(hidden=1024, q=1024, kv=1024, head=64, ffn=4096),
          "4b": dict(hidden=2560, q=4096, kv=1024, head=128, ffn=9728),
          "27b": dict(hidden=5120, q=6144, kv=1024, head=128, ffn=17408)}


def _package():
    if "ggml_xdna_amd" not in sys.modules:
        pkg = Path(__file__).resolve().parents[1] / "ggml-xdna_amd"
        spec = importlib.util.spec_from_file_location("ggml_xdna_amd", pkg / "__init__.py",
                                                      submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["ggml_xdna_amd"] = mod
        spec.loader.exec_module(mod)
        mod.init(0)
    return sys.modules["ggml_xdna_amd"]


# ---- the cases ----------------------------------------------------------------

def listed():
    small, b4, b27 = SHAPES["small"], SHAPES["4b"], SHAPES["27b"]
    return [
        # a prompt's short last chunk, one projection: launch latency and one pass over the weight
        dict(name="mul_mat_short", kind="mul_mat", tokens=48, n=2560, k=2560, type=Q8_0, outliers=0.0),
        # a whole layer of the small model at its smallest chunk: seven matmuls in four launches, all short
        dict(name="layer_small_256", kind="layer", tokens=256, **small, type=Q8_0, type2=Q8_0, qk_norm=False, neox=False,
             yarn=False, pos0=0, glu=SWIGLU, outliers=0.0),
        # one matmul at the gate's smallest batch
        dict(name="mul_mat_1024", kind="mul_mat", tokens=1024, n=2560, k=2560, type=Q8_0, outliers=0.0),
        # the ordinary chunk before attention, as a Qwen3-4B layer has it: norms of every head, NeoX rope
        dict(name="attn_in_2048", kind="attn_in", tokens=2048, **b4, type=Q4_K, qk_norm=True, neox=True, yarn=False,
             pos0=2048, outliers=0.0),
        # and after it
        dict(name="attn_out_2048", kind="attn_out", tokens=2048, **b4, type=Q8_0, outliers=0.0),
        # the ordinary chunk's feed-forward, with outlier channels
        dict(name="ffn_2048", kind="ffn", tokens=2048, **b4, type=Q4_K, type2=Q4_K, glu=SWIGLU, outliers=0.01),
        # the small model's feed-forward on a ragged chunk
        dict(name="ffn_small_1000", kind="ffn", tokens=1000, **small, type=Q8_0, type2=Q8_0, glu=SWIGLU, outliers=0.0),
        # a file that mixes types within a layer: gate and up as a group, GeGLU on its own; a ragged last chunk
        dict(name="ffn_parts_1537", kind="ffn_parts", tokens=1537, **b4, type=Q4_K, type2=Q6_K, glu=GEGLU, outliers=0.01),
        # the 27B-class layer at a 4096-token chunk: before attention, with YaRN positions far out
        dict(name="attn_in_27b_4096", kind="attn_in", tokens=4096, **b27, type=Q4_K, qk_norm=False, neox=False, yarn=True,
             pos0=12288, outliers=0.005),
        # and its feed-forward, the largest case
        dict(name="ffn_27b_4096", kind="ffn", tokens=4096, **b27, type=Q4_K, type2=Q4_K, glu=SWIGLU, outliers=0.005),
        # every row's logits (perplexity, speculative checks), one chunk of 512 tokens
        dict(name="head_512", kind="head", tokens=512, hidden=2560, n=151936, type=Q6_K, outliers=0.0),
        # loading: a layer's gate/up pair into the weight cache
        dict(name="convert_gate_up", kind="convert", n=9728, k=2560, type=Q4_K, pair=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mul_mat", "attn_in", "attn_out", "ffn", "ffn_parts", "layer", "head", "convert"])
    if kind == "convert":
        # any type a file can carry, at any width it allows
        t = rng.choice([F32, F16, BF16, Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, IQ4_NL, IQ4_XS])
        block = max(8, _blocks(t)[0])
        pair = rng.random() < 0.3
        n = _log_uniform(rng, 256, 17408)
        return dict(kind=kind, n=(n + 31) // 32 * 32 if pair else n, k=max(1, _log_uniform(rng, 512, 17408) // block) * block,
                    type=t, pair=pair)
    tokens = _log_uniform(rng, 32, 4096)
    outliers = rng.choice([0.0, 0.0, 0.005, 0.01])
    if rng.random() < 0.5:
        s = dict(SHAPES[rng.choice(["small", "small", "4b", "4b", "27b"])])
    else:  # a width between the shapes
        head = rng.choice([64, 96, 128])
        kvh, per = rng.randint(2, 8), rng.randint(1, 5)
        s = dict(hidden=256 * rng.randint(3, 16), q=kvh * per * head, kv=kvh * head, head=head)
        s["ffn"] = 256 * max(3, int(s["hidden"] * rng.uniform(2.5, 4.0)) // 256)
    types = [Q8_0, Q4_K, Q6_K]
    if kind == "mul_mat":
        t = rng.choice(types)
        block = 32 if t == Q8_0 else 256
        n, k = _log_uniform(rng, 512, 17408), _log_uniform(rng, 1024, 17408) // block * block
        return dict(kind=kind, tokens=min(tokens, int(1e12 / (n * k))), n=n, k=k, type=t, outliers=outliers)
    if kind == "head":
        return dict(kind=kind, tokens=min(tokens, 1024), hidden=s["hidden"], n=_log_uniform(rng, 32000, 151936), type=Q6_K,
                    outliers=outliers)
    c = dict(kind=kind, tokens=tokens, **s, outliers=outliers)
    if c["q"] % 256:  # the O projection's rows must be whole blocks
        c["type"] = Q8_0
    else:
        c["type"] = rng.choice(types)
    if kind in ("attn_in", "layer"):
        c.update(qk_norm=rng.random() < 0.5, neox=rng.random() < 0.5, yarn=rng.random() < 0.25, pos0=rng.choice([0, 2048, 6144, 12288]))
    if kind in ("ffn", "ffn_parts", "layer"):
        c.update(type2=rng.choice([t for t in types if kind != "ffn_parts" or t != c["type"]]), glu=rng.choice([SWIGLU, SWIGLU, GEGLU]))
        if kind == "layer" and c["q"] % 256:
            c["type2"] = Q8_0
    # no more work than the largest listed case has; the unfused and whole-layer forms cost more a product
    most = 2.1e12 if kind == "ffn" else 1.4e12
    c["tokens"] = min(c["tokens"], int(most / work(dict(c, tokens=1))["flops"]))
    return c


# ---- inputs -------------------------------------------------------------------

def _blocks(t):
    """(values, bytes) of a block of a GGUF type."""
    return {F32: (1, 4), F16: (1, 2), BF16: (1, 2), Q4_0: (32, 18), Q4_1: (32, 20), Q5_0: (32, 22), Q5_1: (32, 24), Q8_0: (32, 34),
            Q2_K: (256, 84), Q3_K: (256, 110), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), IQ4_NL: (32, 18),
            IQ4_XS: (256, 136)}[t]


def _half(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(*v.shape, 2)


def _q8_0(w):
    n, k = w.shape
    x = w.reshape(n, k // 32, 32)
    d = x.abs().amax(dim=2) / 127.0
    q = torch.round(x / d.clamp(min=1e-12)[..., None]).clamp(-128, 127).to(torch.int8)
    return torch.cat([_half(d), q.view(torch.uint8)], dim=2).reshape(n, -1)


def _q4_k(w):
    """Q4_K rows: 4-bit codes under the 6-bit scale and offset of each 32 values."""
    n, k = w.shape
    x = w.reshape(n, k // 256, 8, 32)
    low = (-x.amin(dim=3)).clamp(min=0.0)
    s = (x.amax(dim=3) + low) / 15.0
    d, dmin = ((v.amax(dim=2) / 63.0).clamp(min=1e-7).to(torch.float16) for v in (s, low))
    sc, mn = (torch.round(v / f.float()[..., None]).clamp(0, 63) for v, f in ((s, d), (low, dmin)))
    step, off = d.float()[..., None] * sc, dmin.float()[..., None] * mn
    q = torch.round((x + off[..., None]) / step.clamp(min=1e-12)[..., None]).clamp(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    pairs = [sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6), (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)]
    codes = (q[:, :, 0::2] | (q[:, :, 1::2] << 4)).reshape(n, k // 256, 128)
    return torch.cat([_half(d), _half(dmin)] + pairs + [codes], dim=2).reshape(n, -1)


def _q6_k(w):
    """N x K floats -> Q6_K rows: 16-value scales as int8 multiples of a super-block's fp16 step."""
    n, k = w.shape
    x = w.reshape(n, k // 256, 16, 16)
    s = x.abs().amax(dim=3) / 31.0
    d = (s.amax(dim=2) / 127.0).clamp(min=1e-7).to(torch.float16)
    sc = torch.round(s / d.float()[..., None]).clamp(1, 127)
    q = (torch.round(x / (d.float()[..., None] * sc)[..., None]) + 32).clamp(0, 63).to(torch.uint8)
    # value 128h + 32c + l: low bits nibble c/2 of ql[64h + 32(c%2) + l], high bits 2c of qh[32h + l]
    q = q.reshape(n, k // 256, 2, 4, 32)
    out = torch.empty((n, k // 256, 210), dtype=torch.uint8, device=w.device)
    lo, hi = q & 15, q >> 4
    out[..., :128] = torch.stack([lo[..., 0, :] | (lo[..., 2, :] << 4), lo[..., 1, :] | (lo[..., 3, :] << 4)], dim=3).reshape(n, k // 256, 128)
    out[..., 128:192] = (hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)).reshape(n, k // 256, 64)
    out[..., 192:208] = sc.to(torch.int8).view(torch.uint8)
    out[..., 208:] = _half(d)
    return out.reshape(n, -1)


def _weight(t, n, k, g):
    """A GGUF weight, n rows of k values N(0, 0.02), as its bytes."""
    if t in (Q8_0, Q4_K, Q6_K):
        parts = []
        for r in range(0, n, 16384):  # a slice at a time: the quantisers' intermediates are many times the weight
            w = torch.randn((min(16384, n - r), k), generator=g, device="cuda") * 0.02
            parts.append({Q8_0: _q8_0, Q4_K: _q4_k, Q6_K: _q6_k}[t](w))
        return torch.cat(parts)
    if t in (F32, F16, BF16):
        w = torch.randn((n, k), generator=g, device="cuda") * 0.02
        return w.to({F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[t]).view(torch.uint8)
    # the other types: random codes and sub-block scales under block scales of one magnitude
    values, size = _blocks(t)
    raw = torch.randint(0, 256, (n, k // values, size), generator=g, device="cuda", dtype=torch.uint8)
    d = (torch.rand((n, k // values), generator=g, device="cuda") + 0.5) * {Q4_0: 4e-3, Q4_1: 4e-3, Q5_0: 2e-3, Q5_1: 2e-3,
                                                                          IQ4_NL: 3e-4, IQ4_XS: 2e-5}.get(t, 2e-4)
    at = {Q2_K: 80, Q3_K: 108}.get(t, 0)
    raw[..., at:at + 2] = _half(d)
    if t in (Q4_1, Q5_1, Q2_K, Q5_K):  # the offset, or the scale of the offsets
        raw[..., at + 2:at + 4] = _half(d if t in (Q2_K, Q5_K) else -8 * d if t == Q4_1 else -16 * d)
    return raw.reshape(n, -1)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _activations(c, width, g):
    x = torch.randn((c["tokens"], width), generator=g, device="cuda")
    if c["outliers"] > 0:
        ch = torch.randperm(width, generator=g, device="cuda")[:max(1, int(width * c["outliers"]))]
        x[:, ch] *= 20.0 if c["outliers"] >= 0.01 else 30.0
    return x


def _norm_weight(width, g):
    return 1.0 + 0.1 * torch.randn(width, generator=g, device="cuda")


def _sources(c, seed):
    """The inputs of a case as a file and the layers before give them: GGUF bytes, fp32 rows, positions."""
    g, kind, s = _generator(seed), c["kind"], {}
    if kind == "convert":
        s["raw"] = _weight(c["type"], c["n"], c["k"], g)
        if c["pair"]:
            s["raw2"] = _weight(c["type"], c["n"], c["k"], g)
        return s
    if kind == "mul_mat":
        s["x"] = _activations(c, c["k"], g)
        s["w"] = (c["type"], _weight(c["type"], c["n"], c["k"], g), c["n"], c["k"])
        return s
    h, t = c["hidden"], c["type"]
    if kind == "head":
        s.update(x=_activations(c, h, g), norm=_norm_weight(h, g), w=(t, _weight(t, c["n"], h, g), c["n"], h))
        return s
    s["x"] = _activations(c, h, g)
    if kind in ("attn_in", "layer"):
        s["attn_norm"] = _norm_weight(h, g)
        for name, n in (("wq", c["q"]), ("wk", c["kv"]), ("wv", c["kv"])):
            s[name] = (t, _weight(t, n, h, g), n, h)
        s["pos"] = torch.arange(c["pos0"], c["pos0"] + c["tokens"], dtype=torch.int32, device="cuda")
        if c["qk_norm"]:
            s["q_norm"], s["k_norm"] = _norm_weight(c["head"], g), _norm_weight(c["head"], g)
    if kind in ("attn_out", "layer"):
        to = t if kind == "attn_out" else c["type2"]
        s["wo"] = (to, _weight(to, h, c["q"], g), h, c["q"])
        if kind == "attn_out":
            s["attn"] = torch.randn((c["tokens"], c["q"]), generator=g, device="cuda")
    if kind in ("ffn", "ffn_parts", "layer"):
        s["ffn_norm"] = _norm_weight(h, g)
        tu = c["type2"] if kind == "ffn_parts" else t
        s["gate"], s["up"] = (t, _weight(t, c["ffn"], h, g), c["ffn"], h), (tu, _weight(tu, c["ffn"], h, g), c["ffn"], h)
        s["down"] = (c["type2"], _weight(c["type2"], h, c["ffn"], g), h, c["ffn"])
    return s


def _rope_args(c):
    """n_dims, mode, base, freq_scale, ext_factor, attn_factor, corr dims: plain, or YaRN from a 4096-token context by 4."""
    n, base = c["head"], 1e6 if c["neox"] else 1e4
    if not c["yarn"]:
        return n, 2 if c["neox"] else 0, base, 1.0, 0.0, 1.0, (0.0, 0.0)
    dims = [n * math.log(4096 / (beta * 2 * math.pi)) / (2 * math.log(base)) for beta in (32.0, 1.0)]
    corr = (float(max(0, math.floor(dims[0]))), float(min(n - 1, math.ceil(dims[1]))))
    return n, 2 if c["neox"] else 0, base, 0.25, 1.0, 1.0, corr


def prepare(case, seed):
    z = _package()
    c, s = case, _sources(case, seed)
    kind = c["kind"]
    f32 = dict(dtype=torch.float32, device="cuda")
    if kind == "convert":
        s["out"] = z.empty_packed((2 if c["pair"] else 1) * c["n"], c["k"])
        return dict(s, case=c)
    m = c["tokens"]
    st = {"case": c, "flag": torch.zeros(1, dtype=torch.int32, device="cuda")}
    if kind in ("ffn", "layer"):
        gate, up = s.pop("gate"), s.pop("up")
        st["gate_up"] = z.convert_weight_gu(gate[0], gate[1], up[1], gate[2], gate[3])
    for name, v in s.items():
        st[name] = z.convert_weight(*v) if isinstance(v, tuple) else v
    if kind == "mul_mat":
        st.update(px=z.empty_act(m, c["k"]), out=torch.empty((m, c["n"]), **f32))
    elif kind == "head":
        st.update(px=z.empty_act(m, c["hidden"]), out=torch.empty((m, c["n"]), **f32))
    else:
        st["px"] = z.empty_act(m, c["hidden"])
        if kind in ("attn_in", "layer"):
            for name, n in (("q0", c["q"]), ("k0", c["kv"]), ("v", c["kv"]), ("q", c["q"]), ("k", c["kv"])):
                st[name] = torch.empty((m, n), **f32)
            if c["qk_norm"]:
                st["qn"], st["kn"] = torch.empty((m, c["q"]), **f32), torch.empty((m, c["kv"]), **f32)
            st["rope"] = _rope_args(c)
        if kind in ("attn_out", "layer"):
            st.update(po=z.empty_act(m, c["q"]), h=torch.empty((m, c["hidden"]), **f32))
        if kind in ("ffn", "ffn_parts", "layer"):
            st.update(pd=z.empty_act(m, c["ffn"]), out=torch.empty((m, c["hidden"]), **f32))
        if kind == "ffn_parts":
            st["g0"], st["u0"] = torch.empty((m, c["ffn"]), **f32), torch.empty((m, c["ffn"]), **f32)
    return st


# ---- one pass -----------------------------------------------------------------

def _attn_in(z, c, s):
    m, nf, head = c["tokens"], s["flag"], c["head"]
    z.rms_norm(s["x"], EPS, s["attn_norm"], y=None, packed=s["px"])
    z.gemm_group(s["px"], m, [s["wq"], s["wk"], s["wv"]], [c["q"], c["kv"], c["kv"]], c["hidden"],
                 outs=[s["q0"], s["k0"], s["v"]], nonfinite=nf)
    q, k = s["q0"], s["k0"]
    if c["qk_norm"]:
        q, k = (z.rms_norm(v.view(-1, head), EPS, w, y=o.view(-1, head)).view(m, -1)
                for v, w, o in ((q, s["q_norm"], s["qn"]), (k, s["k_norm"], s["kn"])))
    n, mode, base, scale, ext, attn, corr = s["rope"]
    z.rope(q.view(m, -1, head), s["pos"], None, n, mode, base, scale, ext, attn, corr, y=s["q"].view(m, -1, head))
    z.rope(k.view(m, -1, head), s["pos"], None, n, mode, base, scale, ext, attn, corr, y=s["k"].view(m, -1, head))


def _attn_out(z, c, s, attn):
    z.pack_act_x(attn, out=s["po"])
    z.gemm_residual(s["po"], c["tokens"], s["wo"], c["hidden"], c["q"], s["x"], out=s["h"], nonfinite=s["flag"])


def _ffn(z, c, s, h):
    m, nf = c["tokens"], s["flag"]
    z.rms_norm(h, EPS, s["ffn_norm"], y=None, packed=s["px"])
    if "gate_up" in s:
        z.gemm_glu(c["glu"], s["px"], m, s["gate_up"], c["ffn"], c["hidden"], xout=s["pd"], nonfinite=nf)
    else:
        z.gemm_group(s["px"], m, [s["gate"], s["up"]], [c["ffn"], c["ffn"]], c["hidden"], outs=[s["g0"], s["u0"]], nonfinite=nf)
        z.glu(c["glu"], s["g0"], s["u0"], c["ffn"], y=None, packed=s["pd"])
    z.gemm_residual(s["pd"], m, s["down"], c["hidden"], c["ffn"], h, out=s["out"], nonfinite=nf)


def run(state):
    z, s, c = sys.modules["ggml_xdna_amd"], state, state["case"]
    kind = c["kind"]
    if kind == "convert":
        if c["pair"]:
            return z.convert_weight_gu(c["type"], s["raw"], s["raw2"], c["n"], c["k"], out=s["out"])
        return z.convert_weight(c["type"], s["raw"], c["n"], c["k"], out=s["out"])
    if kind == "mul_mat":
        z.pack_act_x(s["x"], out=s["px"])
        return z.gemm(s["px"], c["tokens"], s["w"], c["n"], c["k"], out=s["out"], nonfinite=s["flag"])
    if kind == "head":
        z.rms_norm(s["x"], EPS, s["norm"], y=None, packed=s["px"])
        return z.gemm(s["px"], c["tokens"], s["w"], c["n"], c["hidden"], out=s["out"], nonfinite=s["flag"])
    out = {"flag": s["flag"]}
    if kind in ("attn_in", "layer"):
        _attn_in(z, c, s)
        out.update(q=s["q"], k=s["k"], v=s["v"])
    if kind in ("attn_out", "layer"):
        _attn_out(z, c, s, s["attn"] if kind == "attn_out" else s["q"])
        out["h"] = s["h"]
    if kind in ("ffn", "ffn_parts", "layer"):
        _ffn(z, c, s, s["h"] if kind == "layer" else s["x"])
        out["out"] = s["out"]
    return out


# ---- what a pass cannot do without ----------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    if kind == "convert":
        size = _blocks(c["type"])
        values = (2 if c["pair"] else 1) * c["n"] * c["k"]
        return {"bytes": values * (size[1] / size[0] + 9 / 8), "flops": 0.0}
    m = c["tokens"]
    if kind == "mul_mat":
        weights, fp32 = c["n"] * c["k"], m * (c["n"] + c["k"])
    elif kind == "head":
        weights, fp32 = c["n"] * c["hidden"], m * (c["n"] + c["hidden"])
    else:
        weights = fp32 = 0
        if kind in ("attn_in", "layer"):
            weights += c["hidden"] * (c["q"] + 2 * c["kv"])
            fp32 += m * (c["hidden"] + c["q"] + 2 * c["kv"])
        if kind in ("attn_out", "layer"):
            weights += c["hidden"] * c["q"]
            fp32 += m * (2 * c["hidden"] + c["q"]) if kind == "attn_out" else m * c["hidden"]
        if kind in ("ffn", "ffn_parts", "layer"):
            weights += 3 * c["hidden"] * c["ffn"]
            fp32 += 2 * m * c["hidden"] if kind != "layer" else m * c["hidden"]
    return {"bytes": weights * 9 / 8 + 4.0 * fp32, "flops": 2.0 * m * weights}


def tolerance(case):
    """A matmul's fp32 sums alone, or, where a norm, a GLU or a residual sum is packed to 8 bits on the way, what a
    last-bit difference in it does: a few of its values round the other way (one step of their block, at most 2^-7
    of the block's largest)."""
    kind = case["kind"]
    if kind == "convert":
        return "exact"
    if kind in ("mul_mat", "attn_out"):
        return {"rel": 4e-6, "max": 1e-4}
    if kind in ("attn_in", "head"):
        return {"rel": 1e-4, "max": 2e-2}
    return {"rel": 1e-3, "max": 5e-2}


# ---- the same in 64 bits --------------------------------------------------------

def _dequantized(t, raw, n, k):
    """GGUF rows -> float64 values (each exact in fp32, or rounded to it once, as the format defines them)."""
    if t == Q8_0:
        b = raw.view(n, k // 32, 34)
        d = b[..., :2].contiguous().view(torch.float16).float()
        return (d * b[..., 2:].contiguous().view(torch.int8).float()).reshape(n, k).double()
    if t == Q4_K:
        b = raw.view(n, k // 256, 144)
        d, dmin = (b[..., i:i + 2].contiguous().view(torch.float16).float() for i in (0, 2))
        sb = b[..., 4:16]
        sc = torch.cat([sb[..., :4] & 63, (sb[..., 8:] & 15) | ((sb[..., :4] >> 6) << 4)], dim=2).float()
        mn = torch.cat([sb[..., 4:8] & 63, (sb[..., 8:] >> 4) | ((sb[..., 4:8] >> 6) << 4)], dim=2).float()
        qs = b[..., 16:].reshape(n, k // 256, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], dim=3).reshape(n, k // 256, 8, 32).float()
        return ((d * sc)[..., None] * q - (dmin * mn)[..., None]).reshape(n, k).double()
    assert t == Q6_K
    b = raw.view(n, k // 256, 210)
    ql, qh = b[..., :128].reshape(n, k // 256, 2, 2, 32), b[..., 128:192].reshape(n, k // 256, 2, 32)
    sc = b[..., 192:208].contiguous().view(torch.int8).float()
    d = b[..., 208:].contiguous().view(torch.float16).float()
    low = torch.stack([ql[..., 0, :] & 15, ql[..., 1, :] & 15, ql[..., 0, :] >> 4, ql[..., 1, :] >> 4], dim=3)
    high = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], dim=3)
    q = (low | (high << 4)).reshape(n, k // 256, 16, 16).float() - 32.0
    return ((d * sc)[..., None] * q).reshape(n, k).double()


def _bfp16(x):
    """The nearest bfp16 blocks: eight values share their largest one's exponent, 8-bit signed mantissas."""
    b = x.reshape(x.shape[0], -1, 8)
    e = torch.frexp(b.abs().amax(dim=2, keepdim=True))[1].double() - 1.0
    step = torch.exp2(e - 6.0)
    return (torch.round(b / step).clamp(-128, 127) * step).reshape(x.shape)


def _product(x, w):
    """Packed x times a packed weight, a slice of its rows at a time."""
    t, raw, n, k = w
    a = _bfp16(x)
    return torch.cat([a @ _bfp16(_dequantized(t, raw[r:r + 16384], min(16384, n - r), k)).T for r in range(0, n, 16384)], dim=1)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS) * w.double()


def _rotated(x, c, pos):
    """Rope by the angles its definition gives: one 32-bit multiplication a pair, from the position on."""
    n, mode, base, scale, ext, attn, corr = _rope_args(c)
    f = np.float32
    step, theta, angles = f(math.pow(base, -2.0 / n)), pos.cpu().numpy().astype(f), []
    for _ in range(n // 2):
        angles.append(theta)
        theta = theta * step
    t = np.stack(angles, axis=1)
    th, mscale = f(scale) * t, attn
    if ext:
        ramp = (np.arange(n // 2, dtype=f) - f(corr[0])) / max(f(0.001), f(corr[1]) - f(corr[0]))
        mix = (f(1) - np.minimum(f(1), np.maximum(f(0), ramp))) * f(ext)
        th, mscale = th * (f(1) - mix) + t * mix, attn * (1.0 + 0.1 * math.log(1.0 / scale))
    a = torch.from_numpy(th.astype(np.float64)).cuda()[:, None, :]
    cos, sin = torch.cos(a) * mscale, torch.sin(a) * mscale
    x = x.reshape(x.shape[0], -1, n)
    x0, x1 = (x[..., :n // 2], x[..., n // 2:]) if mode == 2 else (x[..., 0::2], x[..., 1::2])
    y0, y1 = x0 * cos - x1 * sin, x0 * sin + x1 * cos
    y = torch.cat([y0, y1], dim=2) if mode == 2 else torch.stack([y0, y1], dim=3)
    return y.reshape(x.shape[0], -1)


def _activated(kind, g):
    return g * torch.sigmoid(g) if kind == SWIGLU else 0.5 * g * (1.0 + torch.tanh(0.7978845608 * g * (1.0 + 0.044715 * g * g)))


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "convert":
        return None  # bytes
    s = _sources(c, seed)
    x = s["x"].double()
    if kind == "mul_mat":
        return _product(x, s["w"])
    if kind == "head":
        return _product(_rms(x, s["norm"]), s["w"])
    out, head = {"flag": None}, c.get("head")
    if kind in ("attn_in", "layer"):
        a = _rms(x, s["attn_norm"])
        q, k, out["v"] = (_product(a, s[n]) for n in ("wq", "wk", "wv"))
        if c["qk_norm"]:
            q, k = (_rms(v.reshape(-1, head), s[n]).reshape(c["tokens"], -1) for v, n in ((q, "q_norm"), (k, "k_norm")))
        out["q"], out["k"] = _rotated(q, c, s["pos"]), _rotated(k, c, s["pos"])
    if kind in ("attn_out", "layer"):
        out["h"] = x = x + _product(s["attn"].double() if kind == "attn_out" else out["q"], s["wo"])
    if kind in ("ffn", "ffn_parts", "layer"):
        a = _rms(x, s["ffn_norm"])
        out["out"] = x + _product(_activated(c["glu"], _product(a, s["gate"])) * _product(a, s["up"]), s["down"])
    return out
