"""The work that users of samhip have it do, as cases that can be timed and compared.

Each case goes through the public binding (sam.cpp_amd/samhip.py): single linears, the linear streams of the text encoder and of the
detector, one ViT block, the whole image encode, the feature cache's codec and the packing of weights.  Sizes are those of the
repository's benchmark and tests, or generic ones of the same ranges."""
import ctypes
import importlib.util
import math
import os

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_spec = importlib.util.spec_from_file_location("samhip", os.path.join(ROOT, "sam.cpp_amd", "samhip.py"))
sh = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(sh)

DEV = "cuda"
TYPES = {"q8_0": sh.Q8_0, "q4_k": sh.Q4_K, "q5_k": sh.Q5_K, "q6_k": sh.Q6_K, "f16": sh.F16}
_contexts = {}


def context(compute="native"):
    """A program keeps one context for each arithmetic that it uses."""
    if compute not in _contexts:
        _contexts[compute] = sh.Context(0, sh.COMPUTE_F16 if compute == "f16" else sh.COMPUTE_Q8_NATIVE, sh.ROUND_X86)
    return _contexts[compute]


# --- cases ------------------------------------------------------------------


def listed():
    return [
        # The text encoder's out_proj on its 32 tokens as one eager call: the smallest product, where launches and latency count.
        {"name": "text_out_proj_q8_0", "kind": "linear", "m": 32, "n": 1024, "k": 1024, "type": "q8_0", "compute": "native"},
        # A prompt through the text encoder: the token embedding's rows, then every linear of its 24 layers and the resizer, replayed
        # as one graph.  The weights are read once each, from HBM.
        {"name": "text_encoder_q4_k", "kind": "text", "tokens": 32, "width": 1024, "mlp": 4096, "layers": 24, "out": 256, "vocab": 49408,
         "type": "q4_k", "graph": True},
        # The decoder's six layers on 201 queries, 33 prompt tokens and the image tokens, replayed as one graph.
        {"name": "decoder_q8_0", "kind": "detector", "part": "decoder", "layers": 6, "width": 256, "ffn": 2048, "queries": 201, "prompt": 33,
         "image": 5184, "type": "q8_0", "graph": True},
        # The fusion encoder's six layers on the image tokens, as eager calls, with a K-quant checkpoint.
        {"name": "fusion_q6_k", "kind": "detector", "part": "fusion", "layers": 6, "width": 256, "ffn": 2048, "queries": 201, "prompt": 33,
         "image": 5184, "type": "q6_k", "graph": False},
        # One ViT linear on the tokens of one 1008-pixel image.
        {"name": "vit_qkv_q4_k", "kind": "linear", "m": 5184, "n": 3072, "k": 1024, "type": "q4_k", "compute": "native"},
        # The MLP's first linear on a batch of eight images: the largest single product.
        {"name": "batch8_fc1_q5_k", "kind": "linear", "m": 41472, "n": 4736, "k": 1024, "type": "q5_k", "compute": "native"},
        # A linear of odd sizes on strided rows in the fp16 arithmetic (the F32-decode policy's counterpart).
        {"name": "ragged_linear_q8_0_f16", "kind": "linear", "m": 777, "n": 1000, "k": 1056, "pad": 32, "type": "q8_0", "compute": "f16"},
        # The first block of the image encoder behind ln_pre: windowed attention, K-quant linears (fc2 in Q8_0, 4736 being no multiple of 256).
        {"name": "vit_block_window_q4_k", "kind": "block", "grid_w": 72, "grid_h": 72, "window": 24, "embed": 1024, "mlp": 4736, "type": "q4_k",
         "attention": "f32"},
        # A block with global attention, every linear in Q8_0.
        {"name": "vit_block_global_q8_0", "kind": "block", "grid_w": 72, "grid_h": 72, "window": 0, "embed": 1024, "mlp": 4736, "type": "q8_0",
         "attention": "f32"},
        # One image through the encoder: prefix, blocks (every eighth with global attention) and the neck's levels 0 to 2.  16 of the 32
        # blocks: a code of a packed activation that rounding tips over travels on, and past that depth it hides other differences.
        {"name": "encode_q4_k", "kind": "encode", "patch": 14, "grid": 72, "window": 24, "embed": 1024, "mlp": 4736, "depth": 16, "mid": 512,
         "dim": 256, "type": "q4_k"},
        # The feature cache of one image: levels 0 to 2 to Q8_0 rows and back.
        {"name": "feature_cache_q8_0", "kind": "cache", "grid": 72, "dim": 256, "type": "q8_0"},
        # Packing one ViT linear's weight when a checkpoint is converted.
        {"name": "pack_fc1_q4_k", "kind": "pack", "n": 4736, "k": 1024, "type": "q4_k"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "text", "detector", "block", "block", "encode", "cache", "pack"])
    quant = rng.choice(["q8_0", "q4_k", "q5_k", "q6_k"])
    if kind == "linear":
        m, n = _log(rng, 1, 41472), _log(rng, 48, 4736)
        k = 32 * _log(rng, 8, 148) if quant == "q8_0" else 256 * _log(rng, 1, 18)
        c = {"m": m, "n": n, "k": k, "type": quant, "compute": rng.choice(["native", "native", "native", "f16"])}
        if rng.random() < 0.3:
            c["pad"] = rng.choice([1, 4, 32, 256])
    elif kind == "text":
        width = rng.choice([512, 768, 1024])
        c = {"tokens": rng.randint(8, 77), "width": width, "mlp": 4 * width, "layers": rng.randint(1, 16), "out": 256,
             "vocab": _log(rng, 1000, 49408), "type": quant, "graph": rng.random() < 0.5}
    elif kind == "detector":
        c = {"part": rng.choice(["decoder", "fusion"]), "layers": rng.randint(1, 6), "width": 256, "ffn": rng.choice([1024, 2048]),
             "queries": _log(rng, 16, 250), "prompt": rng.randint(2, 64), "image": _log(rng, 300, 5184), "type": quant, "graph": rng.random() < 0.5}
    elif kind == "block":
        embed = 256 * rng.randint(1, 5)
        if rng.random() < 0.5:
            w = rng.choice([7, 8, 12, 14, 16, 24])
            gw, gh = w * rng.randint(1, 72 // w), w * rng.randint(1, 72 // w)
        else:
            w, gw, gh = 0, rng.randint(9, 72), rng.randint(9, 72)
        c = {"grid_w": gw, "grid_h": gh, "window": w, "embed": embed, "mlp": 128 * round(embed * rng.uniform(2, 4.6) / 128 - 0.49), "type": quant,
             "attention": rng.choice(["f32", "f32", "f16"])}
        c["mlp"] = min(c["mlp"], 5120)
    elif kind == "encode":
        w = rng.choice([8, 12, 16, 24])
        c = {"patch": rng.choice([14, 16]), "grid": w * rng.randint(1, 3), "window": w, "embed": 256 * rng.randint(2, 4), "depth": rng.randint(2, 8),
             "mid": 512, "dim": 256, "type": quant}
        c["mlp"] = 4 * c["embed"] + rng.choice([0, 128])
    elif kind == "cache":
        c = {"grid": rng.randint(16, 72), "dim": 32 * rng.randint(2, 12), "type": rng.choice(["q8_0", "f16"])}
    else:
        c = {"n": _log(rng, 256, 9472), "k": 256 * _log(rng, 1, 18), "type": quant}
    return {"kind": kind, **c}


# --- weights in the GGUF block formats ----------------------------------------
# A plain packer (smallest and largest value of each sub-block), so that inputs do not depend on the packer under test; the quants'
# distributions are those of packed N(0, 0.02^2) weights.


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def pack_rows(kind, w):
    n, k = w.shape
    if kind == "q8_0":
        b = w.view(n, k // 32, 32)
        d = (b.abs().amax(-1) / 127).to(torch.float16)
        q = torch.round(b / d.float().clamp_min(1e-30)[..., None]).clamp(-127, 127).to(torch.int8)
        return torch.cat([_half_bytes(d), q.view(torch.uint8)], -1).reshape(n, -1)
    b = w.view(n, k // 256, 256)
    if kind == "q6_k":
        s = b.view(n, -1, 16, 16)
        scale = s.abs().amax(-1) / 31.5
        d = (scale.amax(-1) / 127).to(torch.float16)
        sc = torch.round(scale / d.float().clamp_min(1e-30)[..., None]).clamp(1, 127)
        q = torch.round(s / (d.float()[..., None] * sc).clamp_min(1e-30)[..., None]).clamp(-32, 31).to(torch.int32) + 32
        q = q.view(n, -1, 2, 4, 32)
        lo, hi = q & 15, q >> 4
        ql = torch.stack([lo[..., 0, :] | (lo[..., 2, :] << 4), lo[..., 1, :] | (lo[..., 3, :] << 4)], -2).reshape(n, -1, 128)
        qh = (hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)).reshape(n, -1, 64)
        return torch.cat([ql.to(torch.uint8), qh.to(torch.uint8), sc.to(torch.int8).view(torch.uint8), _half_bytes(d)], -1).reshape(n, -1)
    top = 15 if kind == "q4_k" else 31
    s = b.view(n, -1, 8, 32)
    low = s.amin(-1).clamp_max(0)
    scale = (s.amax(-1) - low) / top
    d, dm = (scale.amax(-1) / 63).to(torch.float16), ((-low).amax(-1) / 63).to(torch.float16)
    ls = torch.round(scale / d.float().clamp_min(1e-30)[..., None]).clamp(1, 63)
    lm = torch.round(-low / dm.float().clamp_min(1e-30)[..., None]).clamp(0, 63)
    q = (s + (dm.float()[..., None] * lm)[..., None]) / (d.float()[..., None] * ls).clamp_min(1e-30)[..., None]
    q = torch.round(q).clamp(0, top).to(torch.int32)
    ls, lm = ls.to(torch.int32), lm.to(torch.int32)
    sc = torch.cat([ls[..., :4] | ((ls[..., 4:] >> 4) << 6), lm[..., :4] | ((lm[..., 4:] >> 4) << 6), (ls[..., 4:] & 15) | ((lm[..., 4:] & 15) << 4)], -1)
    nib = q & 15
    qs = (nib[..., 0::2, :] | (nib[..., 1::2, :] << 4)).reshape(n, -1, 128)
    parts = [_half_bytes(d), _half_bytes(dm), sc.to(torch.uint8)]
    if kind == "q5_k":
        bit = torch.arange(8, device=w.device, dtype=torch.int32)[:, None]
        parts.append(((q >> 4) << bit).sum(-2).to(torch.uint8))
    return torch.cat(parts + [qs.to(torch.uint8)], -1).reshape(n, -1)


def unpack_rows(kind, rows, k):
    """The 64-bit values of packed rows."""
    n = rows.shape[0]

    def half(b):
        return b.contiguous().view(torch.float16).double()

    if kind == "q8_0":
        b = rows.view(n, k // 32, 34)
        return (half(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(n, k)
    if kind == "q6_k":
        b = rows.view(n, k // 256, 210)
        ql, qh = b[..., :128].int().view(n, -1, 2, 2, 32), b[..., 128:192].int().view(n, -1, 2, 32)
        lo = torch.stack([ql[..., 0, :] & 15, ql[..., 1, :] & 15, ql[..., 0, :] >> 4, ql[..., 1, :] >> 4], -2)
        hi = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], -2)
        q = (lo | (hi << 4)).double().view(n, -1, 16, 16) - 32
        return (half(b[..., 208:]) * b[..., 192:208].contiguous().view(torch.int8).double()).unsqueeze(-1).mul(q).reshape(n, k)
    b = rows.view(n, k // 256, 144 if kind == "q4_k" else 176)
    s = b[..., 4:16].int()
    ls = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], -1).double()
    lm = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
    qs = b[..., -128:].int().view(n, -1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], -2).reshape(n, -1, 8, 32)
    if kind == "q5_k":
        bit = torch.arange(8, device=rows.device, dtype=torch.int32)[:, None]
        q = q | (((b[..., 16:48].int().unsqueeze(-2) >> bit) & 1) << 4)
    return ((half(b[..., :2]) * ls).unsqueeze(-1) * q.double() - (half(b[..., 2:4]) * lm).unsqueeze(-1)).reshape(n, k)


def packed_activation(x, wtype):
    """F32 rows as the native arithmetic packs them (Q8_0 for Q8_0 weights, Q8_K for the others), as 64-bit values."""
    x = x.float()
    m, k = x.shape
    if wtype == "q8_0":
        b = x.view(m, k // 32, 32)
        a = b.abs().amax(-1, keepdim=True)
        # quotients as F32 rounds them: formed in 64 bits first
        q = torch.round(b * torch.where(a > 0, (127 / a.double()).float(), torch.zeros_like(a)))
        return (q.double() * (a.double() / 127).float().to(torch.float16).double()).view(m, k)
    b = x.view(m, k // 256, 256)
    at = b.abs().argmax(-1, keepdim=True)
    s = b.gather(-1, at)
    i = torch.where(s != 0, (-127 / s.double()).float(), torch.zeros_like(s))
    d = torch.where(i != 0, (1 / i.double()).float(), torch.zeros_like(i))
    return (torch.round(i * b).clamp_max(127).double() * d.double()).view(m, k)


def product64(x, wtype, rows, compute="native"):
    k = x.shape[1]
    a = x.double() if compute == "f16" else packed_activation(x, wtype)
    return a @ unpack_rows(wtype, rows, k).t()


def row_bytes(kind, k):
    return sh.row_bytes(TYPES[kind], k)


class Draws:
    """Seeded normal draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        v = torch.randn(*shape, generator=self.g, device=DEV)
        return v.mul_(std).add_(mean) if mean or std != 1 else v

    def weight(self, kind, n, k):
        """Packed rows of an [n][k] linear weight N(0, 0.02^2)."""
        return pack_rows(kind, self.normal(n, k, std=0.02))


def tensor(t, kind, ne0, ne1, row0=0, stride=None):
    """The descriptor of rows row0 .. row0 + ne1 of a device tensor (F32 rows of `stride` floats, or packed rows)."""
    if kind == "f32":
        return sh.tensor(sh.F32, ne0, ne1, t.data_ptr(), nb1=4 * (stride or ne0))
    rb = row_bytes(kind, ne0)
    return sh.tensor(TYPES[kind], ne0, ne1, t.data_ptr() + row0 * rb, nb1=rb)


# --- streams of linears ---------------------------------------------------------


def stream_plan(case):
    """(weights, activations, products) of the linear streams.  weights: key -> (rows, k); activations: key -> (m, k, after GELU);
    products: (weight key, first row, n, k, activation key)."""
    weights, acts, prods = {}, {}, []
    if case["kind"] == "text":
        m, w, f = case["tokens"], case["width"], case["mlp"]
        for i in range(case["layers"]):
            p = "l%d." % i
            weights.update({p + "in": (3 * w, w), p + "out": (w, w), p + "fc1": (f, w), p + "fc2": (w, f)})
            acts.update({p + "ln1": (m, w, False), p + "att": (m, w, False), p + "ln2": (m, w, False), p + "act": (m, f, True)})
            prods += [(p + "in", 0, 3 * w, w, p + "ln1"), (p + "out", 0, w, w, p + "att"), (p + "fc1", 0, f, w, p + "ln2"), (p + "fc2", 0, w, f, p + "act")]
        weights["resizer"], acts["last"] = (case["out"], w), (m, w, False)
        prods.append(("resizer", 0, case["out"], w, "last"))
        return weights, acts, prods
    d, f, rows = case["width"], case["ffn"], {"img": case["image"], "prompt": case["prompt"], "query": case["queries"]}

    def attention(p, q, kv):
        weights.update({p + "in": (3 * d, d), p + "out": (d, d)})
        for src, tag in ((q, "q"), (kv, "kv"), (q, "o")):
            acts[p + tag] = (rows[src], d, False)
        # q, k and v are row-offset views of the fused in-projection
        prods.extend([(p + "in", 0, d, d, p + "q"), (p + "in", d, d, d, p + "kv"), (p + "in", 2 * d, d, d, p + "kv"), (p + "out", 0, d, d, p + "o")])

    for i in range(case["layers"]):
        p = "l%d." % i
        if case["part"] == "fusion":
            attention(p + "sa.", "img", "img")
            attention(p + "ca.", "img", "prompt")
            own = rows["img"]
        else:
            attention(p + "sa.", "query", "query")
            attention(p + "text.", "query", "prompt")
            attention(p + "img.", "query", "img")
            own = rows["query"]
        weights.update({p + "fc1": (f, d), p + "fc2": (d, f)})
        acts.update({p + "ln": (own, d, False), p + "act": (own, f, False)})
        prods += [(p + "fc1", 0, f, d, p + "ln"), (p + "fc2", 0, d, f, p + "act")]
    return weights, acts, prods


def output_place(i, prods):
    """(the product's place within a layer, the layer) of product i."""
    layer = prods[i][0].split(".")[0]
    if not layer.startswith("l") or not layer[1:].isdigit():
        return prods[i][0], 0
    per = sum(p[0].startswith("l0.") for p in prods)
    return "%02d" % (i % per), int(layer[1:])


def stream_inputs(case, seed):
    g = Draws(seed)
    weights, acts, prods = stream_plan(case)
    w = {key: g.weight(case["type"], n, k) for key, (n, k) in weights.items()}
    x = {}
    for key, (m, k, gelu) in acts.items():
        v = g.normal(m, k)
        # behind the text encoder's MLP a GELU, behind the detector's a ReLU
        x[key] = torch.nn.functional.gelu(v) if gelu else v.relu_() if key.endswith("act") else v
    if case["kind"] == "text":
        w["embedding"] = g.weight(case["type"], case["vocab"], case["width"])
        x["ids"] = torch.randint(0, case["vocab"], (case["tokens"],), generator=g.g, device=DEV, dtype=torch.int32)
    return w, x, prods


# --- the vision encoder -----------------------------------------------------------

NORMS = ("norm1_w", "norm1_b", "norm2_w", "norm2_b")


def rope_table(width, height, hd=64, theta=10000.0):
    """Axial 2-D table (cos, sin) [width*height][hd/2][2], token t = y*width + x."""
    freqs = 1.0 / theta ** (np.arange(0, hd, 4)[: hd // 4].astype(np.float64) / hd)
    t = np.arange(width * height)
    ang = np.concatenate([np.outer(t % width, freqs), np.outer(t // width, freqs)], axis=1)
    return torch.from_numpy(np.stack([np.cos(ang), np.sin(ang)], axis=-1).astype(np.float32)).to(DEV)


def fc2_type(case):
    return case["type"] if case["type"] == "q8_0" or case["mlp"] % 256 == 0 else "q8_0"


def block_weights(case, g):
    """One block's tensors; *_w of the linears are packed rows."""
    e, f = case["embed"], case["mlp"]
    b = {"norm1_w": g.normal(e, std=0.1, mean=1), "norm1_b": g.normal(e, std=0.05), "norm2_w": g.normal(e, std=0.1, mean=1), "norm2_b": g.normal(e, std=0.05)}
    for name, n, k in (("qkv", 3 * e, e), ("proj", e, e), ("fc1", f, e), ("fc2", e, f)):
        kind = fc2_type(case) if name == "fc2" else case["type"]
        b[name] = g.weight(kind, n, k)
        b[name + "_b"] = g.normal(n, std=0.02)
    return b


def block_desc(case, b, gw, gh, window, freqs, attention="f32"):
    e, f = case["embed"], case["mlp"]
    d = sh.VitBlockDesc()
    d.version = sh.ABI_VERSION
    d.embed, d.heads, d.mlp, d.grid_w, d.grid_h, d.window = e, e // 64, f, gw, gh, window
    d.attention_type = sh.F16 if attention == "f16" else sh.F32
    for name in NORMS:
        setattr(d, name, b[name].data_ptr())
    for name, n, k in (("qkv", 3 * e, e), ("proj", e, e), ("fc1", f, e), ("fc2", e, f)):
        setattr(d, name + "_w", tensor(b[name], fc2_type(case) if name == "fc2" else case["type"], k, n))
        setattr(d, name + "_b", b[name + "_b"].data_ptr())
    d.freqs_cis = freqs.data_ptr()
    return d


def prefix_weights(case, g):
    e, p, pg = case["embed"], case["patch"], case["window"]
    return {"patch_w": g.normal(e, 3, p, p, std=0.02), "pos_embed": g.normal(pg, pg, e, std=0.1), "ln_pre_w": g.normal(e, std=0.1, mean=1),
            "ln_pre_b": g.normal(e, std=0.05)}


def neck_weights(case, g):
    """Scales 0 to 2 in the layouts of the descriptor: deconvolutions [cin][cout][2][2], convolutions [cout][cin][k][k]."""
    e, mid, dim = case["embed"], case["mid"], case["dim"]
    shapes = [{"deconv1": (e, mid, 2), "deconv2": (mid, dim, 2), "conv1x1": (dim, dim, 1), "conv3x3": (dim, dim, 3)},
              {"deconv1": (e, mid, 2), "conv1x1": (dim, mid, 1), "conv3x3": (dim, dim, 3)}, {"conv1x1": (dim, e, 1), "conv3x3": (dim, dim, 3)}]
    scales = []
    for s in shapes:
        one = {}
        for name, (a, b, k) in s.items():
            one[name + "_w"] = g.normal(a, b, k, k, std=0.02)
            one[name + "_b"] = g.normal(b if name.startswith("deconv") else a, std=0.02)
        scales.append(one)
    return scales


def is_global(case, i):
    return i % 8 == 7 or (case["depth"] < 8 and i == case["depth"] - 1)


def norm64(x, w, b):
    x = x.double()
    c = x - x.mean(-1, keepdim=True)
    return c / (c.square().mean(-1, keepdim=True) + 1e-5).sqrt() * w.double() + b.double()


def gelu64(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))


def block64(case, b, x, gw, gh, window, freqs):
    e = case["embed"]
    h = e // 64
    t = gw * gh
    if window:
        order = torch.arange(t, device=DEV).view(gh // window, window, gw // window, window).permute(0, 2, 1, 3).reshape(-1)
        per = window * window
    else:
        order, per = torch.arange(t, device=DEV), t
    y = norm64(x, b["norm1_w"], b["norm1_b"])[order]
    qkv = product64(y, case["type"], b["qkv"]) + b["qkv_b"].double()
    c, s = freqs.double().unbind(-1)
    out = torch.empty(t, e, dtype=torch.float64, device=DEV)
    for w0 in range(0, t, per):
        for i in range(h):
            q, k, v = (qkv[w0:w0 + per, j * e + 64 * i:j * e + 64 * (i + 1)] for j in range(3))
            q, k = (torch.stack([a[:, 0::2] * c - a[:, 1::2] * s, a[:, 0::2] * s + a[:, 1::2] * c], -1).reshape(per, 64) for a in (q, k))
            out[w0:w0 + per, 64 * i:64 * (i + 1)] = torch.softmax(0.125 * (q @ k.t().contiguous()), -1) @ v
    y = product64(out, case["type"], b["proj"]) + b["proj_b"].double()
    back = torch.empty_like(y)
    back[order] = y
    x = x.double() + back
    y = product64(norm64(x, b["norm2_w"], b["norm2_b"]), case["type"], b["fc1"]) + b["fc1_b"].double()
    return x + product64(gelu64(y), fc2_type(case), b["fc2"]) + b["fc2_b"].double()


def prefix64(case, p, image):
    n, k, e = case["grid"], case["patch"], case["embed"]
    cols = image.double().view(3, n, k, n, k).permute(1, 3, 0, 2, 4).reshape(n * n, -1)
    x = cols @ p["patch_w"].double().view(e, -1).t()
    r = n // case["window"]
    x = x + p["pos_embed"].double().repeat(r, r, 1).reshape(n * n, e)
    return norm64(x, p["ln_pre_w"], p["ln_pre_b"])


def neck64(case, scales, x):
    n = case["grid"]

    def deconv(v, side, w, b):
        cin, cout = w.shape[:2]
        y = v @ w.double().permute(0, 2, 3, 1).reshape(cin, -1)
        return y.view(side, side, 2, 2, cout).permute(0, 2, 1, 3, 4).reshape(4 * side * side, cout) + b.double()

    def conv(v, side, w, b):
        cout, cin, k = w.shape[:3]
        if k == 1:
            return v @ w.double().view(cout, cin).t() + b.double()
        pad = torch.zeros(side + 2, side + 2, cin, dtype=torch.float64, device=DEV)
        pad[1:-1, 1:-1] = v.view(side, side, cin)
        y = b.double().expand(side * side, cout).clone()
        for ky in range(3):
            for kx in range(3):
                y += pad[ky:ky + side, kx:kx + side].reshape(side * side, cin) @ w[:, :, ky, kx].double().t()
        return y

    out = []
    for level, s in enumerate(scales):
        v, side = x.double(), n
        if "deconv1_w" in s:
            v, side = deconv(v, side, s["deconv1_w"], s["deconv1_b"]), 2 * side
        if "deconv2_w" in s:
            v, side = deconv(gelu64(v), side, s["deconv2_w"], s["deconv2_b"]), 2 * side
        v = conv(v, side, s["conv1x1_w"], s["conv1x1_b"])
        out.append(conv(v, side, s["conv3x3_w"], s["conv3x3_b"]))
    return out


# --- the four functions --------------------------------------------------------


def linear_inputs(case, seed):
    g = Draws(seed)
    stride = case["k"] + case.get("pad", 0)
    return g.weight(case["type"], case["n"], case["k"]), g.normal(case["m"], stride), stride


def cache_rows(case):
    return [(4 * case["grid"] >> i) ** 2 for i in range(3)]


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "ctx": context(case.get("compute", "native"))}
    if kind == "linear":
        w, x, stride = linear_inputs(case, seed)
        y = torch.empty(case["m"], case["n"], device=DEV)
        s.update(hold=(w, x), y=y, ops=[(tensor(w, case["type"], case["k"], case["n"]), tensor(x, "f32", case["k"], case["m"], stride=stride),
                                         tensor(y, "f32", case["n"], case["m"]))])
    elif kind in ("text", "detector"):
        w, x, prods = stream_inputs(case, seed)
        s["ops"], s["y"] = [], {}
        for i, (key, row0, n, k, act) in enumerate(prods):
            m, (group, layer) = x[act].shape[0], output_place(i, prods)
            # one buffer for the same product of every layer
            y = s["y"].setdefault(group, torch.empty(case["layers"] if group != "resizer" else 1, m, n, device=DEV))[layer]
            s["ops"].append((tensor(w[key], case["type"], k, n, row0=row0), tensor(x[act], "f32", k, m), tensor(y, "f32", n, m)))
        if kind == "text":
            emb = torch.empty(case["tokens"], case["width"], device=DEV)
            s["rows"] = (tensor(w["embedding"], case["type"], case["width"], case["vocab"]), sh.tensor(sh.I32, case["tokens"], 1, x["ids"].data_ptr()),
                         tensor(emb, "f32", case["width"], case["tokens"]))
            s["y"]["embedding"] = emb
        s["hold"] = (w, x)
        if case["graph"]:
            # the products run once before they are recorded, so that the context's staging is large enough
            torch.cuda.synchronize()
            for op in s["ops"]:
                s["ctx"].mul_mat(*op)
            s["ctx"].capture_begin()
            for op in s["ops"]:
                s["ctx"].mul_mat(*op)
            s["graph"] = Replay(s["ctx"].capture_end())
            s["ctx"].synchronize()
    elif kind == "block":
        g = Draws(seed)
        gw, gh, win = case["grid_w"], case["grid_h"], case["window"]
        b, freqs = block_weights(case, g), rope_table(win or gw, win or gh)
        ln = (g.normal(case["embed"], std=0.1, mean=1), g.normal(case["embed"], std=0.05))
        x0 = g.normal(gw * gh, case["embed"])
        s.update(hold=(b, freqs, ln, x0), x=torch.empty_like(x0), desc=block_desc(case, b, gw, gh, win, freqs, case["attention"]))
    elif kind == "encode":
        g = Draws(seed)
        n, e, win = case["grid"], case["embed"], case["window"]
        image = g.normal(3, n * case["patch"], n * case["patch"])
        p = prefix_weights(case, g)
        d = sh.VitPrefixDesc()
        d.version, d.image_size, d.patch, d.embed, d.pos_grid = sh.ABI_VERSION, n * case["patch"], case["patch"], e, win
        for name, v in p.items():
            setattr(d, name, v.data_ptr())
        tables = {True: rope_table(n, n), False: rope_table(win, win)}
        blocks = [block_weights(case, g) for _ in range(case["depth"])]
        descs = [block_desc(case, b, n, n, 0 if is_global(case, i) else win, tables[is_global(case, i)]) for i, b in enumerate(blocks)]
        scales = neck_weights(case, g)
        nd = sh.VitNeckDesc()
        nd.version, nd.grid, nd.embed, nd.mid, nd.dim, nd.columns_type = sh.ABI_VERSION, n, e, case["mid"], case["dim"], sh.F32
        for i, sc in enumerate(scales):
            for name, v in sc.items():
                setattr(nd.scales[i], name, v.data_ptr())
        s.update(hold=(image, p, tables, blocks, scales), image=image, prefix=d, blocks=descs, neck=nd, x=torch.empty(n * n, e, device=DEV),
                 levels=[torch.empty(r, case["dim"], device=DEV) for r in cache_rows(case)])
    elif kind == "cache":
        g = Draws(seed)
        s["x"] = [g.normal(r, case["dim"]) for r in cache_rows(case)]
        s["packed"] = [torch.empty(x.shape[0], row_bytes(case["type"], case["dim"]), dtype=torch.uint8, device=DEV) for x in s["x"]]
        s["back"] = [torch.empty_like(x) for x in s["x"]]
    else:
        s["w"] = Draws(seed).normal(case["n"], case["k"], std=0.02)
        s["packed"] = torch.empty(case["n"], row_bytes(case["type"], case["k"]), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    return s


class Replay:
    """A captured graph that is given back with the state that holds it."""

    def __init__(self, graph):
        self.graph = graph

    def __del__(self):
        if self.graph.ctx.handle:
            self.graph.destroy()


def run(s):
    case, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    if kind == "linear":
        ctx.mul_mat(*s["ops"][0])
        return s["y"]
    if kind in ("text", "detector"):
        if kind == "text":
            ctx.get_rows(*s["rows"])
        if "graph" in s:
            s["graph"].graph.launch()
        else:
            for op in s["ops"]:
                ctx.mul_mat(*op)
        return s["y"]
    lib = sh.lib()
    if kind == "block":
        _, _, ln, x0 = s["hold"]
        x, e = s["x"], case["embed"]
        sh.check(lib.samhip_layer_norm(ctx.handle, x0.data_ptr(), x.data_ptr(), x0.shape[0], e, ln[0].data_ptr(), ln[1].data_ptr(), 1e-5))
        sh.check(lib.samhip_vit_block(ctx.handle, ctypes.byref(s["desc"]), x.data_ptr()))
        return x
    if kind == "encode":
        x = s["x"].data_ptr()
        sh.check(lib.samhip_vit_prefix(ctx.handle, ctypes.byref(s["prefix"]), s["image"].data_ptr(), x))
        for d in s["blocks"]:
            sh.check(lib.samhip_vit_block(ctx.handle, ctypes.byref(d), x))
        sh.check(lib.samhip_vit_neck(ctx.handle, ctypes.byref(s["neck"]), x, *[v.data_ptr() for v in s["levels"]], None))
        return [s["x"]] + s["levels"]
    t = TYPES[case["type"]]
    if kind == "cache":
        k = case["dim"]
        for x, p, y in zip(s["x"], s["packed"], s["back"]):
            ctx.quantize_rows(t, x.data_ptr(), 4 * k, p.data_ptr(), x.shape[0], k, sh.ROUND_X86)
            ctx.dequantize_rows(t, p.data_ptr(), row_bytes(case["type"], k), y.data_ptr(), x.shape[0], k)
        return s["packed"] + s["back"]
    ctx.quantize_rows(t, s["w"].data_ptr(), 4 * case["k"], s["packed"].data_ptr(), case["n"], case["k"], sh.ROUND_REF)
    return s["packed"]


def work(case):
    kind = case["kind"]

    def linear(m, n, k, t):
        return n * row_bytes(t, k) + 4 * m * (n + k), 2 * m * n * k

    if kind == "linear":
        b, f = linear(case["m"], case["n"], case["k"], case["type"])
        return {"bytes": b, "flops": f}
    if kind in ("text", "detector"):
        weights, acts, prods = stream_plan(case)
        b = sum(n * row_bytes(case["type"], k) for n, k in weights.values()) + sum(4 * m * k for m, k, _ in acts.values())
        f = 0
        for _, _, n, k, act in prods:
            b += 4 * acts[act][0] * n
            f += 2 * acts[act][0] * n * k
        if kind == "text":
            b += case["tokens"] * (row_bytes(case["type"], case["width"]) + 4 * case["width"])
        return {"bytes": b, "flops": f}

    def block(t, per):
        e, f = case["embed"], case["mlp"]
        weights = (5 * e + f) * row_bytes(case["type"], e) - e * row_bytes(case["type"], e) + e * row_bytes(fc2_type(case), f)
        return weights + 8 * t * e, 2 * t * (4 * e * e + 2 * e * f) + 4 * t * per * e

    if kind == "block":
        t = case["grid_w"] * case["grid_h"]
        b, f = block(t, case["window"] ** 2 or t)
        return {"bytes": b, "flops": f}
    if kind == "encode":
        t, e, mid, dim = case["grid"] ** 2, case["embed"], case["mid"], case["dim"]
        pw = 3 * case["patch"] ** 2
        b, f = 4 * t * pw + 4 * e * pw + 8 * t * e, 2 * t * e * pw
        for i in range(case["depth"]):
            bb, ff = block(t, t if is_global(case, i) else case["window"] ** 2)
            b, f = b + bb - 8 * t * e, f + ff
        f += 2 * (2 * t * e * 4 * mid + 4 * t * mid * 4 * dim + 16 * t * dim * dim + 4 * t * mid * dim + t * e * dim + 21 * t * 9 * dim * dim)
        b += 4 * (8 * e * mid + 4 * mid * dim + dim * (dim + mid + e) + 27 * dim * dim) + 4 * 21 * t * dim
        return {"bytes": b, "flops": f}
    if kind == "cache":
        n, k = sum(cache_rows(case)), case["dim"]
        return {"bytes": n * (8 * k + 2 * row_bytes(case["type"], k)), "flops": 2 * n * k}
    return {"bytes": case["n"] * (4 * case["k"] + row_bytes(case["type"], case["k"])), "flops": 100 * case["n"] * case["k"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("cache", "pack"):
        return "exact"
    # Q8_0 products of few rows or of a 256 x 256 weight: exact integer block dots, F32 sums (1.7e-7 from 64 bits)
    if kind in ("linear", "text", "detector") and case["type"] == "q8_0" and case.get("compute", "native") == "native":
        if kind == "text" or case.get("part") == "decoder" or (kind == "linear" and case["m"] < 256):
            return {"rel": 1e-6}
    # products with operands rounded to fp16: 2.9e-4 from 64 bits
    if kind in ("linear", "text", "detector"):
        return {"rel": 1.2e-3}
    # a block: 2e-3 to 3e-3 from 64 bits, nearly all of it codes of the packed activations that a rounding of the operands tips over
    if kind == "block":
        return {"rel": 1e-2}
    # the encoder: the same, block upon block (about 1.3e-2 from 64 bits)
    return {"rel": 3e-2}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("cache", "pack"):
        return None
    if kind == "linear":
        w, x, _ = linear_inputs(case, seed)
        return product64(x[:, :case["k"]].contiguous(), case["type"], w, case["compute"])
    if kind in ("text", "detector"):
        w, x, prods = stream_inputs(case, seed)
        out = {}
        for i, (key, row0, n, k, act) in enumerate(prods):
            group, layer = output_place(i, prods)
            y = out.setdefault(group, torch.empty(case["layers"] if group != "resizer" else 1, x[act].shape[0], n, dtype=torch.float64, device=DEV))
            y[layer] = product64(x[act], case["type"], w[key][row0:row0 + n].contiguous())
        if kind == "text":
            out["embedding"] = unpack_rows(case["type"], w["embedding"][x["ids"].long()], case["width"])
        return out
    g = Draws(seed)
    if kind == "block":
        gw, gh, win = case["grid_w"], case["grid_h"], case["window"]
        b = block_weights(case, g)
        ln = (g.normal(case["embed"], std=0.1, mean=1), g.normal(case["embed"], std=0.05))
        x0 = g.normal(gw * gh, case["embed"])
        return block64(case, b, norm64(x0, *ln), gw, gh, win, rope_table(win or gw, win or gh))
    n, win = case["grid"], case["window"]
    image = g.normal(3, n * case["patch"], n * case["patch"])
    x = prefix64(case, prefix_weights(case, g), image)
    for i in range(case["depth"]):
        b, glob = block_weights(case, g), is_global(case, i)
        x = block64(case, b, x, n, n, 0 if glob else win, rope_table(n if glob else win, n if glob else win))
    return [x] + neck64(case, neck_weights(case, g), x)
