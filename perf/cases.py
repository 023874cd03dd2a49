"""Timed cases: the work a program has this framework do, each through its public entry points.

Kinds (case["kind"]):
- "mlp":       mk_gemm twice, a transformer FFN (GELU-tanh up, plain down) over the rows of one prompt or image;
- "attention": mk_attention alone over prepared heads (the joint attention of a block, or a causal text prefix);
- "step":      the dual-stream MMDiT through Engine: one or two blocks with the time embedding, both inputs and the
               output head around them, as a whole guided Euler step on device buffers (step_cfg_device) or as one
               sample's velocity from host buffers (step);
- "q21":       the single-stream 2.1 graph through Engine.step: a later step against the cached text keys, or the first
               step after begin;
- "sdxl":      the SDXL spatial transformer through Engine.sdxl_forward;
- "vae":       the VAE decoder through Vae.decode_device.

Widths are those of the benchmark's workloads and of the tests; the number of blocks is cut to one or two, so a pass is a
layer stack of the full width. Token grids are image sizes / 16 (SDXL: / 16 for its first transformer stage, / 32 for
the second), prompts 16 to 512 rows. Weights are N(0, 0.02) (convolutions N(0, 1 / fan-in)), prompts and latents N(0, 1).
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mako-image_amd"))
import mkimage as M  # noqa: E402

DIM, HEADS, FFN, TEXT, LATENT = 3072, 24, 12288, 3584, 64        # the dual-stream model
QDIM, QHEADS, QFFN, QTEXT = 4096, 32, 12288, 4096                # the 2.1 graph
CTX_ROWS, CTX_DIM = 77, 2048                                     # SDXL's context
VAE_BASE, VAE_Z = 96, 16
GUIDANCE = 4.0
F64 = torch.float64


def listed():
    return [
        # the FFN over one short prompt's rows: every call reads all the weights for 77 rows
        dict(name="mlp_77_rows", kind="mlp", rows=77, wdt="bf16"),
        # the standalone joint attention at 1024 x 1024 (4096 image + 256 text keys), both guidance samples, any scale
        dict(name="attention_1024px", kind="attention", batch=2, heads=24, d=128, rows=4352, block=0, dt="bf16"),
        # a thumbnail preview: one unguided pass from host latents, a short prompt
        dict(name="step_256px", kind="step", blocks=1, h=16, w=16, s0=64, s1=0, fp8=False),
        # a draft at 512 x 512: guided, the negative prompt shorter than the positive one
        dict(name="step_512px_ragged", kind="step", blocks=1, h=32, w=32, s0=131, s1=23, fp8=False),
        # the headline size: guided step at 1024 x 1024, prompts of 256 rows
        dict(name="step_1024px", kind="step", blocks=2, h=64, w=64, s0=256, s1=256, fp8=False),
        # a portrait image on fp8 weights, prompts of different lengths
        dict(name="step_832x1216_fp8", kind="step", blocks=1, h=76, w=52, s0=200, s1=77, fp8=True),
        # the largest: 2048 x 2048 on fp8 weights
        dict(name="step_2048px_fp8", kind="step", blocks=1, h=128, w=128, s0=512, s1=512, fp8=True),
        # the 2.1 graph at 1024 x 1024: one sample's later step against its cached prompt of 256 rows
        dict(name="q21_1024px", kind="q21", h=64, w=64, s=256, first=False),
        # SDXL's second stage at 1024 x 1024, both guidance samples, an F16 checkpoint
        dict(name="sdxl_b_1024px_f16", kind="sdxl", dim=1280, depth=2, h=32, w=32, batch=2, f16=True),
        # SDXL's first stage on a portrait image, one sample, bf16 matrices
        dict(name="sdxl_a_832x1216", kind="sdxl", dim=640, depth=2, h=76, w=52, batch=1, f16=False),
        # the decoder on the headline image
        dict(name="vae_1024px", kind="vae", h=64, w=64),
        # the decoder on a portrait image, whose widths no tile height divides
        dict(name="vae_832x1216", kind="vae", h=76, w=52),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp", "attention", "step", "step", "step", "q21", "sdxl", "sdxl", "vae"])
    if kind == "mlp":
        return dict(kind=kind, rows=_log(rng, 16, 9000), wdt=rng.choice(["bf16", "fp8"]))
    if kind == "attention":
        d = rng.choice([64, 128])
        rows = _log(rng, 77, 4608)
        return dict(kind=kind, batch=rng.choice([1, 2]), heads=24 if d == 128 else rng.choice([10, 20]), d=d, rows=rows,
                    block=rng.choice([0, 0, min(rows, rng.randint(16, 512))]), dt=rng.choice(["bf16", "f16"]))
    if kind == "step":
        area = _log(rng, 12 * 12, 100 * 100)
        h = max(8, int(math.sqrt(area * rng.uniform(0.5, 2.0))))
        return dict(kind=kind, blocks=1, h=h, w=max(8, area // h), s0=_log(rng, 16, 512),
                    s1=rng.choice([0, _log(rng, 16, 512), _log(rng, 16, 512)]), fp8=rng.random() < 0.4)
    if kind == "q21":
        area = _log(rng, 12 * 12, 90 * 90)
        h = max(8, int(math.sqrt(area * rng.uniform(0.5, 2.0))))
        return dict(kind=kind, h=h, w=max(8, area // h), s=_log(rng, 16, 512), first=rng.random() < 0.25)
    if kind == "sdxl":
        dim = rng.choice([640, 1280])
        side = 64 if dim == 640 else 32
        return dict(kind=kind, dim=dim, depth=rng.choice([1, 2]), h=rng.randint(side // 4, side * 5 // 4),
                    w=rng.randint(side // 4, side * 5 // 4), batch=rng.choice([1, 2]), f16=rng.random() < 0.5)
    area = _log(rng, 8 * 8, 70 * 70)
    h = max(6, int(math.sqrt(area * rng.uniform(0.5, 2.0))))
    return dict(kind=kind, h=h, w=max(6, area // h))


# ---------------------------------------------------------------------------------------------------------------------
# inputs and weights, from the seed alone
# ---------------------------------------------------------------------------------------------------------------------

class Rng:
    """Normal draws on the device: call number i of a seed is the same tensor everywhere."""

    def __init__(self, seed):
        self.g = torch.Generator("cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(std).add_(mean)


def _store(t, dt):
    """fp32 draws as a stored matrix: (values, per-row scales or None)."""
    if dt == "fp8":
        s = t.abs().amax(1).clamp_(min=1e-30) / 448.0
        return (t / s[:, None]).to(torch.float8_e4m3fn), s
    return t.to({"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dt]), None


def _names(case):
    """(name, shape, stored type, mean, std) of every weight of an engine case, in the order they are drawn."""
    out = []

    def mat(name, n, k, dt="bf16", bias=True):
        out.append((name + ".weight", (n, k), dt, 0.0, 0.02))
        if bias:
            out.append((name + ".bias", (n,), "f32", 0.0, 0.02))

    def vec(name, n, mean):
        out.append((name, (n,), "f32", mean, 0.02))

    if case["kind"] == "step":
        w = "fp8" if case["fp8"] else "bf16"
        mat("img_in", DIM, LATENT)
        vec("txt_norm.weight", TEXT, 1.0)
        mat("txt_in", DIM, TEXT)
        mat("time_text_embed.timestep_embedder.linear_1", DIM, 256)
        mat("time_text_embed.timestep_embedder.linear_2", DIM, DIM)
        mat("norm_out.linear", 2 * DIM, DIM)
        mat("proj_out", LATENT, DIM)
        for i in range(case["blocks"]):
            p = "transformer_blocks.%d." % i
            for s in ("img_mod.1", "txt_mod.1"):
                mat(p + s, 6 * DIM, DIM)
            for s in ("to_q", "to_k", "to_v", "add_q_proj", "add_k_proj", "add_v_proj", "to_out.0", "to_add_out"):
                mat(p + "attn." + s, DIM, DIM, w)
            for s in ("norm_q", "norm_k", "norm_added_q", "norm_added_k"):
                vec(p + "attn.%s.weight" % s, 128, 1.0)
            for s in ("img_mlp", "txt_mlp"):
                mat(p + s + ".net.0.proj", FFN, DIM, w)
                mat(p + s + ".net.2", DIM, FFN, w)
    elif case["kind"] == "q21":
        mat("img_in", QDIM, LATENT, bias=False)
        vec("txt_in.text_norm.weight", QTEXT, 0.0)
        mat("txt_in.in_layer", QDIM, QTEXT, bias=False)
        mat("txt_in.out_layer", QDIM, QDIM, bias=False)
        mat("time_text_embed.timestep_embedder.linear_1", QDIM, 256, bias=False)
        mat("time_text_embed.timestep_embedder.linear_2", QDIM, QDIM, bias=False)
        mat("modulation.1", 4 * QDIM, QDIM, bias=False)
        mat("norm_out.linear", QDIM, QDIM, bias=False)
        mat("proj_out", LATENT, QDIM, bias=False)
        p = "transformer_blocks.0."
        for s in ("to_q", "to_k", "to_v", "to_out.0"):
            mat(p + "attn." + s, QDIM, QDIM, bias=False)
        for s in ("norm_q", "norm_k"):
            vec(p + "attn.%s.weight" % s, 128, 1.0)
        mat(p + "img_mlp.gate_layer", QFFN, QDIM, bias=False)
        mat(p + "img_mlp.proj", QFFN, QDIM, bias=False)
        mat(p + "img_mlp.out", QDIM, QFFN, bias=False)
    else:
        c, m = case["dim"], "f16" if case["f16"] else "bf16"
        vec("norm.weight", c, 1.0)
        vec("norm.bias", c, 0.0)
        mat("proj_in", c, c, m)
        mat("proj_out", c, c, m)
        for i in range(case["depth"]):
            p = "transformer_blocks.%d." % i
            for j in (1, 2, 3):
                vec(p + "norm%d.weight" % j, c, 1.0)
                vec(p + "norm%d.bias" % j, c, 0.0)
            for s in ("to_q", "to_k", "to_v"):
                mat(p + "attn1." + s, c, c, bias=False)
            mat(p + "attn1.to_out.0", c, c, m)
            mat(p + "attn2.to_q", c, c, m, bias=False)
            mat(p + "attn2.to_k", c, CTX_DIM, bias=False)
            mat(p + "attn2.to_v", c, CTX_DIM, bias=False)
            mat(p + "attn2.to_out.0", c, c, m)
            mat(p + "ff.net.0.proj", 8 * c, c, m)
            mat(p + "ff.net.2", c, 4 * c, m)
    return out


def _weights(case, rng):
    for name, shape, dt, mean, std in _names(case):
        yield name, *_store(rng.normal(*shape, std=std, mean=mean), dt)


def _vae_names():
    """(name, shape) of the decoder's weights."""
    b, d0, out = VAE_BASE, 4 * VAE_BASE, []

    def conv(name, co, ci, k):
        out.append((name + ".weight", (co, ci, k, k)))
        out.append((name + ".bias", (co,)))

    def res(name, ci, co):
        out.append((name + ".norm1.gamma", (ci,)))
        conv(name + ".conv1", co, ci, 3)
        out.append((name + ".norm2.gamma", (co,)))
        conv(name + ".conv2", co, co, 3)
        if ci != co:
            conv(name + ".conv_shortcut", co, ci, 1)

    conv("post_quant_conv", VAE_Z, VAE_Z, 1)
    conv("decoder.conv_in", d0, VAE_Z, 3)
    res("decoder.mid_block.resnets.0", d0, d0)
    out.append(("decoder.mid_block.attentions.0.norm.gamma", (d0,)))
    conv("decoder.mid_block.attentions.0.to_qkv", 3 * d0, d0, 1)
    conv("decoder.mid_block.attentions.0.proj", d0, d0, 1)
    res("decoder.mid_block.resnets.1", d0, d0)
    ins, outs = (4 * b, 2 * b, 2 * b, b), (4 * b, 4 * b, 2 * b, b)
    for i in range(4):
        for j in range(3):
            res("decoder.up_blocks.%d.resnets.%d" % (i, j), outs[i] if j else ins[i], outs[i])
        if i < 3:
            conv("decoder.up_blocks.%d.upsamplers.0.resample.1" % i, outs[i] // 2, outs[i], 3)
    out.append(("decoder.norm_out.gamma", (b,)))
    conv("decoder.conv_out", 3, b, 3)
    return out


def _vae_weights(rng):
    """fp32 tensors whose convolution weights are half values, as an F16 checkpoint's."""
    for name, shape in _vae_names():
        if len(shape) == 4:
            t = rng.normal(*shape, std=1.0 / math.sqrt(shape[1] * shape[2] * shape[3])).half().float()
        else:
            t = rng.normal(*shape, std=0.1, mean=1.0) if name.endswith("gamma") else rng.normal(*shape, std=0.02)
        yield name, t


def _engine_inputs(case, rng):
    """Prompts and latents (or SDXL's contexts and input) of an engine case, fp32 on the device."""
    if case["kind"] == "step":
        prompts = [rng.normal(s, TEXT) for s in (case["s0"], case["s1"]) if s]
        return prompts, rng.normal(case["h"] * case["w"], LATENT)
    if case["kind"] == "q21":
        return [rng.normal(case["s"], QTEXT)], rng.normal(case["h"] * case["w"], LATENT)
    return [rng.normal(CTX_ROWS, CTX_DIM) for _ in range(2)], rng.normal(case["batch"], case["h"] * case["w"],
                                                                         case["dim"])


def _mlp_inputs(case, rng):
    x = rng.normal(case["rows"], DIM).bfloat16()
    w1 = _store(rng.normal(FFN, DIM, std=0.02), case["wdt"])
    w2 = _store(rng.normal(DIM, FFN, std=0.02), case["wdt"])
    return x, w1, rng.normal(FFN, std=0.02), w2, rng.normal(DIM, std=0.02)


def _attention_inputs(case, rng):
    shape = (case["batch"], case["heads"], case["rows"], case["d"])
    dt = {"bf16": torch.bfloat16, "f16": torch.float16}[case["dt"]]
    return [rng.normal(*shape).to(dt) for _ in range(3)]


def _pad(n, m):
    return -(-n // m) * m


_side = []


def _stream():
    """The program's own stream: the engines' device calls are ordered after it and before what follows on it."""
    if not _side:
        _side.append(torch.cuda.Stream())
    return _side[0]


_CODES = {"bf16": M.BF16, "f16": M.F16, "fp8": M.FP8, "f32": M.F32}


def _host(t):
    """A stored tensor as the host array Engine.load takes."""
    if t.dtype in (torch.bfloat16, torch.float16):
        return t.view(torch.int16).cpu().numpy().view(np.uint16)
    if t.dtype == torch.float8_e4m3fn:
        return t.view(torch.uint8).cpu().numpy()
    return t.cpu().numpy()


def _engine(case, rng):
    if case["kind"] == "step":
        eng = M.Engine(M.FAMILY_DUAL, case["blocks"], DIM, HEADS, 128, FFN, TEXT, LATENT,
                       M.FP8 if case["fp8"] else M.BF16, 2)
    elif case["kind"] == "q21":
        eng = M.Engine(M.FAMILY_Q21, 1, QDIM, QHEADS, 128, QFFN, QTEXT, LATENT, M.BF16, 2)
    else:
        c = case["dim"]
        eng = M.Engine(M.FAMILY_SDXL, case["depth"], c, c // 64, 64, 4 * c, CTX_DIM,
                       weight_dtype=M.F16 if case["f16"] else M.BF16)
    types = {name: dt for name, _, dt, _, _ in _names(case)}
    for name, t, scale in _weights(case, rng):
        eng.load(name, _host(t), _CODES[types[name]])
        if scale is not None:
            eng.load(name + ".scale", scale.cpu().numpy(), M.F32)
    return eng


def prepare(case, seed):
    M.call("mk_set_device", 0)
    rng, kind = Rng(seed), case["kind"]
    s = {"case": case}
    if kind == "mlp":
        x, (w1, s1), b1, (w2, s2), b2 = _mlp_inputs(case, rng)
        rows = case["rows"]
        hid = torch.empty(rows, FFN, dtype=torch.bfloat16, device="cuda")
        out = torch.empty(rows, DIM, dtype=torch.float32, device="cuda")
        up, down = M.GemmArgs(), M.GemmArgs()
        for g, a, w, sc, b, c, n, k, epi, cdt in ((up, x, w1, s1, b1, hid, FFN, DIM, M.EPI_GELU_TANH, M.BF16),
                                                  (down, hid, w2, s2, b2, out, DIM, FFN, M.EPI_STORE, M.F32)):
            g.a, g.w, g.bias, g.c = a.data_ptr(), w.data_ptr(), b.data_ptr(), c.data_ptr()
            g.wscale = sc.data_ptr() if sc is not None else None
            g.M, g.N, g.K, g.lda, g.ldc, g.batch = rows, n, k, k, n, 1
            g.w_dtype, g.c_dtype, g.epilogue = _CODES[case["wdt"]], cdt, epi
        s.update(up=up, down=down, hid=hid, out=out, keep=(x, w1, s1, b1, w2, s2, b2))
    elif kind == "attention":
        q, k, v = _attention_inputs(case, rng)
        b, h, n, d = q.shape
        q_pad, k_pad = _pad(n, 256), _pad(n, 64)
        Q, K = q.new_zeros(b, h, q_pad, d), k.new_zeros(b, h, k_pad, d)
        VT = v.new_zeros(b, h, d, k_pad)
        Q[:, :, :n] = q
        K[:, :, :n] = k
        VT[:, :, :, torch.from_numpy(M.vt_col(np.arange(n))).cuda()] = v.transpose(2, 3)
        out = torch.empty(b, n, h * d, dtype=torch.bfloat16, device="cuda")
        s.update(q=Q, k=K, vt=VT, out=out, q_pad=q_pad, k_pad=k_pad)
    elif kind == "vae":
        vae = M.Vae(VAE_BASE, VAE_Z, mean=np.linspace(-0.5, 0.5, VAE_Z), std=np.linspace(1.0, 2.0, VAE_Z))
        for name, t in _vae_weights(rng):
            vae.load(name, t.cpu().numpy())
        s.update(vae=vae, stream=vae.stream(), tokens=rng.normal(case["h"] * case["w"], 4 * VAE_Z),
                 out=torch.empty(16 * case["h"], 16 * case["w"], 4, device="cuda"))
    else:
        eng = _engine(case, rng)
        prompts, x = _engine_inputs(case, rng)
        h, w = case["h"], case["w"]
        hosts = [p.cpu().numpy() for p in prompts]
        for slot, p in enumerate(hosts):
            eng.begin(p, h, w, slot)
        s.update(eng=eng, prompts=hosts)
        if kind == "sdxl":
            s.update(x=x, out=torch.empty_like(x))
        elif kind == "step" and case["s1"]:
            s.update(x=x, out=torch.empty_like(x), stream=_stream().cuda_stream)
        else:
            s.update(x=x.cpu().numpy())
            if kind == "q21" and not case["first"]:
                eng.step(s["x"], 1.0)  # the run's first step: it caches the prompt's keys and values
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "mlp":
        M.call("mk_gemm", C.byref(s["up"]), None)
        M.call("mk_gemm", C.byref(s["down"]), None)
        return {"hidden": s["hid"], "out": s["out"]}
    if kind == "attention":
        b, h, n, d = case["batch"], case["heads"], case["rows"], case["d"]
        M.call("mk_attention", s["q"].data_ptr(), s["k"].data_ptr(), s["vt"].data_ptr(), s["out"].data_ptr(),
               _CODES[case["dt"]], b, h, h, d, n, s["q_pad"], n, s["k_pad"], h * d, n * h * d, 0, case["block"],
               1.0 / math.sqrt(d), None, None)
        return s["out"]
    if kind == "vae":
        s["vae"].decode_device(s["tokens"].data_ptr(), case["h"], case["w"], s["out"].data_ptr())
        M.call("mk_stream_synchronize", s["stream"])  # the decoder's stream is its own: a program waits for it
        return s["out"]
    eng = s["eng"]
    if kind == "sdxl":
        eng.sdxl_forward(s["x"].data_ptr(), case["batch"], case["h"] * case["w"], s["out"].data_ptr())
        return s["out"]
    if kind == "q21":
        if case["first"]:
            eng.begin(s["prompts"][0], case["h"], case["w"], 0)
            return eng.step(s["x"], 1.0)
        return eng.step(s["x"], 0.7)
    if case["s1"]:
        # the one step of a one-step schedule: sigma 1 -> 0
        eng.step_cfg_device(s["x"].data_ptr(), 1.0, 0.0, GUIDANCE, s["out"].data_ptr(), s["stream"])
        return s["out"]
    return eng.step(s["x"], 0.7)


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------

def _vae_flops(h, w):
    """Multiply-adds of the decoder's convolutions and attention, twice."""
    f = 0
    shapes = dict(_vae_names())
    px = 4 * h * w
    for name, shape in shapes.items():
        if len(shape) != 4:
            continue
        level = 0
        if ".up_blocks." in name:
            level = int(name.split(".up_blocks.")[1][0]) + ("upsamplers" in name)
        elif "conv_out" in name:
            level = 3
        f += 2 * px * 4 ** level * math.prod(shape)
    return f + 4 * px * px * 4 * VAE_BASE


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        r, e = case["rows"], 1 if case["wdt"] == "fp8" else 2
        return {"bytes": 2 * DIM * FFN * e + r * (2 * DIM + 2 * 2 * FFN + 4 * DIM), "flops": 4 * r * DIM * FFN}
    if kind == "attention":
        b, h, n, d = case["batch"], case["heads"], case["rows"], case["d"]
        # rows below `block` see their causal prefix, the others all keys
        pairs = case["block"] * (case["block"] + 1) // 2 + (n - case["block"]) * n
        return {"bytes": 4 * 2 * b * h * n * d, "flops": 4 * pairs * d * h * b}
    if kind == "vae":
        n = sum(math.prod(s) * (2 if len(s) == 4 else 4) for _, s in _vae_names())
        px = 256 * case["h"] * case["w"]
        return {"bytes": n + case["h"] * case["w"] * 4 * VAE_Z * 4 + px * 16, "flops": _vae_flops(case["h"], case["w"])}
    size = {"bf16": 2, "f16": 2, "fp8": 1, "f32": 4}
    weights = sum(math.prod(shape) * size[dt] for _, shape, dt, _, _ in _names(case))
    n = case["h"] * case["w"]
    if kind == "sdxl":
        c, b, s = case["dim"], case["batch"], CTX_ROWS
        block = 2 * 18 * c * c * n + 4 * n * n * c + 4 * n * s * c
        weights -= case["depth"] * 2 * c * CTX_DIM * 2  # the context's projections run at begin
        return {"bytes": weights + 2 * b * n * c * 4, "flops": b * (case["depth"] * block + 4 * c * c * n)}
    if kind == "q21":
        s = case["s"]
        rows = n + (s if case["first"] else 0)
        if not case["first"]:
            weights -= 2 * (QTEXT + QDIM) * QDIM  # the text's input layers
        pairs = n * (n + s) + (s * (s + 1) // 2 if case["first"] else 0)
        lin = 2 * rows * (4 * QDIM * QDIM + 3 * QDIM * QFFN) + 4 * n * LATENT * QDIM
        return {"bytes": weights + 2 * n * LATENT * 4, "flops": lin + 4 * pairs * 128 * QHEADS}
    f = 0
    for s in (case["s0"], case["s1"]):
        if s:
            lin = 2 * (n + s) * DIM * (4 * DIM + 2 * FFN)
            f += case["blocks"] * (lin + 4 * (n + s) ** 2 * 128 * HEADS) + 4 * n * LATENT * DIM + 2 * s * TEXT * DIM
    return {"bytes": weights + (2 if case["s1"] else 1) * n * LATENT * 4 + (case["s0"] + case["s1"]) * TEXT * 4,
            "flops": f}


def tolerance(case):
    # about four times each kind's measured distance from exact(), which is its 16-bit operands' and results' rounding
    # (mlp 1.7e-3, attention 2.3e-3, steps 3e-3 to 1e-2 with guidance, q21 4e-3, sdxl 1e-4 to 8e-4, vae 5e-4)
    return {"mlp": {"rel": 6e-3}, "attention": {"rel": 8e-3}, "step": {"rel": 3e-2}, "q21": {"rel": 1.6e-2},
            "sdxl": {"rel": 3e-3}, "vae": {"rel": 2e-3}}[case["kind"]]


# ---------------------------------------------------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------------------------------

class W64:
    """The stored weights' values by name, in 64 bits, and a linear layer over them."""

    def __init__(self, pairs):
        self.t = {}
        for name, t, *scale in pairs:
            t = t.to(F64) if t.dtype != torch.float8_e4m3fn else t.float().to(F64)
            self.t[name] = t * scale[0].to(F64)[:, None] if scale and scale[0] is not None else t

    def __getitem__(self, name):
        return self.t[name]

    def lin(self, name, x):
        y = x @ self.t[name + ".weight"].t()
        b = self.t.get(name + ".bias")
        return y if b is None else y + b


def _silu(x):
    return x / (1 + torch.exp(-x))


def _gelu_tanh(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _ln(x, eps):
    m = x - x.mean(-1, keepdim=True)
    return m / torch.sqrt((m * m).mean(-1, keepdim=True) + eps)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _softmax_v(q, k, v, scale, block=0):
    """[n][d] queries against [m][d] keys: query i sees every key when i >= block, else keys <= i."""
    out = torch.empty(q.shape[0], v.shape[1], dtype=F64, device=q.device)
    for i in range(0, q.shape[0], 4096):
        s = (q[i:i + 4096] @ k.t()).mul_(scale)
        if i < block:
            r = torch.arange(i, i + s.shape[0], device=q.device)[:, None]
            s.masked_fill_((r < block) & (torch.arange(k.shape[0], device=q.device)[None] > r), -math.inf)
        s.sub_(s.amax(1, keepdim=True)).exp_()
        out[i:i + 4096] = (s @ v).div_(s.sum(1, keepdim=True))
    return out


def _attend(q, k, v, heads, scale, block=0):
    """[n][heads d] against [m][heads d]."""
    d = q.shape[1] // heads
    return torch.cat([_softmax_v(q[:, i * d:(i + 1) * d], k[:, i * d:(i + 1) * d], v[:, i * d:(i + 1) * d], scale, block)
                      for i in range(heads)], 1)


def _rope(text, image_frame, h, w):
    """(cos, sin) [text + h w][64] of the three-axis rotary table."""
    t = torch.arange(text, dtype=F64, device="cuda")
    y = torch.arange(h, dtype=F64, device="cuda") - (h - h // 2)
    x = torch.arange(w, dtype=F64, device="cuda") - (w - w // 2)
    pos = [torch.cat([t, torch.full((h * w,), float(image_frame), dtype=F64, device="cuda")]),
           torch.cat([t, y.repeat_interleave(w)]), torch.cat([t, x.repeat(h)])]
    ang = [p[:, None] * 10000.0 ** (-2 * torch.arange(n // 2, dtype=F64, device="cuda") / n)[None]
           for p, n in zip(pos, (16, 56, 56))]
    ang = torch.cat(ang, 1)
    return torch.cos(ang), torch.sin(ang)


def _norm_rotate(x, weight, cs):
    """Per-head RMS norm and rotation of interleaved pairs, x [n][heads 128]."""
    n = x.shape[0]
    y = (_rms(x.reshape(n, -1, 128), 1e-6) * weight).reshape(n, -1, 64, 2)
    c, s = cs[0][:, None], cs[1][:, None]
    return torch.stack([y[..., 0] * c - y[..., 1] * s, y[..., 0] * s + y[..., 1] * c], -1).reshape(n, -1)


def _time(W, sigma):
    f = torch.exp(-math.log(10000.0) * torch.arange(128, dtype=F64, device="cuda") / 128)
    a = 1000.0 * sigma * f
    e = "time_text_embed.timestep_embedder.linear_"
    return _silu(W.lin(e + "2", _silu(W.lin(e + "1", torch.cat([torch.cos(a), torch.sin(a)])[None]))))


def _dual64(W, case, prompt, lat, sigma):
    s, t = prompt.shape[0], _time(W, sigma)
    cs = _rope(s, s, case["h"], case["w"])
    txt = W.lin("txt_in", _rms(prompt, 1e-6) * W["txt_norm.weight"])
    img = W.lin("img_in", lat)
    for i in range(case["blocks"]):
        p = "transformer_blocks.%d." % i
        mi, mt = W.lin(p + "img_mod.1", t)[0].chunk(6), W.lin(p + "txt_mod.1", t)[0].chunk(6)
        xi, xt = _ln(img, 1e-6) * (1 + mi[1]) + mi[0], _ln(txt, 1e-6) * (1 + mt[1]) + mt[0]
        both = lambda a, b: torch.cat([W.lin(p + "attn." + a, xt), W.lin(p + "attn." + b, xi)])  # noqa: E731
        q, k, v = both("add_q_proj", "to_q"), both("add_k_proj", "to_k"), both("add_v_proj", "to_v")
        nw = lambda x, a, b: torch.cat([  # noqa: E731  each stream's own norm weights
            _norm_rotate(x[:s], W[p + "attn.%s.weight" % a], (cs[0][:s], cs[1][:s])),
            _norm_rotate(x[s:], W[p + "attn.%s.weight" % b], (cs[0][s:], cs[1][s:]))])
        o = _attend(nw(q, "norm_added_q", "norm_q"), nw(k, "norm_added_k", "norm_k"), v, HEADS, 1 / math.sqrt(128))
        txt = txt + mt[2] * W.lin(p + "attn.to_add_out", o[:s])
        img = img + mi[2] * W.lin(p + "attn.to_out.0", o[s:])
        for x, m, f in ((img, mi, "img_mlp"), (txt, mt, "txt_mlp")):
            y = _ln(x, 1e-6) * (1 + m[4]) + m[3]
            x += m[5] * W.lin(p + f + ".net.2", _gelu_tanh(W.lin(p + f + ".net.0.proj", y)))
    scale, shift = W.lin("norm_out.linear", t)[0].chunk(2)
    return W.lin("proj_out", _ln(img, 1e-6) * (1 + scale) + shift)


def _q21_64(W, case, prompt, lat, sigma):
    s, p = prompt.shape[0], "transformer_blocks.0."
    rows = lambda name: torch.cat([W.lin(name, _time(W, 0.0)).expand(s, -1),  # noqa: E731  text rows at t = 0
                                   W.lin(name, _time(W, sigma)).expand(lat.shape[0], -1)])
    txt = W.lin("txt_in.out_layer", _gelu_tanh(W.lin("txt_in.in_layer",
                                                     _rms(prompt, 1e-6) * (1 + W["txt_in.text_norm.weight"]))))
    x = torch.cat([txt, W.lin("img_in", lat)])
    cs = _rope(s, s, case["h"], case["w"])
    sc1, g1, sc2, g2 = rows("modulation.1").chunk(4, 1)
    xn = _ln(x, 1e-6) * (1 + sc1)
    q = _norm_rotate(W.lin(p + "attn.to_q", xn), W[p + "attn.norm_q.weight"], cs)
    k = _norm_rotate(W.lin(p + "attn.to_k", xn), W[p + "attn.norm_k.weight"], cs)
    o = _attend(q, k, W.lin(p + "attn.to_v", xn), QHEADS, 1 / math.sqrt(128), s)
    x = x + torch.tanh(g1) * W.lin(p + "attn.to_out.0", o)
    xn = _ln(x, 1e-6) * (1 + sc2)
    m = _silu(W.lin(p + "img_mlp.gate_layer", xn)) * W.lin(p + "img_mlp.proj", xn)
    x = x + torch.tanh(g2) * W.lin(p + "img_mlp.out", m)
    return W.lin("proj_out", (_ln(x, 1e-6) * (1 + rows("norm_out.linear")))[s:])


def _sdxl64(W, case, ctx, x):
    c, n = case["dim"], x.shape[0]
    g = x.reshape(n, 32, c // 32)
    g = g - g.mean((0, 2), keepdim=True)
    g = (g / torch.sqrt((g * g).mean((0, 2), keepdim=True) + 1e-6)).reshape(n, c)
    hs = W.lin("proj_in", g * W["norm.weight"] + W["norm.bias"])
    heads = c // 64
    for i in range(case["depth"]):
        p = "transformer_blocks.%d." % i
        ln = lambda j: _ln(hs, 1e-5) * W[p + "norm%d.weight" % j] + W[p + "norm%d.bias" % j]  # noqa: E731
        y = ln(1)
        q, k, v = (W.lin(p + "attn1.to_" + s, y) for s in "qkv")
        hs = hs + W.lin(p + "attn1.to_out.0", _attend(q, k, v, heads, 0.125))
        q, k, v = W.lin(p + "attn2.to_q", ln(2)), W.lin(p + "attn2.to_k", ctx), W.lin(p + "attn2.to_v", ctx)
        hs = hs + W.lin(p + "attn2.to_out.0", _attend(q, k, v, heads, 0.125))
        a, b = W.lin(p + "ff.net.0.proj", ln(3)).chunk(2, 1)
        hs = hs + W.lin(p + "ff.net.2", a * 0.5 * b * (1 + torch.erf(b / math.sqrt(2))))
    return W.lin("proj_out", hs) + x


def _vae64(W, case, tokens):
    def conv(x, name):  # x [h][w][c], as the sum of its taps' products
        wt, (h, w, c) = W[name + ".weight"], x.shape
        if wt.shape[2] == 1:
            return x @ wt[:, :, 0, 0].t() + W[name + ".bias"]
        xp = torch.zeros(h + 2, w + 2, c, dtype=F64, device=x.device)
        xp[1:-1, 1:-1] = x
        y = W[name + ".bias"].expand(h, w, -1).clone()
        for dy in range(3):
            for dx in range(3):
                y += xp[dy:dy + h, dx:dx + w] @ wt[:, :, dy, dx].t()
        return y

    def norm(x, name):
        return _silu(x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-24) * math.sqrt(x.shape[-1]) * W[name])

    def res(x, p):
        y = conv(norm(conv(norm(x, p + ".norm1.gamma"), p + ".conv1"), p + ".norm2.gamma"), p + ".conv2")
        return y + (conv(x, p + ".conv_shortcut") if p + ".conv_shortcut.weight" in W.t else x)

    h, w = case["h"], case["w"]
    mean = torch.linspace(-0.5, 0.5, VAE_Z, dtype=F64, device="cuda")
    std = torch.linspace(1.0, 2.0, VAE_Z, dtype=F64, device="cuda")
    x = tokens.reshape(h, w, VAE_Z, 2, 2).permute(0, 3, 1, 4, 2).reshape(2 * h, 2 * w, VAE_Z) * std + mean
    x = conv(conv(x, "post_quant_conv"), "decoder.conv_in")
    x = res(x, "decoder.mid_block.resnets.0")
    a, c = "decoder.mid_block.attentions.0.", x.shape[-1]
    y = x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-24) * math.sqrt(c) * W[a + "norm.gamma"]
    q, k, v = conv(y, a + "to_qkv").reshape(-1, 3 * c).chunk(3, 1)
    x = x + conv(_softmax_v(q, k, v, 1 / math.sqrt(c)).reshape(x.shape), a + "proj")
    x = res(x, "decoder.mid_block.resnets.1")
    for i in range(4):
        for j in range(3):
            x = res(x, "decoder.up_blocks.%d.resnets.%d" % (i, j))
        if i < 3:
            x = x.repeat_interleave(2, 0).repeat_interleave(2, 1)
            x = conv(x, "decoder.up_blocks.%d.upsamplers.0.resample.1" % i)
    x = conv(norm(x, "decoder.norm_out.gamma"), "decoder.conv_out").clamp(-1, 1)
    return torch.cat([x, torch.ones_like(x[..., :1])], -1)


def exact(case, seed):
    rng, kind = Rng(seed), case["kind"]
    with torch.no_grad():
        if kind == "mlp":
            x, w1, b1, w2, b2 = _mlp_inputs(case, rng)
            W = W64([("a.weight", *w1), ("a.bias", b1), ("b.weight", *w2), ("b.bias", b2)])
            hid = _gelu_tanh(W.lin("a", x.to(F64)))
            return {"hidden": hid, "out": W.lin("b", hid)}
        if kind == "attention":
            q, k, v = (t.to(F64) for t in _attention_inputs(case, rng))
            return torch.stack([torch.cat([_softmax_v(q[b, i], k[b, i], v[b, i], 1 / math.sqrt(case["d"]), case["block"])
                                           for i in range(case["heads"])], 1) for b in range(case["batch"])])
        if kind == "vae":
            W = W64(_vae_weights(rng))
            return _vae64(W, case, rng.normal(case["h"] * case["w"], 4 * VAE_Z).to(F64))
        W = W64(_weights(case, rng))
        prompts, x = _engine_inputs(case, rng)
        prompts, x = [p.to(F64) for p in prompts], x.to(F64)
        if kind == "sdxl":
            return torch.stack([_sdxl64(W, case, prompts[b], x[b]) for b in range(case["batch"])])
        if kind == "q21":
            return _q21_64(W, case, prompts[0], x, 1.0 if case["first"] else 0.7)
        if not case["s1"]:
            return _dual64(W, case, prompts[0], x, 0.7)
        pos, neg = (_dual64(W, case, p, x, 1.0) for p in prompts)
        return x + (0.0 - 1.0) * (neg + GUIDANCE * (pos - neg))
