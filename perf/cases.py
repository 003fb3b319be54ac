"""Performance cases of the quantised-matmul path: the calls a decode or prefill
program makes through the Python surface, over the sizes it makes them at.

A case is a dict of plain values; `listed()` names twelve, `draw(rng)` gives
more of the same ranges.  `prepare` builds what the program holds before the
call (weights in the device layouts, inputs, workspaces, and for the small
steps the HIP graph that a decode loop replays), `run` is one pass, `exact`
the same outputs from plain torch in 64 bits.

Kinds:
  gemm_w4a16     one projection, matmul_w4a16, any M
  layer_w4a16    every projection of a decoder layer with its norms: rms_norm,
                 the shared-input projections, the output projection, rms_norm,
                 gate + up + silu and down (the one-launch MLP at M = 1)
  lm_head_w4a16  vocabulary projection and greedy token (fused at M = 1,
                 matmul + argmax for several rows)
  lm_head_w8a8   the same over an int8 weight
  mlp_w8a8       the W8A8 MLP block with its norm and activation quantisation
"""
from __future__ import annotations

import gc
import importlib.util
import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

ROOT = Path(__file__).resolve().parent.parent
GROUP, SLAB = 128, 64
EPS = 1e-6
H, I = 1024, 3584                                    # hidden and MLP width of the 24-layer model
PROJ = {"linear": (6144, 2048), "full": (4096, 512, 512)}   # qkv + z; q (with its gate), k, v
ATTN = 2048                                          # width of the attention output
SHAPES = ((1024, 1024), (1024, 3584), (3584, 1024), (1024, 6144), (2048, 1024), (1024, 2048), (1024, 1000), (2048, 1031))
VOCAB = 248094
GRAPH_ROWS = 256                                     # steps of up to this many rows are replayed from a HIP graph


def _pkg():
    name = "minicpmv_amd"
    if name not in sys.modules:
        pkg = ROOT / "minicpm-v-4.6-orangepi_amd"
        spec = importlib.util.spec_from_file_location(name, pkg / "__init__.py", submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ---------------------------------------------------------------------- cases --
def listed():
    return [
        # the smallest call: one decode projection, where the launch is most of the time
        {"name": "gemv_1024", "kind": "gemm_w4a16", "M": 1, "K": 1024, "N": 1024, "zero_bias": 0},
        # one token through the 24 layers' projections, replayed from a graph
        {"name": "decode_layers_w4a16", "kind": "layer_w4a16", "M": 1, "layers": 24, "attn": "linear", "zero_bias": 0},
        # five tokens at once: a small batch, or drafted tokens being verified
        {"name": "batch5_layers_w4a16", "kind": "layer_w4a16", "M": 5, "layers": 24, "attn": "linear", "zero_bias": 0},
        # a short text prompt
        {"name": "prompt77_layers_w4a16", "kind": "layer_w4a16", "M": 77, "layers": 4, "attn": "full", "zero_bias": 1},
        # an image's tokens with a question
        {"name": "prefill1100_layer_w4a16", "kind": "layer_w4a16", "M": 1100, "layers": 1, "attn": "linear", "zero_bias": 0},
        # one projection of a long multi-image prompt, the largest call
        {"name": "prefill8192_gemm_w4a16", "kind": "gemm_w4a16", "M": 8192, "K": 1024, "N": 3584, "zero_bias": 0},
        # the greedy token of a decode step over the whole vocabulary
        {"name": "lm_head_w4a16", "kind": "lm_head_w4a16", "M": 1, "V": VOCAB, "zero_bias": 0},
        # logits and tokens of several rows (batched decode, verification)
        {"name": "lm_head_batch6_w4a16", "kind": "lm_head_w4a16", "M": 6, "V": VOCAB, "zero_bias": 0},
        # the int8 head's greedy token
        {"name": "lm_head_w8a8", "kind": "lm_head_w8a8", "M": 1, "V": VOCAB, "scales": "reference"},
        # one token through the 24 layers' W8A8 MLP blocks
        {"name": "decode_mlp_w8a8", "kind": "mlp_w8a8", "M": 1, "layers": 24, "scales": "reference"},
        # a short prompt through W8A8 MLP blocks
        {"name": "prompt40_mlp_w8a8", "kind": "mlp_w8a8", "M": 40, "layers": 4, "scales": "f32"},
        # a long prompt through one W8A8 MLP block
        {"name": "prefill3000_mlp_w8a8", "kind": "mlp_w8a8", "M": 3000, "layers": 1, "scales": "f32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layers(M):
    return 24 if M <= 16 else 4 if M <= GRAPH_ROWS else 1


def draw(rng):
    kind = rng.choice(("gemm_w4a16", "gemm_w4a16", "layer_w4a16", "layer_w4a16", "lm_head_w4a16", "lm_head_w8a8",
                       "mlp_w8a8", "mlp_w8a8"))
    case = {"kind": kind}
    if kind == "gemm_w4a16":
        K, N = rng.choice(SHAPES)
        case.update(M=_log_int(rng, 1, min(8192, 8192 * 1024 * 3584 // (K * N))), K=K, N=N, zero_bias=rng.randrange(2))
    elif kind == "layer_w4a16":
        M = _log_int(rng, 1, 1100)
        case.update(M=M, layers=_layers(M), attn=rng.choice(sorted(PROJ)), zero_bias=rng.randrange(2))
    elif kind == "lm_head_w4a16":
        case.update(M=_log_int(rng, 1, 32), V=_log_int(rng, 15506, VOCAB), zero_bias=rng.randrange(2))
    elif kind == "lm_head_w8a8":
        case.update(M=_log_int(rng, 1, 32), V=_log_int(rng, 15506, VOCAB), scales=rng.choice(("reference", "f32")))
    else:
        M = _log_int(rng, 1, 3000)
        case.update(M=M, layers=_layers(M), scales=rng.choice(("reference", "f32")))
    return case


# -------------------------------------------------------------------- weights --
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 2654435761 % (1 << 62))


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std


def _w4_parts(g, K, N, zero_bias):
    """q, z [int32] and s [fp16] of N(0, 0.02) weights, asymmetric int4 per group of 128 k."""
    w = _randn(g, K // GROUP, GROUP, N, std=0.02)
    lo, hi = w.amin(1), w.amax(1)
    s = ((hi - lo) / 15).half()
    z = torch.round(-lo / s.float()).clamp_(1, 15)
    q = (torch.round(w / s.float()[:, None]) + z[:, None]).clamp_(0, 15).to(torch.int32)
    return q.view(K, N), z.to(torch.int32), s


def _pack_w4(q, z, s, zero_bias):
    """The slab-64 layout of include/mcv_quant.h."""
    K, N = q.shape
    ns = -(-N // SLAB)
    pad = ns * SLAB - N
    q, zs, sp = (torch.nn.functional.pad(t, (0, pad)) for t in (q, z - zero_bias, s))
    zs[:, N:] = 0
    order = torch.tensor([0, 2, 4, 6, 1, 3, 5, 7], device=q.device)
    nib = q.view(K // 32, 4, 8, ns, SLAB).index_select(2, order)
    words = torch.zeros(K // 32, 4, ns, SLAB, dtype=torch.int32, device=q.device)
    zw = torch.zeros(K // GROUP, ns * 8, dtype=torch.int32, device=q.device)
    zn = zs.view(K // GROUP, ns * 8, 8)
    for i in range(8):
        words |= nib[:, :, i] << (4 * i)
        zw |= zn[:, :, i] << (4 * i)
    qw = words.permute(2, 0, 3, 1).contiguous().view(torch.uint8).reshape(-1)
    return _pkg().W4A16QuantizedWeight(qw, sp.contiguous().view(torch.int16), zw, K, N, zero_bias)


def _w4(g, K, N, zero_bias, keep):
    q, z, s = _w4_parts(g, K, N, zero_bias)
    if keep:                                         # exact(): the weight's values
        return ((q.view(K // GROUP, GROUP, N) - z[:, None]) * s.double()[:, None]).view(K, N)
    return _pack_w4(q, z, s, zero_bias)


def _w8(g, K, N, keep):
    """Per-channel int8 of N(0, 0.02) weights; the fp16 scale truncated as a loader stores it."""
    w = _randn(g, K, N, std=0.02)
    s32 = (w.abs().amax(0) / 127).clamp_min(1e-8)
    s16 = s32.half()
    s16 = torch.where(s16.float() > s32, (s16.view(torch.int16) - 1).view(torch.float16), s16)
    q = torch.round(w / s32).clamp_(-127, 127).to(torch.int8)
    if keep:
        return SimpleNamespace(q=q.double(), f32=s32.double(), reference=s16.double())
    ns, kb = -(-N // SLAB), -(-K // GROUP) * 4
    t = torch.nn.functional.pad(q, (0, ns * SLAB - N, 0, kb * 32 - K))
    t = t.view(kb, 2, 16, ns, 2, 32).permute(3, 0, 4, 1, 5, 2).contiguous().reshape(-1)
    pkg = _pkg()
    return pkg.W8A8QuantizedWeight(t, s16, s32, K, N, pkg.W8_TILED)


def _rows(g, M, K):
    return _randn(g, M, K).half()


def _inputs(case, seed, keep):
    """Weights (their values where `keep`) and activations of a case, from the seed alone."""
    g, kind, M = _gen(seed), case["kind"], case["M"]
    st = SimpleNamespace(case=case, M=M)
    if kind == "gemm_w4a16":
        st.w = _w4(g, case["K"], case["N"], case["zero_bias"], keep)
        st.x = _rows(g, M, case["K"])
    elif kind in ("lm_head_w4a16", "lm_head_w8a8"):
        V = case["V"]
        st.w = _w4(g, H, V, case["zero_bias"], keep) if kind == "lm_head_w4a16" else _w8(g, H, V, keep)
        # a hidden state leans towards the embedding of the token it predicts
        pick = torch.randint(V, (M,), generator=g, device="cuda")
        lean = _lean(st.w, pick, keep, kind)
        st.x = (_randn(g, M, H) + lean).half()
    else:
        st.layers = []
        for _ in range(case["layers"]):
            y = SimpleNamespace()
            if kind == "layer_w4a16":
                zb = case["zero_bias"]
                y.proj = [_w4(g, H, n, zb, keep) for n in PROJ[case["attn"]]]
                y.o = _w4(g, ATTN, H, zb, keep)
                y.gate, y.up, y.down = (_w4(g, k, n, zb, keep) for k, n in ((H, I), (H, I), (I, H)))
                y.x, y.h, y.attn = _rows(g, M, H), _rows(g, M, H), _rows(g, M, ATTN)
                y.gx, y.gh = ((1 + _randn(g, H, std=0.1)).half() for _ in range(2))
            else:
                y.gate, y.up, y.down = (_w8(g, k, n, keep) for k, n in ((H, I), (H, I), (I, H)))
                y.h, y.gh = _rows(g, M, H), (1 + _randn(g, H, std=0.1)).half()
            st.layers.append(y)
    return st


def _lean(w, pick, keep, kind):
    """Rows of about unit size along the picked columns, read back from the packed weight (or its values)."""
    if keep:
        cols = (w if kind == "lm_head_w4a16" else w.q * w.f32)[:, pick].t()
        return (cols / cols.norm(dim=1, keepdim=True) * 12.0).float()
    slab, lane = pick // SLAB, pick % SLAB
    ns = -(-w.N // SLAB)
    if kind == "lm_head_w4a16":
        words = w.qweight.view(torch.int32).view(ns, H // 32, SLAB, 4)[slab, :, lane]            # [M, C, 4]
        shift = torch.tensor([0, 16, 4, 20, 8, 24, 12, 28], device=words.device, dtype=torch.int32)
        q = ((words[..., None] >> shift) & 15).reshape(len(pick), H)
        z = ((w.zeros[:, pick >> 3] >> ((pick & 7) * 4).int()) & 15) + w.zero_bias               # [G, M]
        s = w.scales.view(torch.float16)[:, pick].double()
        cols = ((q.view(-1, H // GROUP, GROUP) - z.t()[..., None]) * s.t()[..., None]).reshape(len(pick), H)
    else:
        t = w.w_int8.view(ns, H // 32, 2, 2, 32, 16)[slab, :, lane // 32, :, lane % 32]
        cols = t.reshape(len(pick), H).double() * w.w_scale_f32[pick].double()[:, None]
    return (cols / cols.norm(dim=1, keepdim=True) * 12.0).float()


# ------------------------------------------------------------------------ run --
def _step_gemm(st):
    return _pkg().matmul_w4a16(st.x, st.w)


def _step_lm_head_w4a16(st):
    pkg = _pkg()
    if st.M == 1:
        return st.head.launch(st.x, st.logits[0]), st.logits
    pkg.matmul_w4a16(st.x, st.w, out=st.logits)
    return pkg.argmax_last_dim(st.logits, out=st.tokens), st.logits


def _step_lm_head_w8a8(st):
    pkg = _pkg()
    if st.M == 1:
        return pkg.lm_head_argmax_w8a8_fused(st.x, st.w, st.case["V"], st.workspace, logits=st.logits, token=st.tokens,
                                             use_f32_scale=st.f32), st.logits
    xq, xs = _quant(pkg, st.x, st.f32)
    pkg.matmul_w8a8(xq, xs, st.w, out=st.logits, use_f32_scale=st.f32)
    return pkg.argmax_last_dim(st.logits, out=st.tokens), st.logits


def _step_layer_w4a16(st):
    pkg = _pkg()
    for y in st.layers:
        pkg.matmul_w4a16_multi(pkg.rms_norm(y.x, y.gx, EPS, out=y.nx), y.proj, outs=y.outs)
        pkg.matmul_w4a16(y.attn, y.o, out=y.oo)
        pkg.rms_norm(y.h, y.gh, EPS, out=y.nh)
        if y.mlp is not None:
            y.mlp(y.nh, out=y.mo)
        else:
            pkg.mlp_gate_up_silu_w4a16(y.nh, y.gate, y.up, out=y.act)
            pkg.matmul_w4a16(y.act, y.down, out=y.mo)
    return [*st.proj, st.oo, st.mo]


def _step_mlp_w8a8(st):
    pkg, f32, M = _pkg(), st.f32, st.M
    for y in st.layers:
        if y.mlp is not None:
            y.mlp(pkg.rms_norm(y.h, y.gh, EPS, out=y.nh), out=y.mo)
            continue
        s16 = None if f32 else torch.empty(M, dtype=torch.float16, device="cuda")
        _, xq, xs, xs16 = pkg.rms_norm_w8a8_quantize(y.h, y.gh, EPS, want_normed=False, x_scale_f16=s16)
        xs = xs if f32 else xs16
        if M <= 4:
            act = pkg.mlp_gate_up_silu_w8a8(xq, xs, y.gate, y.up, use_f32_scale=f32)
        else:
            act = pkg.silu_mul(pkg.matmul_w8a8(xq, xs, y.gate, use_f32_scale=f32),
                               pkg.matmul_w8a8(xq, xs, y.up, use_f32_scale=f32))
        aq, asc = _quant(pkg, act, f32)
        pkg.matmul_w8a8(aq, asc, y.down, out=y.mo, use_f32_scale=f32)
    return st.mo


STEPS = {"gemm_w4a16": _step_gemm, "lm_head_w4a16": _step_lm_head_w4a16, "lm_head_w8a8": _step_lm_head_w8a8,
         "layer_w4a16": _step_layer_w4a16, "mlp_w8a8": _step_mlp_w8a8}


def prepare(case, seed):
    pkg = _pkg()
    st = _inputs(case, seed, keep=False)
    kind, M = case["kind"], case["M"]
    half = dict(dtype=torch.float16, device="cuda")
    st.f32 = case.get("scales") == "f32"
    st.graph = None
    if kind in ("lm_head_w4a16", "lm_head_w8a8"):
        st.logits = torch.empty(M, case["V"], **half)
        st.tokens = torch.empty(M, dtype=torch.int64, device="cuda")
        if M == 1 and kind == "lm_head_w4a16":
            st.head = pkg.LmHeadW4A16(st.w, case["V"])
        elif M == 1:
            st.workspace = torch.zeros(pkg.lm_head_workspace_bytes(case["V"]), dtype=torch.uint8, device="cuda")
    elif kind == "layer_w4a16":
        L = case["layers"]
        st.proj = [torch.empty(L, M, n, **half) for n in PROJ[case["attn"]]]
        st.oo, st.mo = torch.empty(L, M, H, **half), torch.empty(L, M, H, **half)
        for i, y in enumerate(st.layers):
            y.outs, y.oo, y.mo = [t[i] for t in st.proj], st.oo[i], st.mo[i]
            y.nx, y.nh, y.act = torch.empty(M, H, **half), torch.empty(M, H, **half), torch.empty(M, I, **half)
            y.mlp = pkg.DecodeMlpW4A16(y.gate, y.up, y.down) if M == 1 else None
    elif kind == "mlp_w8a8":
        st.mo = torch.empty(case["layers"], M, H, **half)
        for i, y in enumerate(st.layers):
            y.nh, y.mo = torch.empty(M, H, **half), st.mo[i]
            y.mlp = pkg.DecodeMlpW8A8(y.gate, y.up, y.down, precision=case["scales"]) if M == 1 else None
    if kind in ("layer_w4a16", "mlp_w8a8") and M <= GRAPH_ROWS:
        # a decode loop (or a server's short prompts) replays its step from a graph
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            STEPS[kind](st)
        torch.cuda.synchronize()
        gc.collect()                                 # no older graph may be destroyed while this one is captured
        st.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st.graph, stream=side):
            st.out = STEPS[kind](st)
    return st


def _quant(pkg, x, f32):
    if f32:
        q, s, _ = pkg.w8a8_quantize(x)
        return q, s
    q, s, s16 = pkg.w8a8_quantize(x, x_scale_f16=torch.empty(x.shape[0], dtype=torch.float16, device=x.device))
    return q, s16


def run(state):
    if state.graph is not None:
        state.graph.replay()
        return state.out
    return STEPS[state.case["kind"]](state)


# ------------------------------------------------------------------- measures --
def _w4_bytes(K, N):
    return K * N // 2 + (K // GROUP) * N * 5 // 2


def work(case):
    kind, M = case["kind"], case["M"]
    if kind == "gemm_w4a16":
        K, N = case["K"], case["N"]
        return {"bytes": _w4_bytes(K, N) + 2 * M * (K + N), "flops": 2 * M * K * N}
    if kind == "lm_head_w4a16":
        V = case["V"]
        return {"bytes": _w4_bytes(H, V) + 2 * M * (H + V) + 8 * M, "flops": 2 * M * H * V}
    if kind == "lm_head_w8a8":
        V = case["V"]
        scale = 4 if case["scales"] == "f32" else 2
        return {"bytes": V * (H + scale) + 2 * M * (H + V) + 8 * M, "flops": 2 * M * H * V}
    if kind == "layer_w4a16":
        ns = PROJ[case["attn"]]
        b = sum(_w4_bytes(H, n) for n in ns) + _w4_bytes(ATTN, H) + 2 * _w4_bytes(H, I) + _w4_bytes(I, H) + 4 * H
        b += 2 * M * (H + sum(ns) + ATTN + H + H + H)
        f = 2 * M * (H * sum(ns) + ATTN * H + 3 * H * I)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    scale = 4 if case["scales"] == "f32" else 2
    b = 3 * H * I + scale * (2 * I + H) + 2 * H + 4 * M * H
    return {"bytes": case["layers"] * b, "flops": case["layers"] * 6 * M * H * I}


def tolerance(case):
    # One rounding of the output to fp16 and, for the W4A16 prefill kernels,
    # one of each weight; the layers and MLPs add the fp16 roundings of the
    # normed row and of the activation.  W8A8 sums are exact, but an
    # activation one ulp off can move its int8 value by one step.  Measured
    # against exact(): 2.1e-4 (one output rounding) to 2.7e-4 (rounded
    # weights), layers 2.1e-4 to 5.6e-4, W8A8 MLPs 4e-4 to 1.8e-3.
    if case["kind"] == "gemm_w4a16" or case["kind"] == "lm_head_w4a16":
        return {"rel": 1.2e-3, "max": 8e-3}
    if case["kind"] == "layer_w4a16":
        return {"rel": 1.6e-3, "max": 1.2e-2}
    if case["kind"] == "lm_head_w8a8":
        return {"rel": 1e-3, "max": 4e-3}
    return {"rel": 2e-3, "max": 2e-2}


def _rms64(x, gamma):
    v = x.double()
    return v * torch.rsqrt(v.square().mean(1, keepdim=True) + EPS) * gamma.double()


def _quant64(x, f32):
    """The activation quantiser's definition over fp16 rows: int values and scale."""
    x = x.half().float()
    s = (x.abs().amax(1) / torch.tensor(127.0, device=x.device)).clamp_min(1e-8)
    v = (x * (1.0 / s)[:, None]).clamp(-128, 127)
    q = torch.trunc(torch.where(v >= 0, v + 0.5, v - 0.5)).double()
    return q, (s if f32 else s.half()).double()


def _mm8(q, xs, w, scales):
    return (q @ w.q) * getattr(w, scales) * xs[:, None]


def exact(case, seed):
    st = _inputs(case, seed, keep=True)
    kind = case["kind"]
    if kind == "gemm_w4a16":
        return st.x.double() @ st.w
    if kind == "lm_head_w4a16":
        return None, st.x.double() @ st.w
    if kind == "lm_head_w8a8":
        q, xs = _quant64(st.x, case["scales"] == "f32")
        return None, _mm8(q, xs, st.w, case["scales"])
    proj, oo, mo = [], [], []
    for y in st.layers:
        if kind == "layer_w4a16":
            nx, nh = _rms64(y.x, y.gx), _rms64(y.h, y.gh)
            proj.append([nx @ w for w in y.proj])
            oo.append(y.attn.double() @ y.o)
            mo.append((torch.nn.functional.silu(nh @ y.gate) * (nh @ y.up)) @ y.down)
        else:
            sc = case["scales"]
            q, xs = _quant64(_rms64(y.h, y.gh), sc == "f32")
            g, u = _mm8(q, xs, y.gate, sc).half().double(), _mm8(q, xs, y.up, sc).half().double()
            q, xs = _quant64(torch.nn.functional.silu(g) * u, sc == "f32")
            mo.append(_mm8(q, xs, y.down, sc))
    if kind == "mlp_w8a8":
        return torch.stack(mo)
    return [*(torch.stack(t) for t in zip(*proj)), torch.stack(oo), torch.stack(mo)]
