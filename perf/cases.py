"""The work that a user of the backend has it do, as cases that can be timed and checked.

Five families, each through a public entry point of ggml_mi355x:
  mul_mat   MUL_MAT on one device-resident weight: tiled fp16, or a quantized type decoded per call
  group     MUL_MATs that share their activations: one pack, one fused launch (Q/K/V, gate/up)
  attn      FLASH_ATTN_EXT on strided views of a KV cache
  moe       MUL_MAT_ID on a quantized expert stack
  layer     one layer's claimed ops handed to graph_compute as host tensors, as ggml hands them over
Quantized weights are ggml blocks quantized here from N(0, 0.02), a trained weight's spread.
Activations are N(0, 1), as after a norm. Sizes are those of the 8B prefill, the quantized MUL_MAT
sweep, the attention and the 128-expert configurations of bench.py and the tests.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ggml-rocket_amd"))
import ggml_mi355x as mx  # noqa: E402

TYPES = {"F16_T": mx.F16_T, "Q8_0": mx.Q8_0, "Q4_0": mx.Q4_0, "Q4_K": mx.Q4_K, "Q6_K": mx.Q6_K, "MXFP4": mx.MXFP4}
EXPERT = {"Q8_0": mx.Q8_0_X, "Q4_K": mx.Q4_K_X, "Q6_K": mx.Q6_K_X, "MXFP4": mx.MXFP4_X}
BITS = {"F16_T": 16.0, "Q8_0": 8.5, "Q4_0": 4.5, "Q4_K": 4.5, "Q6_K": 6.5625, "MXFP4": 4.25}


def listed():
    return [
        # the quantized sweep's smallest call: 32 rows (MIN_M) on a small projection; latency counts
        dict(name="mul_mat_q8_0_m32", kind="mul_mat", wtype="Q8_0", M=32, N=3072, K=3072),
        # a short, ragged prompt on a wide projection
        dict(name="mul_mat_q4_k_m100", kind="mul_mat", wtype="Q4_K", M=100, N=8192, K=3072),
        # a micro-batch on a weight kept in its quantized form (the per-call route)
        dict(name="mul_mat_q6_k_m512", kind="mul_mat", wtype="Q6_K", M=512, N=8192, K=3072),
        # the sweep's largest batch, on a deep and narrow weight
        dict(name="mul_mat_q4_k_m2048", kind="mul_mat", wtype="Q4_K", M=2048, N=3072, K=8192),
        # the 8B model's projections at a 512-token micro-batch, weights resident as tiled fp16
        dict(name="qkv_m512", kind="group", M=512, K=4096, N="4096,1024,1024"),
        dict(name="gate_up_m512", kind="group", M=512, K=4096, N="14336,14336"),
        dict(name="down_m512", kind="mul_mat", wtype="F16_T", M=512, N=4096, K=14336),
        # attention of the 8B model at the last micro-batch of a 2048-token prefill
        dict(name="attn_kv2048", kind="attn", T=512, KV=2048, H=32, HK=8, dk=128, dv=128, softcap=0.0),
        # the same model deep in a long context
        dict(name="attn_kv8192", kind="attn", T=512, KV=8192, H=32, HK=8, dk=128, dv=128, softcap=0.0),
        # absorbed MLA: every query head on one latent KV head
        dict(name="attn_mla_kv4096", kind="attn", T=512, KV=4096, H=16, HK=1, dk=576, dv=512, softcap=0.0),
        # experts' gate / up projection, 512 tokens, top 8 of 128
        dict(name="moe_q4_k_t512", kind="moe", wtype="Q4_K", T=512, E=128, U=8, K=2048, N=768, per_slot=False),
        # one 8B layer through the plugin boundary: host tensors in and out
        dict(name="layer_host_m512", kind="layer", T=512, n_kv=2048, d=4096, ffn=14336, kv_heads=8),
    ]


def _log(rng, lo, hi, step=1):
    """A size spread over the logarithm of [lo, hi], a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(max(round(v / step), -(-lo // step)), hi // step)) * step


def draw(rng):
    kind = rng.choice(["mul_mat"] * 4 + ["group"] * 2 + ["attn"] * 3 + ["moe"] * 2 + ["layer"])
    most = 512 * 28672 * 4096
    if kind == "mul_mat":
        c = dict(kind=kind, wtype=rng.choice(list(TYPES)), M=_log(rng, 1, 2048), N=_log(rng, 1024, 14336, 16),
                 K=_log(rng, 1024, 14336, 256))
        c["M"] = max(1, min(c["M"], most // (c["N"] * c["K"])))
        return c
    if kind == "group":
        K, d = _log(rng, 2048, 5120, 64), _log(rng, 1024, 14336, 64)
        N = rng.choice([[d, d], [d, d // 4 // 16 * 16, d // 4 // 16 * 16]])
        return dict(kind=kind, M=min(_log(rng, 129, 2048), most // (K * sum(N))), K=K, N=",".join(map(str, N)))
    if kind == "attn":
        dk, dv, H, HK = rng.choice([(64, 64, 32, 8), (64, 64, 24, 8), (128, 128, 32, 8), (128, 128, 32, 4), (128, 128, 16, 16),
                                    (192, 128, 16, 16), (256, 256, 16, 8), (576, 512, 16, 1)])
        return dict(kind=kind, T=_log(rng, 16, 512), KV=_log(rng, 1024, 4096 if dk > 128 else 8192), H=H, HK=HK, dk=dk, dv=dv,
                    softcap=rng.choice([0.0, 0.0, 0.0, 50.0]) if dk <= 256 else 0.0)
    if kind == "moe":
        K, N = rng.choice([(2048, 768), (768, 2048), (2048, 1024), (1024, 2048), (2816, 704), (1536, 512)])
        wt = rng.choice(list(EXPERT))
        if wt in ("Q4_K", "Q6_K"):
            K = K // 256 * 256
        return dict(kind=kind, wtype=wt, T=_log(rng, 64, 1024), E=rng.choice([32, 64, 128]), U=rng.choice([2, 4, 6, 8]), K=K, N=N,
                    per_slot=bool(rng.getrandbits(1)))
    d = rng.choice([2048, 3072, 4096])
    return dict(kind=kind, T=512, n_kv=_log(rng, 1024, 2048, 32), d=d, ffn=_log(rng, 2 * d, 3 * d, 256), kv_heads=rng.choice([4, 8]))


# ---- inputs ---------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, device="cuda", generator=g).mul_(std)


def _f16(x):
    """fp16 values as their two bytes."""
    return x.half().contiguous().view(torch.uint8).reshape(*x.shape, 2)


def quantize(wtype, W):
    """(ggml blocks of the rows of W as uint8 [rows][bytes], a function giving the values they stand
    for in 64 bits). Plain round-to-nearest quantizers of the published block formats."""
    rows, K = W.shape
    if wtype == "F16_T":
        h = W.half()
        return h.view(torch.uint8), lambda: h.double()
    if wtype in ("Q8_0", "Q4_0", "MXFP4"):
        x = W.view(rows, K // 32, 32)
        top = x.abs().amax(-1).clamp_min(1e-8)
        if wtype == "MXFP4":
            e = (torch.floor(torch.log2(top)) - 2).clamp(-126, 120)
            v = x / torch.exp2(e)[..., None]
            grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], device=W.device)
            mid = (grid[1:] + grid[:-1]) / 2
            c = torch.bucketize(v.abs().contiguous(), mid)
            code = (c + 8 * (v < 0)).to(torch.uint8)
            q = code[..., :16] | (code[..., 16:] << 4)
            p = torch.cat([(e + 127).to(torch.uint8)[..., None], q], -1)
            return p.reshape(rows, -1), lambda: (torch.where(v < 0, -grid[c], grid[c]).double() * torch.exp2(e.double())[..., None]).view(rows, K)
        d = (top / (127 if wtype == "Q8_0" else 7)).half()
        q = torch.round(x / d.float()[..., None]).clamp(-127 if wtype == "Q8_0" else -8, 127 if wtype == "Q8_0" else 7)
        if wtype == "Q8_0":
            p = torch.cat([_f16(d), q.to(torch.int8).view(torch.uint8)], -1)
        else:
            u = (q + 8).to(torch.uint8)
            p = torch.cat([_f16(d), u[..., :16] | (u[..., 16:] << 4)], -1)
        return p.reshape(rows, -1), lambda: (q.double() * d.double()[..., None]).view(rows, K)
    nb = K // 256
    if wtype == "Q4_K":
        x = W.view(rows, nb, 8, 32)
        lo = (-x.amin(-1)).clamp_min(0)
        s = ((x.amax(-1) + lo) / 15).clamp_min(1e-8)
        d, dm = (s.amax(-1) / 63).half(), (lo.amax(-1) / 63).clamp_min(1e-7).half()
        sc = torch.round(s / d.float()[..., None]).clamp(1, 63)
        mn = torch.round(lo / dm.float()[..., None]).clamp(0, 63)
        ds, dmn = d.float()[..., None] * sc, dm.float()[..., None] * mn
        q = torch.round((x + dmn[..., None]) / ds[..., None]).clamp(0, 15)
        S, Mn, u = sc.to(torch.uint8), mn.to(torch.uint8), q.to(torch.uint8)
        b = torch.cat([S[..., :4] | ((S[..., 4:] >> 4) << 6), Mn[..., :4] | ((Mn[..., 4:] >> 4) << 6),
                       (S[..., 4:] & 15) | ((Mn[..., 4:] & 15) << 4)], -1)
        qs = (u[..., 0::2, :] | (u[..., 1::2, :] << 4)).reshape(rows, nb, 128)
        p = torch.cat([_f16(d), _f16(dm), b, qs], -1)
        return p.reshape(rows, -1), lambda: (q.double() * (d.double()[..., None] * sc.double())[..., None]
                                             - (dm.double()[..., None] * mn.double())[..., None]).view(rows, K)
    assert wtype == "Q6_K", wtype
    x = W.view(rows, nb, 16, 16)
    s = (x.abs().amax(-1) / 31).clamp_min(1e-8)
    d = (s.amax(-1) / 127).half()
    sc = torch.round(s / d.float()[..., None]).clamp(1, 127)
    q = torch.round(x / (d.float()[..., None] * sc)[..., None]).clamp(-32, 31)
    u = (q + 32).to(torch.uint8).view(rows, nb, 2, 4, 32)
    a, b, c, e = u.unbind(3)
    ql = torch.cat([(a & 15) | ((c & 15) << 4), (b & 15) | ((e & 15) << 4)], -1).reshape(rows, nb, 128)
    qh = ((a >> 4) | ((b >> 4) << 2) | ((c >> 4) << 4) | ((e >> 4) << 6)).reshape(rows, nb, 64)
    p = torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _f16(d)], -1)
    return p.reshape(rows, -1), lambda: (q.double() * (d.double()[..., None] * sc.double())[..., None]).view(rows, K)


def _weight(g, wtype, rows, K):
    return quantize(wtype, _normal(g, rows, K, std=0.02))


def _widths(case):
    return [int(n) for n in case["N"].split(",")]


def _attn_inputs(g, case):
    """Q [H][T][dk] as the view ggml permutes it to, K and V as views of a [KV][HK][d] cache (MLA: V is
    the first dv dims of K), a causal mask whose last query sees every key, rows padded to 64."""
    T, KV, H, HK, dk, dv = (case[n] for n in ("T", "KV", "H", "HK", "dk", "dv"))
    q = _normal(g, T, H, dk).transpose(0, 1)
    kc = _normal(g, KV, HK, dk).half()
    k = kc.transpose(0, 1)
    v = k[..., :dv] if dk > 256 else _normal(g, KV, HK, dv).half().transpose(0, 1)
    pad = (KV + 63) // 64 * 64
    j, t = torch.arange(pad, device="cuda")[None, :], torch.arange(T, device="cuda")[:, None]
    mask = torch.zeros(T, pad, dtype=torch.float16, device="cuda").masked_fill_(j > KV - T + t, float("-inf"))
    return q, k, v, mask


def _moe_inputs(g, case):
    T, E, U, K = (case[n] for n in ("T", "E", "U", "K"))
    b = _normal(g, T, U if case["per_slot"] else 1, K)
    # router logits with some experts more popular than others
    logits = _normal(g, T, E) + _normal(g, E, std=0.5)
    return b, logits.topk(U, dim=1).indices.to(torch.int32).contiguous()


LAYER = ("q", "k", "v", "o", "gate", "up", "down")


def _layer_shapes(case):
    d, ffn, kvd = case["d"], case["ffn"], case["kv_heads"] * 128
    return dict(q=(d, d), k=(kvd, d), v=(kvd, d), o=(d, d), gate=(ffn, d), up=(ffn, d), down=(d, ffn))


def _layer_inputs(g, case):
    T, n_kv, kvh = case["T"], case["n_kv"], case["kv_heads"]
    x, act = _normal(g, T, case["d"]), _normal(g, T, case["ffn"])
    kc, vc = _normal(g, n_kv, kvh, 128).half(), _normal(g, n_kv, kvh, 128).half()
    j, t = torch.arange(n_kv, device="cuda")[None, :], torch.arange(T, device="cuda")[:, None]
    mask = torch.zeros(T, n_kv, dtype=torch.float16, device="cuda").masked_fill_(j > n_kv - T + t, float("-inf"))
    return x, act, kc, vc, mask


def _prepare_layer(g, case):
    T, n_kv, d, ffn, kvh = (case[n] for n in ("T", "n_kv", "d", "ffn", "kv_heads"))
    heads, hd = d // 128, 128
    be = mx.Backend()
    be.set_quant_resident(1)   # quantized weights held as fp16, the setting to use on this card
    gr = mx.Graph()
    host = lambda t: t.contiguous().cpu().numpy().reshape(-1)
    shapes = _layer_shapes(case)
    w = {}
    for n in LAYER:
        blocks, _ = _weight(g, "Q4_K", *shapes[n])
        w[n] = gr._new(mx.Q4_K, [shapes[n][1], shapes[n][0]], name=f"blk.0.{n}.weight", data=host(blocks))
    x, act, kc, vc, mask = _layer_inputs(g, case)
    X, A = gr._new(mx.F32, [d, T], data=host(x)), gr._new(mx.F32, [ffn, T], data=host(act))
    K, V = gr._new(mx.F16, [hd, kvh, n_kv], data=host(kc)), gr._new(mx.F16, [hd, kvh, n_kv], data=host(vc))
    Mk = gr._new(mx.F16, [n_kv, T], data=host(mask))
    out = {n: np.zeros((T, shapes[n][0]), dtype=np.float32) for n in LAYER}
    out["attn"] = np.zeros((T, d), dtype=np.float32)
    mm = lambda n, src: gr._new(mx.F32, [shapes[n][0], T], op=mx.OP_MUL_MAT, srcs=(w[n], src), data=out[n])
    q, k, v = mm("q", X), mm("k", X), mm("v", X)
    qv = gr.permute_view(q, [hd, T, heads, 1], [4, d * 4, hd * 4, d * 4 * T])
    kv = gr.permute_view(K, [hd, n_kv, kvh, 1], [2, kvh * hd * 2, hd * 2, kvh * hd * 2 * n_kv])
    vv = gr.permute_view(V, [hd, n_kv, kvh, 1], [2, kvh * hd * 2, hd * 2, kvh * hd * 2 * n_kv])
    fa = gr._new(mx.F32, [hd, heads, T], op=mx.OP_FLASH_ATTN_EXT, srcs=(qv, kv, vv, Mk), data=out["attn"])
    ctypes.memmove(ctypes.addressof(fa.op_params), (ctypes.c_float * 3)(1.0 / math.sqrt(hd), 0.0, 0.0), 12)
    fa2 = gr.permute_view(fa, [d, T, 1, 1], [4, d * 4, d * 4 * T, d * 4 * T])
    calls = [[q, k, v], [fa, fa2, mm("o", fa2)], [mm("gate", X), mm("up", X)], [mm("down", A)]]
    return dict(kind="layer", be=be, graph=gr, calls=calls, out=out)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "layer":
        return _prepare_layer(g, case)
    s = dict(kind=kind, case=dict(case))
    if kind == "mul_mat":
        M, N, K, wt = case["M"], case["N"], case["K"], case["wtype"]
        blocks, _ = _weight(g, wt, N, K)
        if wt == "F16_T":
            s["w"] = mx.tile_f16(mx.F16, blocks.view(torch.uint8).reshape(-1), N, K)
        else:
            s["w"] = mx.upload_weight(TYPES[wt], blocks, N, K)
        s["x"], s["out"] = _normal(g, M, K), torch.empty(M, N, device="cuda")
        need = int(mx.lib().mi355x_mul_mat_workspace_for(TYPES[wt], N, K, M))
        s["ws"] = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")
    elif kind == "group":
        M, K = case["M"], case["K"]
        s["x"], s["outs"] = _normal(g, M, K), []
        for N in _widths(case):
            blocks, _ = _weight(g, "F16_T", N, K)
            w = mx.tile_f16(mx.F16, blocks.view(torch.uint8).reshape(-1), N, K)
            s["outs"].append((w, N, 0, N, torch.empty(M, N, device="cuda")))
    elif kind == "attn":
        s["q"], s["k"], s["v"], s["mask"] = _attn_inputs(g, case)
        s["out"] = torch.empty(case["T"], case["H"], case["dv"], device="cuda")
        need = mx.flash_attn_workspace(s["q"], s["k"], s["v"], s["mask"], s["out"], 1.0 / math.sqrt(case["dk"]), case["softcap"])
        s["ws"] = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")
    else:
        N, K, E = case["N"], case["K"], case["E"]
        blocks, _ = _weight(g, case["wtype"], E * N, K)
        s["w"] = mx.upload_weight(EXPERT[case["wtype"]], blocks, E * N, K)
        s["b"], s["ids"] = _moe_inputs(g, case)
        s["out"] = torch.empty(case["T"], case["U"], N, device="cuda")
    return s


def run(s):
    if s["kind"] == "layer":
        for nodes in s["calls"]:
            if s["be"].compute(nodes) != mx.STATUS_SUCCESS:
                raise RuntimeError("graph_compute failed")
        return s["out"]
    c = s["case"]
    if s["kind"] == "mul_mat":
        return mx.mul_mat(TYPES[c["wtype"]], s["w"], c["N"], c["K"], s["x"], out=s["out"], workspace=s["ws"])
    if s["kind"] == "group":
        a16, sc = mx.pack_act(s["x"], tiled=True)
        mx.gemm(mx.F16_T, a16, sc, c["K"], s["outs"])
        return [o[4] for o in s["outs"]]
    if s["kind"] == "attn":
        return mx.flash_attn(s["q"], s["k"], s["v"], s["mask"], 1.0 / math.sqrt(c["dk"]), softcap=c["softcap"], out=s["out"],
                             workspace=s["ws"])
    return mx.mul_mat_id(EXPERT[c["wtype"]], s["w"], c["E"], c["N"], c["K"], s["b"], s["ids"], out=s["out"])


# ---- what a pass cannot do without, and how far a correct result may be off -------------------------

def work(case):
    kind = case["kind"]
    if kind == "mul_mat":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=N * K * BITS[case["wtype"]] / 8 + 4 * M * (N + K), flops=2 * M * N * K)
    if kind == "group":
        M, N, K = case["M"], sum(_widths(case)), case["K"]
        return dict(bytes=2 * N * K + 4 * M * (N + K), flops=2 * M * N * K)
    if kind == "attn":
        T, KV, H, HK, dk, dv = (case[n] for n in ("T", "KV", "H", "HK", "dk", "dv"))
        seen = T * KV - T * (T - 1) // 2   # the (query, key) pairs the causal mask leaves
        kv = HK * KV * 2 * (dk if dk > 256 else dk + dv)
        return dict(bytes=4 * T * H * (dk + dv) + kv + 2 * T * KV, flops=2 * H * seen * (dk + dv))
    if kind == "moe":
        T, E, U, K, N = (case[n] for n in ("T", "E", "U", "K", "N"))
        rows = T * U
        return dict(bytes=min(E, rows) * N * K * BITS[case["wtype"]] / 8 + 4 * rows * N + 4 * T * (U if case["per_slot"] else 1) * K,
                    flops=2 * rows * N * K)
    T, n_kv, shapes = case["T"], case["n_kv"], _layer_shapes(case)
    mm = sum(n * k for n, k in shapes.values())
    seen = T * n_kv - T * (T - 1) // 2
    host = 4 * T * (3 * case["d"] + case["ffn"] + sum(n for n, _ in shapes.values())) + 2 * n_kv * (2 * case["kv_heads"] * 128 + T)
    return dict(bytes=2 * mm + host, flops=2 * T * mm + 4 * case["d"] * seen)


def tolerance(case):
    """About four times what the path shows against exact(): fp16 operands and P with 32-bit sums are
    2e-4 to 3e-4 off (the layer's chained attention and O projection 6e-4); a Q4_K weight decoded in
    packed fp16, its scale and minimum rounded first, 7e-4."""
    if case["kind"] == "layer" or case.get("wtype") == "Q4_K":
        return {"rel": 2.5e-3, "max": 2.5e-2}
    return {"rel": 1.2e-3, "max": 1.2e-2}


# ---- the results in 64 bits -------------------------------------------------------------------------

def _attend(q, k, v, mask, scale, softcap):
    """softmax(cap(scale q.k) + mask) . v per head in 64 bits: [T][H][dv]."""
    H, HK = q.shape[0], k.shape[0]
    out = torch.empty(q.shape[1], H, v.shape[2], dtype=torch.float64, device=q.device)
    m = mask[:, :k.shape[1]].double()
    for h in range(H):
        kh, vh = k[h // (H // HK)].double().contiguous(), v[h // (H // HK)].double().contiguous()
        s = (q[h].double() @ kh.t().contiguous()) * scale
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        out[:, h] = torch.softmax(s + m, dim=-1) @ vh
    return out


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "mul_mat":
        W = _weight(g, case["wtype"], case["N"], case["K"])[1]()
        return _normal(g, case["M"], case["K"]).double() @ W.t()
    if kind == "group":
        x = _normal(g, case["M"], case["K"]).double()
        return [x @ _weight(g, "F16_T", N, case["K"])[1]().t() for N in _widths(case)]
    if kind == "attn":
        return _attend(*_attn_inputs(g, case), 1.0 / math.sqrt(case["dk"]), case["softcap"])
    if kind == "moe":
        T, E, U, K, N = (case[n] for n in ("T", "E", "U", "K", "N"))
        W = _weight(g, case["wtype"], E * N, K)[1]().view(E, N, K)
        b, ids = _moe_inputs(g, case)
        rows = b.double().expand(T, U, K).reshape(T * U, K)
        out = torch.empty(T * U, N, dtype=torch.float64, device="cuda")
        flat = ids.reshape(-1)
        for e in range(E):
            sel = (flat == e).nonzero().reshape(-1)
            if sel.numel():
                out[sel] = rows[sel] @ W[e].t()
        return out.view(T, U, N)
    shapes = _layer_shapes(case)
    w = {n: _weight(g, "Q4_K", *shapes[n])[1]() for n in LAYER}
    x, act, kc, vc, mask = _layer_inputs(g, case)
    T, d = case["T"], case["d"]
    out = {n: x.double() @ w[n].t() for n in ("q", "k", "v", "gate", "up")}
    out["down"] = act.double() @ w["down"].t()
    q = out["q"].view(T, d // 128, 128).transpose(0, 1)
    out["attn"] = _attend(q, kc.transpose(0, 1), vc.transpose(0, 1), mask, 1.0 / math.sqrt(128), 0.0).reshape(T, d)
    out["o"] = out["attn"] @ w["o"].t()
    return out
