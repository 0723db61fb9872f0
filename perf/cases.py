"""The performance cases of this library: what a program that serves a model
with a foveated KV cache has it do, through the public entry points.

Three kinds of call:

  decode    one decode step's attention on handles that the program keeps:
            ``FoveatedHandle`` / ``TurboFoveatedHandle`` called once
            (``layers`` 0), or a step over several layers captured in one HIP
            graph and replayed (``layers`` > 0); with ``drain`` the step's
            spike drain on the device follows the call.
  compress  a layer's prompt K and V into tiers: ``CompressHandle`` (fp8
            keys, INT4 values) or ``turbo_compress_keys`` / ``_values``.
  prefill   the whole way from a layer's prompt K and V to the first decode
            token: ``FoveatedKVCache.update``, ``compress`` and the first
            ``attend_fused_with_spikes`` (which builds the layer's handle).

Shapes are B sequences, ``Hkv`` KV heads of ``D`` dims serving ``G`` query
heads each, ``S`` prompt tokens and ``n_dec`` decoded ones.  Inputs are made
on the GPU from the seed: K, V ~ N(0, 1) with a few outlier key channels, as
the benchmark's.
"""

import math

import torch

from foveated_kv_amd import FoveatedKVCache, TierConfig, ext, turbo
from foveated_kv_amd.promotion import PromotionPipeline

MARGIN = 10.0  # the spike margin the cache layers use

_DEFAULTS = {"dtype": "float16", "format": "fp8", "v_group": 0, "k_scale": False, "importance": False,
             "spike_k": 1, "n_dec": 0, "layers": 0, "drain": False}


def _case(name, kind, B, Hkv, G, D, S, **options):
    c = {"kind": kind, "B": B, "Hkv": Hkv, "G": G, "D": D, "S": S, **_DEFAULTS, **options}
    return {"name": name, **c} if name else c


def listed():
    return [
        # a short chat on a half-billion-parameter model, called layer by
        # layer: host time, launch and latency
        _case("decode_small_512", "decode", 1, 2, 7, 64, 512, n_dec=16),
        # a 7B model at 4K with a chat's answer under way: a decode step's
        # attention over eight layers replayed as one HIP graph
        _case("decode_7b_4k_graph", "decode", 1, 8, 4, 128, 4096, n_dec=64, dtype="bfloat16", layers=8),
        # batched serving at 16K, the benchmark's headline shape
        _case("decode_7b_16k_b8", "decode", 8, 8, 4, 128, 16384),
        # a 70B model's long document: up to 32 spiking tokens a head and
        # their drain, the near tier's headroom being used up
        _case("decode_70b_64k_top32_drain", "decode", 1, 8, 8, 128, 65536, importance=True, spike_k=32,
              n_dec=32, drain=True),
        # the TurboQuant far tier at 8K, four layers in a graph
        _case("decode_turbo_8k_b4_graph", "decode", 4, 8, 4, 128, 8192, format="turbo", layers=4),
        # per-head-scaled keys and group-32 values at an odd length and an
        # odd group, float32 activations
        _case("decode_scaled_g32_odd", "decode", 3, 4, 5, 128, 11003, dtype="float32", v_group=32, k_scale=True,
              n_dec=37),
        # prompt compression: the smallest (latency), the batched one, the
        # long one with every option (bf16 activations)
        _case("compress_small_512", "compress", 1, 2, 7, 64, 512, dtype="float32"),
        _case("compress_7b_16k_b8", "compress", 8, 8, 4, 128, 16384),
        _case("compress_70b_64k_importance", "compress", 1, 8, 8, 128, 65536, dtype="bfloat16", importance=True,
              k_scale=True, v_group=32),
        # TurboQuant prompt compression, an odd length
        _case("compress_turbo_8k_b4", "compress", 4, 8, 4, 128, 8191, format="turbo"),
        # time to the first decode token after the model's prefill
        _case("prefill_7b_8k_b4", "prefill", 4, 8, 4, 128, 8192),
        _case("prefill_turbo_3k_d64", "prefill", 2, 4, 7, 64, 3001, format="turbo", dtype="bfloat16"),
    ]


# most elements of K that a drawn case of a kind has (the largest listed one's)
_MOST = {"decode": 8 * 8 * 16384 * 128, "compress": 8 * 8 * 16384 * 128, "prefill": 4 * 8 * 8192 * 128}


def draw(rng):
    kind = rng.choice(["decode", "decode", "compress", "compress", "prefill"])
    fmt = rng.choice(["fp8", "fp8", "turbo"])
    D = rng.choice([64, 128, 128])
    most = _MOST["prefill"] if fmt == "turbo" else _MOST[kind]
    B, Hkv = rng.choice([1, 1, 2, 3, 4, 8]), rng.choice([1, 2, 4, 8, 8])
    S = int(math.exp(rng.uniform(math.log(256), math.log(65536))))
    S = max(256, min(S, most // (B * Hkv * D)))
    o = {"dtype": rng.choice(["float16", "float16", "bfloat16", "float32"])}
    if fmt == "turbo":
        o["format"] = "turbo"
    else:
        o["v_group"] = rng.choice([0, 0, 32])
        o["k_scale"] = rng.random() < 0.25
    if kind == "compress" and fmt == "fp8":
        o["importance"] = rng.random() < 0.4
    if kind == "decode":
        o["n_dec"] = rng.choice([0, rng.randint(1, 128)])
        o["layers"] = rng.choice([0, 0, 4])
        if fmt == "fp8" and Hkv <= 4 and rng.random() < 0.4:
            o.update(spike_k=rng.choice([4, 32]), drain=rng.random() < 0.5, layers=0)
    return _case(None, kind, B, Hkv, rng.choice([1, 4, 5, 7, 8]), D, S, **o)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _dtype(case):
    return getattr(torch, case["dtype"])


def _layer_inputs(case, seed, layer=0):
    """Prompt K, V, the query, decode rows and importance of one layer."""
    B, H, D, S = case["B"], case["Hkv"], case["D"], case["S"]
    g = torch.Generator(device="cuda").manual_seed(1000003 * seed + layer)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)

    # activations of the case's type (a decode step's tiers come from fp16 ones)
    dt = torch.float16 if case["kind"] == "decode" else _dtype(case)
    k = normal(B, H, S, D)
    k[..., torch.randperm(D, generator=g, device="cuda")[:4]] *= 8.0
    x = {"k": k.to(dt), "v": normal(B, H, S, D).to(dt), "q": normal(B, H * case["G"], 1, D).to(_dtype(case))}
    x["dk"] = normal(B, H, case["n_dec"], D).half() if case["n_dec"] else None
    x["dv"] = normal(B, H, case["n_dec"], D).half() if case["n_dec"] else None
    x["imp"] = normal(B, H, S) if case["importance"] else None
    return x


def _config(case):
    c = TierConfig(compress_method=case["format"], v_group=case["v_group"], k_scale=case["k_scale"],
                   spike_k=case["spike_k"])
    if case["drain"]:  # late in a long answer: promotions have used the near tier's headroom up
        c.promo_headroom_pct, c.promo_headroom_min = 0.0, 0
    return c


def _cache(case, x):
    cache = FoveatedKVCache(_config(case))
    cache.update(x["k"], x["v"], 0)
    cache.compress(importance=x["imp"])
    return cache


def _handle(case, layer):
    if case["format"] == "turbo":
        tc = layer._turbo_constants
        return turbo.TurboFoveatedHandle(layer.near_k, layer.near_v, layer.turbo_far_k_indices,
                                         layer.turbo_far_k_signs, layer.turbo_far_k_norm, layer.turbo_far_k_gamma,
                                         layer.turbo_far_v_packed, layer.turbo_far_v_scale, layer.near_valid,
                                         tc.Pi, tc.S, tc.centroids, spike_margin=MARGIN)
    return ext.FoveatedHandle(layer.near_k, layer.near_v, layer.far_k, layer.far_v, layer.far_v_scale,
                              layer.far_v_zero, layer.near_valid, spike_margin=MARGIN,
                              far_k_scale=layer.far_k_scale, spike_k=case["spike_k"])


def _prepare_decode(case, seed):
    calls, state = [], {"case": case, "step": 0}
    for i in range(max(case["layers"], 1)):
        x = _layer_inputs(case, seed, i)
        layer = _cache(case, x).layers[0]
        handle = _handle(case, layer)
        calls.append((handle, x["q"], x["dk"], x["dv"]))
        if case["drain"]:
            pipe = PromotionPipeline(1, max_per_drain=32 * case["Hkv"], spike_k=case["spike_k"])
            pipe.register_archive_tensors(0, layer.archive_k, layer.archive_v, layer.archive_idx, device=True)
            pipe.register_blob(0, handle)
            state.update(pipe=pipe, far_idx=layer.far_idx.contiguous())
    state["calls"] = calls
    if case["layers"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for handle, q, dk, dv in calls:
                handle(q, dk, dv)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["outs"] = [handle(q, dk, dv) for handle, q, dk, dv in calls]
    return state


def prepare(case, seed):
    if case["kind"] == "decode":
        return _prepare_decode(case, seed)
    x = _layer_inputs(case, seed)
    if case["kind"] == "compress":
        if case["format"] == "turbo":
            return {"case": case, "x": x, "constants": turbo.get_turbo_constants(case["D"])}
        return {"case": case, "x": x, "handle": ext.CompressHandle(_config(case).to_native())}
    return {"case": case, "x": x, "config": _config(case)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _tensors(layer, names):
    return {n: getattr(layer, n) for n in names if getattr(layer, n) is not None}


_FP8_TIERS = ("near_k", "near_v", "far_k", "far_v", "far_v_scale", "far_v_zero", "near_valid", "archive_k",
              "archive_v", "near_idx", "far_idx", "far_k_scale")
_TURBO_TIERS = ("near_k", "near_v", "near_valid", "archive_k", "archive_v", "near_idx", "far_idx",
                "turbo_far_k_indices", "turbo_far_k_signs", "turbo_far_k_norm", "turbo_far_k_gamma",
                "turbo_far_v_packed", "turbo_far_v_scale")


def run(state):
    case = state["case"]
    if case["kind"] == "decode":
        if case["layers"]:
            state["graph"].replay()
            return state["outs"]
        handle, q, dk, dv = state["calls"][0]
        out, flags, tokens = handle(q, dk, dv)
        if case["drain"]:
            state["pipe"].drain_spikes_device(0, flags, tokens, state["far_idx"], state["step"])
            state["step"] += 1
        return [out, flags, tokens]
    x = state["x"]
    if case["kind"] == "compress":
        if case["format"] == "turbo":
            return list(turbo.turbo_compress_keys(x["k"], state["constants"])) + \
                list(turbo.turbo_compress_values(x["v"]))
        return _tensors(state["handle"].compress_layer(x["k"], x["v"], importance=x["imp"]), _FP8_TIERS)
    cache = FoveatedKVCache(state["config"])
    cache.update(x["k"], x["v"], 0)
    cache.compress(importance=x["imp"])
    layer = cache.layers[0]
    out, flags, tokens = layer.attend_fused_with_spikes(x["q"])
    return {"out": out, "flags": flags, "tokens": tokens,
            "tiers": _tensors(layer, _TURBO_TIERS if case["format"] == "turbo" else _FP8_TIERS)}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _bounds(case):
    """Sinks, window, near tokens of the middle, far tokens, near slots."""
    S = case["S"]
    sinks = min(4, S)
    window = min(32, S - sinks)
    mid = S - sinks - window
    near_mid = min(max(max(int(S * 0.10), sinks + window) - sinks - window, 0), mid)
    R = sinks + window + near_mid
    slots = R if case["drain"] else R + max(int(R * 0.5), 8)
    return sinks, window, near_mid, mid - near_mid, R, slots


def work(case):
    B, H, G, D, S = case["B"], case["Hkv"], case["G"], case["D"], case["S"]
    F, R, slots = _bounds(case)[3:]
    item = torch.finfo(_dtype(case)).bits // 8
    if case["format"] == "turbo":
        far = D // 4 + D // 8 + 4 + D // 4 + 2 * (D // 32)
    else:
        far = D + D // 2 + 4 * (D // 32 if case["v_group"] else 1)
    q = B * H * G * D * (item + 2) + B * H * G * 4 * (1 + case["spike_k"])  # query, output, spikes
    if case["kind"] == "decode":
        row = q + B * H * (4 * D * (R + case["n_dec"]) + far * F) + 4 * H
        flops = 4 * B * H * G * D * (R + F + case["n_dec"])
        n = max(case["layers"], 1)
        return {"bytes": n * row, "flops": n * flops}
    tokens = B * H * S
    if case["kind"] == "compress" and case["format"] == "turbo":
        return {"bytes": tokens * (2 * D * item + far), "flops": tokens * 6 * D * D}
    nbytes = tokens * 2 * D * item + B * H * (4 * D * slots + (far + 4 * D) * F)
    nbytes += B * H * (4 * S + 4 * slots + 4 * F) if case["importance"] else 0
    flops = B * H * F * 6 * D * D if case["format"] == "turbo" else 0
    if case["kind"] == "prefill":
        nbytes += q + 4 * B * H * (slots + F)  # and the index sets
        flops += 4 * B * H * G * D * (R + F)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # tiers are copies, codes and correctly rounded scales: the same bits
    if case["kind"] == "compress" and case["format"] == "fp8":
        return "exact"
    # TurboQuant codes and signs follow from 32-bit sums of D products: one
    # that lies within rounding of a boundary may fall on either side, and
    # with it its token's residual and signs (measured against 64 bits: 4e-6
    # of the bytes), and a norm may round to the next fp16 (7e-6 of their 2-norm)
    if case["kind"] == "compress":
        return {"rel": 3e-5, "max": 2e-3, "differ": 2e-5 + 1.0 / (case["B"] * case["Hkv"] * case["S"])}
    # attention: fp16 softmax weights and an fp16 result over fp32 sums
    # (2.3e-4 from 64 bits, 2e-3 of the root mean square at most), for
    # TurboQuant on an fp16 rotated query and matrices (1.1e-3); a spike may
    # fall on either side of its threshold, two tokens with scores within
    # rounding may swap
    k = 4.0 if case["format"] == "turbo" else 1.0
    return {"rel": 1e-3 * k, "max": 1e-2 * k, "differ": 5e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _e4m3(x):
    """fp16 -> the value of its E4M3 code: 3 mantissa bits to nearest even,
    zero below 2^-6, 448 from 256 on (before or after rounding)."""
    m, e = torch.frexp(x.double())
    r = torch.round(m * 16) / 16 * torch.exp2(e.double())
    big = torch.sign(r) * 448.0
    r = torch.where((x.double().abs() >= 256.0) | (r.abs() >= 256.0), big, r)
    return torch.where(x.double().abs() < 2.0 ** -6, torch.zeros_like(r), r)


def _int4(v, group):
    """Rows of `group` values -> (dequantised values, scale, zero): 16 levels
    from the row's minimum, in fp32 as the format asks, scale and zero fp16."""
    f = v.float().unflatten(-1, (-1, group))
    lo, hi = f.amin(-1, keepdim=True), f.amax(-1, keepdim=True)
    # (torch divides by a Python number through its reciprocal on a GPU)
    scale = ((hi - lo) / torch.full_like(lo, 15.0)).clamp_min(1e-8)
    code = torch.floor(((f - lo) / scale).double() + 0.5).clamp(0, 15)
    deq = code.double() * scale.half().double() + lo.half().double()
    return deq.flatten(-2), scale.double().squeeze(-1), lo.double().squeeze(-1)


def _split(case, x):
    """Token positions (B, H, .) of the near and the far tier, in slot order."""
    sinks, window, near_mid, _, _, _ = _bounds(case)
    B, H, S = case["B"], case["Hkv"], case["S"]
    rank = x["imp"][..., sinks:S - window] if x["imp"] is not None else \
        torch.arange(S - window - sinks, device="cuda", dtype=torch.float32).expand(B, H, -1)
    order = torch.sort(rank, dim=-1, stable=True).indices + sinks  # later tokens win ties
    n = order.shape[-1] - near_mid
    far, mid = order[..., :n].sort(-1).values, order[..., n:].sort(-1).values
    first = torch.arange(sinks, device="cuda").expand(B, H, -1)
    last = torch.arange(S - window, S, device="cuda").expand(B, H, -1)
    return torch.cat([first, mid, last], -1), far


def _take(t, idx):
    return t.half().gather(2, idx.unsqueeze(-1).expand(-1, -1, -1, t.shape[-1]))


_LEVELS = (-1.0, -0.333333, 0.333333, 1.0)


def _turbo_keys(k):
    """Effective keys, norms and residual norms of fp16 keys."""
    D = k.shape[-1]
    tc = turbo.get_turbo_constants(D)  # the format's matrices and levels
    Pi, S, c, b = (t.cuda().double() for t in (tc.Pi, tc.S, tc.centroids, tc.boundaries))
    k = k.double()
    n = k.norm(dim=-1, keepdim=True)
    coarse = c[torch.bucketize((k / n.clamp_min(1e-8)) @ Pi.T.contiguous(), b, right=True)] @ Pi
    r = k - n * coarse
    gamma = r.norm(dim=-1, keepdim=True)
    sign = torch.where(r @ S.T.contiguous() >= 0, 1.0, -1.0).double()
    eff = n.half().double() * coarse + (math.sqrt(math.pi / 2) / D) * gamma.half().double() * (sign @ S)
    return eff, n.squeeze(-1), gamma.squeeze(-1)


def _turbo_values(v):
    f = v.float().unflatten(-1, (-1, 32))
    scale = f.abs().amax(-1, keepdim=True).clamp_min(1e-8)
    code = torch.round((f / scale + 1.0) * 1.5).clamp(0, 3).long()
    lv = torch.tensor(_LEVELS, device="cuda", dtype=torch.float64)[code]
    return (lv * scale.half().double()).flatten(-2), scale.double().squeeze(-1)


def _exact_layer(case, x, attend=True):
    """Tiers (float ones in 64 bits) and, with ``attend``, the output."""
    B, H, G, D = case["B"], case["Hkv"], case["G"], case["D"]
    near, far = _split(case, x)
    R, slots = near.shape[-1], _bounds(case)[5]
    fk, fv = _take(x["k"], far), _take(x["v"], far)
    pad = (0, 0, 0, slots - R)
    nk, nv = (torch.nn.functional.pad(_take(x[t], near), pad) for t in ("k", "v"))
    t = {"near_k": nk, "near_v": nv, "archive_k": fk, "archive_v": fv}
    if case["format"] == "turbo":
        ek, t["turbo_far_k_norm"], t["turbo_far_k_gamma"] = _turbo_keys(fk)
        ev, t["turbo_far_v_scale"] = _turbo_values(fv)
    else:
        ks = torch.ones((B, H), device="cuda")
        if case["k_scale"]:
            ks = fk.float().abs().amax((2, 3)) / torch.full_like(ks, 240.0)
            t["far_k_scale"] = ks
        ek = _e4m3((fk.float() / ks[..., None, None]).half()) * ks[..., None, None].double()
        ev, t["far_v_scale"], t["far_v_zero"] = _int4(fv, case["v_group"] or D)
        if not case["v_group"]:
            t["far_v_scale"], t["far_v_zero"] = t["far_v_scale"].squeeze(-1), t["far_v_zero"].squeeze(-1)
    if not attend:
        return {n: u.double() for n, u in t.items()}, None
    q = x["q"].half().double().reshape(B, H, G, D)
    out = torch.empty((B, H * G, 1, D), dtype=torch.float64, device="cuda")
    for i in range(B):
        ka = [nk[i, :, :R].double(), ek[i]] + ([x["dk"][i].double()] if x["dk"] is not None else [])
        va = [nv[i, :, :R].double(), ev[i]] + ([x["dv"][i].double()] if x["dv"] is not None else [])
        s = q[i] @ torch.cat(ka, 1).transpose(1, 2).contiguous() / math.sqrt(D)
        out[i] = (torch.softmax(s, -1) @ torch.cat(va, 1)).reshape(H * G, 1, D)
    return {n: u.double() for n, u in t.items()}, out


def exact(case, seed):
    if case["kind"] == "decode":
        outs = [[_exact_layer(case, _layer_inputs(case, seed, i))[1], None, None]
                for i in range(max(case["layers"], 1))]
        return outs if case["layers"] else outs[0]
    x = _layer_inputs(case, seed)
    if case["kind"] == "compress":
        if case["format"] == "turbo":
            _, n, gamma = _turbo_keys(x["k"].half())
            return [None, None, n, gamma, None, _turbo_values(x["v"].half())[1]]
        return _exact_layer(case, x, attend=False)[0]
    tiers, out = _exact_layer(case, x)
    return {"out": out, "flags": None, "tokens": None, "tiers": tiers}
