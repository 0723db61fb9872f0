"""GPU parity: the HIP library (through the C ABI) against the CPU oracle.

Codes and tier partitions must be bit-exact; attention outputs within
max-abs 2e-3 and cosine >= 0.9999 of the oracle (kernel semantics and the
reference dequant+SDPA formulation); spike flags/tokens equal except where
the oracle itself shows a near tie.
"""

import ctypes
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from _parity import ATOL, COS, run_attention  # noqa: F401  (ATOL/COS: the tolerance of every case)
from _parity import flush as _flush


@pytest.fixture(scope="module")
def fkv():
    import foveated_kv_amd
    from foveated_kv_amd import _lib

    _lib.load()
    assert torch.cuda.is_available(), "GPU tests need a ROCm device"
    assert foveated_kv_amd.is_available(), "libfkv.so loaded but no gfx950 device"
    return foveated_kv_amd


def _np(t):
    return t.detach().cpu().numpy()


def _cfg(fkv, **kw):
    from foveated_kv_amd import ext

    c = ext.TierConfig()
    c.promo_headroom_min = kw.get("promo_headroom_min", 8)
    c.v_group = kw.get("v_group", 0)
    return c


# ---------------------------------------------------------------------------
# compression: bit-exact vs the oracle
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("B,H,S,D,dtype", [
    (1, 2, 512, 64, "f16"), (1, 8, 4096, 128, "f16"), (2, 2, 300, 128, "bf16"),
    (1, 2, 700, 64, "f32"), (1, 1, 37, 128, "f16"), (1, 2, 20, 64, "f16"), (3, 3, 1000, 128, "f16"),
])
def test_compress_bit_exact(fkv, orc, B, H, S, D, dtype):
    from foveated_kv_amd import ext, synthetic

    _flush(f"compress B={B} H={H} S={S} D={D} {dtype}")
    k, v = synthetic.make_kv(B, H, S, D, seed=S + D)
    if dtype == "bf16":
        kt = torch.from_numpy(k.astype(np.float32)).to(torch.bfloat16)
        vt = torch.from_numpy(v.astype(np.float32) * 3).to(torch.bfloat16)
        k16 = kt.float().numpy().astype(np.float16)
        v16 = vt.float().numpy().astype(np.float16)
    elif dtype == "f32":
        rng = np.random.default_rng(1)
        kf = rng.standard_normal((B, H, S, D)).astype(np.float32)
        vf = rng.standard_normal((B, H, S, D)).astype(np.float32)
        kt, vt = torch.from_numpy(kf), torch.from_numpy(vf)
        k16, v16 = kf.astype(np.float16), vf.astype(np.float16)
    else:
        kt, vt = torch.from_numpy(k), torch.from_numpy(v)
        k16, v16 = k, v
    cl = ext.CompressHandle(_cfg(fkv)).compress_layer(kt.cuda(), vt.cuda())
    torch.cuda.synchronize()
    ref = orc.compress_layer(k16, v16)
    assert np.array_equal(_np(cl.near_k).view(np.uint16), ref["near_k"].view(np.uint16))
    assert np.array_equal(_np(cl.near_v).view(np.uint16), ref["near_v"].view(np.uint16))
    assert np.array_equal(_np(cl.far_k), ref["far_k"])
    assert np.array_equal(_np(cl.far_v), ref["far_v"])
    assert np.array_equal(_np(cl.far_v_scale).view(np.uint16), ref["far_v_scale"].view(np.uint16))
    assert np.array_equal(_np(cl.far_v_zero).view(np.uint16), ref["far_v_zero"].view(np.uint16))
    assert np.array_equal(_np(cl.near_valid), ref["near_valid"])
    assert np.array_equal(_np(cl.archive_k).view(np.uint16), ref["archive_k"].view(np.uint16))
    assert np.array_equal(_np(cl.archive_v).view(np.uint16), ref["archive_v"].view(np.uint16))
    assert cl.n_near_actual == ref["tb"]["R_actual"]


def test_compress_exhaustive_fp16_patterns(fkv, orc):
    """Every fp16 bit pattern through the GPU E4M3 encoder, plus INT4 rows
    with exact .5 ties, constant rows and saturating magnitudes."""
    from foveated_kv_amd import ext

    D, S = 128, 1024
    tb = orc.tier_boundaries(S)
    F = tb["far_count"]
    assert F * D >= 65536
    rng = np.random.default_rng(9)
    k = rng.standard_normal((1, 1, S, D)).astype(np.float16)
    pats = np.arange(65536, dtype=np.uint16).view(np.float16)
    far = k[0, 0, tb["mid_start"]:tb["mid_start"] + F].reshape(-1)
    far[:65536] = pats
    k[0, 0, tb["mid_start"]:tb["mid_start"] + F] = far.reshape(F, D)
    v = rng.standard_normal((1, 1, S, D)).astype(np.float16)
    fv = v[0, 0, tb["mid_start"]:tb["mid_start"] + F]
    fv[0] = 0.0
    fv[0, 1] = 15.0
    fv[0, 2:10] = np.arange(8) + 0.5  # exact ties with scale 1
    fv[1] = 3.0  # constant row
    fv[2] = np.linspace(-60000, 60000, D).astype(np.float16)  # near fp16 max
    fv[3] = np.linspace(-1e-6, 1e-6, D).astype(np.float16)  # subnormal range
    cl = ext.CompressHandle(_cfg(fkv)).compress_layer(torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    torch.cuda.synchronize()
    ref = orc.compress_layer(k, v)
    assert np.array_equal(_np(cl.far_k), ref["far_k"])
    assert np.array_equal(_np(cl.far_v), ref["far_v"])
    assert np.array_equal(_np(cl.far_v_scale).view(np.uint16), ref["far_v_scale"].view(np.uint16))
    assert np.array_equal(_np(cl.far_v_zero).view(np.uint16), ref["far_v_zero"].view(np.uint16))


# ---------------------------------------------------------------------------
# fused attention
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("args", [
    dict(B=1, Hq=14, Hkv=2, D=64, S=512, n_dec=16, seed=1),      # config 1
    dict(B=1, Hq=32, Hkv=8, D=128, S=4096, n_dec=64, seed=2, heavy_tail=True),  # config 2
    dict(B=1, Hq=4, Hkv=4, D=64, S=256, n_dec=0, seed=3),        # no GQA
    dict(B=2, Hq=8, Hkv=2, D=128, S=512, n_dec=7, seed=4),
    dict(B=1, Hq=64, Hkv=8, D=128, S=2048, n_dec=3, seed=5),     # G = 8, small grid: rows of 4 heads
    dict(B=1, Hq=32, Hkv=2, D=64, S=700, n_dec=5, seed=6),       # G = 16, small grid: four rows of 4 heads
    dict(B=1, Hq=6, Hkv=2, D=128, S=36, n_dec=2, seed=7),        # no far tier
    dict(B=1, Hq=8, Hkv=2, D=64, S=40, n_dec=0, seed=8),         # 4 far tokens
    dict(B=3, Hq=12, Hkv=4, D=64, S=333, n_dec=70, seed=9),      # ragged tiles
    dict(B=1, Hq=64, Hkv=8, D=128, S=32768, n_dec=5, seed=10),   # 32 splits x 8 heads: records exceed LDS
    dict(B=1, Hq=32, Hkv=4, D=64, S=16384, n_dec=3, seed=11),    # the same at D = 64
    dict(B=4, Hq=40, Hkv=2, D=128, S=4096, n_dec=5, seed=12),    # G = 20: a 16-head and a 4-head row
    dict(B=1, Hq=12, Hkv=2, D=64, S=600, n_dec=2, seed=13),      # small grid: rows of 4 heads, G = 6
    dict(B=2, Hq=48, Hkv=4, D=128, S=8192, n_dec=9, seed=14),    # G = 12: rows of three head quads
    dict(B=1, Hq=40, Hkv=4, D=64, S=16384, n_dec=4, seed=15),    # G = 10 at D = 64: three quads
])
def test_attention_parity(fkv, orc, args):
    run_attention(fkv, orc, **args)


@pytest.mark.parametrize("sharp", ["near", "all"])
@pytest.mark.parametrize("args", [dict(B=1, Hq=14, Hkv=2, D=64, S=512, n_dec=16, seed=61),     # C1 shape
                                  dict(B=1, Hq=32, Hkv=8, D=128, S=4096, n_dec=64, seed=62)],  # C2 shape
                         ids=["c1", "c2"])
def test_attention_sharp_softmax_value_outliers(fkv, orc, args, sharp):
    """Every head's weight on three tokens (near, far, decode) at scores
    30-31 with value rows x8 (plant_sharp): the P.V weights of such tokens
    are the large ones, so their rounding to fp16 matrix-core operands shows
    most here.  The outputs reach ~20, where the fp16 output's own rounding
    (half an ulp: 3.9e-3 to 7.8e-3) exceeds 2e-3, so the bar applies beyond
    that rounding (run_attention).  Checked against the kernel restatement,
    and against the formulation: at the bar when the far row keeps its
    values ("near"); with the far row x8 too ("all") the formulation's fp16
    dequantisation of far values alone moves it 5e-3 from the kernel
    semantics, which the check allows on top of the bar."""
    run_attention(fkv, orc, sharp=sharp, **args)


# Rows of 16-head workgroups whose last head quad is only partly filled
# (fkv_attn_plan gives 16 heads per row for each): G = 7 and 5 fill two
# quads with 3 and 1 heads in the second, G = 14 four quads with 2 in the
# last -- common model shapes (Hq 28 / Hkv 4, Hq 40 / Hkv 8, Hq 56 / Hkv 4).
PARTIAL = [
    dict(B=1, Hq=28, Hkv=4, D=128, S=32768, n_dec=5, seed=51),   # G = 7, 64 splits
    dict(B=8, Hq=28, Hkv=4, D=128, S=8192, n_dec=0, seed=52, spikes=0.02),  # G = 7, 8 splits
    dict(B=1, Hq=40, Hkv=8, D=128, S=32768, n_dec=3, seed=53),   # G = 5
    dict(B=1, Hq=56, Hkv=4, D=128, S=16384, n_dec=2, seed=54),   # G = 14: four quads
    dict(B=2, Hq=28, Hkv=4, D=64, S=8192, n_dec=0, seed=55),     # G = 7 at D = 64
]


@pytest.mark.parametrize("vg", [0, 32])
@pytest.mark.parametrize("args", PARTIAL, ids=[f"B{a['B']}_Hq{a['Hq']}_Hkv{a['Hkv']}_D{a['D']}_S{a['S']}"
                                               for a in PARTIAL])
def test_attention_partial_quad_rows(fkv, orc, args, vg):
    from foveated_kv_amd import _lib

    out = (ctypes.c_int64 * 8)()
    tb = orc.tier_boundaries(args["S"], promo_headroom_min=8)
    assert _lib.load().fkv_attn_plan(args["B"], args["Hkv"], args["D"], tb["N_near_padded"], tb["far_count"],
                                     args["Hq"], args["n_dec"], 256, 2 if vg else 0, out) == 0
    assert out[0] == 16 and (args["Hq"] // args["Hkv"]) % 4 != 0  # 16-head rows, last quad partial
    run_attention(fkv, orc, v_group=vg, **args)


# D = 64 rows split for two workgroups per CU: many rows of one and two
# quads, in whole groups of 8 rows (split merge within an XCD) and not
TWO_PER_CU = [
    dict(B=33, Hq=16, Hkv=4, D=64, S=2200, n_dec=3, seed=56),                # 132 rows, 3 splits
    dict(B=18, Hq=28, Hkv=4, D=64, S=4400, n_dec=0, seed=57, spikes=0.02),   # 72 rows of two quads, 7 splits
]


@pytest.mark.parametrize("vg", [0, 32])
@pytest.mark.parametrize("args", TWO_PER_CU, ids=[f"B{a['B']}_Hq{a['Hq']}_S{a['S']}" for a in TWO_PER_CU])
def test_attention_two_workgroups_per_cu(fkv, orc, args, vg):
    from foveated_kv_amd import _lib

    out = (ctypes.c_int64 * 8)()
    tb = orc.tier_boundaries(args["S"], promo_headroom_min=8)
    assert _lib.load().fkv_attn_plan(args["B"], args["Hkv"], 64, tb["N_near_padded"], tb["far_count"],
                                     args["Hq"], args["n_dec"], 256, 2 if vg else 0, out) == 0
    assert 256 < out[1] * out[2] <= 512
    # against the kernel's oracle only: at these sizes the formulation's fp16
    # dequantisation leaves that oracle by up to 1.6e-3 by itself, and half an
    # fp16 unit of an output past 2 is 1e-3 more
    run_attention(fkv, orc, v_group=vg, check_formulation=False, **args)


GROUP32 = [
    dict(B=1, Hq=14, Hkv=2, D=64, S=512, n_dec=16, seed=31),
    dict(B=1, Hq=32, Hkv=8, D=128, S=4096, n_dec=64, seed=32, heavy_tail=True),
    dict(B=2, Hq=8, Hkv=2, D=128, S=700, n_dec=7, seed=33, spikes=0.02),
    dict(B=1, Hq=32, Hkv=2, D=64, S=700, n_dec=5, seed=34),      # two head groups
    dict(B=3, Hq=12, Hkv=4, D=64, S=333, n_dec=70, seed=35),     # ragged tiles
    dict(B=1, Hq=8, Hkv=2, D=128, S=1000, n_dec=3, seed=36, near_valid_delta=5),
    dict(B=2, Hq=36, Hkv=4, D=128, S=8192, n_dec=5, seed=37),    # G = 9: rows of three head quads
]


@pytest.mark.parametrize("args", GROUP32, ids=[f"B{a['B']}_Hq{a['Hq']}_D{a['D']}_S{a['S']}" for a in GROUP32])
def test_attention_group32_parity(fkv, orc, args):
    """fp8 K + group-32 INT4 V: compress and fused attention against the
    oracle with one value scale / zero per 32 dims."""
    run_attention(fkv, orc, v_group=32, **args)


@pytest.mark.parametrize("B,H,S,D", [(1, 2, 512, 64), (2, 3, 1000, 128), (1, 1, 37, 128)])
def test_compress_group32_bit_exact(fkv, orc, B, H, S, D):
    from foveated_kv_amd import ext, synthetic

    _flush(f"compress group-32 B={B} H={H} S={S} D={D}")
    k, v = synthetic.make_kv(B, H, S, D, seed=S + 1)
    v = (v * (4.0 ** np.arange(D // 32)).repeat(32)).astype(np.float16)
    cl = ext.CompressHandle(_cfg(fkv, v_group=32)).compress_layer(torch.from_numpy(k).cuda(),
                                                                  torch.from_numpy(v).cuda())
    torch.cuda.synchronize()
    ref = orc.compress_layer(k, v, v_group=32)
    for n in ("near_k", "near_v", "far_k", "far_v", "far_v_scale", "far_v_zero", "archive_k", "archive_v"):
        got, want = _np(getattr(cl, n)), ref[n]
        assert got.shape == want.shape, n
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), n


def test_attention_bf16_and_f32_query(fkv, orc):
    run_attention(fkv, orc, 1, 8, 2, 128, 600, 4, seed=11, q_dtype=torch.bfloat16, check_formulation=False)
    run_attention(fkv, orc, 1, 8, 2, 64, 600, 4, seed=12, q_dtype=torch.float32, check_formulation=False)


def test_attention_spikes(fkv, orc):
    _, flags, tokens, kf = run_attention(fkv, orc, 2, 16, 4, 128, 2048, 8, seed=13, spikes=0.02)
    assert kf.sum() > 0 and flags.sum() > 0  # the injected tokens are flagged


def test_attention_uneven_near_valid(fkv, orc):
    """Per-head near_valid after promotions (kernel reads near_valid[kv_head])."""
    run_attention(fkv, orc, 1, 8, 2, 128, 1000, 3, seed=14, near_valid_delta=5)


def test_attention_split_invariance(fkv, orc):
    outs = []
    for target in ("1", "64", "1024", "4096"):
        os.environ["FKV_TARGET_WGS"] = target
        try:
            outs.append(run_attention(fkv, orc, 1, 8, 2, 128, 3000, 5, seed=15, check_formulation=False))
        finally:
            del os.environ["FKV_TARGET_WGS"]
    for o, f, t, _ in outs[1:]:
        assert np.abs(o - outs[0][0]).max() < 5e-4
        assert np.array_equal(t, outs[0][2])


def test_attention_config3_8k(fkv, orc):
    run_attention(fkv, orc, 8, 32, 8, 128, 8192, 0, seed=16, spikes=0.02, check_formulation=False)


def test_attention_repeat_calls_stable(fkv, orc):
    """Split counters self-reset: back-to-back calls give identical results."""
    from foveated_kv_amd import ext, synthetic

    k, v = synthetic.make_kv(2, 4, 3000, 128, 17)
    q = torch.from_numpy(synthetic.make_query(2, 16, 128, 17)).cuda()
    cl = ext.CompressHandle(_cfg(fkv)).compress_layer(torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda())
    h = ext.FoveatedHandle(cl.near_k, cl.near_v, cl.far_k, cl.far_v, cl.far_v_scale, cl.far_v_zero,
                           cl.near_valid, spike_margin=10.0)
    first = [t.clone() for t in h(q[:, :, None])]
    for _ in range(5):
        again = h(q[:, :, None])
        for a, b in zip(first, again):
            assert torch.equal(a, b)


def test_handle_rejects_nan_codes(fkv):
    from foveated_kv_amd import _lib, ext

    B, H, Na, F, D = 1, 1, 8, 64, 64
    nk = torch.zeros((B, H, Na, D), dtype=torch.float16, device="cuda")
    fk = torch.zeros((B, H, F, D), dtype=torch.uint8, device="cuda")
    fk[0, 0, 3, 5] = 0x7F
    fv = torch.zeros((B, H, F, D // 2), dtype=torch.uint8, device="cuda")
    sc = torch.ones((B, H, F), dtype=torch.float16, device="cuda")
    with pytest.raises(_lib.FkvDataError):
        ext.FoveatedHandle(nk, nk, fk, fv, sc, sc, torch.full((H,), Na, dtype=torch.int32, device="cuda"))


def test_e4m3_converter_matches_reference_lut(fkv, orc):
    """The fused kernel's fp8 converter against the reference decode LUT on
    all 256 codes: equal on every code the encoder emits (228), and the blob
    packer zeroes exponent-0 codes as the LUT does."""
    from foveated_kv_amd import _lib

    codes = torch.arange(256, dtype=torch.int32).to(torch.uint8).cuda()
    out = torch.empty(256, dtype=torch.float16, device="cuda")
    _lib.check(_lib.load().fkv_e4m3_decode(_lib.ptr(codes), _lib.ptr(out), 256, _lib.stream_ptr()),
               "fkv_e4m3_decode")
    torch.cuda.synchronize()
    got = out.cpu().numpy().view(np.uint16)
    lut = orc.decode_fp8(np.arange(256, dtype=np.uint8)).view(np.uint16)
    reach = np.unique(orc.encode_fp8(np.arange(65536, dtype=np.uint16)))
    assert np.array_equal(got[reach], lut[reach])


@pytest.mark.parametrize("B,Hq,Hkv,D,S,n_dec,vg", [(8, 32, 8, 128, 8192, 0, 0), (2, 32, 2, 64, 3000, 9, 0),
                                                   (8, 32, 8, 128, 8192, 0, 32), (1, 64, 8, 128, 65536, 7, 0)])
def test_fused_split_merge_back_to_back(fkv, orc, B, Hq, Hkv, D, S, n_dec, vg):
    """The last-arriving split merges the partial records in-kernel; its
    arrival counters are re-armed by the kernel itself.  200 launches queued
    back to back (no host sync between them) must all be bit-identical, and
    must equal the separate merge launch bit for bit (both merges follow the
    same arithmetic in the same order), and the merge through memory
    (FKV_XCD_LOCAL=0) must equal the XCD-local merge bit for bit."""
    from foveated_kv_amd import ext, synthetic

    _flush(f"fused merge stress B={B} Hq={Hq} Hkv={Hkv} D={D} S={S} n_dec={n_dec} v_group={vg}")
    k, v = synthetic.make_kv(B, Hkv, S, D, 21)
    q = torch.from_numpy(synthetic.make_query(B, Hq, D, 21)).cuda()[:, :, None]
    dk, dv = synthetic.make_decode(B, Hkv, n_dec, D, 21)
    dkt = torch.from_numpy(dk).cuda() if dk is not None else None
    dvt = torch.from_numpy(dv).cuda() if dv is not None else None
    cl = ext.CompressHandle(_cfg(fkv, v_group=vg)).compress_layer(
        torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), with_archive=False)
    h = ext.FoveatedHandle(cl.near_k, cl.near_v, cl.far_k, cl.far_v, cl.far_v_scale, cl.far_v_zero,
                           cl.near_valid, spike_margin=10.0)
    os.environ["FKV_FUSED_MERGE"] = "0"  # read once, when a handle is created
    try:
        h_sep = ext.FoveatedHandle(cl.near_k, cl.near_v, cl.far_k, cl.far_v, cl.far_v_scale, cl.far_v_zero,
                                   cl.near_valid, spike_margin=10.0)
    finally:
        del os.environ["FKV_FUSED_MERGE"]
    os.environ["FKV_XCD_LOCAL"] = "0"  # read once, when a handle is created
    try:
        h_mem = ext.FoveatedHandle(cl.near_k, cl.near_v, cl.far_k, cl.far_v, cl.far_v_scale, cl.far_v_zero,
                                   cl.near_valid, spike_margin=10.0)
    finally:
        del os.environ["FKV_XCD_LOCAL"]
    ref = [t.clone() for t in h_sep(q, dkt, dvt)]
    del h_sep
    assert h_mem.dispatch_info() == 0
    ref_mem = [t.clone() for t in h_mem(q, dkt, dvt)]
    del h_mem
    outs = [h(q, dkt, dvt) for _ in range(200)]
    torch.cuda.synchronize()
    first = outs[0]
    for o in outs[1:]:
        for a, b in zip(first, o):
            assert torch.equal(a, b)
    assert torch.equal(first[1], ref[1]) and torch.equal(first[2], ref[2])
    diff = (first[0].float() - ref[0].float()).abs().max().item()
    assert diff <= 1e-3 * max(1.0, ref[0].float().abs().max().item()), diff
    assert torch.equal(first[0], ref[0])
    for a, b in zip(first, ref_mem):
        assert torch.equal(a, b)
    assert h.dispatch_info() > 0, "the workgroup -> XCD dispatch rule did not hold on this device"
    # every one of the 200 dispatches kept each row on one XCD (the watch
    # words the merging workgroups check and clear)
    assert h.dispatch_check() == 0 and h.dispatch_info() > 0


@pytest.mark.parametrize("B,Hq,Hkv,D,S,n_dec", [(8, 32, 8, 128, 8192, 0), (4, 32, 8, 64, 4096, 5)])
def test_xcd_local_merge_across_concurrent_streams(fkv, orc, B, Hq, Hkv, D, S, n_dec):
    """The XCD-local merge relies on the dispatch rule holding for every
    dispatch, whatever hardware queue it comes from (the rule's XCD offset
    differs between queues) and whatever else runs: handles on three
    streams, launched back to back without host synchronisation, must all
    match the merge through memory bit for bit."""
    from foveated_kv_amd import ext, synthetic

    _flush(f"xcd-local merge, 3 streams B={B} Hq={Hq} Hkv={Hkv} D={D} S={S} n_dec={n_dec}")
    k, v = synthetic.make_kv(B, Hkv, S, D, 23)
    q = torch.from_numpy(synthetic.make_query(B, Hq, D, 23)).cuda()[:, :, None]
    dk, dv = synthetic.make_decode(B, Hkv, n_dec, D, 23)
    dkt = torch.from_numpy(dk).cuda() if dk is not None else None
    dvt = torch.from_numpy(dv).cuda() if dv is not None else None
    cl = ext.CompressHandle(_cfg(fkv)).compress_layer(torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(),
                                                      with_archive=False)
    args = (cl.near_k, cl.near_v, cl.far_k, cl.far_v, cl.far_v_scale, cl.far_v_zero, cl.near_valid)
    os.environ["FKV_XCD_LOCAL"] = "0"
    try:
        h_mem = ext.FoveatedHandle(*args, spike_margin=10.0)
    finally:
        del os.environ["FKV_XCD_LOCAL"]
    ref = [t.clone() for t in h_mem(q, dkt, dvt)]
    torch.cuda.synchronize()
    hs = [ext.FoveatedHandle(*args, spike_margin=10.0) for _ in range(3)]
    assert all(h.dispatch_info() > 0 for h in hs)
    streams = [torch.cuda.Stream() for _ in hs]
    outs = []
    for _ in range(40):
        for h, st in zip(hs, streams):
            with torch.cuda.stream(st):
                outs.append(h(q, dkt, dvt))
    torch.cuda.synchronize()
    for o in outs:
        for a, b in zip(o, ref):
            assert torch.equal(a, b)
    assert [h.dispatch_check() for h in hs] == [0, 0, 0]


@pytest.mark.parametrize("K", [1, 8])
def test_one_handle_called_from_three_streams(fkv, orc, K):
    """One handle called from three streams, back to back without host
    synchronisation: every call reuses the handle's split records, arrival
    counters and (K > 1) selection buffers, so the library orders a call
    after the handle's previous eager call when that ran on another stream;
    every output equals the single-stream one bit for bit."""
    from foveated_kv_amd import ext, synthetic

    B, Hq, Hkv, D, S, n_dec = 1, 32, 8, 128, 4096, 64
    _flush(f"one handle, 3 streams B={B} Hq={Hq} Hkv={Hkv} D={D} S={S} n_dec={n_dec} spike_k={K}")
    k, v = synthetic.make_kv(B, Hkv, S, D, 29)
    q0 = synthetic.make_query(B, Hq, D, 29)
    tb = orc.tier_boundaries(S)
    synthetic.inject_spikes(k, q0, tb["mid_start"], tb["far_count"], 0.02, 29)
    q = torch.from_numpy(q0).cuda()[:, :, None]
    dk, dv = synthetic.make_decode(B, Hkv, n_dec, D, 29)
    dkt, dvt = torch.from_numpy(dk).cuda(), torch.from_numpy(dv).cuda()
    cl = ext.CompressHandle(_cfg(fkv)).compress_layer(torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(),
                                                      with_archive=False)
    h = ext.FoveatedHandle(cl.near_k, cl.near_v, cl.far_k, cl.far_v, cl.far_v_scale, cl.far_v_zero,
                           cl.near_valid, spike_margin=10.0, spike_k=K)
    ref = [t.clone() for t in h(q, dkt, dvt)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs = []
    for _ in range(30):
        for st in streams:
            with torch.cuda.stream(st):
                outs.append(h(q, dkt, dvt))
    torch.cuda.synchronize()
    for o in outs:
        for a, b in zip(o, ref):
            assert torch.equal(a, b)
    if K > 1:
        assert int(ref[1].sum()) > 0
