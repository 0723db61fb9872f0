"""GPU cases of the prompt-side kernels at the edges of their work splits:
the per-head key scale's reduction, the importance partition, TurboQuant
compression and the blob packers.  Everything is compared bit for bit with
the oracle or with plain torch / numpy unless a test says otherwise.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def flush(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def fkv():
    import foveated_kv_amd

    assert foveated_kv_amd.is_available(), "libfkv.so loaded but no gfx950 device"
    return foveated_kv_amd


def _cfg(**kw):
    from foveated_kv_amd import ext

    c = ext.TierConfig()
    c.promo_headroom_min = 8
    for k, v in kw.items():
        setattr(c, k, v)
    return c


# far rows below one lane group's batch, just past one, several workgroups
# with a ragged last one, and more rows than one sweep of the grid; the most
# rows that one workgroup takes and one more
@pytest.mark.parametrize("B,H,D,S,near_pct", [(1, 1, 128, 44, 0.0), (1, 2, 64, 166, 0.0), (2, 3, 128, 101, 0.0),
                                              (1, 1, 128, 4099, 0.1), (40, 8, 64, 1500, 0.1),
                                              (1, 2, 128, 1060, 0.0), (1, 2, 128, 1061, 0.0),
                                              (2, 1, 64, 2084, 0.0), (2, 1, 64, 2085, 0.0)])
def test_k_scale_reduction_edges(fkv, B, H, D, S, near_pct):
    """The scale is the exact maximum over every far row: a maximum planted in
    the first, the last and a middle far row of each head is found, one
    planted in a near row is not."""
    from foveated_kv_amd import ext

    cfg = _cfg(k_scale=1, near_pct=near_pct)
    tb = ext.tier_boundaries_c(cfg, S)
    F, m0 = tb["far_count"], tb["mid_start"]
    g = torch.Generator(device="cuda").manual_seed(S)
    k = torch.randn((B, H, S, D), generator=g, device="cuda").half()
    k[:, :, 0, 0] = 1000.0  # a sink: near
    for where, dim in ((0, 0), (F - 1, D - 1), (F // 2, 17)):
        flush(f"k_scale B={B} H={H} D={D} S={S} far={F} planted at {where}")
        kk = k.clone()
        kk[:, :, m0 + where, dim] = -77.0
        cl = ext.CompressHandle(cfg).compress_layer(kk, kk, with_archive=False)
        want = np.full((B, H), np.float32(77.0) / np.float32(240.0), np.float32)
        assert np.array_equal(cl.far_k_scale.cpu().numpy(), want)


def test_k_scale_without_far_rows(fkv):
    from foveated_kv_amd import ext

    k = torch.randn((2, 3, 30, 64), device="cuda").half()
    cl = ext.CompressHandle(_cfg(k_scale=1)).compress_layer(k, k)
    assert cl.far_k.shape[2] == 0 and torch.equal(cl.far_k_scale, torch.ones((2, 3), device="cuda"))


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("top", [65504.0, 65519.0, 65520.0, 65280.0, 65536.0, float("inf"), float("nan"), 6e-8, 2e-8, 0.0])
def test_k_scale_finite_in_fp16(fkv, dt, top):
    """The maximum is over the keys as fp16: one that overflows there is left
    out, as infinities and NaN are, whatever type it came in (one workgroup
    per head, and several)."""
    from foveated_kv_amd import ext

    for S in (300, 3000):
        flush(f"k_scale of {top} from {dt} S={S}")
        k = torch.full((1, 2, S, 64), 1e-8 if 0 < top < 1e-3 or top == 0 else 3.0)
        k[0, 0, 150, 5], k[0, 0, 151, 6] = top, -top
        k = k.to(dt).cuda()
        cl = ext.CompressHandle(_cfg(k_scale=1)).compress_layer(k, k)
        far = cl.archive_k.float()
        far = torch.where(torch.isfinite(far), far.abs(), torch.zeros_like(far)).amax((2, 3)).cpu().numpy()
        want = np.where(far > 0, far / np.float32(240), np.float32(1)).astype(np.float32)
        assert np.array_equal(cl.far_k_scale.cpu().numpy(), want)


# the edges of the tokens a thread holds (4, 16, 64 per thread of 1,024),
# the first middle past them, and one whose last wave is partly empty
@pytest.mark.parametrize("mid", [1, 63, 65, 4096, 4097, 16384, 16385, 50001, 65536, 65537])
@pytest.mark.parametrize("kind", ["normal", "ties", "equal", "special"])
def test_partition_size_edges(orc, fkv, mid, kind):
    _check_partition(orc, mid, kind)


# registers in use: all but the last, one chunk of four more than a multiple
# of 1,024 fills, one chunk of a few waves only, the lowest key below and
# beside the places past the middle
@pytest.mark.parametrize("mid", [1023, 1024, 1025, 3073, 4100, 5121, 8192, 8193, 17408, 20481, 61440, 61441])
@pytest.mark.parametrize("kind", ["normal", "special"])
def test_partition_registers_in_use(orc, fkv, mid, kind):
    _check_partition(orc, mid, kind)


def _check_partition(orc, mid, kind):
    from foveated_kv_amd import ext

    S = mid + 36
    rng = np.random.default_rng(mid)
    imp = rng.standard_normal((1, 2, S)).astype(np.float32)
    if kind == "ties":
        imp = rng.integers(-1, 2, imp.shape).astype(np.float32)
    elif kind == "equal":
        imp[:] = 3.25
    elif kind == "special":
        imp.reshape(-1)[rng.integers(0, imp.size, imp.size // 3)] = np.nan
        imp.reshape(-1)[rng.integers(0, imp.size, imp.size // 9)] = -np.inf
        imp.reshape(-1)[rng.integers(0, imp.size, imp.size // 9)] = np.finfo(np.float32).min
        imp.reshape(-1)[rng.integers(0, imp.size, imp.size // 9)] = -0.0
    for pct in (0.1, 0.9):
        flush(f"partition mid={mid} {kind} near_pct={pct}")
        near, far = ext.partition_importance(_cfg(near_pct=pct), torch.from_numpy(imp).cuda(), 1, 2, S)
        torch.cuda.synchronize()
        wn, wf, _ = orc.partition_importance(imp, S, 1, 2, promo_headroom_min=8, near_pct=pct)
        assert np.array_equal(near.cpu().numpy(), wn)
        assert np.array_equal(far.cpu().numpy(), wf)


def _int4_numpy(v, group):
    """The INT4 quantiser on fp16 rows, fp32 as the format defines it
    (foveated_compress.metal:153-205): NaN ignored by the extrema and coded 0."""
    f = v.astype(np.float32).reshape(v.shape[:-1] + (-1, group))
    with np.errstate(all="ignore"):
        # the extrema start from +inf / -inf: what a row of NaN keeps
        mn = np.fmin.reduce(f, -1, keepdims=True, initial=np.inf)
        mx = np.fmax.reduce(f, -1, keepdims=True, initial=-np.inf)
        scale = np.fmax((mx - mn) / np.float32(15), np.float32(1e-8))
        q = (f - mn) / scale
        code = np.fmin(np.fmax(np.trunc(q) + (q - np.trunc(q) >= 0.5), 0), 15)
    code = np.nan_to_num(code).astype(np.uint8).reshape(v.shape)
    return code[..., 0::2] | (code[..., 1::2] << 4), scale[..., 0].astype(np.float16), mn[..., 0].astype(np.float16)


@pytest.mark.parametrize("D,vg", [(64, 0), (128, 0), (64, 32), (128, 32)])
@pytest.mark.parametrize("dt", [torch.float16, torch.float32])
@pytest.mark.parametrize("importance", [False, True])
def test_far_rows_special_values(fkv, D, vg, dt, importance):
    """Far rows with infinities, NaN, -0, subnormals, constant rows and exact
    ties, with and without key scales: codes as the formats define them."""
    from foveated_kv_amd import ext

    H, S = 2, 700
    rng = np.random.default_rng(D + vg)
    x = rng.standard_normal((1, H, S, D)).astype(np.float16)
    x[0, 0, 40:60] = rng.integers(-15, 16, (20, D))     # ties: half-integer quotients
    x[0, 0, 60:70] *= np.float16(2.0 ** -20)            # subnormal rows
    x[0, 0, 70:75] = 3.5                                # constant rows
    x[0, 0, 75, :8] = [-0.0, 0.0, 2.0 ** -24, -2.0 ** -24, 65504, -65504, 247.9, 248]
    x[0, 1, 40:100, 3] = np.nan
    x[0, 1, 50:60, 5] = np.inf
    x[0, 1, 60:70, 7] = -np.inf
    x[0, 1, 70] = np.nan
    x[0, 1, 71] = np.inf
    t = torch.from_numpy(x).cuda().to(dt)
    imp = torch.arange(S, dtype=torch.float32, device="cuda") if importance else None
    for ks in (0, 1):
        flush(f"special values D={D} v_group={vg} {dt} importance={importance} k_scale={ks}")
        cl = ext.CompressHandle(_cfg(v_group=vg, k_scale=ks)).compress_layer(t, t, importance=imp)
        far = cl.archive_k.cpu().numpy()
        m0 = 4
        assert np.array_equal(far.view(np.uint16), x[:, :, m0:m0 + far.shape[2]].view(np.uint16))
        codes, scale, zero = _int4_numpy(far, vg or D)
        assert np.array_equal(cl.far_v.cpu().numpy(), codes)
        gs, gz = cl.far_v_scale.cpu().numpy().reshape(scale.shape), cl.far_v_zero.cpu().numpy().reshape(zero.shape)
        assert np.array_equal(gs, scale, equal_nan=True) and np.array_equal(gz, zero, equal_nan=True)
        import oracle

        if ks:
            want = oracle.encode_fp8_scaled(far, oracle.k_head_scale(far))
            assert np.array_equal(cl.far_k_scale.cpu().numpy(), oracle.k_head_scale(far))
        else:
            want = oracle.encode_fp8(far)
        assert np.array_equal(cl.far_k.cpu().numpy(), want)


@pytest.mark.parametrize("exponent", [15, 0, -15])
def test_scaled_keys_every_pair(fkv, exponent):
    """Every fp16 key against every mantissa that a head's largest key can
    have: the code of fp16(fp32(key / scale)), both roundings apart (one
    rounding to fp16 of the quotient gives another code where fp32's has
    moved it onto a tie: 0.958 / (5 / 240) among others)."""
    import oracle
    from foveated_kv_amd import ext

    B, H, D = 16, 64, 64
    keys = np.arange(0x7C00, dtype=np.uint16).view(np.float16)
    keys[1::2] *= -1
    # mantissas of one binade (the subnormal one for the least exponent)
    top = (np.arange(1024, dtype=np.float64) + 1024) * 2.0 ** (exponent - 10)
    if exponent == -15:
        top = (np.arange(1024, dtype=np.float64) + 1) * 2.0 ** -24
    top = top.astype(np.float16).reshape(B, H, 1)
    flat = np.clip(keys, -top, top)
    flat[..., 0] = top[..., 0]
    rows = flat.reshape(B, H, 496, D)
    pad = [np.zeros((B, H, n, D), np.float16) for n in (4, 32)]
    k = torch.from_numpy(np.concatenate([pad[0], rows, pad[1]], 2)).cuda()
    flush(f"scaled keys, every pair, largest key 2^{exponent}")
    cl = ext.CompressHandle(_cfg(k_scale=1, near_pct=0.0)).compress_layer(k, k, with_archive=False)
    scale = top.astype(np.float32) / np.float32(240)
    assert np.array_equal(cl.far_k_scale.cpu().numpy(), scale[..., 0])
    with np.errstate(all="ignore"):
        want = oracle.encode_fp8((rows.astype(np.float32) / scale[..., None]).astype(np.float16))
    bad = cl.far_k.cpu().numpy() != want
    assert not bad.any(), (int(bad.sum()), rows[bad][:4])


def _unpack(p, bits):
    per = 8 // bits
    return ((p[..., None] >> (bits * np.arange(per))) & ((1 << bits) - 1)).reshape(p.shape[:-1] + (-1,))


def _check_turbo_keys(k, Pi, S, cb, bd, got):
    """Codes, signs and norms against fp64.  A decision may differ only where
    its fp64 value lies within a worst-case fp32 evaluation of its boundary:
    D sums and the operands' rounding, (D + 16) 2^-24 of the sum of the
    products' magnitudes; the residual follows from the codes returned."""
    idx, sgn, nrm, gam = (t.cpu().numpy() for t in got)
    k, Pi, S, cb, bd = (np.asarray(a, np.float64) for a in (k, Pi, S, cb, bd))
    D = k.shape[-1]
    eps = (D + 16) * 2.0 ** -24
    n = np.linalg.norm(k, axis=-1, keepdims=True)
    y, tol = k @ Pi.T, eps * (np.abs(k) @ np.abs(Pi).T)
    codes = _unpack(idx, 2)
    nc = np.maximum(n, np.float64(np.float32(1e-8)))
    lo = sum((y - tol >= b * nc + abs(b) * nc * 2.0 ** -23).astype(int) for b in bd)
    hi = sum((y + tol >= b * nc - abs(b) * nc * 2.0 ** -23).astype(int) for b in bd)
    assert ((codes >= lo) & (codes <= hi)).all()
    c = cb[codes]
    r = k - n * (c @ Pi)
    rtol = 2.0 ** -22 * np.abs(k) + n * eps * (np.abs(c) @ np.abs(Pi))
    p, ptol = r @ S.T, rtol @ np.abs(S).T + eps * (np.abs(r) @ np.abs(S).T)
    signs = _unpack(sgn, 1).astype(bool)
    assert (signs == (p >= 0))[np.abs(p) > ptol].all()
    g = np.linalg.norm(r, axis=-1)
    assert (np.abs(nrm - n[..., 0]) <= 2.0 ** -11 * n[..., 0] + 2.0 ** -24).all()
    assert (np.abs(gam - g) <= 2.0 ** -11 * g + np.linalg.norm(rtol, axis=-1) + 2.0 ** -24).all()


def _turbo_keys(_lib, k, Pi, S, cb, bd, offset=0):
    """fkv_turbo_compress_keys on (n, D) keys, the buffers ``offset`` elements
    past a 16-byte boundary."""
    n, D = k.shape

    def at(numel, dtype):
        return torch.zeros(numel + offset, dtype=dtype, device="cuda")[offset:]

    kk = at(n * D, k.dtype)
    kk.copy_(k.reshape(-1))
    idx, sgn = at(n * D // 4, torch.uint8), at(n * D // 8, torch.uint8)
    nrm, gam = at(n, torch.float16), at(n, torch.float16)
    ms = [torch.as_tensor(np.asarray(a, np.float32)).cuda().contiguous() for a in (Pi, S, cb, bd)]
    _lib.check(_lib.load().fkv_turbo_compress_keys(
        _lib.ptr(kk), _lib.dtype_code(k.dtype), n, D, *(_lib.ptr(m) for m in ms), _lib.ptr(idx), _lib.ptr(sgn),
        _lib.ptr(nrm), _lib.ptr(gam), _lib.stream_ptr(torch.device("cuda"))), "fkv_turbo_compress_keys")
    torch.cuda.synchronize()
    return idx.view(n, D // 4), sgn.view(n, D // 8), nrm, gam


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 128, 129, 1000])
@pytest.mark.parametrize("dt,offset", [(torch.float16, 0), (torch.bfloat16, 0), (torch.float32, 0),
                                       (torch.float16, 1), (torch.bfloat16, 3), (torch.float32, 1)])
def test_turbo_keys_edges(fkv, D, n, dt, offset):
    """Token counts at the edges of a wave and a workgroup, every input type,
    unaligned buffers; keys of very different magnitudes."""
    from foveated_kv_amd import _lib
    from foveated_kv_amd.turbo import get_turbo_constants

    flush(f"turbo keys D={D} n={n} {dt} offset={offset}")
    rng = np.random.default_rng(n + D)
    k = rng.standard_normal((n, D)) * 2.0 ** rng.integers(-12, 11, (n, 1))
    k[:, :4] *= 8
    k[n // 2] = 0
    kt = torch.from_numpy(k.astype(np.float32)).cuda().to(dt)
    c = get_turbo_constants(D)
    args = [t.numpy() for t in (c.Pi, c.S, c.centroids, c.boundaries)]
    got = _turbo_keys(_lib, kt, *args, offset=offset)
    _check_turbo_keys(kt.half().cpu().numpy(), *args, got)


@pytest.mark.parametrize("D", [64, 128])
def test_turbo_keys_general_matrices(fkv, D):
    """Any matrices, centroids and boundaries the entry point takes: rows of
    very different scales, a zero row, centroids far from 1, boundaries not
    in order."""
    from foveated_kv_amd import _lib

    rng = np.random.default_rng(D)
    Pi = rng.standard_normal((D, D)).astype(np.float32) * 2.0 ** rng.integers(-9, 10, (D, 1)).astype(np.float32)
    S = rng.standard_normal((D, D)).astype(np.float32) * np.float32(1e-6)
    Pi[3] = 0
    for cb, bd in (([-300.0, -7.0, 12.0, 500.0], [0.3, -0.4, 0.05]), ([-3e-7, -1e-7, 2e-7, 4e-7], [0.0, 1.0, -1.0])):
        cb, bd = np.asarray(cb, np.float32), np.asarray(bd, np.float32)
        kt = torch.from_numpy(rng.standard_normal((200, D)).astype(np.float16)).cuda()
        flush(f"turbo keys general D={D} cb={cb} bd={bd}")
        got = _turbo_keys(_lib, kt, Pi, S, cb, bd)
        idx, sgn, nrm, gam = got
        ok = torch.isfinite(gam)  # residual norms past fp16 are infinite, as before
        assert (ok | (gam == float("inf"))).all()
        g = gam.clone()
        g[~ok] = 0
        sel = ok.cpu().numpy()
        if sel.any():
            _check_turbo_keys(kt.cpu().numpy()[sel], Pi, S, cb, bd, (idx[ok], sgn[ok], nrm[ok], gam[ok]))


def test_turbo_keys_non_finite(fkv):
    """A key row with an infinity or NaN: code 0 and sign 0 everywhere, as a
    sum of NaN compares; the other rows are untouched by it."""
    from foveated_kv_amd import _lib
    from foveated_kv_amd.turbo import get_turbo_constants

    for D in (64, 128):
        rng = np.random.default_rng(7)
        k = rng.standard_normal((64, D)).astype(np.float16)
        k[5, 3], k[6, 9], k[7, 0] = np.inf, -np.inf, np.nan
        c = get_turbo_constants(D)
        args = [t.numpy() for t in (c.Pi, c.S, c.centroids, c.boundaries)]
        flush(f"turbo keys non-finite D={D}")
        got = _turbo_keys(_lib, torch.from_numpy(k).cuda(), *args)
        bad = torch.tensor([5, 6, 7], device="cuda")
        assert (got[0][bad] == 0).all() and (got[1][bad] == 0).all() and not torch.isfinite(got[2][bad]).any()
        keep = np.ones(64, bool)
        keep[[5, 6, 7]] = False
        m = torch.from_numpy(keep).cuda()
        _check_turbo_keys(k[keep], *args, tuple(t[m] for t in got))


@pytest.mark.parametrize("dt,offset", [(torch.float16, 0), (torch.float16, 1), (torch.bfloat16, 3), (torch.float32, 0),
                                       (torch.float32, 1)])
@pytest.mark.parametrize("D,n", [(32, 1), (64, 3), (128, 67), (96, 1001)])
def test_turbo_values_edges(fkv, D, n, dt, offset):
    """TurboQuant values bit for bit against fp32 numpy: ties, zero groups,
    infinities, NaN, subnormals, any head dim of whole groups, unaligned values."""
    from foveated_kv_amd import _lib

    flush(f"turbo values D={D} n={n} {dt} offset={offset}")
    rng = np.random.default_rng(D + n)
    v = rng.standard_normal((n, D)).astype(np.float32)
    v[0, :32] = 0
    v[0, :9] = [3, -3, 1, -1, 0.5, 2, -2, -0.0, 0]
    flat = v.reshape(-1, 32)
    if len(flat) > 40:
        flat[7] = 0
        flat[8] *= 2.0 ** -22
        flat[9, 3], flat[10, 4], flat[11, 5] = np.inf, -np.inf, np.nan
        flat[12] = np.nan
        flat[13] = rng.integers(-6, 7, 32)
    buf = torch.zeros(n * D + offset, dtype=dt, device="cuda")[offset:]
    buf.copy_(torch.from_numpy(v.reshape(-1)).cuda().to(dt))
    packed = torch.empty(n * D // 4, dtype=torch.uint8, device="cuda")
    scale = torch.empty(n * D // 32, dtype=torch.float16, device="cuda")
    _lib.check(_lib.load().fkv_turbo_compress_values(_lib.ptr(buf), _lib.dtype_code(dt), n, D, _lib.ptr(packed),
                                                     _lib.ptr(scale), _lib.stream_ptr(torch.device("cuda"))),
               "fkv_turbo_compress_values")
    f = buf.half().float().cpu().numpy().reshape(-1, 32)
    with np.errstate(all="ignore"):
        sc = np.fmax(np.fmax.reduce(np.abs(f), -1, keepdims=True, initial=0), np.float32(1e-8))
        x = np.rint((f / sc + np.float32(1)) * np.float32(1.5))
        codes = np.nan_to_num(np.fmin(np.fmax(x, 0), 3)).astype(np.uint8)
    want = (codes.reshape(-1, 4) << np.array([0, 2, 4, 6], np.uint8)).sum(-1).astype(np.uint8)
    assert np.array_equal(packed.cpu().numpy(), want)
    assert np.array_equal(scale.cpu().numpy(), sc[:, 0].astype(np.float16))


def _moved(t, offset):
    """A contiguous copy of ``t`` whose storage starts ``offset`` elements in."""
    flat = torch.empty(t.numel() + offset, dtype=t.dtype, device=t.device)[offset:]
    flat.copy_(t.reshape(-1))
    return flat.view(t.shape)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("fmt", ["fp8", "g32", "turbo"])
@pytest.mark.parametrize("S", [700, 1000])
def test_blob_from_any_alignment_and_type(fkv, orc, D, fmt, S):
    """The blob packed from unaligned arrays, and from bf16 / fp32 near tiers,
    gives the outputs of the aligned fp16 one bit for bit; the near tier
    comes back as it went in (token counts off the tile edges)."""
    from foveated_kv_amd import FoveatedKVCache, TierConfig, ext, turbo

    B, H, G = 2, 3, 5
    rng = np.random.default_rng(S + D)
    # near values that every type holds exactly
    k, v = (torch.from_numpy(rng.integers(-31, 32, (B, H, S, D)).astype(np.float16) / 16).cuda() for _ in range(2))
    q = torch.from_numpy(rng.standard_normal((B, H * G, 1, D)).astype(np.float16)).cuda()
    cache = FoveatedKVCache(TierConfig(compress_method="turbo" if fmt == "turbo" else "fp8",
                                       v_group=32 if fmt == "g32" else 0))
    cache.update(k, v, 0)
    cache.compress()
    lay = cache.layers[0]

    def build(near=lambda t: t, other=lambda t: t):
        if fmt == "turbo":
            tc = lay._turbo_constants
            return turbo.TurboFoveatedHandle(
                near(lay.near_k), near(lay.near_v), *(other(t) for t in (
                    lay.turbo_far_k_indices, lay.turbo_far_k_signs, lay.turbo_far_k_norm, lay.turbo_far_k_gamma,
                    lay.turbo_far_v_packed, lay.turbo_far_v_scale)), lay.near_valid, tc.Pi, tc.S, tc.centroids, 10.0)
        return ext.FoveatedHandle(near(lay.near_k), near(lay.near_v), *(other(t) for t in (
            lay.far_k, lay.far_v, lay.far_v_scale, lay.far_v_zero)), lay.near_valid, 10.0)

    flush(f"blob alignment and types D={D} {fmt} S={S} near={lay.near_k.shape[2]}")
    want = build()(q)
    for near, other in ((lambda t: _moved(t, 1), lambda t: _moved(t, 3)), (lambda t: t.bfloat16(), lambda t: t),
                        (lambda t: _moved(t.float(), 1), lambda t: t), (lambda t: t.float(), lambda t: _moved(t, 1))):
        h = build(near, other)
        got = h(q)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        ek, ev = h.export_near()
        assert torch.equal(ek, lay.near_k) and torch.equal(ev, lay.near_v)


def test_far_nan_codes_refused(fkv):
    """A NaN code anywhere in the far keys (first, last, inside a dword) is refused."""
    from foveated_kv_amd import _lib, ext

    k = torch.randn((1, 2, 300, 64), device="cuda").half()
    cl = ext.CompressHandle(_cfg()).compress_layer(k, k)
    flat = cl.far_k.view(-1)
    for at in (0, 5, flat.numel() // 2 + 2, flat.numel() - 1):
        for code in (0x7F, 0xFF):
            old = flat[at].clone()
            flat[at] = code
            with pytest.raises(Exception, match="NaN codes"):
                ext.FoveatedHandle(cl.near_k, cl.near_v, cl.far_k, cl.far_v, cl.far_v_scale, cl.far_v_zero, cl.near_valid)
            flat[at] = old
    ext.FoveatedHandle(cl.near_k, cl.near_v, cl.far_k, cl.far_v, cl.far_v_scale, cl.far_v_zero, cl.near_valid)


def test_tier_index_rows_match_host(fkv):
    """The index kernel against the torch construction, over tier configs and
    lengths down to empty tiers."""
    from foveated_kv_amd.tier_cache import TierConfig, tier_index_tensors

    for kw in ({}, dict(n_sinks=0, window_size=0), dict(near_pct=0.5), dict(near_pct=1.0),
               dict(promo_headroom_pct=0.0, promo_headroom_min=0)):
        for S in (0, 1, 3, 36, 37, 500, 4097):
            tb = TierConfig(**kw).tier_boundaries(S)
            flush(f"tier index rows {kw} S={S}")
            for a, b in zip(tier_index_tensors(tb, S, 2, 3, "cuda"), tier_index_tensors(tb, S, 2, 3, "cpu")):
                assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a.cpu(), b)


def test_layer_next_position(fkv):
    """The position after the prompt, as counted from the index tensors."""
    from foveated_kv_amd import FoveatedKVCache, FoveatedLayer, TierConfig

    for kw in ({}, dict(compress_method="turbo"), dict(window_size=0, n_sinks=0)):
        for S in (40, 333):
            k = torch.randn((1, 2, S, 64), device="cuda").half()
            cache = FoveatedKVCache(TierConfig(**kw))
            cache.update(k, k, 0)
            cache.compress(importance=torch.rand(S, device="cuda") if S == 333 else None)
            lay = cache.layers[0]
            want = max(int(lay.near_idx.max()), int(lay.far_idx.max()) if lay.far_idx.numel() else -1) + 1
            assert lay._next_pos == want == S


def test_blob_memory_outlives_calls_in_flight(fkv):
    """A handle dropped right after calls on another stream and a graph replay:
    its blob's memory is not handed out again while they run."""
    from foveated_kv_amd import FoveatedKVCache, TierConfig

    k, v = (torch.randn((2, 4, 6000, 128), device="cuda").half() for _ in range(2))
    q = torch.randn((2, 16, 1, 128), device="cuda").half()
    cache = FoveatedKVCache(TierConfig())
    cache.update(k, v, 0)
    cache.compress()
    lay = cache.layers[0]
    want = [t.clone() for t in lay.attend_fused_with_spikes(q)]
    side = torch.cuda.Stream()
    for _ in range(5):
        lay._kcache = None
        lay._ensure_kcache()
        h = lay._kcache["cpp_handle"]
        outs = [torch.empty_like(t) for t in want]
        h(q, out=outs)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            h(q, out=outs)
        nbytes = h._blob.numel()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(20):
                got = h(q)
            g.replay()
        lay._kcache = None
        del h
        junk = torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda")  # likely the same memory
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want)) and all(torch.equal(a, b) for a, b in zip(outs, want))
        del junk, g


def test_create_at_checks_the_blob(fkv):
    """A blob that is too small or not aligned is refused before any use."""
    import ctypes

    from foveated_kv_amd import _lib, ext

    k = torch.randn((1, 2, 300, 64), device="cuda").half()
    cl = ext.CompressHandle(_cfg()).compress_layer(k, k)
    lib = _lib.load()
    Na, F = cl.near_k.shape[2], cl.far_k.shape[2]
    n = lib.fkv_attn_blob_bytes(1, 2, 64, Na, F, 0)
    mem = torch.empty(n + 512, dtype=torch.uint8, device="cuda")
    for off, size, ok in ((0, n, True), (0, n - 1, False), (16, n, False), (256, n, True)):
        h = ctypes.c_void_p()
        rc = lib.fkv_attn_create_at(
            ctypes.byref(h), 0, 1, 2, 64, Na, F, _lib.ptr(cl.near_k), _lib.ptr(cl.near_v), 0, _lib.ptr(cl.far_k),
            _lib.ptr(cl.far_v), _lib.ptr(cl.far_v_scale), _lib.ptr(cl.far_v_zero), 0, _lib.ptr(cl.near_valid), 10.0,
            ctypes.c_void_p(mem.data_ptr() + off), size, _lib.stream_ptr(torch.device("cuda")))
        assert (rc == 0) == ok
        if ok:
            lib.fkv_attn_destroy(h)
    assert lib.fkv_attn_blob_bytes(1, 2, 96, Na, F, 0) < 0 and lib.fkv_attn_blob_bytes(1, 2, 64, Na, F, 3) < 0


@pytest.mark.parametrize("importance", [False, True])
def test_compress_past_the_cache(fkv, importance):
    """Large tiers (stores that pass the caches by) hold the bytes that
    the same heads compressed a few at a time do."""
    from foveated_kv_amd import ext

    B, H, S, D = 8, 8, 17000, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    k, v = (torch.randn((B, H, S, D), generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    imp = torch.rand((B, H, S), generator=g, device="cuda") if importance else None
    h = ext.CompressHandle(_cfg())
    flush(f"compress past the cache importance={importance}")
    big = h.compress_layer(k, v, importance=imp)
    nbytes = sum(getattr(big, n).numel() * getattr(big, n).element_size() for n in ("near_k", "near_v", "far_k", "far_v"))
    assert nbytes > 192 << 20
    for b in range(0, B, 4):
        part = h.compress_layer(k[b:b + 4], v[b:b + 4], importance=None if imp is None else imp[b:b + 4])
        for n in ("near_k", "near_v", "far_k", "far_v", "far_v_scale", "far_v_zero", "archive_k", "archive_v"):
            assert torch.equal(getattr(big, n)[b:b + 4], getattr(part, n)), n


def test_float32_compress_past_the_cache(fkv):
    """float32 K and V of 262 MB (read past the caches) give the bytes that a
    batch at a time gives (65 MB, read through them), with key scales too."""
    from foveated_kv_amd import ext

    B, H, S, D = 4, 8, 8000, 128
    g = torch.Generator(device="cuda").manual_seed(4)
    k, v = (torch.randn((B, H, S, D), generator=g, device="cuda") for _ in range(2))
    flush("float32 compress past the cache")
    for ks in (0, 1):
        h = ext.CompressHandle(_cfg(k_scale=ks))
        big = h.compress_layer(k, v)
        for b in range(B):
            part = h.compress_layer(k[b:b + 1], v[b:b + 1])
            for n in ("near_k", "near_v", "far_k", "far_v", "far_v_scale", "far_v_zero", "archive_k", "archive_v"):
                assert torch.equal(getattr(big, n)[b:b + 1], getattr(part, n)), n


@pytest.mark.parametrize("importance", [False, True])
@pytest.mark.parametrize("dt,S,D", [(torch.float16, 700, 128), (torch.bfloat16, 37, 64), (torch.float32, 2100, 64),
                                    (torch.float16, 20, 128)])
def test_archive_layer_is_the_compress_layer_without_far_codes(fkv, importance, dt, S, D):
    from foveated_kv_amd import ext

    g = torch.Generator(device="cuda").manual_seed(S)
    k, v = (torch.randn((2, 3, S, D), generator=g, device="cuda").to(dt) for _ in range(2))
    imp = torch.rand((2, 3, S), generator=g, device="cuda") if importance else None
    flush(f"archive layer S={S} D={D} {dt} importance={importance}")
    h = ext.CompressHandle(_cfg())
    a, b = h.archive_layer(k, v, importance=imp), h.compress_layer(k, v, importance=imp)
    for n in ("near_k", "near_v", "near_valid", "archive_k", "archive_v", "near_idx", "far_idx"):
        x, y = getattr(a, n), getattr(b, n)
        assert (x is None) == (y is None) and (x is None or torch.equal(x, y)), n
    assert a.far_k is None and a.n_near_actual == b.n_near_actual


@pytest.mark.parametrize("D,dt", [(64, torch.float16), (128, torch.float16), (128, torch.float32)])
def test_turbo_codes_are_the_64_bit_ones(fkv, D, dt):
    """Over 200,000 random tokens (with zero and padded ones) every code is the
    one that fp64 gives.  About 30 of them lie near a boundary, of which plain
    fp32 sums would miss one or two: the 64-bit decision itself is held by
    test_turbo_codes_next_to_a_boundary."""
    from foveated_kv_amd.turbo import get_turbo_constants, turbo_compress_keys

    g = torch.Generator(device="cuda").manual_seed(D)
    n = 200_003
    k = torch.randn((1, 1, n, D), generator=g, device="cuda")
    k[..., :4] *= 8
    k[0, 0, 5] = 0
    k = k.to(dt)
    tc = get_turbo_constants(D)
    flush(f"turbo codes against fp64 D={D} {dt} n={n}")
    idx = turbo_compress_keys(k, tc)[0]
    got = ((idx.unsqueeze(-1) >> torch.tensor([0, 2, 4, 6], device="cuda", dtype=torch.uint8)) & 3).flatten(-2)
    kd = k.half().double()
    y = (kd @ tc.Pi.cuda().double().T.contiguous()) / kd.norm(dim=-1, keepdim=True).clamp_min(np.float32(1e-8))
    want = torch.bucketize(y, tc.boundaries.cuda().double(), right=True)
    assert int((got != want).sum()) == 0


def test_turbo_keys_refused_under_capture(fkv):
    from foveated_kv_amd.turbo import get_turbo_constants, turbo_compress_keys

    k = torch.randn((1, 1, 64, 64), device="cuda").half()
    tc = get_turbo_constants(64)
    turbo_compress_keys(k, tc)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        with pytest.raises(Exception, match="graph capture"):
            turbo_compress_keys(k, tc)
    want = turbo_compress_keys(k, tc)
    assert all(torch.equal(a, b) for a, b in zip(turbo_compress_keys(k, tc), want))


def test_archive_layer_ignores_the_key_scale_option(fkv):
    """It has no far keys to scale: a configuration with k_scale set (by hand,
    on a TurboQuant one) gives the layer that one without it does."""
    from foveated_kv_amd import FoveatedKVCache, TierConfig

    k, v = (torch.randn((1, 2, 300, 64), device="cuda").half() for _ in range(2))
    layers = []
    for k_scale in (False, True):
        cfg = TierConfig(compress_method="turbo")
        cfg.k_scale = k_scale
        cache = FoveatedKVCache(cfg)
        cache.update(k, v, 0)
        cache.compress()
        layers.append(cache.layers[0])
    for n in ("near_k", "near_v", "near_valid", "archive_k", "archive_v", "turbo_far_k_indices", "turbo_far_k_signs",
              "turbo_far_v_packed"):
        assert torch.equal(getattr(layers[0], n), getattr(layers[1], n)), n


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("e", [-6, -9, -16, -20, -22])
def test_turbo_codes_of_small_keys(fkv, D, e):
    """Keys down to a few units of fp16's subnormals, alone and beside large
    ones in a wave: every code is the one of fp64, norms and residual norms
    are those of the keys, and so are the signs away from rounding."""
    from foveated_kv_amd import _lib
    from foveated_kv_amd.turbo import get_turbo_constants

    g = torch.Generator(device="cuda").manual_seed(D - e)
    k = (torch.randn((200_003, D), generator=g, device="cuda") * 2.0 ** e).half()
    k[7::64] = (k[7::64].float() * 2.0 ** (3 - e)).half()
    k[5] = 0
    k[6] = 2.0 ** -24
    flush(f"turbo codes of small keys D={D} 2^{e}")
    tc = get_turbo_constants(D)
    args = [t.numpy() for t in (tc.Pi, tc.S, tc.centroids, tc.boundaries)]
    got = _turbo_keys(_lib, k, *args)
    kd = k.double()
    y = (kd @ tc.Pi.cuda().double().T.contiguous()) / kd.norm(dim=-1, keepdim=True).clamp_min(np.float32(1e-8))
    want = torch.bucketize(y, tc.boundaries.cuda().double(), right=True)
    codes = ((got[0].unsqueeze(-1) >> torch.tensor([0, 2, 4, 6], device="cuda", dtype=torch.uint8)) & 3).flatten(-2)
    assert int((codes != want).sum()) == 0
    _check_turbo_keys(k[:20000].cpu().numpy(), *args, tuple(t[:20000] for t in got))


def _keys_near_a_boundary(tc, rng):
    """fp16 keys, one for every dim, boundary and side, whose rotated
    coordinate lies 1e-9 to 3e-8 of their norm from the boundary in fp64:
    random keys moved along the dim's row of Pi, then the nearest of 16^4
    combinations of steps of four of their elements."""
    Pi, bd = tc.Pi.numpy().astype(np.float64), tc.boundaries.numpy().astype(np.float64)
    D = Pi.shape[0]
    grid = np.arange(-8.0, 8.0)
    out = []
    for i in range(D):
        for b in bd:
            for side in (-1.0, 1.0):
                k = rng.standard_normal(D)
                k[:4] *= 8
                for _ in range(4):
                    k = k + (b * np.linalg.norm(k) - k @ Pi[i]) * Pi[i]
                k = k.astype(np.float16).astype(np.float64)
                # elements well inside their binade: eight steps stay fp16 numbers
                m, e = np.frexp(np.abs(k))
                dims = rng.permutation(np.flatnonzero((m > 0.55) & (m < 0.95) & (np.abs(k) > 0.1)))[:4]
                dot, sq = k @ Pi[i], k @ k
                for a, d in enumerate(dims):
                    shape = [1] * 4
                    shape[a] = 16
                    s = (grid * 2.0 ** (e[d] - 11.0)).reshape(shape)
                    dot = dot + s * Pi[i, d]
                    sq = sq + s * (2 * k[d] + s)
                off = side * (dot / np.sqrt(sq) - b)
                at = np.unravel_index(np.argmin(np.where(off >= 1e-9, off, np.inf)), off.shape)
                for a, d in enumerate(dims):
                    k[d] += grid[at[a]] * 2.0 ** (e[d] - 11.0)
                h = k.astype(np.float16)
                assert np.array_equal(h.astype(np.float64), k)
                gap = side * (k @ Pi[i] / np.linalg.norm(k) - b)
                if 1e-9 <= gap <= 3e-8:
                    out.append(h)
    return np.stack(out)


@pytest.mark.parametrize("D", [64, 128])
def test_turbo_codes_next_to_a_boundary(fkv, D):
    """Keys with a coordinate closer to a boundary than the fp32-precision
    sums decide (their error has a standard deviation of about 5e-9 of the
    norm): every code is the one of fp64.  Waves of such keys only, and waves
    that hold some among others."""
    from foveated_kv_amd import _lib
    from foveated_kv_amd.turbo import get_turbo_constants

    rng = np.random.default_rng(D)
    tc = get_turbo_constants(D)
    near = _keys_near_a_boundary(tc, rng)
    assert len(near) > 5 * D  # of 6 D
    other = rng.standard_normal((3 * len(near), D)).astype(np.float16)
    mixed = np.concatenate([near, other])
    rng.shuffle(mixed)
    k = np.concatenate([near, mixed])
    flush(f"turbo codes next to a boundary D={D} keys={len(near)}")
    args = [t.numpy() for t in (tc.Pi, tc.S, tc.centroids, tc.boundaries)]
    got = _turbo_keys(_lib, torch.from_numpy(k).cuda(), *args)
    kd = k.astype(np.float64)
    y = (kd @ args[0].astype(np.float64).T) / np.linalg.norm(kd, axis=-1, keepdims=True)
    want = (y[..., None] >= args[3].astype(np.float64)).sum(-1)
    assert int((_unpack(got[0].cpu().numpy(), 2) != want).sum()) == 0
    _check_turbo_keys(k, *args, got)
