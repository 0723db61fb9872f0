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
# with a ragged last one, and more rows than one sweep of the grid
@pytest.mark.parametrize("B,H,D,S,near_pct", [(1, 1, 128, 44, 0.0), (1, 2, 64, 166, 0.0), (2, 3, 128, 101, 0.0),
                                              (1, 1, 128, 4099, 0.1), (40, 8, 64, 1500, 0.1)])
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


# the edges of the tokens a thread holds (4, 16, 64 per thread of 1,024),
# the first middle past them, and one whose last wave is partly empty
@pytest.mark.parametrize("mid", [1, 63, 65, 4096, 4097, 16384, 16385, 50001, 65536, 65537])
@pytest.mark.parametrize("kind", ["normal", "ties", "equal", "special"])
def test_partition_size_edges(orc, fkv, mid, kind):
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
