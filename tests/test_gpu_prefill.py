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
