"""bf16 and float32 queries give the bits of the same query cast to fp16 first,
whichever kernel rounds them: rows of one, two and three head quads, partly
filled quads, every far format, short and long contexts, no far tier, device
decode counts, unaligned queries."""

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(2, 3, 4, 128, 1500, 5), (1, 2, 1, 64, 300, 0), (1, 2, 7, 64, 512, 16), (3, 4, 5, 128, 3003, 7),
         (2, 8, 8, 128, 4096, 0), (2, 8, 8, 64, 4100, 70), (1, 4, 12, 128, 2500, 3), (1, 2, 4, 128, 33, 2)]


def _handle(B, H, D, S, fmt):
    from foveated_kv_amd import FoveatedKVCache, TierConfig

    g = torch.Generator(device="cuda").manual_seed(S)
    k, v = (torch.randn((B, H, S, D), generator=g, device="cuda").half() for _ in range(2))
    cache = FoveatedKVCache(TierConfig(compress_method="turbo" if fmt == "turbo" else "fp8",
                                       v_group=32 if fmt == "g32" else 0, k_scale=fmt == "scaled"))
    cache.update(k, v, 0)
    cache.compress()
    lay = cache.layers[0]
    lay._ensure_kcache()
    return lay._kcache["cpp_handle"], g


@pytest.mark.parametrize("B,H,G,D,S,nd", CASES)
@pytest.mark.parametrize("fmt", ["fp8", "g32", "scaled", "turbo"])
def test_query_types_bit_equal(B, H, G, D, S, nd, fmt):
    print(f"query types B={B} H={H} G={G} D={D} S={S} n_dec={nd} {fmt}", flush=True)
    h, g = _handle(B, H, D, S, fmt)
    q = torch.randn((B, H * G, 1, D), generator=g, device="cuda") * 1.5
    q[0, 0, 0, :4] = torch.tensor([0.0, -0.0, 1e-7, -3e-8])  # fp16 subnormals and zeros
    dk = torch.randn((B, H, nd, D), generator=g, device="cuda").half() if nd else None
    for dt in (torch.bfloat16, torch.float32):
        qd = q.to(dt)
        want = h(qd.half(), dk, dk)
        for off in (0, 1):  # one element past a 4-byte boundary for bf16
            buf = torch.empty(qd.numel() + off, dtype=dt, device="cuda")[off:]
            buf.copy_(qd.reshape(-1))
            got = h(buf.view(qd.shape), dk, dk)
            assert all(torch.equal(a, b) for a, b in zip(got, want)), (dt, off)
        if nd:
            n = torch.tensor([nd], dtype=torch.int32, device="cuda")
            assert all(torch.equal(a, b) for a, b in zip(h(qd, dk, dk, n_decode=n), want)), dt
