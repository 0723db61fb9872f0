"""Device copies of TurboQuant constants: each object gets its own, whatever
became of other objects at its address, and tracks writes to its tensors."""

import copy
import gc
import pickle
import types

import numpy as np
import pytest
import torch

from foveated_kv_amd.turbo import TurboConstants, get_turbo_constants


def _constants(seed, D=16):
    rng = np.random.default_rng(seed)
    f = [torch.from_numpy(rng.standard_normal(s).astype(np.float32)) for s in ((D, D), (D, D), (4,), (3,))]
    f[2], f[3] = f[2].sort().values, f[3].sort().values
    return TurboConstants(*f)


def test_constants_of_dropped_objects_are_not_reused():
    for i in range(50):
        tc = _constants(i, D=(8, 16)[i % 2])
        on = tc.on("cpu")
        assert torch.equal(on.Pi, tc.Pi) and torch.equal(on.S, tc.S)
        assert torch.equal(on.centroids, tc.centroids) and torch.equal(on.boundaries, tc.boundaries)
        del tc, on
        gc.collect()


def test_constants_are_copied_once_and_again_after_a_write():
    tc = _constants(0)
    # a device whose copies are other tensors, without a GPU
    first = tc.on("meta")
    assert tc.on(torch.device("meta")) is first
    tc.S.mul_(2)
    assert tc.on("meta") is not first and tc.on("meta") is tc.on("meta")


def test_constants_copies_stay_out_of_saved_and_copied_objects():
    tc = _constants(1)
    tc.on("cpu")
    for other in (pickle.loads(pickle.dumps(tc)), copy.copy(tc), copy.deepcopy(tc)):
        assert set(vars(other)) == {"Pi", "S", "centroids", "boundaries"}
        assert torch.equal(other.on("cpu").Pi, tc.Pi)


def test_constants_from_arrays():
    tc = _constants(2)
    arrays = TurboConstants(*(t.numpy() for t in (tc.Pi, tc.S, tc.centroids, tc.boundaries)))
    arrays.Pi[0, 0] = 7
    assert float(arrays.on("cpu").Pi[0, 0]) == 7.0
    arrays.Pi[0, 0] = 8
    assert float(arrays.on("cpu").Pi[0, 0]) == 8.0


def test_built_in_constants_are_ordinary_tensors_in_inference_mode():
    with torch.inference_mode():
        tc = get_turbo_constants(64, 1001, 1002)  # seeds of their own: not built before
        assert not tc.Pi.is_inference() and tc.on("meta") is tc.on("meta")


@pytest.mark.parametrize("name,shape", [("Pi", (8, 8)), ("S", (8, 8)), ("S", (32, 16)), ("centroids", (3,)),
                                        ("boundaries", (2,))])
def test_constants_of_another_head_dim_are_refused(monkeypatch, name, shape):
    """Before the library is called: its kernel would read past their end."""
    import dataclasses

    from foveated_kv_amd import _lib, ext, turbo

    class Reached(Exception):
        pass

    def load():
        raise Reached

    monkeypatch.setattr(ext, "_require_device", lambda *a: None)
    monkeypatch.setattr(_lib, "load", load)
    keys = torch.zeros((1, 1, 3, 16), dtype=torch.float16)
    with pytest.raises(Reached):
        turbo.turbo_compress_keys(keys, _constants(3))
    with pytest.raises(ValueError, match=name):
        turbo.turbo_compress_keys(keys, dataclasses.replace(_constants(3), **{name: torch.zeros(shape)}))


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
def test_fused_attention_takes_the_layers_own_constants(D):
    """Layers with constants of their own, built and dropped in turn: the
    fused handle of each is the one built from its matrices, also when they
    come as arrays or in a plain object, and after a write to them."""
    import dataclasses

    from foveated_kv_amd import FoveatedKVCache, TierConfig, turbo

    g = torch.Generator(device="cuda").manual_seed(D)
    k, v = (torch.randn((1, 2, 500, D), generator=g, device="cuda").half() for _ in range(2))
    q = torch.randn((1, 8, 1, D), generator=g, device="cuda").half()
    cache = FoveatedKVCache(TierConfig(compress_method="turbo"))
    cache.update(k, v, 0)
    cache.compress()
    lay = cache.layers[0]

    def direct(tc):
        h = turbo.TurboFoveatedHandle(
            lay.near_k, lay.near_v, lay.turbo_far_k_indices, lay.turbo_far_k_signs, lay.turbo_far_k_norm,
            lay.turbo_far_k_gamma, lay.turbo_far_v_packed, lay.turbo_far_v_scale, lay.near_valid, tc.Pi, tc.S,
            tc.centroids, 10.0)
        return h(q)

    def through_layer(tc):
        return dataclasses.replace(lay, _turbo_constants=tc).attend_fused_with_spikes(q)

    def same(a, b):
        return all(torch.equal(x, y) for x, y in zip(a, b))

    seen = []
    for i in range(6):
        print(f"own constants D={D} object {i}", flush=True)
        tc = get_turbo_constants.__wrapped__(D, 500 + i, 600 + i)
        want = direct(tc)
        assert same(through_layer(tc), want)
        assert not any(torch.equal(want[0], s) for s in seen)
        seen.append(want[0])
        if i == 0:
            arrays = TurboConstants(*(t.numpy() for t in (tc.Pi, tc.S, tc.centroids, tc.boundaries)))
            plain = types.SimpleNamespace(Pi=tc.Pi, S=tc.S, centroids=tc.centroids)
            assert same(through_layer(arrays), want) and same(through_layer(plain), want)
            tc.Pi.copy_(tc.Pi.flip(0).contiguous())
            want = direct(tc)
            assert same(through_layer(tc), want) and not torch.equal(want[0], seen[0])
        del tc
        gc.collect()
