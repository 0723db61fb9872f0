"""The next token's position of a layer: the builder's, else one past the
largest index of the layer's own index tensors."""

import dataclasses

import torch


def test_replaced_layer_takes_its_position_from_its_own_indices():
    from foveated_kv_amd import FoveatedLayer

    def index(*values):
        return torch.tensor(values, dtype=torch.int32).view(1, 1, -1)

    z = torch.zeros((1, 1, 4, 64), dtype=torch.float16)
    layer = FoveatedLayer(near_k=z, near_v=z, near_idx=index(0, 1, 98, 99), far_k=z, far_v=z, far_v_scale=z,
                          far_v_zero=z, far_idx=index(2, 3), archive_k=z, archive_v=z, archive_idx=index(2, 3),
                          next_position=100)
    assert layer._next_pos == 100
    layer.add_token(z[:, :, :1], z[:, :, :1])
    assert layer._next_pos == 101
    assert dataclasses.replace(layer, spike_k=2)._next_pos == 100
    assert dataclasses.replace(layer, near_idx=index(0, 1, -1, -1), far_idx=index(2, 41))._next_pos == 42
    assert dataclasses.replace(layer, next_position=7)._next_pos == 7
