"""QWeight.pack, the weights' bytes of the per-step calls, against the C struct's bytes:
tensors and raw addresses, given and derived lengths, values out of a field's range."""
import ctypes

import pytest
import torch

import dyninfer_amd as d

W8 = torch.zeros(64, dtype=torch.uint8)
S = torch.zeros(4, 2, dtype=torch.bfloat16)


@pytest.mark.parametrize("w,lens", [
    (d.QWeight(d.ENC_Q4_0, 4, 64, W8), (64, 0, 0)),
    (d.QWeight(d.ENC_Q4_0, 4, 64, 4096), (144, 0, 0)),
    (d.QWeight(d.ENC_Q6_K, 3, 512, W8, data_bytes=7), (7, 0, 0)),
    (d.QWeight(d.ENC_MLX_U4, 4, 64, W8, S, S[:2], 32), (64, 16, 8)),
    (d.QWeight(d.ENC_MLX_U4, 4, 64, 4096, 8192, 12288, 32, d.DTYPE_F32, biases_bytes=5), (128, 32, 5)),
    (d.QWeight(d.ENC_MLX_U4, 4, 64, None, None, None, 0), (128, 0, 0)),
    (d.QWeight(d.ENC_Q8_0, -1, 64, W8), (64, 0, 0)),
    (d.QWeight(1 << 33, 4, 64, W8, group_size=-2), (64, -256 % 2**64, -256 % 2**64)),
])
def test_pack_is_the_struct(w, lens):
    c = w.c()
    assert w.pack() == bytes(c) and len(w.pack()) == ctypes.sizeof(c)
    assert (c.data_bytes, c.scales_bytes, c.biases_bytes) == lens
    assert (c.rows, c.cols) == (w.rows % 2**64, w.cols)


def test_out_of_range_is_refused_by_the_library():
    with pytest.raises(d.DyninferError):
        d.prefill_workspace_bytes([d.QWeight(d.ENC_Q4_0, -1, 64, W8)], 64)
