"""The quantizer's rule on how rows move - pieces of 8 elements, of 4, or one by
one - over head dimensions, row strides and displaced bases on both sides of
each condition, with last blocks of one row and of all but one, special values
in every block, and guard elements after the outputs. Bytes and scales equal
the C oracle's.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import dev_half, host
from test_quantize_special_gpu import check_side, special_rows

pytestmark = pytest.mark.gpu

GUARD = 5


@pytest.mark.parametrize("heads,M,N,d,pad,shift,shift8", [
    (2, 129, 65, 4, 0, 0, 0), (3, 255, 127, 100, 0, 0, 0), (3, 1, 1, 12, 0, 0, 0), (2, 1000, 577, 124, 0, 0, 0),
    (2, 300, 200, 60, 0, 4, 4),  # half the registers (d <= 64), 8-byte and 4-byte aligned bases
    (2, 300, 200, 128, 4, 0, 0), (2, 300, 200, 64, 4, 0, 0),  # row strides that are multiples of 4
    (2, 300, 200, 100, 8, 0, 0), (2, 130, 66, 100, 2, 0, 0),  # the second: element by element
    (2, 300, 200, 128, 0, 4, 0), (2, 300, 200, 128, 0, 0, 4), (2, 300, 200, 128, 0, 0, 1), (2, 300, 200, 100, 0, 2, 0),
    (2, 300, 200, 102, 0, 0, 0), (70, 130, 65, 36, 0, 0, 0),
])
def test_pieces_match_oracle(tm, oracle_lib, cuda, heads, M, N, d, pad, shift, shift8):
    import torch

    print(f"quantizer pieces heads={heads} M={M} N={N} d={d} pad={pad} shift={shift}/{shift8}", flush=True)
    rng = np.random.default_rng(M * d + pad + shift + shift8)
    inputs, ins, flats, outs, scales = [], [], [], [], []
    for rows, block in ((M, 128), (N, 64)):
        x = np.stack([special_rows(rows, d, block, rng) for _ in range(heads)])
        wide = np.full((heads, rows, d + pad), 0x7C00, np.uint16)  # an infinity would show in the maximum
        wide[:, :, :d] = x
        inputs.append(x)
        ins.append(dev_half(np.concatenate([np.full(shift, 0x7C00, np.uint16), wide.reshape(-1)]))[shift:])
        flats.append(torch.full((shift8 + x.size + GUARD,), -128, dtype=torch.int8, device=cuda))
        outs.append(flats[-1][shift8:])
        scales.append(torch.full((heads, -(-rows // block)), 0x7B53, dtype=torch.int16, device=cuda))
    row = d + pad
    tm.check(tm.quantize_tilemix_qk_strided(ins[0], ins[1], outs[0], outs[1], scales[0], scales[1], heads, M, N, d,
                                            M * row, N * row, row, row))
    torch.cuda.synchronize()
    for x, out, flat, s, block, label in zip(inputs, outs, flats, scales, (128, 64), "QK"):
        check_side(oracle_lib, x, host(out)[:x.size].reshape(x.shape), host(s, np.uint16), block, label)
        whole = host(flat)
        assert (whole[:shift8] == -128).all() and (whole[-GUARD:] == -128).all(), f"{label}: written past its end"


@pytest.mark.parametrize("heads,M,N,d,pad", [
    (3, 300, 200, 128, 0), (5, 129, 65, 64, 0), (2, 130, 1, 128, 64),  # the grid runs over heads first
    (3, 300, 200, 96, 0), (3, 300, 200, 64, 8), (3, 300, 200, 100, 0),  # over blocks first
    (1, 300, 200, 128, 0),
])
def test_interleaved_heads_match_oracle(tm, oracle_lib, cuda, heads, M, N, d, pad):
    """[rows, heads, d + pad] inputs, both grid orders."""
    import torch

    print(f"quantizer interleaved heads={heads} M={M} N={N} d={d} pad={pad}", flush=True)
    rng = np.random.default_rng(M * d + pad)
    row = heads * (d + pad)
    inputs, ins, outs, scales = [], [], [], []
    for rows, block in ((M, 128), (N, 64)):
        inputs.append(np.stack([special_rows(rows, d, block, rng) for _ in range(heads)]))
        wide = np.full((rows, heads, d + pad), 0x7C00, np.uint16)
        wide[:, :, :d] = inputs[-1].transpose(1, 0, 2)
        ins.append(dev_half(wide))
        outs.append(torch.full((heads, rows, d), -128, dtype=torch.int8, device=cuda))
        scales.append(torch.full((heads, -(-rows // block)), 0x7B53, dtype=torch.int16, device=cuda))
    tm.check(tm.quantize_tilemix_qk_strided(ins[0], ins[1], outs[0], outs[1], scales[0], scales[1], heads, M, N, d,
                                            d + pad, d + pad, row, row))
    torch.cuda.synchronize()
    for x, out, s, block, label in zip(inputs, outs, scales, (128, 64), "QK"):
        check_side(oracle_lib, x, host(out), host(s, np.uint16), block, label)
