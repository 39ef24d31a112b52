"""Rows that are no multiple of 16 elements, or not 16-byte aligned, in the
prefill kernel: tiles come in 16-byte pieces where every piece of a row is
whole (d a multiple of 8), in pieces that may carry the next row's first bytes
(d a multiple of 4, or dword-aligned tensors), or element by element. The
routing trace makes the kernel take elements, so each call is made with and
without it: O must agree to the bit, and with the fp64 oracle within the
batched bounds (2e-3 / 2e-4, or 1e-5 + 1e-4|x| with precise P.V).

Shapes: the last tile full and ragged, one key past a tile, M and N odd, every
d class of the kernel (up to 32, 64, 96, 128), heads packed with nothing
between them (what a piece carries past a head would be the next head's), and
an infinity in the element that follows a row's end.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import compare, dev, dev_half

pytestmark = pytest.mark.gpu

# heads, M, N, d, g, causal, precise, quantize, shift (elements by which Q, K, V and O are displaced)
CASES = [
    (2, 130, 128, 72, 1, False, True, 1, 0), (3, 100, 193, 72, 2, False, False, 2, 0), (2, 257, 257, 40, 2, True, True, 0, 0),
    (3, 90, 127, 120, 1, False, False, 1, 0), (2, 200, 333, 104, 2, True, False, 0, 0), (2, 129, 320, 24, 1, False, True, 1, 0),
    (2, 70, 65, 8, 1, False, False, 1, 0), (2, 150, 270, 100, 1, False, True, 1, 0), (3, 129, 192, 100, 2, False, False, 0, 0),
    (2, 260, 260, 76, 2, True, True, 2, 0), (2, 64, 191, 36, 1, False, False, 1, 0), (2, 130, 64, 12, 1, False, True, 0, 0),
    (2, 90, 129, 4, 1, False, False, 1, 0), (2, 200, 200, 128, 2, True, False, 1, 2), (2, 150, 129, 64, 1, False, True, 0, 2),
    (2, 100, 200, 72, 1, False, False, 1, 4), (2, 100, 200, 96, 1, False, True, 1, 1), (1, 300, 700, 88, 2, False, True, 1, 0),
    (2, 120, 100, 22, 1, False, False, 1, 0),
    # K8 rows of 4 bytes: pieces of the tile before the last that would end past the head
    (2, 70, 65, 4, 1, False, False, 1, 0), (3, 130, 194, 4, 2, False, True, 2, 0), (2, 90, 131, 4, 1, False, False, 0, 0),
]


def _shifted(bits, shift):
    """The fp16 bits as a device tensor whose data starts `shift` elements into an allocation."""
    import torch

    flat = dev_half(np.concatenate([np.zeros(shift, np.uint16), bits.reshape(-1)]))
    return flat[shift:].view(torch.float16).view(bits.shape)


def _calls(tm, c, q, k, v, codes, routed=True):
    """O of the call without and with the trace."""
    import torch

    from tilemix import routing

    heads, M, N, d, g, causal, precise, quantize, shift = c
    Q, K, V = (_shifted(x, shift) for x in (q, k, v))
    packed = [routing.pack_cells(x, g) for x in codes]
    empty = np.zeros(routing.word_count(M, N, g), np.uint64)
    route = dev(np.concatenate([r for r, _ in packed]))
    skip = dev(np.concatenate([empty if s is None else s for _, s in packed]))
    Q8 = torch.empty((heads, M, d), dtype=torch.int8, device="cuda:0")
    K8 = torch.empty((heads, N, d), dtype=torch.int8, device="cuda:0")
    qs = torch.empty((heads, (M + 127) // 128), dtype=torch.int16, device="cuda:0")
    ks = torch.empty((heads, (N + 63) // 64), dtype=torch.int16, device="cuda:0")
    tm.check(tm.quantize_tilemix_qk_batched(Q, K, Q8, K8, qs, ks, heads, M, N, d))
    outs = []
    for traced in (False, True):
        flat = torch.full((shift + heads * M * d + 4,), 96.0, device="cuda:0")
        trace = torch.empty(codes.size, dtype=torch.uint8, device="cuda:0")
        options = dict(quantize=quantize, route_words=route, skip_words=skip, Q8=Q8, K8=K8, q_scales=qs,
                       k_scales=ks) if routed else dict(quantize=0)
        args = tm.BatchedArgs(Q=Q, K=K, V=V, O=flat[shift:], heads=heads, M=M, N=N, d=d, score_scale=d ** -0.5,
                              causal=causal, precise=precise, key_tiles_per_group=g,
                              decoded_bits=trace if traced else None, **options)
        tm.check(tm.attention_batched(args))
        torch.cuda.synchronize()
        flat = flat.cpu().numpy()
        assert (flat[:shift] == 96.0).all() and (flat[-4:] == 96.0).all(), "written outside O"
        outs.append(flat[shift:-4].reshape(heads, M, d))
    return outs


def _problem(oracle_lib, c):
    heads, M, N, d, g = c[:5]
    rng = np.random.default_rng(M * 31 + N * 7 + d)
    q, k, v = (oracle_lib.float_to_half(rng.standard_normal((heads, r, d)).astype(np.float32)) for r in (M, N, N))
    groups = ((N + 31) // 32 + g - 1) // g
    codes = np.repeat(rng.choice([0, 1, 1, 2], (heads, (M + 15) // 16, groups)).astype(np.uint8), g, axis=2)
    return q, k, v, np.ascontiguousarray(codes[:, :, :(N + 31) // 32])


@pytest.mark.parametrize("case", CASES, ids=["-".join(map(str, c)) for c in CASES])
def test_pieces_equal_elements(tm, oracle_lib, cuda, case):
    q, k, v, codes = _problem(oracle_lib, case)
    print(f"row pieces {case}", flush=True)
    pieces, elements = _calls(tm, case, q, k, v, codes)
    assert np.array_equal(pieces.view(np.uint32), elements.view(np.uint32))
    heads, M, N, d, g, causal, precise = case[:7]
    for h in range(heads):
        q8, qs = oracle_lib.quantize(q[h], 128)
        k8, ks = oracle_lib.quantize(k[h], 64)
        want = oracle_lib.tilemix(q[h], k[h], v[h], q8, k8, qs, ks, codes[h], float(np.float32(d ** -0.5)), causal)
        if precise:
            compare(pieces[h], want, 1e-5, 1e-4, f"head {h}")
        else:
            err = np.abs(pieces[h].astype(np.float64) - want)
            assert err.max() <= 2e-3 and err.mean() <= 2e-4, (h, float(err.max()), float(err.mean()))


@pytest.mark.parametrize("d", [100, 36, 4, 72])
def test_infinity_after_a_row(tm, oracle_lib, cuda, d):
    """-inf in the first element of some keys, positive first elements of Q: those keys weigh nothing, and the keys
    before them, whose last piece carries that element, stay as they are."""
    case = (2, 100, 300, d, 1, False, True, 0, 0)
    q, k, v, codes = _problem(oracle_lib, case)
    q[:, :, 0] = oracle_lib.float_to_half(np.full(1, 0.5, np.float32))[0]
    k[:, 5::7, 0] = 0xFC00
    print(f"infinity after a row, d={d}", flush=True)
    pieces, elements = _calls(tm, case, q, k, v, codes, routed=False)
    assert np.isfinite(pieces).all()
    assert np.array_equal(pieces.view(np.uint32), elements.view(np.uint32))
