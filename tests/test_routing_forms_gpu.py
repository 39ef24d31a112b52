"""The routing producer's kernels where their work is divided: a wave per tile
row of the three-way builder (fewer tiles than lanes, one lane more, rows that
stay entirely skipped, more rows than one launch has waves), and the tile
maxima's 16-byte loads (heads that are dword-aligned only, blocks that end
inside such a load, NaN and the largest value among the elements past the last
whole one). Codes equal the host restatement exactly.
"""
from __future__ import annotations

import numpy as np
import pytest

import routing_reference as ref
from test_routing_gpu import _codes, _host_importance

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,M,N,tr,tk,p_skip,p_int8", [
    (3, 100, 20, 16, 32, 0.5, 0.3),  # one tile a row
    (2, 200, 63 * 32, 16, 32, 0.97, 0.02),
    (2, 200, 64 * 32, 16, 32, 1.0, 0.0),  # every row skipped: every forced column
    (5, 333, 65 * 32, 16, 32, 0.99, 0.0),
    (1, 17, 8191, 16, 32, 0.3, 0.4),
    (1, 16 * ((1 << 22) + 3), 40, 16, 32, 0.6, 0.2),  # rows past one launch's waves
])
def test_three_way_rows(tm, cuda, heads, M, N, tr, tk, p_skip, p_int8):
    import torch

    print(f"three-way heads={heads} M={M} N={N} skip={p_skip}", flush=True)
    c = _codes(torch, heads, M, N, tr, tk)
    tm.check(tm.tiles_three_way(c, heads, M, N, tr, tk, p_skip, p_int8, 91))
    torch.cuda.synchronize()
    assert np.array_equal(c.cpu().numpy(), ref.three_way(heads, M, N, tr, tk, p_skip, p_int8, 91))


@pytest.mark.parametrize("heads,M,N,d,shift", [
    (3, 331, 999, 100, 0),  # heads 8-byte aligned, last blocks end inside a load
    (2, 258, 514, 33, 0),  # odd d, even heads
    (2, 259, 515, 33, 0),  # odd heads: element by element
    (2, 129, 65, 6, 0),
    (2, 300, 300, 64, 2),  # dword-aligned base
    (2, 300, 300, 64, 1),  # 2-byte aligned base
    (1, 1, 1, 2, 0),
])
def test_importance_alignment(tm, cuda, heads, M, N, d, shift):
    import torch

    print(f"importance heads={heads} M={M} N={N} d={d} shift={shift}", flush=True)
    tr, tk, fraction = 64, 64, 0.4
    rng = np.random.default_rng(M * d + shift)
    sides = []
    for rows in (M, N):
        x = rng.standard_normal((heads, rows, d)).astype(np.float16)
        x[0, -1, -1] = 60000.0  # the last element of the last block decides its maximum
        if heads > 1:
            x[1, -1, -1] = np.nan
        flat = torch.empty(shift + x.size, dtype=torch.float16, device="cuda")
        flat[shift:] = torch.from_numpy(x.reshape(-1)).cuda()
        sides.append((x, flat[shift:].view(x.shape)))
    (qn, q), (kn, k) = sides
    need = tm.importance_workspace_bytes(heads, M, N, tr, tk)
    ws = torch.empty(need // 4, dtype=torch.float32, device="cuda")
    c = _codes(torch, heads, M, N, tr, tk)
    tm.check(tm.tiles_importance(q, k, heads, M, N, d, tr, tk, fraction, ws, need, c))
    torch.cuda.synchronize()
    tq, tkk = ref.tile_grid(M, N, tr, tk)
    maxima = ws.cpu().numpy().reshape(heads, tq + tkk)
    for h in range(heads):
        with np.errstate(invalid="ignore"):
            expected = [np.nanmax(np.append(np.abs(x[h, i * t:(i + 1) * t].astype(np.float32)), 0.0))
                        for x, t, n in ((qn, tr, tq), (kn, tk, tkk)) for i in range(n)]
        assert np.array_equal(maxima[h], np.array(expected, np.float32)), f"maxima of head {h}"
        assert np.array_equal(c[h].cpu().numpy(), _host_importance(qn[h], kn[h], M, N, d, tr, tk, fraction)), f"head {h}"
