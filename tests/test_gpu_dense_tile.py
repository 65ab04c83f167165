"""Dense projections of more than 32 rows: every row has the bits of a run of that row alone, at the
edges of the 32-row tiles and the 64-row chunks, for one K step (three of the four K quarters empty),
step counts that the quarters and the ring do not divide, K splits (uneven ones too), and column counts
on both sides of the chunk rule (strips that leave CUs idle, fill them, spill into a second round)."""

from __future__ import annotations

import pytest
import torch

import metile_amd as mt
from metile_amd import _lib

# K, N, projections, residual
CASES = [
    (64, 32, 1, True),
    (64, 96, 2, False),
    (320, 64, 2, False),
    (576, 160, 1, False),
    (1088, 8224, 2, False),    # 257 strips: a second round
    (704, 6112, 2, False),     # 191: a quarter of the CUs idle
    (704, 6144, 2, False),     # 192
    (704, 4096, 2, False),     # 128: both row chunks at once, a workgroup a CU
    (704, 4128, 2, False),     # 129: one chunk, strips that 8 does not divide
    (192, 1024, 2, False),     # two chunks of an even number of strips, empty quarters
    (4160, 320, 1, True),      # K splits of unequal length
    (8192, 2048, 1, True),
    (9216, 4096, 1, True),     # above 64 MiB of weights: one chunk
    (2112, 64, 2, False),      # SwiGLU over K splits
]


def _run(x, weights, residual, y):
    lib = _lib.lib()
    m, k = x.shape
    n = weights[0].shape[0]
    need = lib.mt_dense_workspace_bytes(m, k, n, len(weights))
    ws = torch.zeros(max(int(need), 4), dtype=torch.uint8, device=x.device)
    dtype = 0 if x.dtype == torch.bfloat16 else 1
    stream = torch.cuda.current_stream().cuda_stream
    if len(weights) == 2:
        _lib.check(lib.mt_dense_swiglu(x.data_ptr(), weights[0].data_ptr(), weights[1].data_ptr(),
                                       y.data_ptr(), m, k, n, dtype, ws.data_ptr(), ws.numel(),
                                       stream))
    else:
        _lib.check(lib.mt_dense_residual_qmv(
            x.data_ptr(), weights[0].data_ptr(), None if residual is None else residual.data_ptr(),
            y.data_ptr(), m, k, n, dtype, ws.data_ptr(), ws.numel(), stream))
    torch.cuda.synchronize()
    if need:  # the arrival counters are left at zero
        assert int(ws[:65536].max()) == 0
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k,n,nproj,with_residual", CASES)
def test_rows_equal_single_row_runs(k, n, nproj, with_residual, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    g = torch.Generator(device="cuda").manual_seed(k + n)
    weights = [(torch.randn(n, k, generator=g, device="cuda") / k**0.5).to(dtype)
               for _ in range(nproj)]
    x = torch.randn(128, k, generator=g, device="cuda").to(dtype)
    res = torch.randn(128, n, generator=g, device="cuda").to(dtype) if with_residual else None
    alone = torch.empty(128, n, dtype=dtype, device="cuda")
    for r in (0, 31, 32, 63, 64, 65, 95, 96, 127):
        _run(x[r:r + 1], weights, None if res is None else res[r:r + 1], alone[r:r + 1])
    for m in (33, 64, 65, 96, 97, 128):
        print(f"[dense tile] {m}x{k}x{n} nproj={nproj} {dtype}", flush=True)
        got = _run(x[:m], weights, None if res is None else res[:m],
                   torch.full((m + 1, n), 7.0, dtype=dtype, device="cuda"))
        for r in (0, 31, 32, 63, 64, 65, 95, 96, 127):
            if r < m:
                assert torch.equal(got[r], alone[r]), (m, r)
        assert bool((got[m] == 7.0).all())  # nothing behind the last row


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k,n,nproj", [(320, 64, 2), (576, 160, 1), (4160, 320, 1)])
def test_residual_and_output_at_an_odd_element(k, n, nproj, dtype):
    """Neither needs alignment: the same bits as with aligned ones, nothing written beside them."""
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    m = 100
    g = torch.Generator(device="cuda").manual_seed(k)
    weights = [(torch.randn(n, k, generator=g, device="cuda") / k**0.5).to(dtype)
               for _ in range(nproj)]
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    res = torch.randn(m, n, generator=g, device="cuda").to(dtype) if nproj == 1 else None
    want = _run(x, weights, res, torch.empty(m, n, dtype=dtype, device="cuda"))
    if nproj == 1:
        odd = torch.empty(m * n + 1, dtype=dtype, device="cuda")[1:].view(m, n).copy_(res)
        assert odd.data_ptr() % 4 == 2
        assert torch.equal(_run(x, weights, odd, torch.empty_like(want)), want)
    buf = torch.full((m * n + 9,), 7.0, dtype=dtype, device="cuda")
    got = _run(x, weights, res, buf[1:1 + m * n].view(m, n))
    assert got.data_ptr() % 4 == 2 and torch.equal(got, want)
    assert float(buf[0]) == 7.0 and bool((buf[1 + m * n:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("k,n,nproj", [(704, 4128, 2), (4160, 320, 1), (192, 1024, 2)])
def test_rows_beyond_one_launch_equal_single_row_runs(k, n, nproj):
    """More than 128 rows: launches that others follow (weights read without the hint) and the last
    one, of one row, of a row kernel's and of a tile's size."""
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    g = torch.Generator(device="cuda").manual_seed(k + n)
    weights = [(torch.randn(n, k, generator=g, device="cuda") / k**0.5).bfloat16()
               for _ in range(nproj)]
    x = torch.randn(300, k, generator=g, device="cuda").bfloat16()
    rows = (0, 63, 64, 127, 128, 129, 159, 160, 255, 256, 299)
    alone = {r: _run(x[r:r + 1], weights, None, torch.empty(1, n, dtype=x.dtype, device="cuda"))
             for r in rows}
    for m in (129, 160, 200, 256, 300):
        got = _run(x[:m], weights, None, torch.empty(m, n, dtype=x.dtype, device="cuda"))
        for r in rows:
            assert r >= m or torch.equal(got[r], alone[r][0]), (m, r)
