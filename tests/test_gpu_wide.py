"""Calls of more rows than one small-row dispatch takes, through the entry points: the wide kernel's
tile edges (rows and columns beside multiples of 32, 64, 96 and 128), one K step and step counts
beside its four- and eight-step loop and its 16-group chunks, odd group counts (scale rows that start
inside a dword), K splits, both code widths, groups of 32 to 4096, both types, both layouts, residuals and
the SwiGLU epilogue, against the oracle.

The bars are the contract's: 2e-3 of the largest output after removing the final rounding, and at
least 98% (bf16) or 90% (f16) of outputs equal to the correctly rounded reference."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import metile_amd as mt
from metile_amd import _lib
from oracle import affine as O
from tests.helpers import act_to_torch, affine_to_torch, torch_to_act

TOL = 2e-3

# rows, K, N, bits, group, dtype, projections, residual, repacked
CASES = [
    (33, 64, 32, 4, 64, "bf16", 1, False, False),       # one K step, one column block
    (33, 320, 96, 4, 64, "f16", 1, True, True),         # five steps, odd groups a row
    (64, 1088, 288, 4, 64, "bf16", 1, True, False),     # 17 groups: a chunk and one more
    (65, 1024, 256, 4, 128, "f16", 1, False, True),
    (96, 2112, 96, 4, 64, "bf16", 2, False, False),     # SwiGLU, 33 groups
    (97, 768, 160, 4, 256, "bf16", 2, False, True),
    (128, 1536, 1024, 4, 64, "bf16", 1, True, True),
    (129, 1536, 320, 4, 64, "f16", 2, False, False),
    (300, 576, 544, 4, 64, "bf16", 1, False, False),
    (48, 8960, 192, 4, 64, "bf16", 1, True, False),     # few columns, long K: K splits
    (40, 4096, 64, 4, 128, "f16", 1, True, True),
    (17, 64, 32, 8, 32, "bf16", 1, False, False),       # groups of 32 leave small rows at 16
    (40, 544 * 2, 96, 8, 32, "f16", 2, False, True),    # 34 groups of 32
    (64, 640, 128, 8, 64, "bf16", 2, False, False),
    (100, 1152, 96, 8, 128, "f16", 1, True, False),
    (130, 2048, 288, 8, 32, "bf16", 1, True, True),
    (36, 5120, 64, 8, 64, "f16", 1, False, True),       # K splits
    (300, 2048, 544, 4, 64, "f16", 1, True, False),     # the same over ten row dispatches
    (17, 2560, 64, 8, 32, "f16", 1, False, True),
    (64, 8192, 64, 4, 512, "bf16", 1, True, True),      # groups beyond four steps: splits of whole ones
    (40, 8192, 96, 8, 1024, "f16", 2, False, False),
    (100, 4096, 96, 4, 4096, "bf16", 1, False, False),  # one group a row
]


def _shifted(t):
    """``t`` at an odd element offset of its buffer (2 bytes behind a 16-byte boundary)."""
    out = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)[1:1 + t.numel()].view(t.shape)
    assert out.data_ptr() % 16 == 2
    return out.copy_(t)


def _fn(nproj, repacked):
    lib = _lib.lib()
    if nproj == 2:
        return lib.mt_affine_swiglu_repacked if repacked else lib.mt_affine_swiglu
    return lib.mt_affine_qmv_repacked if repacked else lib.mt_affine_qmv


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,bits,g,dtype,nproj,residual,repacked", CASES)
def test_wide_meets_the_contract(m, k, n, bits, g, dtype, nproj, residual, repacked):
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    print(f"[wide] {m}x{k}x{n} bits={bits} g={g} {dtype} nproj={nproj}", flush=True)
    x = O.make_activations(m, k, 51, dtype=dtype)
    res = O.make_activations(m, n, 51, tensor_id=3, dtype=dtype) if residual else None
    weights = [O.make_affine_weight(n, k, bits, g, 51, 10 + 2 * p, dtype=dtype)
               for p in range(nproj)]
    xt = act_to_torch(x, dtype)
    triples = [affine_to_torch(w, dtype) for w in weights]
    if repacked:
        triples = [(mt.affine_repack(w, bits=bits), s, b) for w, s, b in triples]
    if nproj == 2:
        ref = O.affine_swiglu(x, *weights, g, bits, dtype=dtype)
        got = mt.affine_swiglu(xt, *triples[0], *triples[1], group_size=g, bits=bits)
    else:
        rt = act_to_torch(res, dtype) if residual else None
        ref = O.affine_qmv(x, *weights[0], g, bits, dtype=dtype, residual=res)
        got = mt.affine_qmv(xt, *triples[0], group_size=g, bits=bits, residual=rt)
    y = torch_to_act(got, dtype)
    err = O.tolerance_error(y, ref, dtype)
    rounded = O.to_f32(O.from_f32(ref.astype(np.float32), dtype), dtype)
    same = np.mean(O.to_f32(y, dtype) == rounded)
    print(f"[wide] tolerance_error={err:.2e} exact={same:.5f}", flush=True)
    assert err <= TOL and same >= (0.98 if dtype == "bf16" else 0.90)
    # With the workspace of the row dispatches the call runs as them (where the wide kernel needs no
    # more, it runs all the same): the bits of the slices.
    lib = _lib.lib()
    need = lib.mt_affine_qmv_workspace_bytes(m, k, n, g, bits, nproj)
    ws = torch.zeros(max(need, 1), dtype=torch.uint8, device="cuda")
    out = torch.empty_like(got)
    args = [xt.data_ptr(), *(t.data_ptr() for triple in triples for t in triple)]
    if nproj == 1:
        args.append(rt.data_ptr() if residual else None)
    _lib.check(_fn(nproj, repacked)(
        *args, out.data_ptr(), m, k, n, g, bits, _lib.MT_BF16 if dtype == "bf16" else _lib.MT_F16,
        ws.data_ptr() if need else None, need, torch.cuda.current_stream().cuda_stream))
    assert O.tolerance_error(torch_to_act(out, dtype), ref, dtype) <= TOL
    if lib.mt_affine_rows_workspace_bytes(m, k, n, g, bits, nproj) <= need:
        return
    chunk = 16 if g == 32 else 32
    for i in range(0, m, chunk):
        part = xt[i:i + chunk]
        alone = (mt.affine_swiglu(part, *triples[0], *triples[1], group_size=g, bits=bits)
                 if nproj == 2 else
                 mt.affine_qmv(part, *triples[0], group_size=g, bits=bits,
                               residual=rt[i:i + chunk] if residual else None))
        assert torch.equal(out[i:i + chunk].view(torch.int16), alone.view(torch.int16))


def test_cases_cover_row_dispatches_in_place_of_the_wide_kernel():
    """Some cases' second half runs row dispatches: several chunks, groups of 32, both projections."""
    lib = _lib.lib()
    split = [c for c in CASES if lib.mt_affine_rows_workspace_bytes(c[0], c[1], c[2], c[4], c[3], c[6])
             > lib.mt_affine_qmv_workspace_bytes(c[0], c[1], c[2], c[4], c[3], c[6])]
    assert any(c[0] > 64 for c in split) and {c[3] for c in split} == {4, 8}
    assert {c[6] for c in split if c[4] == 32} == {1, 2} and any(c[4] > 256 for c in split)


@pytest.mark.gpu
def test_wide_reads_both_layouts_alike_and_replays_in_a_graph():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    h, i, m = 512, 4096, 70
    weights = [affine_to_torch(O.make_affine_weight(n, k, 4, 64, 52, 10 + 2 * p), "bf16")
               for p, (n, k) in enumerate(((i, h), (i, h), (h, i)))]
    packed = [(mt.affine_repack(w, bits=4), s, b) for w, s, b in weights]
    x = act_to_torch(O.make_activations(m, h, 52), "bf16")
    r = act_to_torch(O.make_activations(m, h, 52, tensor_id=3), "bf16")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = mt.affine_mlp(x, *weights, residual=r)
        other = mt.affine_mlp(x, *packed, residual=r)
    side.synchronize()
    assert torch.equal(want.view(torch.int16), other.view(torch.int16))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        got = mt.affine_mlp(x, *packed, residual=r)
    for _ in range(3):
        got.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_wide_workspace_sizes():
    """No device: few rows need nothing, the MLP's size covers its stages and the older query, and
    formats and sizes that the kernel does not take ask for nothing."""
    lib = _lib.lib()
    assert lib.mt_affine_rows_workspace_bytes(32, 8960, 1536, 64, 4, 1) == 0
    split = lib.mt_affine_rows_workspace_bytes(48, 8960, 1536, 64, 4, 1)
    assert split > 64 * 1024  # few columns, long K: split
    assert lib.mt_affine_rows_workspace_bytes(48, 8960, 1536, 32, 4, 1) == 0  # 4-bit groups of 32
    assert lib.mt_affine_rows_workspace_bytes(1 << 20, 8960, 1536, 64, 4, 1) == 0  # x beyond 2 GiB
    for m in (1, 32, 48, 333):
        whole = lib.mt_affine_mlp_rows_workspace_bytes(m, 1536, 8960, 64, 4)
        assert whole >= lib.mt_affine_mlp_workspace_bytes(m, 1536, 8960, 64, 4)
        assert whole >= (lib.mt_affine_rows_workspace_bytes(m, 8960, 1536, 64, 4, 1)
                         + m * 8960 * 2)
    assert (lib.mt_affine_mlp_rows_workspace_bytes(32, 1536, 8960, 64, 4)
            == lib.mt_affine_mlp_workspace_bytes(32, 1536, 8960, 64, 4))
    buf = ctypes.c_void_p(256)  # never dereferenced: too small a workspace is refused as before
    st = lib.mt_affine_mlp(*([buf] * 10), None, buf, 48, 1536, 8960, 64, 4, 0, buf, 1 << 10, None)
    assert st == _lib.MT_ERR_WORKSPACE


@pytest.mark.parametrize("m,k,n", [(333, 8960, 1536), (2048, 4864, 896), (512, 14336, 4096)])
def test_wide_refuses_what_the_row_kernels_refuse(m, k, n):
    """A workspace below the plain queries is refused, also where the wide kernel could do with it."""
    lib = _lib.lib()
    buf = ctypes.c_void_p(256)  # never dereferenced
    need = lib.mt_affine_qmv_workspace_bytes(m, k, n, 64, 4, 1)
    assert need > 0 and lib.mt_affine_rows_workspace_bytes(m, k, n, 64, 4, 1) >= need
    assert lib.mt_affine_qmv(buf, buf, buf, buf, None, buf, m, k, n, 64, 4, 0, buf, need - 1,
                             None) == _lib.MT_ERR_WORKSPACE
    need = lib.mt_affine_gemm_workspace_bytes(m, k, n, 64, 4)
    if need:
        assert lib.mt_affine_gemm(buf, buf, buf, buf, buf, m, k, n, 64, 4, 0, buf, need - 1,
                                  None) == _lib.MT_ERR_WORKSPACE


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n", [(40, 1536, 8960), (64, 1536, 2048), (129, 1024, 4096)])
def test_wide_repeats_to_the_bit(m, k, n):
    """Short K on a full chip, where the first steps' loads arrive last: every call and both layouts
    give the same bits (a wait that ends before the loads it counts shows here)."""
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    w = affine_to_torch(O.make_affine_weight(n, k, 4, 64, 53, 10), "bf16")
    packed = mt.affine_repack(w[0], bits=4)
    x = act_to_torch(O.make_activations(m, k, 53, dtype="bf16"), "bf16")
    want = mt.affine_qmv(x, *w, group_size=64, bits=4)
    for _ in range(20):
        assert torch.equal(mt.affine_qmv(x, *w, group_size=64, bits=4), want)
        assert torch.equal(mt.affine_qmv(x, packed, w[1], w[2], group_size=64, bits=4), want)


# rows, K, N, bits: codes of 512 MiB and more (a range in bits wraps at 2^32), a vocabulary head
# among them
@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,bits", [(33, 3584, 152064, 8), (40, 8192, 131072, 4)])
def test_wide_reaches_every_column_of_large_codes(m, k, n, bits):
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    print(f"[wide] {m}x{k}x{n} bits={bits}: {n * k * bits // 8 >> 20} MiB of codes", flush=True)
    g = torch.Generator(device="cuda").manual_seed(54)
    words = torch.randint(-2**31, 2**31, (n, k * bits // 32), generator=g, device="cuda",
                          dtype=torch.int64).to(torch.int32)
    coef, zero = (0.02, 8.0) if bits == 4 else (0.002, 128.0)
    scales = (torch.randn(n, k // 64, generator=g, device="cuda").abs() * coef).bfloat16()
    biases = (scales.float() * -zero).bfloat16()
    x = O.make_activations(m, k, 54)
    xt = act_to_torch(x, "bf16")
    got = [mt.affine_qmv(xt, words, scales, biases, bits=bits),
           mt.affine_qmv(xt, mt.affine_repack(words, bits=bits), scales, biases, bits=bits)]
    if bits == 4:
        got.append(mt.affine_matmul(xt, words, scales, biases))
    for first in (0, n // 2, n - 64):
        cols = slice(first, first + 64)
        ref = O.affine_qmv(x, words[cols].cpu().numpy().view(np.uint32),
                           torch_to_act(scales[cols], "bf16"), torch_to_act(biases[cols], "bf16"),
                           64, bits)
        for y in got:
            assert O.tolerance_error(torch_to_act(y[:, cols], "bf16"), ref) <= TOL, first


@pytest.mark.gpu
@pytest.mark.parametrize("repacked", [False, True])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_residual_and_output_at_an_odd_element(dtype, repacked):
    """They need no alignment: such calls run as row dispatches, bit for bit those of the slices of
    up to 32 rows, and write nothing beside the output."""
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    m, k, n = 70, 512, 96
    x = act_to_torch(O.make_activations(m, k, 55, dtype=dtype), dtype)
    r = act_to_torch(O.make_activations(m, n, 55, tensor_id=3, dtype=dtype), dtype)
    w, s, b = affine_to_torch(O.make_affine_weight(n, k, 4, 64, 55, 10, dtype=dtype), dtype)
    if repacked:
        w = mt.affine_repack(w, bits=4)
    want = torch.cat([mt.affine_qmv(x[i:i + 32], w, s, b, residual=r[i:i + 32])
                      for i in range(0, m, 32)])
    bits = lambda t: t.contiguous().view(torch.int16)  # noqa: E731
    assert torch.equal(bits(mt.affine_qmv(x, w, s, b, residual=_shifted(r))), bits(want))
    lib = _lib.lib()
    code = _lib.MT_BF16 if dtype == "bf16" else _lib.MT_F16
    buf = torch.full((m * n + 9,), 7.0, dtype=x.dtype, device="cuda")
    ws = torch.zeros(1 << 22, dtype=torch.uint8, device="cuda")
    assert ws.numel() >= lib.mt_affine_rows_workspace_bytes(m, k, n, 64, 4, 1)
    _lib.check(_fn(1, repacked)(x.data_ptr(), w.data_ptr(), s.data_ptr(), b.data_ptr(),
                                r.data_ptr(), buf.data_ptr() + 2, m, k, n, 64, 4, code,
                                ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(bits(buf[1:1 + m * n].view(m, n)), bits(want))
    assert float(buf[0]) == 7.0 and bool((buf[1 + m * n:] == 7.0).all())


def _captured(call, warm, monkeypatch):
    """Replays of ``call`` captured on a stream whose only workspace is that of ``warm``."""
    from metile_amd import quantized

    monkeypatch.setattr(quantized, "_workspaces", {})
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    if warm is not None:
        with torch.cuda.stream(side):
            warm()
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call()
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        yield out


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,warm", [(64, 4864, 896, 8),   # K split, a buffer for the row dispatches
                                        (40, 1536, 2048, 0)])  # row dispatches need none at all
def test_capture_with_the_workspace_of_the_row_dispatches(m, k, n, warm, monkeypatch):
    """Inside capture a workspace cannot grow: a call whose row dispatches have room runs as them."""
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    lib = _lib.lib()
    least = lib.mt_affine_qmv_workspace_bytes(m, k, n, 64, 4, 1)
    assert least <= (1 << 20 if warm else 0) < lib.mt_affine_rows_workspace_bytes(m, k, n, 64, 4, 1)
    w = affine_to_torch(O.make_affine_weight(n, k, 4, 64, 56, 10), "bf16")
    x = act_to_torch(O.make_activations(m, k, 56), "bf16")
    want = torch.cat([mt.affine_qmv(x[:32], *w), mt.affine_qmv(x[32:], *w)])
    for out in _captured(lambda: mt.affine_qmv(x, *w),
                         (lambda: mt.affine_qmv(x[:warm], *w)) if warm else None, monkeypatch):
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("bound", [False, True])
def test_mlp_capture_with_the_workspace_of_the_row_dispatches(bound, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    h, i, m = 512, 4096, 48
    lib = _lib.lib()
    assert (lib.mt_affine_mlp_workspace_bytes(m, h, i, 64, 4) <= 1 << 20
            < lib.mt_affine_mlp_rows_workspace_bytes(m, h, i, 64, 4))
    weights = [affine_to_torch(O.make_affine_weight(n, k, 4, 64, 57, 10 + 2 * p), "bf16")
               for p, (n, k) in enumerate(((i, h), (i, h), (h, i)))]
    x = act_to_torch(O.make_activations(m, h, 57), "bf16")
    call = mt.quantized.BoundMlp(*weights) if bound else (lambda v: mt.affine_mlp(v, *weights))
    ws = torch.zeros(lib.mt_affine_mlp_workspace_bytes(m, h, i, 64, 4), dtype=torch.uint8,
                     device="cuda")
    want = torch.empty_like(x)
    _lib.check(lib.mt_affine_mlp(
        x.data_ptr(), *(t.data_ptr() for triple in weights for t in triple), None, want.data_ptr(),
        m, h, i, 64, 4, _lib.MT_BF16, ws.data_ptr(), ws.numel(),
        torch.cuda.current_stream().cuda_stream))
    for out in _captured(lambda: call(x), lambda: call(x[:8]), monkeypatch):
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
