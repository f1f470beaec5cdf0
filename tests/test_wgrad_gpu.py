"""The wide network's weight gradient (nect_wgrad) over alignments, leading dimensions and the edges of its steps and chunks.

Tolerance: 16-bit products are exact in float32; a sum of K of them in float32 is off by at most K 2^-24 of the sum of
magnitudes in the worst order, 2^-24 sqrt(K) of it as roundings of either sign add up; four times that."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,m,n", [(1, 1, 1), (31, 8, 128), (257, 129, 24), (5000, 128, 131), (140_001, 16, 128),
                                   (150_000, 128, 104), (512 * 256 + 33, 128, 256)])
@pytest.mark.parametrize("pad_a,pad_b,offset", [(0, 0, 0), (8, 16, 8), (3, 0, 0), (8, 8, 1)])
def test_alignments(device, dtype, K, m, n, pad_a, pad_b, offset):
    from nect_amd import _lib

    print(f"[wgrad] {dtype} {K}x{m}x{n} pad {pad_a} {pad_b} offset {offset}", flush=True)
    g = torch.Generator(device=device).manual_seed(K + n)
    lda, ldb = m + pad_a, n + pad_b
    a = torch.full((K * lda + offset,), float("nan"), dtype=dtype, device=device)
    b = torch.full((K * ldb + offset,), float("nan"), dtype=dtype, device=device)
    dz, h = (torch.randn(K, c, device=device, generator=g).to(dtype) for c in (m, n))
    a[offset:].view(K, lda)[:, :m] = dz
    b[offset:].view(K, ldb)[:, :n] = h
    dw = torch.full((m, n + 1), 0.5, device=device)
    _lib.call("nect_wgrad", _lib.dtype_code(dtype), a.data_ptr() + 2 * offset, lda, b.data_ptr() + 2 * offset, ldb, K, m, n,
              0.25, dw.data_ptr(), n + 1, _lib.stream_of(device))
    torch.cuda.synchronize()
    want = 0.5 + 0.25 * (dz.double().t() @ h.double())
    tol = 4 * 2.0 ** -24 * (K ** 0.5 + 1) * (0.25 * dz.double().abs().t() @ h.double().abs() + 0.5)
    assert bool(((dw[:, :n].double() - want).abs() <= tol).all())
    assert bool((dw[:, n] == 0.5).all())
