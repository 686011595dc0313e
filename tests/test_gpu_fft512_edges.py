"""The 512 x 512 plane transforms where their launches can go wrong (needs an
MI355X): one and three planes (the last block of columns is partly empty),
both sides of the FP32 rule for 8 or 16 columns per block (95 and 96 planes),
and physical planes that start one real past a complex value's alignment.

Against numpy.fft on the first and the last plane, relative L2 <= 1e-14 (FP64)
and 2e-6 (FP32): log2(512^2) = 18 butterfly levels of a few 2^-53 or 2^-24
each; a wrong column, row or plane is O(1)."""
import numpy as np
import pytest
import torch

from diablo_amd import batched

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("planes,fp32", [(1, False), (3, False), (3, True), (95, True), (96, True)])
def test_fft512_block_edges_and_unaligned_planes(planes, fp32):
    print(f"[batched] fft512 planes={planes} fp32={fp32}", flush=True)
    rdt, cdt, bar = (torch.float32, torch.complex64, 2e-6) if fp32 else (torch.float64, torch.complex128, 1e-14)
    gen = torch.Generator(device="cuda").manual_seed(planes)
    store = torch.randn(planes * 512 * 512 + 1, dtype=rdt, device="cuda", generator=gen)
    phys = store[1:].view(planes, 512, 512)  # one real past the allocation's start
    four = torch.empty(planes, 512, 257, dtype=cdt, device="cuda")
    batched.fft_to_fourier(phys, four, fp32=fp32)
    spec = torch.randn(planes, 512, 257, dtype=cdt, device="cuda", generator=gen)
    keep = spec.clone()
    out = torch.full((planes * 512 * 512 + 1,), float("nan"), dtype=rdt, device="cuda")
    back = out[1:].view(planes, 512, 512)
    batched.fft_to_physical(spec, back, fp32=fp32)
    torch.cuda.synchronize()
    assert torch.equal(spec, keep)
    assert torch.isnan(out[0]) and torch.isfinite(back).all()
    for p in {0, planes - 1}:
        ph = phys[p].cpu().numpy().astype(np.float64)
        assert _rel(four[p].cpu().numpy(), np.fft.rfft2(ph) / 512 ** 2) <= bar
        sp = spec[p].cpu().numpy().astype(np.complex128)
        assert _rel(back[p].cpu().numpy(), np.fft.irfft2(sp, s=(512, 512)) * 512 ** 2) <= bar
