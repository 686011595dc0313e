"""The inverse 512 x 512 transform into memory that it shares with its input
(needs an MI355X): phys = four, and phys ahead of four, at 1 plane, a whole
pass through the static array (16 planes) and parts of it, from two streams at
once, and captured in a graph.

Each result must equal the transform into memory of its own bit for bit (the
same kernels), and what phys does not cover of four must stay."""
import pytest
import torch

from diablo_amd import batched, channel

pytestmark = pytest.mark.gpu


def _call(four_ptr, phys_ptr, n, fp32, stream):
    lib = channel.load_library()
    rc = lib.dh_fft512_xz_to_physical_dev(four_ptr, phys_ptr, n, fp32, stream)
    assert rc == 0, lib.dh_batched_last_error()


def _case(n, fp32, seed, ahead=0):
    """(buffer of reals, four at `ahead` reals into it, the expected planes)"""
    rdt = torch.float32 if fp32 else torch.float64
    g = torch.Generator("cuda:0").manual_seed(seed)
    buf = torch.randn(ahead + n * 512 * 514, dtype=rdt, device="cuda:0", generator=g)
    four = torch.view_as_complex(buf[ahead:].clone().view(n, 512, 257, 2))
    ref = torch.empty((n, 512, 512), dtype=rdt, device="cuda:0")
    batched.fft_to_physical(four, ref, fp32=fp32)
    torch.cuda.synchronize()
    return buf, ref


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("n,ahead", [(1, 0), (16, 0), (19, 0), (19, 1024)])
def test_inverse_into_its_own_input(n, ahead, fp32):
    print(f"[fft512 overlap] n={n} ahead={ahead} fp32={fp32}", flush=True)
    buf, ref = _case(n, fp32, 3, ahead)
    tail = buf[n * 512 * 512:].clone()
    _call(buf.data_ptr() + ahead * buf.element_size(), buf.data_ptr(), n, fp32, None)
    torch.cuda.synchronize()
    assert torch.equal(buf[: n * 512 * 512].view_as(ref), ref)
    assert torch.equal(buf[n * 512 * 512:], tail)


def test_two_streams_take_the_array_in_turn():
    print("[fft512 overlap] two streams", flush=True)
    cases = [_case(33, 0, s) for s in (5, 6)]
    streams = [torch.cuda.Stream() for _ in cases]
    for (buf, _), s in zip(cases, streams):
        _call(buf.data_ptr(), buf.data_ptr(), 33, 0, s.cuda_stream)
    torch.cuda.synchronize()
    for buf, ref in cases:
        assert torch.equal(buf[: ref.numel()].view_as(ref), ref)


def test_captured():
    print("[fft512 overlap] captured", flush=True)
    n = 19
    buf, ref = _case(n, 0, 7)
    src = buf.clone()
    _call(buf.data_ptr(), buf.data_ptr(), n, 0, None)  # the tables of a first call
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        buf.copy_(src)
        _call(buf.data_ptr(), buf.data_ptr(), n, 0, torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(buf[: ref.numel()].view_as(ref), ref)
        buf.normal_()
        torch.cuda.synchronize()
