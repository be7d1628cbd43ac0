"""GPU parity of the one-launch weight layout (r9k_mxfp4_prep) against the torch expressions on the CPU, and of the
magnitude-wise NVFP4 -> MXFP4 search against the oracle on blocks that reach each of its branches: bit for bit."""
import numpy as np
import pytest
import torch

from helpers import make_experts
from oracle import oracle as O
from r9700_vllm.kernels import moe as K
from r9700_vllm.quant import nvfp4 as NV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,N,Kd", [(1, 16, 32), (3, 48, 96), (2, 32, 128), (2, 64, 416), (1, 2064, 5120), (5, 16, 2624)])
def test_prep_equals_torch(dev, E, N, Kd):
    packed, e8 = make_experts(E, N, Kd, torch.Generator().manual_seed(E + N + Kd), lo=0, hi=255)
    ref_q, ref_s = K.permute_fragments(packed), K.pack_scales(e8)          # CPU tensors: the torch expressions
    W = K.prepare_mxfp4_weights(packed.to(dev), e8.to(dev))
    assert torch.equal(W.wq.cpu(), ref_q) and torch.equal(W.wsr.cpu(), ref_s)
    assert torch.equal(K.permute_fragments(packed.to(dev)).cpu(), ref_q)
    assert torch.equal(K.pack_scales(e8.to(dev)).cpu(), ref_s)
    # sources the kernel does not take (strided, off the 16-byte grid) still go through torch
    wide = torch.zeros(E, N, Kd, dtype=torch.uint8, device=dev)
    wide[..., : Kd // 2] = packed.to(dev)
    assert torch.equal(K.permute_fragments(wide[..., : Kd // 2]).cpu(), ref_q)
    off = torch.zeros(packed.numel() + 8, dtype=torch.uint8, device=dev)[8:].view(packed.shape).copy_(packed)
    assert off.data_ptr() % 16 and torch.equal(K.permute_fragments(off).cpu(), ref_q)


def test_prep_output_sizes(dev):
    """An `out` of another size never reaches the kernel: too small is refused, a longer scale tensor keeps its tail."""
    E, N, Kd = 2, 32, 128
    packed, e8 = make_experts(E, N, Kd, torch.Generator().manual_seed(5), lo=0, hi=255)
    small = torch.empty(E * N * Kd // 2 - 16, dtype=torch.uint8, device=dev)
    with pytest.raises(RuntimeError):
        K.permute_fragments(packed.to(dev), out=small)
    with pytest.raises((RuntimeError, IndexError)):
        K.pack_scales(e8.to(dev), out=torch.empty((E, Kd // 32, N), dtype=torch.uint8, device=dev))
    long = torch.full((E, Kd // 32 + 2, N), 7, dtype=torch.uint8, device=dev)
    K.pack_scales(e8.to(dev), out=long)
    assert torch.equal(long[:, :-1].cpu(), K.pack_scales(e8)) and bool((long[:, -1] == 7).all())


def test_nvfp4_conversion_of_strided_tensors_stays_chunked(dev):
    """Codes and scales that lie in wider buffers: the bytes of the contiguous conversion, and no copy of the whole
    tensor (a chunk's rows at a time)."""
    g = torch.Generator().manual_seed(11)
    N, Kd = 8192, 2048
    p = torch.randint(0, 256, (N, Kd // 2 + 64), generator=g, dtype=torch.uint8).to(dev)
    s = (torch.randn(N, Kd // 16 + 32, generator=g).abs() * 20).clamp(2 ** -9, 448).to(torch.float8_e4m3fn).to(dev)
    pv, sv, div = p[:, : Kd // 2], s[:, : Kd // 16], torch.full((N,), 448.0, device=dev)
    want = NV.nvfp4_to_mxfp4(pv.contiguous(), sv.contiguous(), div)
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    got = NV.nvfp4_to_mxfp4(pv, sv, div, rows_per_chunk=512)
    extra = torch.cuda.max_memory_allocated() - base
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    outputs = N * Kd // 2 + N * Kd // 32
    chunk = 512 * (Kd // 2 + Kd // 16)
    assert extra <= outputs + 3 * chunk + (1 << 20), (extra, outputs, chunk)      # two chunks may be alive, and their rounding


def search_blocks(rd):
    """Checkpoint tensors of 256 x 512: uniform blocks, every scale byte (zero, subnormal, negative, NaN), one-magnitude
    and all-zero blocks, groups whose scales lie far apart, exact ties of the two candidates."""
    g = torch.Generator().manual_seed(int(abs(np.log(rd)) * 10) + 1)
    N, Kd = 256, 512
    packed = torch.randint(0, 256, (N, Kd // 2), generator=g, dtype=torch.int32).to(torch.uint8)
    s16 = (torch.randn(N, Kd // 16, generator=g).abs() * 100).clamp(max=448).to(torch.float8_e4m3fn).view(torch.uint8)
    s16[0:32] = torch.arange(256, dtype=torch.int32).to(torch.uint8).repeat(4).view(32, 32)      # every byte
    for r in range(16):                                                     # blocks of one code, of two codes
        packed[32 + r] = r * 17
        packed[48 + r] = r * 16 + (r * 5 & 15)
    packed[64:72] = 0x80                                                    # +-0 only
    s16[72:80] = torch.tensor([1, 0x7e], dtype=torch.uint8).repeat(16)      # smallest and largest scale in one block
    s16[80:128] = (s16[80:128] & 0x78) | 0x08                               # power-of-two scales: exact values, ties
    s16[128:144, 0::2] = 0                                                  # one group of a block all zero
    return packed, s16, torch.full((N,), rd)


DIVISORS = [1.0, 448.0, 2688.0 / 3.7, 1e30, 1e-30, 3.3e38]                  # some leave the exact quotients' range


@pytest.mark.parametrize("rd", DIVISORS)
def test_nvfp4_search_branches(dev, rd):
    """The conversion of a small weight (element by element) on blocks that reach each branch of the search."""
    packed, s16, div = search_blocks(rd)
    pm, em = NV.nvfp4_to_mxfp4(packed.to(dev), s16.view(torch.float8_e4m3fn).to(dev), div.to(dev))
    po, eo = O.nvfp4_to_mxfp4(packed.numpy(), s16.numpy(), div.numpy())
    bad = np.argwhere(em.cpu().numpy() != eo)
    assert bad.size == 0, f"exponents differ at {bad[:4].tolist()}"
    assert np.array_equal(pm.cpu().numpy(), po)


@pytest.mark.parametrize("rd", DIVISORS)
def test_nvfp4_search_by_magnitudes(dev, rd):
    """The same blocks often enough for the kernel of large weights (more than 2^19 blocks; three rows short of whole
    copies, so the last workgroup is partly idle): every row has the oracle's codes and exponents."""
    packed, s16, div = search_blocks(rd)
    po, eo = O.nvfp4_to_mxfp4(packed.numpy(), s16.numpy(), div.numpy())
    n, rows = 129, 129 * 256 - 3
    assert rows * 16 > 1 << 19 and rows * 16 % 256
    many = lambda t: t.to(dev).repeat(n, *[1] * (t.dim() - 1))[:rows].contiguous()
    pm, em = NV.nvfp4_to_mxfp4(many(packed), many(s16).view(torch.float8_e4m3fn), many(div))
    bad = (em != many(torch.from_numpy(eo))).nonzero()
    assert bad.numel() == 0, f"exponents differ at {bad[:4].tolist()}"
    assert torch.equal(pm, many(torch.from_numpy(po)))
