"""torch.library custom ops over libr9k's entries, so the dense linears can sit inside a torch.compile'd
graph (Dynamo cannot trace a call into the library) and be captured into HIP graphs. The reference's r9700_vllm/ops.py surface
for the 4-bit path:

  torch.ops.r9700.mxfp4_linear(x [M, K] bf16, wq, wsr, N, K, fold) -> [M, N] bf16   MXFP4 weight, per-token fp8 act
  torch.ops.r9700.nvfp4_linear(x [M, K] bf16, wq, ws, wg, N, K) -> [M, N] bf16      native NVFP4 weight (exact bits)

plus `mxfp4_gemm_q` (the GEMM on already-quantised rows, which the shared expert uses). A dense linear is the grouped
MoE GEMM with one expert and identity routing tables (`IdentityTables`). At decode widths it is one launch with the
activation quant inside (kernels.moe.dense_mxfp4_qa, dense_nvfp4_qa), then, up to 16 rows, the quant and the dense
kernel's weight stream without tables (dense_mxfp4_a8, dense_nvfp4_a8); wide MXFP4 linears leave these from 12 rows on
for the LDS-ring kernel (kernels.moe.dense_mid_wanted). The reference's fp8_linear / fp8_block_linear
(dense fp8 GEMMs) are outside this build.
"""
from __future__ import annotations

import torch

from ._compat import register_custom_op
from .kernels import moe as KM

_LIB = torch.library.Library("r9700", "FRAGMENT")
_registered = False


class IdentityTables:
    """Routing tables that make the grouped GEMM a dense one: rows 0..Mpad-1 in order, every block on expert 0,
    Mpad = M rounded up to the block. Built once per (device, Mpad, block) and reused (graph capture needs fixed
    addresses, and a decode step asks for the same few shapes every time). A width first met under capture gets tables
    that the graph fills itself: device fills only, and not kept, since they hold nothing before the first replay."""

    _cache: dict = {}

    @staticmethod
    def _build(device: torch.device, mpad: int, block: int):
        i32 = dict(dtype=torch.int32, device=device)
        return torch.arange(mpad, **i32), torch.full((mpad // block,), 0, **i32), torch.full((1,), mpad, **i32)

    @classmethod
    def get(cls, device: torch.device, M: int, block: int):
        mpad = -(-M // block) * block
        key = (device.type, device.index, mpad, block)
        t = cls._cache.get(key)
        if t is None:
            t = cls._build(device, mpad, block)
            if not (device.type == "cuda" and torch.cuda.is_current_stream_capturing()):
                cls._cache[key] = t
        return t


def _decode_mt(M: int) -> int:
    """M-tiles per routing block of a dense decode GEMM (kernels.moe.decode_mt)."""
    return KM.decode_mt(M)


def mxfp4_gemm_q(q: torch.Tensor, s: torch.Tensor, W, out: torch.Tensor, M: int, cfg, topk_w=None) -> None:
    """out [M, W.N] bf16 = dequant(q, s) @ W^T (* topk_w[row]) for one dense MXFP4 weight, on the kernel `cfg` names:
    ("P", prefill cfg) or a decode tuple (WV, SK, NPW[, MT]) whose only meaning here is the optional MT. A decode cfg
    with at most KM.DENSE_A8_MAX_M rows runs on the dense kernel (r9k_dense_mxfp4_a8), the decode GEMM's bits."""
    if (not KM.is_prefill_cfg(cfg) and M <= KM.DENSE_A8_MAX_M and not W.fold
            and KM.dense_mxfp4_a8(q, s, W, out, topk_w)):
        return
    if KM.is_prefill_cfg(cfg):
        tabs = IdentityTables.get(q.device, M, KM.prefill_block(cfg[1]))
        KM.moe_gemm(q, s, W, out, *tabs, M, 1, topk_w, num_experts=1, prefill=cfg[1])
        return
    MT = cfg[3] if len(cfg) > 3 else _decode_mt(M)
    tabs = IdentityTables.get(q.device, M, KM.MOE_BLOCK * MT)
    KM.moe_gemm(q, s, W, out, *tabs, M, 1, topk_w, *cfg[:3], num_experts=1, MT=MT)


def mxfp4_gemm_rows(q: torch.Tensor, s: torch.Tensor, W, out: torch.Tensor, M: int, fold: bool = False,
                    topk_w=None) -> None:
    """mxfp4_gemm_q on pick_cfg's choice (which the rows the dense kernel serves do without)."""
    if M <= KM.DENSE_A8_MAX_M and not W.fold and KM.dense_mxfp4_a8(q, s, W, out, topk_w):
        return
    mxfp4_gemm_q(q, s, W, out, M, KM.pick_cfg(W.N, W.K, M=M, kind="mxfp4", fold=fold), topk_w=topk_w)


# The prefill GEMMs address their activation rows and their output through 32-bit buffer ranges, so one launch may
# touch at most this many bytes of either; a longer dense linear runs as row ranges (row_ranges), each a launch of its
# own over its own identity tables.
BUF_LIMIT = (1 << 31) - 1


def row_ranges(M: int, N: int, K: int, limit: int = BUF_LIMIT) -> list:
    """[(r0, r1), ...] covering rows 0..M, as few and as even as possible, each range's output [r1 - r0, N] bf16 and
    fp8 activation codes [r1 - r0, K] within `limit` bytes."""
    per_row = max(2 * N, K, 1)
    n = -(-M // max(1, limit // per_row)) if M else 0
    bounds = [M * i // n for i in range(n + 1)] if n else [0]
    return list(zip(bounds[:-1], bounds[1:]))


def _mxfp4_linear_rows(x: torch.Tensor, W, out: torch.Tensor, fold: bool) -> None:
    M = x.shape[0]
    if M <= KM.DENSE_QA_MAX_M and not fold and KM.dense_mxfp4_qa(x, W, out):   # decode widths: quant in the launch
        return
    q, s = KM.quant_rows_fp8(x)
    if M < KM.PREFILL_MIN_M and KM.dense_mid_wanted(M, W.N, W.K):
        mxfp4_gemm_q(q, s, W, out, M, ("P", KM.MID_CFG))
    else:
        mxfp4_gemm_rows(q, s, W, out, M, fold)


def _mxfp4_linear(x: torch.Tensor, wq: torch.Tensor, wsr: torch.Tensor, N: int, K: int, fold: bool = False
                  ) -> torch.Tensor:
    M = x.shape[0]
    out = KM._empty(x, torch.bfloat16, M, N)
    W = KM.Mxfp4Experts(wq, wsr, N, K, fold)
    ranges = row_ranges(M, N, K)
    if len(ranges) == 1:
        _mxfp4_linear_rows(x, W, out, fold)
        return out
    for r0, r1 in ranges:
        _mxfp4_linear_rows(x[r0:r1], W, out[r0:r1], fold)
    return out


def _nvfp4_linear_rows(x: torch.Tensor, W, out: torch.Tensor) -> None:
    M = x.shape[0]
    if M <= KM.DENSE_NV_QA_MAX_M and KM.dense_nvfp4_qa(x, W, out):   # decode widths: the quant inside the GEMM launch
        return
    q, s = KM.quant_rows_fp8(x)
    if KM.dense_nvfp4_a8_wanted(M, W.N, W.K) and KM.dense_nvfp4_a8(q, s, W, out):
        return
    if M >= KM.NV_PREFILL_MIN_M and W.K % 32 == 0:
        tabs = IdentityTables.get(x.device, M, KM.prefill_block(KM.NV_PREFILL_CFG))
        KM.moe_gemm(q, s, W, out, *tabs, M, 1, None, num_experts=1, prefill=KM.NV_PREFILL_CFG)
    else:
        MT = _decode_mt(M)
        tabs = IdentityTables.get(x.device, M, KM.MOE_BLOCK * MT)
        KM.moe_gemm(q, s, W, out, *tabs, M, 1, None, num_experts=1, MT=MT)


def _nvfp4_linear(x: torch.Tensor, wq: torch.Tensor, ws: torch.Tensor, wg: torch.Tensor, N: int, K: int
                  ) -> torch.Tensor:
    """Native NVFP4 weights (prepare_nvfp4_weights of one expert) with per-row fp8 activations: one launch with the
    quant inside up to DENSE_NV_QA_MAX_M rows, the quant and the table-less dense kernel up to DENSE_NV_A8_MAX_M
    (dense_nvfp4_a8_wanted), the decode-family kernel below NV_PREFILL_MIN_M rows, the 128 x 128-tile prefill kernel
    (r9k_moe_4bit_prefill nv = 1) from there; row ranges past the 2 GiB buffer range (row_ranges)."""
    M = x.shape[0]
    out = KM._empty(x, torch.bfloat16, M, N)
    W = KM.Nvfp4Experts(wq, ws, wg, N, K)
    ranges = row_ranges(M, N, K)
    if len(ranges) == 1:
        _nvfp4_linear_rows(x, W, out)
        return out
    for r0, r1 in ranges:
        _nvfp4_linear_rows(x[r0:r1], W, out[r0:r1])
    return out


def _rows_out_fake(x: torch.Tensor, N: int) -> torch.Tensor:
    return torch.empty((x.shape[0], N), dtype=torch.bfloat16, device=x.device)


def _mxfp4_linear_fake(x: torch.Tensor, wq: torch.Tensor, wsr: torch.Tensor, N: int, K: int, fold: bool = False
                       ) -> torch.Tensor:
    return _rows_out_fake(x, N)


def _nvfp4_linear_fake(x: torch.Tensor, wq: torch.Tensor, ws: torch.Tensor, wg: torch.Tensor, N: int, K: int
                       ) -> torch.Tensor:
    return _rows_out_fake(x, N)


_OPS = (("mxfp4_linear", _mxfp4_linear, _mxfp4_linear_fake), ("nvfp4_linear", _nvfp4_linear, _nvfp4_linear_fake))


def register() -> None:
    global _registered
    if not _registered:
        for name, fn, fake in _OPS:
            register_custom_op(_LIB, name, fn, [], fake)
        _registered = True


def _call_on_rows(op, x: torch.Tensor, K: int, N: int) -> torch.Tensor:
    """op over x viewed as contiguous bf16 rows [-1, K], the result shaped back to x's leading dims + [N]."""
    register()
    flat = x.dim() == 2 and x.shape[1] == K                    # rows already: no view to make and undo
    rows = x if flat else x.reshape(-1, K)
    if rows.dtype != torch.bfloat16:
        rows = rows.to(torch.bfloat16)
    y = op(rows.contiguous())
    return y if flat else y.reshape(*x.shape[:-1], N)


def mxfp4_linear(x: torch.Tensor, wq: torch.Tensor, wsr: torch.Tensor, N: int, K: int, fold: bool = False
                 ) -> torch.Tensor:
    return _call_on_rows(lambda r: torch.ops.r9700.mxfp4_linear(r, wq, wsr, N, K, fold), x, K, N)


def nvfp4_linear(x: torch.Tensor, wq: torch.Tensor, ws: torch.Tensor, wg: torch.Tensor, N: int, K: int
                 ) -> torch.Tensor:
    return _call_on_rows(lambda r: torch.ops.r9700.nvfp4_linear(r, wq, ws, wg, N, K), x, K, N)
