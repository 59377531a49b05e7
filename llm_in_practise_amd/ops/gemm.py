"""Frozen-base GEMM dispatch: which kernel computes ``x · Wᵀ`` and ``dY · W``.

* Training / prefill sizes (M >= 256): the hand-written MFMA GEMM ``gemm4w`` (csrc/kernels/gemm4w*.hip) —
  forward with the residual in its epilogue, backward dX reading W as stored (transposed-B), split-K by its
  own cost model.  An NF4 base (QLoRA) either feeds its 4-bit codes straight into gemm4w (the NF4
  dequant-GEMM: the codes expanded to bf16 between the load and the LDS B image) or is expanded once per
  step at HBM speed (``nf4_dequant3_k``) when that copy serves two GEMMs (forward + dX): ``_nf4_w4``.
* Decode sizes: the split-K weight-streaming kernels (``skinny.hip``, ``gemv_w4``).
* Shapes no kernel takes (CPU tensors, K % 64): torch.
* ``GEMM_STATS`` counts every GEMM launch by form (bench.py's kernel-provenance record).

The LoRA op built on these is ``ops/linear.py``; the fused SwiGLU MLP ``ops/mlp.py``; the chunked LM-head loss
``ops/loss.py``.  Reference role: bitsandbytes' dequantize + cuBLAS (``Fine-Tuning/qwen3-8b-qlora-dist.py:102-110``).
"""
from __future__ import annotations

import collections
import os

import torch

from ..quant.nf4 import NF4Weight, dequantize_nf4
from ._native import _functorch_active, eager, fn_apply, force_reference, native

_MIN_M = 256     # training / prefill-sized GEMMs: gemm4w and the fused LoRA paths

# GEMM launches by form since the last clear (bench.py provenance): "gemm4w" (bf16 B operand), "gemm4w-nf4"
# (the NF4 codes read in-kernel), "nf4-expansion" (one bf16 copy of an NF4 base), "decode" (skinny / gemv
# weight-streaming kernels), "library" (torch.matmul fallback for shapes gemm4w does not take)
GEMM_STATS: collections.Counter = collections.Counter()


def _count(form: str, n: int = 1):
    GEMM_STATS[form] += n


def _g4w_ok(a: torch.Tensor, w: torch.Tensor, bt: bool) -> bool:
    """Shapes / strides the gemm4w kernel takes for a bf16 weight: a [M, K] row-major (row stride % 8),
    w [N, K] (or [K, N] when bt) with unit inner stride, training-sized M — the same predicate the
    binding enforces (``gemm4w_supported``: K % 64, N % 8, every operand's byte extent < 4 GiB), so an
    oversized operand falls back here instead of failing in the kernel's TORCH_CHECK."""
    if not (a.is_cuda and a.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and a.dim() == 2
            and w.dim() == 2 and a.shape[0] >= _MIN_M and a.stride(1) == 1 and w.stride(1) == 1
            and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0):
        return False
    K = a.shape[1]
    if (w.shape[0] if bt else w.shape[1]) != K:
        return False
    N = w.shape[1] if bt else w.shape[0]
    return bool(native().gemm4w_ok(a.shape[0], N, K, a.stride(0), w.stride(0), bt, False))


def _w4_ok(a: torch.Tensor, q: NF4Weight, bt: bool) -> bool:
    """An NF4 base the gemm4w kernel reads as codes (K9): forward x·deq(W)ᵀ (bt=False, a [M, K_w]) or
    dX = dY·deq(W) (bt=True, a [M, N_w]); blocksize 64, both dims multiples of 64, M > 8."""
    if not (a.is_cuda and a.dtype == torch.bfloat16 and a.dim() == 2 and a.shape[0] > 8
            and a.stride(1) == 1 and a.data_ptr() % 16 == 0 and q.kernel_ok()):
        return False
    n, k = q.shape
    if a.shape[1] != (n if bt else k):
        return False
    return bool(native().gemm4w_ok(a.shape[0], k if bt else n, a.shape[1], a.stride(0), 0, bt, True))


def _w4_gemm(a: torch.Tensor, q: NF4Weight, bt: bool, c: torch.Tensor | None = None) -> torch.Tensor:
    """gemm4w on NF4 codes: a·deq(W)ᵀ (+ c) or, bt, a·deq(W) (+ c)."""
    codes, sc = q.g4w_pack()
    n, k = q.shape
    _count("gemm4w-nf4")
    return native().gemm4w(a, codes, c, 0, bt, 0, 0, sc, k if bt else n)


def _nf4_dequant_bf16(q: NF4Weight) -> torch.Tensor:
    """One bf16 expansion of an NF4 base (HBM speed)."""
    n, k = q.shape
    _count("nf4-expansion")
    return native().nf4_dequant_fast(q.codes, q.gemv_scales(), n, k)


# Which NF4 form a call takes (LIPA_NF4_GEMM = w4 | expand | auto).  Measured per GEMM at the Qwen3-8B
# shapes (profiles/r4/gemm4w_nf4_ab.txt): the in-kernel expansion costs 1.1-1.2x the bf16 gemm4w time
# (the 3-VALU-per-element table lookup is only partly hidden beside 16x16x32 MFMAs), the same as an
# expansion + bf16 GEMM when that copy serves ONE GEMM.  "auto" therefore expands where the copy is
# reused — a training forward whose backward needs dX (the copy is kept for it: ≈14 GB transient for
# Qwen3-8B), a checkpointed layer (one expansion per optimizer step, below) — and feeds the codes
# straight in everywhere else (inference, no-grad prefill, frozen inputs): no transient bf16 weights.
# "w4" everywhere is the memory-lean training mode (peak HBM ≈ the 4-bit model + activations).
_NF4_MODE = os.environ.get("LIPA_NF4_GEMM", "auto")


def _nf4_w4(reused: bool) -> bool:
    if _NF4_MODE == "w4":
        return True
    if _NF4_MODE == "expand":
        return False
    return not (reused or _IN_CKPT[0])


# NF4-aware activation checkpointing: inside a checkpointed layer (its forward AND its backward
# recompute) the bf16 expansion of each frozen NF4 base is made once per optimizer step and reused —
# the reference-faithful step (gradient checkpointing + sequential GA micro-steps) otherwise expands
# every weight 2 × GA times per step.  The copies are held in ONE registry, bounded by
# LIPA_CKPT_NF4_CACHE_GB (default 32; 0 = off: every call expands), and released eagerly when the
# optimizer steps (``nf4_cache_advance``: optim/adamw.py, parallel/zero.py; an optimizer that never
# calls it keeps at most the budget).  Memory: the budget is the cost — Qwen3-8B's bases expand to
# 13.9 GB (peak HBM of the faithful bench step: README §3).
_CKPT_BUDGET = float(os.environ.get("LIPA_CKPT_NF4_CACHE_GB", "32")) * 2 ** 30
_IN_CKPT = [0]
_CACHE: dict = {}        # id(NF4Weight) -> (weight, bf16 expansion)
_CACHE_BYTES = [0]


def nf4_cache_advance():
    """Called by the optimizers at every step: the expanded copies of the finished step are released."""
    _CACHE.clear()
    _CACHE_BYTES[0] = 0


def _nf4_expand(q: NF4Weight) -> torch.Tensor:
    """The bf16 expansion for the "expand" form (cached inside checkpointed layers, see above)."""
    if _IN_CKPT[0]:
        hit = _CACHE.get(id(q))
        if hit is not None and hit[0] is q:
            return hit[1]
    w = _nf4_dequant_bf16(q)
    if _IN_CKPT[0] and _CACHE_BYTES[0] + w.numel() * 2 <= _CKPT_BUDGET:
        _CACHE[id(q)] = (q, w)
        _CACHE_BYTES[0] += w.numel() * 2
    return w


def head_logits(h: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """LM-head logits of serving rows, batch-invariant: on the GPU always gemm4w with one K-split — every logit
    is one lane's fp32 accumulation over K in the same order whatever the tile shape the planner picks for this
    row count — so a request's greedy tokens do not depend on how many rows share the call (continuous batching,
    hipGraph buckets, the pipelined engine).  A library GEMM's algorithm (and rounding) changes with M.  The
    head is weight-streaming at decode sizes (151936 × 4096 bf16 = 1.2 GB per call): the kernel reads each
    weight panel once, as a GEMV would."""
    x = h.reshape(-1, h.shape[-1])
    if not x.is_contiguous():
        x = x.contiguous()
    if (x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and weight.dim() == 2
            and weight.stride(1) == 1 and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
            and weight.shape[1] == x.shape[1]
            and native().gemm4w_ok(x.shape[0], weight.shape[0], x.shape[1], x.stride(0), weight.stride(0), False,
                                   False)):
        _count("gemm4w")
        y = native().gemm4w(x, weight, None, 1, False)
    else:
        y = _base_gemm(x, weight)
    return y.view(*h.shape[:-1], weight.shape[0])


def norms_rows(x: torch.Tensor, weight, base, glu: bool) -> bool:
    """Whether the decode products (csrc/kernels/skinny.hip) take these rows in front of their RMSNorm: few bf16 rows of 512 .. 4096
    that fit into LDS, no gradient and no transform, a norm's weight of their type and a bf16 weight that the product takes."""
    return (not _functorch_active() and x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and 1 <= x.shape[0] <= 4 and x.is_contiguous() and x.data_ptr() % 16 == 0
            and isinstance(weight, torch.Tensor) and weight.is_cuda and weight.dtype == torch.bfloat16 and weight.is_contiguous()
            and weight.shape == x.shape[1:] and weight.data_ptr() % 16 == 0
            and isinstance(base, torch.Tensor) and base.is_cuda and base.dtype == torch.bfloat16 and base.is_contiguous()
            and base.shape[1] == x.shape[1] and base.data_ptr() % 16 == 0 and not base.requires_grad
            and not (torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad)) and not force_reference()
            and native().skinny_norms(x.shape[0], x.shape[1], glu))


class _NormedRowsFn(torch.autograd.Function):
    """(No backward: normed_rows leaves what needs a gradient to the differentiable ops.)"""
    @staticmethod
    def forward(ctx, x, weight, eps, base):
        return native().gemm_skinny(x, base, None, weight, eps)


def normed_rows(x: torch.Tensor, weight, eps: float, base) -> torch.Tensor | None:
    """``rms_norm(x) · baseᵀ`` of a few decode rows in one launch, every bit as from the two kernels, or None where that is not served
    (see :func:`norms_rows`; N as for the product alone).  Norm and product → here, µs at 1 row: 6144 × 4096
    15.4 → 12.5, 6144 × 2560 12.6 → 9.6, 4096 × 1024 5.7 → 4.6."""
    if not norms_rows(x, weight, base, False) or base.shape[0] > 8192 or base.shape[0] % 16:
        return None
    _count("decode")
    return fn_apply(_NormedRowsFn, x, weight, eps, base)


def _narrow_rows(x, base, residual):
    """How the product of up to 64 rows and a narrow bf16 weight runs: 1 in the decode products (csrc/kernels/skinny.hip), 64 or 128 in four
    parts of units of that depth (csrc/kernels/rows.hip), 0 by what stands below.  Up to 32 rows and K = 8192, and below K = 4096, the decode
    products are the fastest or within 10 % of it (1024 × 3072 from 40 rows on 10 to 20 %; it is left at one launch); deeper weights and more rows take
    the parts, one launch more, where x is read by a quarter of the workgroups.
    Library / decode products / parts in µs, W cold, residual included, at 17 / 32 / 48 / 64 rows: 4096 × 12288 26.6 / 30.1 / 35.8 / 39.5, 22.0 / 29.4 /
    35.2 / 37.0 and 23.3 / 25.1 / 25.3 / 26.9, 2560 × 9728 22.4 / 23.6 / 23.7 / 30.9, 15.7 / 19.2 / 25.0 / 27.1 and 15.8 / 16.9 / 19.0 / 19.5, 1024 × 12288
    18.8 / 24.1 / 19.6 / 20.5, 17.5 / 21.9 / 29.5 / 31.8 and 13.0 / 13.4 / 15.1 / 16.5, 4096 × 4096 16.1 / 16.1 / 16.2 / 17.8, 8.9 / 9.9 / 12.4 / 13.1 and 11.1 /
    11.6 / 12.2 / 12.8, 2560 × 4096 14.8 / 14.5 / 14.6 / 16.6, 7.8 / 9.1 / 11.5 / 12.3 and 10.3 / 10.7 / 10.6 / 11.3, 1024 × 3072 13.5 / 11.8 / 13.6 / 13.8, 6.0 /
    7.3 / 9.1 / 9.7 and 6.7 / 7.1 / 7.8 / 8.1.  At 1 / 16 rows library and decode products 4096 × 12288 21.4 / 21.5 and 18.0 / 20.3, 2560 × 9728 18.1 / 16.0 and
    12.1 / 15.0.  (5120 × 4096 at 17 / 32: 15.4 / 14.7 and 14.2 / 16.4.)
    Error against 64 bits, residual included: 1.65e-3 to 1.67e-3 from all three; results that are not the exact one rounded, per 100 000, library
    and here: 4096 × 12288 33 and 33 at 32 rows, 44 and 33 at 48, 39 and 39 at 64, 4096 × 4096 16 and 16, 26 and 18, 18 and 18, 2560 × 9728 33 and 33, 28 and
    28, 34 and 34 (of 500 000 results or more)."""
    M, K = x.shape
    N = base.shape[0]
    if not (x.is_cuda and 1 <= M <= 64 and N <= 4096 and N % 16 == 0 and K % 64 == 0 and K < 1 << 24 and eager(x, base, residual) and x.dtype == base.dtype == torch.bfloat16
            and x.stride(1) == 1 and x.stride(0) % 8 == 0 and base.is_contiguous() and x.data_ptr() % 16 == 0 and base.data_ptr() % 16 == 0
            and x.get_device() == base.get_device() == torch.cuda.current_device()
            and (residual is None or (residual.dtype == torch.bfloat16 and residual.shape == (M, N) and residual.is_contiguous()
                                      and residual.data_ptr() % 16 == 0 and residual.get_device() == x.get_device()))):
        return 0
    if M <= 16:
        return int(K > 8192 and K % 128 == 0)
    if K < 4096 or (M <= 32 and K <= 8192):
        return 1
    return 0 if K % 512 else 128 if M <= 32 else 64


class _RowsNormedFn(torch.autograd.Function):
    """(No backward: rows_normed leaves what needs a gradient to the differentiable ops.)"""
    @staticmethod
    def forward(ctx, x, base, residual, unit, weight, eps):
        return tuple(native().rows_parts_norm(x, base, residual, unit, weight, eps))


def norm_follows(x: torch.Tensor, residual, weight, N: int) -> bool:
    """Whether the launch that adds up a decode product's parts may form the RMSNorm behind it as well (csrc/kernels/rows.hip): bf16 rows and a
    norm's weight of their type, in memory of their own and without gradients, of a width the kernel takes."""
    return (x.is_cuda and isinstance(residual, torch.Tensor) and isinstance(weight, torch.Tensor) and eager(x, residual, weight)
            and x.dim() == 2 and x.dtype == residual.dtype == weight.dtype == torch.bfloat16 and weight.get_device() == residual.get_device() == x.get_device()
            and residual.shape == (x.shape[0], N) and residual.is_contiguous() and residual.data_ptr() % 16 == 0
            and weight.shape == (N,) and weight.is_contiguous() and weight.data_ptr() % 16 == 0 and not force_reference()
            and not (torch.is_grad_enabled() and (x.requires_grad or residual.requires_grad or weight.requires_grad))
            and native().parts_norm_serves(N))


def rows_normed(x: torch.Tensor, base, residual, weight, eps: float):
    """``(y, rms_norm(y))`` of ``y = x · baseᵀ + residual`` for 17 to 64 decode rows whose product adds up parts of K: every bit as from the
    product and the norm behind it, a launch less; None where that is not served."""
    if not (isinstance(base, torch.Tensor) and 16 < x.shape[0] <= 64 and not base.requires_grad
            and norm_follows(x, residual, weight, base.shape[0])):
        return None
    unit = _narrow_rows(x, base, residual)
    if unit <= 1:
        return None
    _count("decode")
    return fn_apply(_RowsNormedFn, x, base, residual, unit, weight, eps)


def _base_gemm(x, base, ext_a=None, ext_b=None, residual=None):
    if isinstance(base, NF4Weight):
        if x.shape[0] <= 8 and base.kernel_ok():   # decode: weight-streaming GEMV, no MFMA tile
            n, k = base.shape
            _count("decode")
            y = native().gemv_w4(x, base.codes, base.gemv_scales(), None, n, base.blocksize,
                                 residual if ext_a is None else None)
            if ext_a is not None:
                y = y + ext_a @ ext_b.t()
                if residual is not None:
                    y = y + residual
            return y
        if _w4_ok(x, base, False):                  # the NF4 dequant-GEMM (gemm4w reads the codes)
            y = _w4_gemm(x, base, False, None if residual is None else residual.contiguous())
            return y if ext_a is None else y.addmm_(ext_a, ext_b.t())
        w = _nf4_dequant_bf16(base) if (base.kernel_ok() and x.is_cuda) else dequantize_nf4(base, x.dtype)
        return _base_gemm(x, w, ext_a, ext_b, residual)
    M, K = x.shape
    N = base.shape[0]
    few = (x.is_cuda and M <= 16 and N <= 8192 and K <= 8192 and N % 16 == 0 and K % 64 == 0 and x.stride(0) % 8 == 0
           and x.stride(1) == 1 and base.is_contiguous())
    narrow = _narrow_rows(x, base, residual) if M <= 64 and not few else 0
    if few or narrow:
        # decode-sized q|k|v / o projections: the weight-streaming MFMA kernel (csrc/kernels/skinny.hip) takes 8.3-9.3 µs for
        # 4096 × 4096 and 1-16 rows, residual included, where hipBLASLt takes 15.3 (12.6-14.2 against 15 for 6144 rows of W,
        # 24 against 29-31 for 8192 × 8192)
        _count("decode")
        y = native().rows_parts(x, base, residual, narrow) if narrow > 1 else native().gemm_skinny(x, base, residual)
        return y if ext_a is None else y.addmm_(ext_a, ext_b.t())
    if _g4w_ok(x, base, False):
        _count("gemm4w")
        y = native().gemm4w(x, base, None if residual is None else residual.contiguous(), 0, False)
        return y if ext_a is None else y.addmm_(ext_a, ext_b.t())
    # shapes gemm4w does not take (CPU, M < 256, K % 64): torch — residual = addmm's beta term, the LoRA
    # K-slice one rank-Σr update
    _count("library")
    if residual is None:
        y = x @ base.t()
    elif x.is_cuda and M <= 64:             # (decode rows: the same product without a launch that copies the residual)
        y = native().lt_addmm(residual, x, base)
    else:
        y = torch.addmm(residual, x, base.t())
    if ext_a is not None:
        y.addmm_(ext_a, ext_b.t())
    return y


def _dense_dx(dy: torch.Tensor, w: torch.Tensor, c: torch.Tensor | None = None) -> torch.Tensor:
    """dX = dY·W (+ c) for a bf16 [N, K] weight: gemm4w's transposed-B form (W read as stored; split-K when
    the output has fewer tiles than CUs, e.g. gate|up dX at M = 2048), else torch."""
    if _g4w_ok(dy, w, True):
        _count("gemm4w")
        return native().gemm4w(dy, w, c, 0, True)
    _count("library")
    return dy @ w if c is None else torch.addmm(c, dy, w)


def _base_gemm_t(dy, base, ext_a=None, ext_b=None, c=None):
    """dX = dY·W (+ c) (+ ext_a · ext_bᵀ, ext_b given as [K, R])."""
    if isinstance(base, NF4Weight):
        if _w4_ok(dy, base, True):
            dx = _w4_gemm(dy, base, True, c)
            return dx if ext_a is None else dx.addmm_(ext_a, ext_b.t())
        base = _nf4_dequant_bf16(base) if (base.kernel_ok() and dy.is_cuda) else dequantize_nf4(base, dy.dtype)
    dx = _dense_dx(dy, base, c)
    return dx if ext_a is None else dx.addmm_(ext_a, ext_b.t())


def matmul_f32(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``x w^T`` with a float result (``x`` ``[T, K]`` and ``w`` ``[N, K]`` of one dtype): bf16 operands accumulate in
    float and the sums are not rounded back (logits, pre-activations of recurrences)."""
    if x.dtype == torch.float32 or not x.is_cuda:
        return x.float() @ w.float().t()
    return torch.mm(x, w.t(), out_dtype=torch.float32)
