"""The EXL3 shard GEMM as PyTorch custom ops (same names and schema as the reference's
orcasaq2/ops.py:37-66), backed by the gfx950 HIP library through its C ABI.

A custom op keeps the shard opaque to Dynamo -- one graph node with a known output shape
(the register_fake below) -- so a torch.compile'd model compiles around it, and its
kernels only enqueue on the current stream, so it can be captured in a HIP graph.

Dispatch on the number of activation rows (reference: orcasaq2/ops.py:25, 46-59):
  * rows <= 16            fused decode-GEMV (exl3_gemv): packed words streamed from HBM and
                          decoded in registers, never stored; rows 1..4: one persistent kernel
                          (MFMA multiply-accumulate; a column group split over workgroups is
                          summed in fixed point in the workspace and finished by the workgroup
                          whose add completes it); rows 5..16, and 2..4-row shards too large for
                          that kernel's tables: the same decode on 4 x 2-tile units, one MFMA
                          serving all rows; output Hadamard and svh at the end;
  * 16 < rows <= SPLIT_MAX_ROWS
                          fused decode-GEMM (exl3_gemm): set-up of x in fragment order, the
                          K-split decode into MFMA operands, a finishing launch; a fused layer's
                          shards together (shards_gemm).  A row knob set lower is the
                          reference's hard switch to the reconstruct branch;
  * above                 the reference's reconstruct branch: had_r_128(x, suh), dense W_q
                          (decoded transposed, (oc, ic)) into a scratch freed on exit, library
                          fp16 transposed-B GEMM, had_r_128(y, svh) -- except, while the row
                          knob is at its default, 8192+ inputs up to WIDE_FUSED_MAX_ROWS rows
                          (faster fused but at 2048 rows, kept fused there for no dense W_q)
                          and 4096..8191 inputs with at least twice as many outputs in
                          WIDE_OUT_FUSED_ROWS, where the fused kernel measured faster
                          (_fused_gemm_faster); a fused layer whose shards all route fused
                          runs them as one grouped launch (shards_gemm).
The op is registered for the "cuda" device type (ROCm) only: there is no CPU path.
"""

import functools
import os

import torch
from torch import Tensor

from . import _native

# Rows at or below which the fused kernels are used (the reference's default and env knob,
# orcasaq2/ops.py:22-25).  Above it the dense W_q is rebuilt once and a library GEMM runs --
# except, while the knob is left at its default, for the shapes where the fused kernel
# measured faster (_fused_gemm_faster).  Setting the knob makes it the hard switch of the
# reference.
GEMM_MAX_ROWS = int(os.environ.get("ORCA_EXL3_GEMM_MAX_ROWS", "144"))
GEMM_MAX_ROWS_SET = "ORCA_EXL3_GEMM_MAX_ROWS" in os.environ
SPLIT_MAX_ROWS = 512                 # every shard: the K-split decode-GEMM up to here
WIDE_FUSED_MAX_ROWS = 2560           # 8192+ inputs: fused up to here
WIDE_OUT_FUSED_ROWS = (1536, 3072)   # 4096..8191 inputs, oc >= 2 ic: fused in (lo, hi] too
GEMV_MAX_ROWS = _native.GEMV_MAX_ROWS


def exl3_K(trellis: Tensor):
    """Bits per weight = trellis.shape[-1] / 16 (16-weight steps per tile row).  Integers
    stay int; the mul1 half rates (1.5/2.5/3.5: 24/40/56 words per tile) stay float, as in
    orcasaq2/ops.py:28-34.  The HIP kernels accept integer K in 1..8 only."""
    k = trellis.shape[-1] / 16
    return int(k) if float(k).is_integer() else k


def _fused_gemm_faster(rows: int, ic: int, oc: int) -> bool:
    """Whether the fused decode-GEMM beats the reconstruct branch for one shard of `rows` >
    GEMV_MAX_ROWS rows.  Measured on MI355X at settled clocks (us per call, HIP graph, fused /
    reconstruct branch; the branch's library GEMM is far from monotone in the row count):
      17408 -> 5120:  144: 116 / 176, 256: 118 / 225, 1024: 221 / 308, 1536: 308 / 430,
                      2048: 388 / 370, 2560: 499 / 652, 3072: 589 / 487, 4096: 732 / 701;
      5120 -> 17408:  64: 60 / 77, 128: 80 / 83, 144: 112 / 95, 384: 143 / 120,
                      1024: 220 / 232, 1536: 300 / 285, 2048: 390 / 478, 2560: 478 / 569,
                      3072: 592 / 644, 4096: 742 / 685;
      5120 -> 6144:   40: 39 / 45, 64: 46 / 46, 80: 60 / 49, 144: 71 / 52, 2048: 166 / 142.
    So: 8192+ inputs fused up to WIDE_FUSED_MAX_ROWS -- at 2048 rows too, 5% slower than the
    reconstruct branch but with no dense W_q (the branch writes and reads a 2 ic oc-byte
    transient, 178 MB for down_proj) and no library GEMM;
    4096..8191 inputs fused up to 64 rows, and with oc >= 2 ic up to 128 rows and within
    WIDE_OUT_FUSED_ROWS; narrower inputs (unmeasured below 4096) fused up to GEMM_MAX_ROWS."""
    if ic >= 8192:
        return rows <= WIDE_FUSED_MAX_ROWS
    if ic < 4096:
        return True
    if oc >= 2 * ic:
        lo, hi = WIDE_OUT_FUSED_ROWS
        return rows <= 128 or lo < rows <= hi
    return rows <= 64


def _fused_route(rows: int, ic: int, oc: int) -> bool:
    """The fused decode-GEMM for rows > GEMV_MAX_ROWS: within GEMM_MAX_ROWS where it measured
    faster; beyond it, while the knob is at its default, for inputs of 4096 or more where it
    measured faster (narrower inputs keep the reference's switch)."""
    if rows <= GEMM_MAX_ROWS:
        return _fused_gemm_faster(rows, ic, oc)
    return not GEMM_MAX_ROWS_SET and ic >= 4096 and _fused_gemm_faster(rows, ic, oc)


def _op_route(rows: int, ic: int, oc: int) -> bool:
    """Whether the ops take the fused path for rows > GEMV_MAX_ROWS.  Up to SPLIT_MAX_ROWS rows the
    library runs the K-split decode-GEMM, measured faster than the reconstruct branch on every
    shape there (us, fused / branch: 5120 -> 6144 at 144 rows 37 / 53, 256: 39 / 73, 384: 48 / 64;
    5120 -> 17408 at 144 rows 78 / 95, 256: 81 / 109, 384: 105 / 118; 17408 -> 5120 at 384 rows
    102 / 183), unless the row knob is set below; above, the stream-K kernel where it measured
    faster (_fused_route)."""
    if rows <= SPLIT_MAX_ROWS:
        return rows <= GEMM_MAX_ROWS or not GEMM_MAX_ROWS_SET
    return _fused_route(rows, ic, oc)


def _shard_gemm_impl(x: Tensor, trellis: Tensor, suh: Tensor, svh: Tensor, oc: int, k: float,
                     mcg: bool, mul1: bool) -> Tensor:
    cb = _native.codebook_id(mcg, mul1)
    if float(k).is_integer():
        k = int(k)
    rows, ic = x.shape
    if rows == 0:
        return x.new_empty((0, oc), dtype=torch.half)
    if rows <= GEMV_MAX_ROWS:
        return _native.gemv(x, trellis, suh, svh, k, cb)
    if _op_route(rows, ic, oc):
        return _native.gemm(x, trellis, suh, svh, k, cb)
    return _reconstruct_branch(x, trellis, suh, svh, k, cb)


def _reconstruct_branch(x: Tensor, trellis: Tensor, suh: Tensor, svh: Tensor, k, cb: int) -> Tensor:
    """The reference's prefill branch (orcasaq2/ops.py:50-59): had_r_128, reconstruct, a dense
    GEMM, had_r_128.  The dense W_q lives only for the duration of the call, decoded as W_q^T
    (oc, ic) so the library runs its transposed-B GEMM (measured 15-20% faster than x @ W_q at
    512-4096 rows on MI355X)."""
    xh = _native.had_r_128(x, pre=suh)
    wt = _native.reconstruct_t(trellis, k, cb)
    y = torch.nn.functional.linear(xh, wt)
    del wt, xh
    return _native.had_r_128(y, out=y, post=svh)


@torch.library.custom_op("orcasaq2::shard_gemm", mutates_args=(), device_types="cuda")
def shard_gemm(x: Tensor, trellis: Tensor, suh: Tensor, svh: Tensor,
               oc: int, k: float, mcg: bool, mul1: bool) -> Tensor:
    return _shard_gemm_impl(x, trellis, suh, svh, oc, k, mcg, mul1)


@shard_gemm.register_fake
def _shard_gemm_fake(x: Tensor, trellis: Tensor, suh: Tensor, svh: Tensor,
                     oc: int, k: float, mcg: bool, mul1: bool) -> Tensor:
    return x.new_empty((x.shape[0], oc), dtype=torch.half)


@torch.library.custom_op("orcasaq2::shards_gemv", mutates_args=(), device_types="cuda")
def shards_gemv(x: Tensor, trellis: list[Tensor], suh: list[Tensor], svh: list[Tensor],
                oc: list[int], k: list[float], mcg: list[bool], mul1: list[bool]) -> Tensor:
    """All shards of a fused layer (q/k/v, gate/up) for rows <= 16 in as few launches as
    there are distinct (K, codebook); outputs are written side by side, which is the
    per-shard loop + torch.cat of orcasaq2/config.py:237-243 without the copy."""
    shards = [dict(trellis=t, suh=a, svh=b, oc=o, K=kk, codebook=_native.codebook_id(m, m1))
              for t, a, b, o, kk, m, m1 in zip(trellis, suh, svh, oc, k, mcg, mul1)]
    return _native.gemv_grouped(x, shards)


@shards_gemv.register_fake
def _shards_gemv_fake(x, trellis, suh, svh, oc, k, mcg, mul1) -> Tensor:
    return x.new_empty((x.shape[0], sum(oc)), dtype=torch.half)


@torch.library.custom_op("orcasaq2::shards_gemm", mutates_args=(), device_types="cuda")
def shards_gemm(x: Tensor, trellis: list[Tensor], suh: list[Tensor], svh: list[Tensor],
                oc: list[int], k: list[float], mcg: list[bool], mul1: list[bool]) -> Tensor:
    """All shards of a fused layer for rows > 16 (up to GEMM_MAX_ROWS, and above it when every
    shard routes fused): one set-up kernel (each shard's Hadamard pass) and one stream-K
    launch per codebook (per K with 256-row tiles) for all of them, outputs side by side --
    the per-shard shard_gemm loop + torch.cat of orcasaq2/config.py:237-243 with one launch
    tail instead of one per shard."""
    shards = [dict(trellis=t, suh=a, svh=b, oc=o, K=kk, codebook=_native.codebook_id(m, m1))
              for t, a, b, o, kk, m, m1 in zip(trellis, suh, svh, oc, k, mcg, mul1)]
    return _native.gemm_grouped(x, shards)


@shards_gemm.register_fake
def _shards_gemm_fake(x, trellis, suh, svh, oc, k, mcg, mul1) -> Tensor:
    return x.new_empty((x.shape[0], sum(oc)), dtype=torch.half)


# Above SPLIT_MAX_ROWS a layer's shards take the K-split decode-GEMM together where it beats their
# own routes, by estimates (us on MI355X) fitted to HIP-graph timings at 520..4096 rows of 2048-,
# 5120-, 6144- and 17408-input layers.  Measured, own routes / K split: qkv 5120 -> 6144 + 2 x 1024 at
# 520, 1024, 1536, 2048 rows 150 / 94, 181 / 135, 217 / 197, 257 / 262; its k and v alone at 2048, 3072,
# 4096 rows 113 / 84, 136 / 133, 162 / 163; gate_up 5120 -> 2 x 17408 at 520, 640, 768 rows 278 / 295,
# 326 / 305, 341 / 365; 2048 -> 2 x 6144 at 1024, 1536 rows 106 / 99, 126 / 149; 17408 -> 5120 (stream-K)
# at 640, 768, 1024 rows 185 / 156, 190 / 187, 225 / 240.
_CUS = 256
_SPLIT_MARGIN = 1.05   # the library GEMM is far from monotone: take the K split where it is clear


def _ksplit_us(rows: int, ic: int, ocs) -> float:
    """Whole rounds of 128 x 128-output segments, one per CU (fill, epilogue, then a step of 32
    inputs per pair of waves), and the segments left over split evenly, with a finishing launch."""
    full, rem = divmod(-(-rows // 128) * (sum(ocs) // 128), _CUS)
    steps = ic / 32
    us = 4 + 1e-6 * rows * ic * len(ocs) + full * (10 + 1.1 * steps / 4)
    return us + (20 + 1.1 * rem * steps / (4 * _CUS) if rem else 0)


def _own_us(rows: int, ic: int, oc: int) -> float:
    """The shard's own route: the stream-K kernel where _fused_route takes it (256-row tiles and a
    tail of its own), else the reconstruct branch (four launches, W_q written and read, the library
    GEMM, two Hadamard passes)."""
    mweights = ic * oc * 1e-6
    if _fused_route(rows, ic, oc):
        return 60 + 0.472 * -(-rows // 256) * mweights
    return 28 + 0.4 * mweights + 0.18 * rows / 128 * mweights + 1e-6 * rows * (ic + oc)


@functools.lru_cache(maxsize=1024)
def _ksplit_shards(rows: int, ic: int, ocs: tuple) -> tuple:
    """Shards (indices) of a layer above SPLIT_MAX_ROWS that run as one K-split call: the narrowest
    ones, as many as give the least estimated time with the wider ones on their own routes."""
    if GEMM_MAX_ROWS_SET:
        return ()
    idx = sorted(range(len(ocs)), key=lambda i: ocs[i])
    own = [_own_us(rows, ic, ocs[i]) for i in idx]
    best, take = sum(own), 0
    for n in range(1, len(idx) + 1):
        us = _SPLIT_MARGIN * _ksplit_us(rows, ic, [ocs[i] for i in idx[:n]]) + sum(own[n:])
        if us < best:
            best, take = us, n
    return tuple(sorted(idx[:take]))


def _shards_linear_impl(x: Tensor, trellis: list[Tensor], suh: list[Tensor], svh: list[Tensor],
                        oc: list[int], k: list[float], mcg: list[bool], mul1: list[bool]) -> Tensor:
    rows, ic = x.shape
    cb = [_native.codebook_id(m, m1) for m, m1 in zip(mcg, mul1)]
    out = x.new_empty((rows, sum(oc)))
    if rows == 0:
        return out
    if x.dtype == torch.bfloat16 and x.data_ptr() % 4:
        x = x.clone()   # the kernels load pairs; a copy converted to fp16 was always aligned
    cols = [0]
    for o in oc:
        cols.append(cols[-1] + o)

    def fused(idx, ksplit=False):
        def pick(v):
            return v if len(idx) == len(oc) else [v[i] for i in idx]
        _native.linear_io(x, out, pick(cols), pick(trellis), pick(suh), pick(svh), pick(oc), pick(k), pick(cb), ksplit)

    every = range(len(oc))
    if rows <= GEMV_MAX_ROWS or (rows <= SPLIT_MAX_ROWS and _op_route(rows, ic, 0)):
        fused(every)
        return out
    split = _ksplit_shards(rows, ic, tuple(oc)) if rows > SPLIT_MAX_ROWS else ()
    if split:
        fused(split, True)
    rest = [i for i in every if i not in split]
    if rest and all(_op_route(rows, ic, oc[i]) for i in rest):
        fused(rest)
        return out
    fn = "orcasaq2::shards_linear"
    for i in rest:
        if _op_route(rows, ic, oc[i]):
            fused([i])
            continue
        # the reconstruct branch (see _reconstruct_branch)
        xh = torch.empty((rows, ic), dtype=torch.half, device=x.device)
        _native.had_r_128_cols(fn, x, xh, 0, pre=suh[i])
        wt = _native.reconstruct_t(trellis[i], k[i], cb[i])
        y = torch.nn.functional.linear(xh, wt)
        del wt, xh
        _native.had_r_128_cols(fn, y, out, cols[i], post=svh[i])
        del y
    return out


@torch.library.custom_op("orcasaq2::shards_linear", mutates_args=(), device_types="cuda")
def shards_linear(x: Tensor, trellis: list[Tensor], suh: list[Tensor], svh: list[Tensor],
                  oc: list[int], k: list[float], mcg: list[bool], mul1: list[bool]) -> Tensor:
    """A layer's shards for any row count, fp16 or bf16 x in and out: what
    orcasaq2/config.py:228-245 does around the shard op -- x to fp16, the shards' outputs side by
    side, back to x's dtype -- with the conversions and the concatenation in the kernels' loads and
    stores.  Separate passes cost a bf16 decoder layer ~40 us at one row (eight launches) and
    ~420 us at 2048 rows; the concatenation 206 us of a gate_up call at 4096 rows."""
    return _shards_linear_impl(x, trellis, suh, svh, oc, k, mcg, mul1)


@shards_linear.register_fake
def _shards_linear_fake(x, trellis, suh, svh, oc, k, mcg, mul1) -> Tensor:
    return x.new_empty((x.shape[0], sum(oc)))


# The same op without custom_op's Python wrapper, for eager calls that need no gradient: the wrapper
# (an autograd kernel that refuses backward, checks of the outputs) costs ~15 us of host time per
# call (23-25 us against 8-10 with three shards), as long as a decode launch runs.
_eager = torch.library.Library("orcasaq2", "FRAGMENT")
_eager.define("shards_linear_eager(Tensor x, Tensor[] trellis, Tensor[] suh, Tensor[] svh, int[] oc, float[] k, "
              "bool[] mcg, bool[] mul1) -> Tensor")
_eager.impl("shards_linear_eager", _shards_linear_impl, "CUDA")
torch.library.register_fake("orcasaq2::shards_linear_eager", _shards_linear_fake, lib=_eager)


def shards_linear_op(x: Tensor):
    """shards_linear, or its eager form where nothing could ask for a derivative of the call:
    not being compiled, no gradient wanted of x, no forward-mode level open."""
    if (torch.compiler.is_compiling() or (x.requires_grad and torch.is_grad_enabled())
            or torch.autograd.forward_ad._current_level >= 0):
        return torch.ops.orcasaq2.shards_linear
    return torch.ops.orcasaq2.shards_linear_eager
