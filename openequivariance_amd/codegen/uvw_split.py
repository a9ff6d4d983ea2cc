"""Split-operand matrix kernels for shared-weight 'uvw' tensor products in fp32: forward, dX / dY and dW.

The fp32 matrix instructions share the datapath of the vector unit and give 157 TFLOP/s; the bf16 ones are a pipe of their
own with 16 times that. Here every fp32 operand is the sum of three bf16 numbers (8 mantissa bits each: together the 24 of
fp32; a remainder is exact), and a product the six cross products of weight 2^-16 and above, accumulated in fp32 by
``v_mfma_f32_16x16x32_bf16``: 6 x 16 cycles for what takes the fp32 instruction 8 x 32. What is dropped is 2^-24.3 of a
product at most and 2^-27.4 root mean square, and 32 products are summed before they are rounded, so the results are nearer to 64 bits than those of the
fp32 instruction. 64x{0e,1o,2e} (x) {0e,1o,2e} -> the same, relative errors of Z, dX, dY, dW at 100 003 rows, before
and now: 2.9e-7, 1.6e-7, 1.7e-7, 5.4e-7 and 0.75e-7, 0.8e-7, 1.0e-7, 1.7e-7.

Three parts hold a magnitude of 2^-110 (7.7e-34) to 3.39e38, and zero. Rows are multiplied by 2^20 on the way and weights divided by it
(``SCALE``): all normal numbers below 1.6e32 = 2^107 are held, and weights from 8.1e-28 on (sums of X times weights beyond 3.4e38
are infinite, where the fp32 kernels' products with a small Y come first). Forward and dX watch
the largest operand; rows with a larger one or an infinity, and all rows where a weight is not held, are formed once more by fp32
instructions (``emit_redo``). Where dW's sums are not finite, a wave forms them once more (``emit_redo_dw``). That costs, on the
problem above, forward / backward, without / with, us: 500 rows 12.6 / 13.7 and 45.6 / 49.1, 4 500 19.7 / 21.1 and 64 / 70, 100 003
155 / 159 and 505 / 502; such rows in every tile take 8 times as long as with the fp32 kernels (2 364 / 311, 6 454 / 772).

Where the fp32 kernels (``uvw_mfma.py``) contract with the coupling coefficients first and multiply the result, forward and dX
multiply first: the matrix cores form W^T x (or W dZ) component by component, the lanes contract what comes out. The
operand that is split, written to LDS and read by every wave is then a row as it lies in memory - 9 components per channel
at l <= 2, where the contraction of 11 paths has 35 - so that a tile's operands are prepared once, and X and dZ are read
once per kernel. The exception are paths whose other side has a single component, l x l -> 0 in the forward and 0 x l -> l in
dW (there the output gradient's side): contracted on the way to LDS they are one product, not 2 l + 1 (``folds``; 35 -> 29
products each; forward 182 -> 175 us, dW 332 -> 318). dX has no such path, since dY needs every component of W dZ. The most
frequent coefficient of a path is a factor of its weights (``Sub.unit``).

* Forward, dX: a block of 4 waves owns 16 rows at a time; wave w result channels 16 w .. 16 w + 15, with the weights
  of all sub-paths of the kernel in registers. The threads split the next tile's rows into LDS (two copies) while
  this one's components are multiplied. dY falls out of dX's products: summed over the lanes of a row in registers, over
  the waves through LDS in wave order. As few kernels as the registers allow (``SplitEmitter.plan``).
* dW: wave w owns input channels 16 w .. 16 w + 15, contracts X and Y for them in registers, eight rows a lane, in the
  layout of the A operand; the output gradient's operands are split once per block. Products of 32 rows are summed from zero
  and then added to the running sums. The bf16 instruction cuts off what it aligns,
  always downwards, and running sums of 12 steps drift by that: every second block works on negated values,
  which the addition turns back (dW above: 1.5e-6 on the running sums directly, 5.4e-7 from zero, 2.3e-7
  with the signs, 1.7e-7 with the folds). Y lies in LDS times the coefficients it is met with, as zeros past the batch.

What bounds them (MI355X, the problem above, 100 003 rows): the registers of a SIMD hold one wave of these kernels, and
a wave issues an instruction in 2.1 ns, one that needs the result before it in 3.6, a matrix instruction takes 8. Counters of
the forward: of 100 wave cycles 54 issue, 31 wait to issue, 15 wait for memory or LDS; matrix cores busy 42. Run back to back the
kernels are also bound by power: random operands lower the clock (2.1 GHz, 2.4 on zeros), fewer matrix instructions raise it.
So the order of the instructions is written out (``interleave``): vector, LDS and memory instructions go between the matrix
instructions that hide them, and what takes several is cut in steps (a split of eight values as one piece: 714 us for a pass through
forward and backward, in steps 695); left to the compiler they clump, and registers spill. The pass: fp32 kernels
1 062 us, these 719 with 35 products each and without the steps, 633 with both, 647 with what keeps operands in range.
"""

from __future__ import annotations

from collections import Counter
from dataclasses import dataclass
from functools import cached_property
from typing import Dict, List, Optional

import numpy as np

from .common import Src
from .lower import Lowered, Path, float_literal

WAVES = 4
# (part of A, part of B), smallest products first
TERMS = ((2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0))
LDS_BUDGET = 160 * 1024 - 1024
# Estimated registers up to which result blocks share a kernel: what mostly compiles without scratch memory (512 registers
# a lane; the estimates are seldom more than 30 below what the compiler takes, and above it for dW). Where one does not,
# uvw_mfma.tp_module finds out.
MAX_REGS, MAX_REGS_DW = 500, 430
# Registers of weight operands kept as accumulation registers, of 256; the others hold results (64x{0e,1o,2e}, forward: with 168 to
# 204 no scratch memory, 8 to 24 bytes a lane below and 72 above).
PARKED = 180
# Two waves per SIMD (256 registers): up to this estimate. 64x0e+16x1o (x) 0e+1o -> the same, 150 000 rows, one wave / two:
# forward 52 / 40 us, dX 71 / 54, dW 69 / 61.
TWO_WAVES = 300
# Operands of weights on their way from memory while one is split (64x{0e,1o,2e}, forward and backward, one after the other /
# with these and the first tile's rows ahead: 4 500 rows 91 / 86 us, 20 000 173 / 167, 131 072 853 / 845).
WEIGHTS_AHEAD = 6
# Components of Y that dW reads from LDS ahead of their use.
AHEAD = 4
# Operands are multiplied by this before they are split, so that three parts hold every normal number; in forward and dX the
# weights are divided by it, in dW the sums by its square. (dW: with Y's coefficients, in place of a copy of X in folded
# sub-paths, and dZ.)
SCALE = 2.0 ** 20


def c16(n: int) -> int:
    return (n + 15) // 16


def c32(n: int) -> int:
    return (n + 31) // 32


@dataclass
class Sub:
    """One channel v of a path's second operand: a mul1 x mul3 weight matrix."""
    index: int
    p: Path
    v: int

    @property
    def key(self):
        return ("fold", self.index)

    @cached_property
    def unit(self) -> float:
        """The magnitude that most coefficients of the path have (one coefficient in seven of the eleven paths up to
        l = 2): a factor of the weights, before they are split, or of their gradient, after the sums."""
        sizes = Counter(f"{abs(c):.12g}" for *_, c in self.p.nnz)
        most = max(sizes.values())
        # (a path of weight zero keeps its coefficients, all of them zero)
        return next(abs(c) for *_, c in self.p.nnz if sizes[f"{abs(c):.12g}"] == most) or 1.0

    def ratio(self, c: float) -> float:
        return float(f"{abs(c) / self.unit:.12g}")


DEVICE = r"""
typedef float oeq_f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float oeq_f2u __attribute__((ext_vector_type(2), aligned(4)));
// a and b as sums of three bf16 numbers each (round to nearest; the remainders are exact in fp32); q<i> holds the i-th
// parts, a's in the low half. A remainder is one dot product with (-1, 0) or (0, -1).
OEQ_DEV void oeq_split3(float a, float b, unsigned& q0, unsigned& q1, unsigned& q2)
{
    unsigned l = 0x0000bf80u, h = 0xbf800000u;
    asm("" : "+s"(l), "+s"(h));
    const oeq_bf2 lo = __builtin_bit_cast(oeq_bf2, l), hi = __builtin_bit_cast(oeq_bf2, h);
    const oeq_bf2 p0 = __builtin_convertvector((oeq_f2{a, b}), oeq_bf2);
    a = __builtin_amdgcn_fdot2_f32_bf16(p0, lo, a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(p0, hi, b, false);
    const oeq_bf2 p1 = __builtin_convertvector((oeq_f2{a, b}), oeq_bf2);
    a = __builtin_amdgcn_fdot2_f32_bf16(p1, lo, a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(p1, hi, b, false);
    const oeq_bf2 p2 = __builtin_convertvector((oeq_f2{a, b}), oeq_bf2);
    q0 = __builtin_bit_cast(unsigned, p0), q1 = __builtin_bit_cast(unsigned, p1), q2 = __builtin_bit_cast(unsigned, p2);
}
// The same in steps, for a caller that puts other instructions between them: q = the next parts of a and b, which keep the
// remainders (a dependent instruction is issued after 3.6 ns, one that is not after 2.1).
OEQ_DEV void oeq_split_part(float& a, float& b, unsigned& q)
{
    unsigned l = 0x0000bf80u, h = 0xbf800000u;
    asm("" : "+s"(l), "+s"(h));
    const oeq_bf2 p = __builtin_convertvector((oeq_f2{a, b}), oeq_bf2);
    a = __builtin_amdgcn_fdot2_f32_bf16(p, __builtin_bit_cast(oeq_bf2, l), a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(p, __builtin_bit_cast(oeq_bf2, h), b, false);
    q = __builtin_bit_cast(unsigned, p);
}
OEQ_DEV void oeq_split_last(float a, float b, unsigned& q)
{
    q = __builtin_bit_cast(unsigned, __builtin_convertvector((oeq_f2{a, b}), oeq_bf2));
}
// The largest magnitude of those seen (NaN does not count; from the compiler, with an instruction to quiet each operand), and whether
// any lane of the wave has met one that three parts do not hold.
OEQ_DEV float oeq_top(float top, float a, float b)
{
    float r;
    asm("v_max3_f32 %0, %1, abs(%2), abs(%3)" : "=v"(r) : "v"(top), "v"(a), "v"(b));
    return r;
}
OEQ_DEV bool oeq_too_large(float top) { return __builtin_amdgcn_ballot_w64(top >= 3.39e38f) != 0; }
// Of eight values: the largest magnitude, and twice the bits of the smallest, zeros aside, less one.
OEQ_DEV void oeq_extent(const float (&r)[8], float& top, unsigned& least)
{
    unsigned v[8];
    #pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (__builtin_bit_cast(unsigned, r[e]) << 1) - 1u;
    const unsigned a = min(min(v[0], v[1]), v[2]), b = min(min(v[3], v[4]), v[5]);
    least = min(min(min(v[6], v[7]), a), b);
    top = oeq_top(top, oeq_top(0.0f, r[0], r[1]), oeq_top(oeq_top(oeq_top(0.0f, r[2], r[3]), r[4], r[5]), r[6], r[7]));
}
// Component I of eight channels (or rows) as three bf16 operands: r[e * D + I], e = 0..7.
template <int D, int I> OEQ_DEV void oeq_split8(const float (&r)[8 * D], oeq_bf8 (&f)[3])
{
    unsigned q[3][4];
    #pragma unroll
    for (int m = 0; m < 4; ++m) oeq_split3(r[2 * m * D + I], r[(2 * m + 1) * D + I], q[0][m], q[1][m], q[2][m]);
    #pragma unroll
    for (int c = 0; c < 3; ++c) f[c] = __builtin_bit_cast(oeq_bf8, oeq_u4{q[c][0], q[c][1], q[c][2], q[c][3]});
}
// The same four registers as accumulation registers.
OEQ_DEV oeq_bf8 oeq_park(oeq_bf8 v)
{
    const oeq_u4 q = __builtin_bit_cast(oeq_u4, v);
    oeq_u4 r;
    #pragma unroll
    for (int m = 0; m < 4; ++m) { unsigned t; asm("v_accvgpr_write_b32 %0, %1" : "=a"(t) : "v"(q[m])); r[m] = t; }
    return __builtin_bit_cast(oeq_bf8, r);
}
// r[n] = lo[n] + (lo[n] of the mirrored lane) in the lanes of the lower half, hi[n] + (hi[n] of it) in the others; r may be lo.
// (Two wait states between the instruction that writes an operand and the one that reads it from other lanes, which the
// compiler does not see.)
#define OEQ_FOLD_LANES(r0, r1, r2, lo0, lo1, lo2, hi0, hi1, hi2, MIRROR, UPPER) \
    { \
        float f0 = lo0, f1 = lo1, f2 = lo2; \
        asm("s_nop 1\n\tv_add_f32_dpp %0, %0, %0 " MIRROR " row_mask:0xf bank_mask:0xf\n\t" \
            "v_add_f32_dpp %1, %1, %1 " MIRROR " row_mask:0xf bank_mask:0xf\n\t" \
            "v_add_f32_dpp %2, %2, %2 " MIRROR " row_mask:0xf bank_mask:0xf\n\t" \
            "v_add_f32_dpp %0, %3, %3 " MIRROR " row_mask:0xf bank_mask:" UPPER "\n\t" \
            "v_add_f32_dpp %1, %4, %4 " MIRROR " row_mask:0xf bank_mask:" UPPER "\n\t" \
            "v_add_f32_dpp %2, %5, %5 " MIRROR " row_mask:0xf bank_mask:" UPPER \
            : "+v"(f0), "+v"(f1), "+v"(f2) : "v"(hi0), "v"(hi1), "v"(hi2)); \
        r0 = f0, r1 = f1, r2 = f2; \
    }
OEQ_DEV void oeq_block_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// One value of four rows, at these byte offsets.
OEQ_DEV v4t oeq_rows4(const float* p, const unsigned (&at)[4]) { return v4t{*oeq_at(p, at[0]), *oeq_at(p, at[1]), *oeq_at(p, at[2]), *oeq_at(p, at[3])}; }
// oeq_block_sync with the block's accesses to memory as well.
OEQ_DEV void oeq_block_sync_all()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
"""


class SplitEmitter:
    def __init__(self, low: Lowered, waves: Optional[Dict[str, int]] = None):
        """``waves``: waves per SIMD of a role ('forward', or 'dx' for the backward pass) where that is not left to the rule."""
        self.low = low
        self.given = {kind: n for kind, n in (waves or {}).items() if n}
        self.subs: List[Sub] = []
        for p in low.paths:
            for v in range(low.in2[p.i2].mul):
                self.subs.append(Sub(len(self.subs), p, v))

    # ------------------------------------------------------------------ shared
    def yat(self, sub: Sub, j: int) -> int:
        b2 = self.low.in2[sub.p.i2]
        return b2.off + sub.v * b2.d + j

    def wpos(self, sub: Sub, u: str, w: str) -> str:
        V, wtot = self.low.in2[sub.p.i2].mul, self.low.out[sub.p.io].mul
        return f"{sub.p.woff + sub.v * wtot} + ({u}) * {V * wtot} + ({w})"

    def lit(self, v):
        return float_literal(v, "float")

    def sides(self, kind: str):
        """(blocks contracted over, blocks of the result tiles, their index in a sub-path)"""
        low = self.low
        if kind == "forward":
            return low.in1, low.out, (lambda q: q.p.i1), (lambda q: q.p.io)
        return low.out, low.in1, (lambda q: q.p.io), (lambda q: q.p.i1)

    def cut(self, blocks, block_of, fits):
        """Sub-paths by kernel: consecutive blocks that fit one together."""
        kernels = []
        for t in range(len(blocks)):
            mine = [q for q in self.subs if block_of(q) == t]
            if mine and kernels and fits(kernels[-1] + mine):
                kernels[-1] += mine
            elif mine:
                kernels.append(mine)
        return kernels

    def plan(self, kind: str):
        A, T, ia, it = self.sides(kind)
        return self.cut(T, it, lambda subs: self.registers(kind, subs) <= MAX_REGS and self.lds(kind, subs) <= LDS_BUDGET)

    def plan_dw(self):
        return self.cut(self.low.out, lambda q: q.p.io,
                        lambda subs: self.registers_dw(subs) <= MAX_REGS_DW and self.lds_dw(subs) <= LDS_BUDGET)

    def registers(self, kind: str, subs) -> int:
        """Estimate for a forward or dX kernel: weights, sums, Y, operands on their way from LDS, results, rows on
        their way from memory; for dX also X (this tile's and the next one's) and dY."""
        A, T, ia, it = self.sides(kind)
        S = lambda q: c32(A[ia(q)].mul)
        used_a, used_t = {ia(q) for q in subs}, {it(q) for q in subs}
        tacc = 4 * sum(T[t].d for t in used_t)
        most = max(sum(1 for q in subs if ia(q) == a) for a in used_a)
        regs = 12 * sum(S(q) for q in subs) + tacc + 4 * self.low.L2 + 24 * max(S(q) for q in subs) + 8 * most + \
            sum(2 * A[a].d * c32(A[a].mul) for a in used_a) + 32
        if kind != "forward":
            regs += 2 * tacc + 4 * self.low.L2
        return regs

    def lds(self, kind: str, subs) -> int:
        A, T, ia, it = self.sides(kind)
        frags = sum(A[a].d * c32(A[a].mul) for a in {ia(q) for q in subs})
        return 2 * (3072 * frags + 64 * self.low.L2 * (1 if kind == "forward" else 5))

    def folds(self, kind: str, subs):
        """Sub-paths of a forward kernel whose result has one component and whose operand has more (l x l -> 0): X and Y
        are contracted by the threads that split the rows, and one component is multiplied, not 2 l + 1. As many as the LDS
        has room for, and two more steps remain."""
        A, T, ia, it = self.sides(kind)
        out, room = [], LDS_BUDGET // self.waves(kind) - self.lds(kind, subs)
        for q in sorted(subs, key=lambda q: -A[ia(q)].d):
            if kind == "forward" and T[it(q)].d == 1 and A[ia(q)].d > 1:
                room -= 2 * 3072 * c32(A[ia(q)].mul)
                raw = {ia(p) for p in subs if p not in out and p is not q}
                if room >= 0 and sum(A[a].d for a in raw) >= 2:
                    out.append(q)
        return out

    def share(self, kind: str) -> float:
        """Of the multiplies of a pass, those with weights that are not padding (a wave's 16 result channels times four,
        32 contracted channels at a time)."""
        A, T, ia, it = self.sides(kind)
        return sum(A[ia(q)].d * A[ia(q)].mul * T[it(q)].mul for q in self.subs) / \
            sum(A[ia(q)].d * 32 * c32(A[ia(q)].mul) * 64 for q in self.subs)

    def waves(self, kind: str) -> int:
        """Waves per SIMD of the kernels of a role: two where the largest of them comes under 256 registers and half
        the LDS."""
        kinds = [kind] if kind == "forward" else ["dx", "dw"]
        if kinds[0] in self.given:
            return self.given[kinds[0]]
        need = [(self.registers_dw(s), self.lds_dw(s)) if k == "dw" else (self.registers(k, s), self.lds(k, s))
                for k in kinds for s in (self.plan_dw() if k == "dw" else self.plan(k))]
        return 2 if all(r <= TWO_WAVES and 2 * m <= LDS_BUDGET for r, m in need) else 1

    def supported(self, kind: str) -> bool:
        """Whether these kernels are the ones to use for a role ('forward', or 'dx' for the whole backward pass).

        Not for blocks of more than 64 channels, whose weights a wave's registers do not hold, nor where a tile would be mostly
        padding. Two waves per SIMD: the share of real multiplies 0.28 (24 channels, l <= 1, 60 000 rows) forward 26 -> 15 us,
        backward 67 -> 49; 0.1 (33 and 17 -> 15 and 7 channels) 23 -> 16 and 54 -> 46; 0.03 (8 channels) 15 -> 14 and
        42 -> 44. One wave: 0.5 (32 channels, l <= 2) 95 -> 59 and 233 -> 161; 0.38 / 0.30 (40, 30 -> 50, 20, 10 channels) 43 ->
        30 and 95 -> 99; 0.12 (16 channels, l <= 2) 57 -> 56 and 133 -> 158."""
        low = self.low
        if low.elem_size != 4 or any(low.in1[q.p.i1].mul > 64 or low.out[q.p.io].mul > 64 for q in self.subs):
            return False
        A, T, ia, it = self.sides(kind)
        for subs in self.plan(kind):
            # (two components at least: the pipeline over them has a step that writes LDS and one that reads it)
            if self.registers(kind, subs) > MAX_REGS or self.lds(kind, subs) > LDS_BUDGET or \
                    sum(A[a].d for a in {ia(q) for q in subs}) < 2:
                return False
        # (scalars alone: one component of dX for many of dZ, 64x0e -> 64x0e+32x1o+16x2e backward 78 -> 81 us)
        if sum(low.in1[a].d for a in {q.p.i1 for q in self.subs}) < 2:
            return False
        if kind != "forward" and any(self.registers_dw(s) > MAX_REGS_DW or self.lds_dw(s) > LDS_BUDGET or
                                     len(self.stages_dw(s)) < 2 for s in self.plan_dw()):
            return False
        least = 0.08 if self.waves(kind) == 2 else 0.35 if kind == "forward" else 0.45
        return self.share(kind) >= least

    def open_kernel(self, s: Src, name: str, sig: str, waves: int):
        s.open(f'extern "C" __global__ __launch_bounds__({64 * WAVES}) '
               f'__attribute__((amdgpu_waves_per_eu({waves}, {waves}))) void {name}{sig}')
        s("const int lane = oeq_lane(), wave = oeq_wave(), l16 = lane & 15, lq = lane >> 4;")
        s("(void)lane; (void)wave; (void)l16; (void)lq;")

    # ------------------------------------------------------------- forward and dX
    def weights(self, s: Src, kind: str, subs, park: int = 0):
        """B operands of the sub-paths in registers: the lane's result channel 16 wave + lane % 16 and, of every 32
        contracted channels, the eight from 8 (lane / 16) on; zeros past either block. The first ``park`` registers of them go
        to accumulation registers. Memory is WEIGHTS_AHEAD operands ahead of the splits."""
        A, T, ia, it = self.sides(kind)
        loads, splits = [], []
        for q in subs:
            a, t, S = A[ia(q)], T[it(q)], c32(A[ia(q)].mul)
            ld = self.low.in2[q.p.i2].mul * self.low.out[q.p.io].mul
            cu, ct = (ld, 1) if kind == "forward" else (1, ld)   # distance of two contracted / two result channels
            base = q.p.woff + q.v * self.low.out[q.p.io].mul
            s(f"oeq_bf8 w{q.index}[{S}][3];")
            for st in range(S):
                r = f"r{q.index}_{st}"
                get, use = [f"float {r}[8];"], [f"oeq_extent({r}, top, least);"]
                for e in range(8):
                    full = 32 * st + 32 <= a.mul
                    u = f"{32 * st + e} + 8 * lq"
                    get.append(f"{r}[{e}] = W[{base} + ({u if full else f'min({u}, {a.mul - 1})'}) * {cu} + min(16 * wave + l16, {t.mul - 1}) * {ct}];")
                    conds = ([] if t.mul >= 64 else [f"16 * wave + l16 < {t.mul}"]) + ([] if full else [f"{u} < {a.mul}"])
                    val = f"({self.lit(q.unit / SCALE)} * sign) * {r}[{e}]"
                    use.append(f"{r}[{e}] = " + (f"oeq_sel({' && '.join(conds)}, {val});" if conds else f"{val};"))
                use.append(f"oeq_split8<1, 0>({r}, w{q.index}[{st}]);")
                # (a weight that is 2^-110 or more when it is split is held by three parts)
                small = 2 * int(np.float32(2.0 ** -110 * SCALE / q.unit).view(np.uint32))
                use.insert(1, f"wout |= __builtin_amdgcn_ballot_w64(least < {small}u) != 0;")
                if park > 0:
                    use.append(f"for (int c = 0; c < 3; ++c) w{q.index}[{st}][c] = oeq_park(w{q.index}[{st}][c]);")
                park -= 12
                loads.append(get)
                splits.append(use)
        for n in range(-WEIGHTS_AHEAD, len(loads)):
            for line in (loads[n + WEIGHTS_AHEAD] if n + WEIGHTS_AHEAD < len(loads) else []) + (splits[n] if n >= 0 else []):
                s(line)
            if n >= 0:
                s("__builtin_amdgcn_sched_barrier(0);")

    def rows_request(self, kind: str, a: int, st: int):
        """ra<a>_<st>: two neighbouring channels of one of the tile's 16 rows, for the thread to split (in scope:
        ``rows``, the tile's first row, and ``own``, the byte offset of the thread's row from there)."""
        b = self.sides(kind)[0][a]
        if b.mul % 2 == 0:
            ch = f"2 * (tid & 15) * {b.d}"
            if 32 * st + 32 > b.mul:
                ch = f"min(2 * (tid & 15), {b.mul - 2 - 32 * st}) * {b.d}"
            out = f"{{ const float* ap = oeq_at(rows + {b.off + 32 * st * b.d}, own + 4u * (unsigned)({ch})); "
            for m in range(b.d):
                out += f"{{ const oeq_f2u v = *(const oeq_f2u*)(ap + {2 * m}); ra{a}_{st}[{2 * m}] = v[0]; ra{a}_{st}[{2 * m + 1}] = v[1]; }} "
            return [(3, out + "}")]
        out = []
        for e in range(2):
            t = f"{{ const float* ap = oeq_at(rows + {b.off}, own + 4u * (unsigned)(min({32 * st + e} + 2 * (tid & 15), {b.mul - 1}) * {b.d})); "
            out.append((3, t + " ".join(f"ra{a}_{st}[{e * b.d + i}] = ap[{i}];" for i in range(b.d)) + " }"))
        return out

    def rows_write(self, kind: str, a: int, st: int, at: int, buf: str):
        """ra<a>_<st> as A operands: (part, lane, pair) at 16 bytes a lane. The lanes of a quarter are turned by four
        times its number, so that a wave's stores fall into 64 banks."""
        b = self.sides(kind)[0][a]
        out = []
        for i in range(b.d):
            v = [f"ra{a}_{st}[{e * b.d + i}]" for e in range(2)]
            if 32 * st + 32 > b.mul:
                # channels past the block meet zero weights: zeros here too, not other channels' values
                v = [f"oeq_sel({32 * st + e} + 2 * (tid & 15) < {b.mul}, {v[e]})" for e in range(2)]
            out += self.split_pair(f"{a}_{st}_{i}", v, [f"{buf}[{at + 768 * i + 256 * c} + put]" for c in range(3)])
        return out

    def fold_write(self, q: Sub, st: int, at: int, buf: str):
        """The one component of a folded sub-path from ra<a>_<st> and yt<q>, as ``rows_write`` has it."""
        b, n = self.low.in1[q.p.i1], q.index
        out = []
        for e in range(2):
            out += [(1, line) for line in self.fold_terms(q, f"tf{n}_{st}_{e}", lambda i: f"ra{q.p.i1}_{st}[{e * b.d + i}]")]
        v = [f"tf{n}_{st}_{e}" for e in range(2)]
        if 32 * st + 32 > b.mul:
            v = [f"oeq_sel({32 * st + e} + 2 * (tid & 15) < {b.mul}, {v[e]})" for e in range(2)]
        return out + self.split_pair(f"f{n}_{st}", v, [f"{buf}[{at + 256 * c} + put]" for c in range(3)])

    def fold_terms(self, q: Sub, name: str, x):
        """The sum of a folded sub-path's terms; ``x(i)``: component i of the channel, yt<q>: Y of its row."""
        out = []
        for m, (i, j, _, c) in enumerate(q.p.nnz):
            r = q.ratio(c)
            y = f"yt{q.index}[{j}]" if r == 1.0 else f"({self.lit(r)} * yt{q.index}[{j}])"
            op = ("= -" if c < 0 else "= ") if m == 0 else "-= " if c < 0 else "+= "
            out.append(f"{'float ' if m == 0 else ''}{name} {op}{y} * {x(i)};")
        return out

    @staticmethod
    def split_pair(name: str, v, to):
        """Two values, times SCALE, to three places, in steps."""
        q, large = [f"q{name}_{c}" for c in range(3)], float_literal(SCALE, "float")
        return [(2, f"float s{name}_0 = {large} * {v[0]}, s{name}_1 = {large} * {v[1]}; unsigned {', '.join(q)};"),
                (1, f"top = oeq_top(top, s{name}_0, s{name}_1);")] + \
            [(3, f"oeq_split_part(s{name}_0, s{name}_1, {q[c]});") for c in range(2)] + \
            [(1, f"oeq_split_last(s{name}_0, s{name}_1, {q[2]});")] + [(1, f"{to[c]} = {q[c]};") for c in range(3)]

    @staticmethod
    def split_tasks(v: str, q: str):
        """Eight values as the parts ``q[part][pair]``, pair by pair and part by part; the values are used up."""
        out = [(3, f"oeq_split_part({v}[{2 * m}], {v}[{2 * m + 1}], {q}[{c}][{m}]);") for c in range(2) for m in range(4)]
        return out + [(1, f"oeq_split_last({v}[{2 * m}], {v}[{2 * m + 1}], {q}[2][{m}]);") for m in range(4)]

    @staticmethod
    def put(s: Src, tasks):
        for _, line in tasks:
            s(line)

    @staticmethod
    def spread_reads(reads, tasks):
        """``reads`` from LDS at equal distances among the first two thirds of ``tasks``: the four waves of a block come
        to them together."""
        out, total = [], sum(w for w, _ in tasks)
        done, at = 0, 0
        for t in tasks:
            while at < len(reads) and done * len(reads) * 3 >= 2 * total * at:
                out.append(reads[at])
                at += 1
            out.append(t)
            done += t[0]
        return out + reads[at:]

    @staticmethod
    def interleave(s: Src, lead, tasks):
        """The matrix instructions ``lead`` with ``tasks`` (weight, line) shared out between them, in this order:
        the wave issues in order, and what is issued while the matrix cores are at work costs nothing."""
        total, done, at = sum(w for w, _ in tasks) or 1, 0, 0
        for n, m in enumerate(lead):
            s(m)
            some = False
            while at < len(tasks) and (done + tasks[at][0] / 2) * len(lead) <= total * (n + 1):
                s(tasks[at][1])
                done += tasks[at][0]
                at += 1
                some = True
            if some:
                s("__builtin_amdgcn_sched_barrier(0);")
        for w, line in tasks[at:]:
            s(line)
        s("__builtin_amdgcn_sched_barrier(0);")

    def emit_pass(self, s: Src, kind: str, name: str, sig: str):
        names = []
        for n, subs in enumerate(self.plan(kind)):
            names.append(name if n == 0 else f"{name}_{n}")
            self.emit_kernel(s, kind, names[-1], sig, subs, n)
        return names

    def emit_kernel(self, s: Src, kind: str, name: str, sig: str, subs, number: int):
        low = self.low
        A, T, ia, it = self.sides(kind)
        L2, fwd = low.L2, kind == "forward"
        dst, LT = ("L3_out", low.L3) if fwd else ("L1_grad", low.L1)
        used_a, used_t = sorted({ia(q) for q in subs}), sorted({it(q) for q in subs})
        folds = self.folds(kind, subs)
        raw_a = sorted({ia(q) for q in subs if q not in folds})   # blocks whose components are multiplied
        at, total = {}, 0
        for a in raw_a:
            for st in range(c32(A[a].mul)):
                at[(a, st)] = total
                total += 768 * A[a].d
        for q in folds:
            for st in range(c32(A[ia(q)].mul)):
                at[(q.key, st)] = total
                total += 768
        self.open_kernel(s, name, sig, self.waves(kind))
        s("const int tid = (int)threadIdx.x;")
        s(f"__shared__ __attribute__((aligned(16))) unsigned s_a[2][{total}];")
        s(f"__shared__ __attribute__((aligned(16))) float s_y[2][{L2}][16];")
        if not fwd:
            s(f"__shared__ float s_dy[2][{WAVES}][{16 * L2}];")
        s("const i64 ntiles = (num_batch + 15) / 16;")
        # where a thread's pair of channels goes within an operand, and where a lane's operand lies
        s("const int put = 4 * (((tid & 15) >> 2) * 16 + (((tid >> 4) + 4 * ((tid & 15) >> 2)) & 15)) + (tid & 3);")
        s("const int get = 4 * (lq * 16 + ((l16 + 4 * lq) & 15));")
        park = PARKED if self.waves(kind) == 1 else 0
        for a in used_a:
            for st in range(c32(A[a].mul)):
                s(f"float ra{a}_{st}[{2 * A[a].d}];")
        ny = (16 * L2 + 255) // 256
        s(f"float ry[{ny}];")

        src, LA = ("L1_in", low.L1) if fwd else ("L3_grad", low.L3)

        def where(tile, const="const "):
            """Where the rows of ``tile`` lie; past the batch: its last row."""
            s(f"{const}first = min(({tile}) * 16, num_batch - 1);")
            s(f"{'const int ' if const else ''}end = (int)min((i64)15, num_batch - 1 - first);")

        def request_y():
            for n in range(ny):
                v = f"min(tid + {256 * n}, {16 * L2 - 1})"
                s(f"ry[{n}] = *oeq_at(L2_in + first * {L2}, 4u * (unsigned)min({v}, end * {L2} + {v} % {L2}));")

        # (threads past the tile repeat its last value: a store under a lane's condition makes the compiler wait for more
        # than it has to afterwards)
        def write_y(buf):
            for n in range(ny):
                v = f"min(tid + {256 * n}, {16 * L2 - 1})"
                s(f"s_y[{buf}][{v} % {L2}][{v} / {L2}] = sign * ry[{n}];")

        # byte offsets of the lane's four rows in a tile of X or the results; past the batch: its last row
        s(f"unsigned lr[4];")
        s(f"for (int r = 0; r < 4; ++r) lr[r] = {4 * LT}u * (4 * lq + r);")
        row_at = lambda r, end: f"min(lr[{r}], {4 * LT}u * (unsigned){end})"

        def request_x(t):
            b = T[t]
            return [(4, f"{{ const float* xp = oeq_at(L1_in + xfirst * {low.L1} + {b.off}, {row_at(r, 'xend')} + ch{t}); "
                        + " ".join(f"xn{t}[{i}][{r}] = xp[{i}];" for i in range(b.d)) + " }") for r in range(4)]

        for t in used_t:
            s(f"const unsigned ch{t} = {4 * T[t].d}u * min(16 * wave + l16, {T[t].mul - 1});")
            if not fwd:
                s(f"v4t xn{t}[{T[t].d}];")
        for q in folds:
            s(f"float yt{q.index}[{low.in2[q.p.i2].d}];  // Y of the thread's row")

        def y_request(q):
            b2 = low.in2[q.p.i2]
            return [(3, f"{{ const float* yp = oeq_at(L2_in + first * {L2} + {self.yat(q, 0)}, 4u * (unsigned)(min(tid >> 4, end) * {L2})); "
                     + " ".join(f"yt{q.index}[{j}] = yp[{j}];" for j in range(b2.d)) + " }")]

        def request(a, st):
            """The rows of a unit, and the Y that its folds will meet once the last of them is written."""
            out = self.rows_request(kind, a, st)
            if st == c32(A[a].mul) - 1:
                for q in folds:
                    out += y_request(q) if ia(q) == a else []
            return out

        def write(a, st, buf):
            out = self.rows_write(kind, a, st, at[(a, st)], buf) if a in raw_a else []
            for q in folds:
                if ia(q) == a:
                    out += self.fold_write(q, st, at[(q.key, st)], buf)
            return out

        # The matrix instruction cuts off downwards (see dW): weights are negated in every second block, and what comes of them is
        # turned back with Y or, where no Y follows, by itself. Mean error of 30 011 rows of 64x0e+16x1o, Y of l = 0 one, over
        # the results' size, without / with: Z -5.7e-9 / 0.04e-9, dX -3.8e-9 / -0.02e-9 (errors of elements 6e-8).
        s("const float sign = (blockIdx.x & 1) ? -1.0f : 1.0f;")
        # Tiles with operands that three parts do not hold: a bit each, by the tile's number among the block's modulo 32.
        # top: the largest operand of the next tile that the thread has split; next: that tile's bit.
        s("unsigned redo = 0, next = 2, least;")
        s("float top = 0.0f;")
        s("bool wout = false;  // a weight is not held")
        units = [(a, st) for a in used_a for st in range(c32(A[a].mul))]
        where("(i64)blockIdx.x", "const i64 ")
        s(f"const float* rows = {src} + first * {LA};")
        s(f"const unsigned own = (unsigned)min(tid >> 4, end) * {4 * LA}u;")
        for a, st in units:
            self.put(s, request(a, st))
        request_y()
        if not fwd:
            s("const i64 xfirst = first;")
            s("const int xend = end;")
            for t in used_t:
                self.put(s, request_x(t))
        self.weights(s, kind, subs, park)   # (the first tile's rows are on their way meanwhile)
        s("const unsigned wrows = wout || oeq_too_large(top) ? 0xffffu : 0u;")
        s("top = 0.0f;")
        for a, st in units:
            self.put(s, write(a, st, "s_a[0]"))
        write_y("0")
        s("redo = wrows ? ~0u : oeq_too_large(top) ? 1u : 0u;")
        s("top = 0.0f;")
        s.open("")
        where("((i64)blockIdx.x + gridDim.x)", "const i64 ")
        s(f"const float* rows = {src} + first * {LA};")
        s(f"const unsigned own = (unsigned)min(tid >> 4, end) * {4 * LA}u;")
        for a, st in units:
            self.put(s, request(a, st))
        request_y()
        s.close()
        # Software pipeline over the components of the contracted rows, across tiles: while the matrix cores work on one,
        # the lanes contract the results of the one before with the coupling coefficients, and its successor's operands
        # are on their way from LDS. The last component of a tile is contracted, and its rows are stored, beside the first
        # matrix instructions of the next.
        steps = [(a, i) for a in sorted(raw_a, key=lambda a: -A[a].d) for i in range(A[a].d)] + [(q.key, 0) for q in folds]
        mine = {a: [q for q in subs if ia(q) == a and q not in folds] for a in raw_a} | {q.key: [q] for q in folds}
        slots = {a: c32(A[a].mul) for a in raw_a} | {q.key: c32(A[ia(q)].mul) for q in folds}
        N = len(steps)

        def fetch(n, buf="cur"):
            a, i = steps[n]
            return [(1, f"f{n}[{st}][{c}] = __builtin_bit_cast(oeq_bf8, *(const oeq_u4*)(s_a[{buf}] + "
                        f"{at[(a, st)] + 768 * i + 256 * c} + get));") for st in range(slots[a]) for c in range(3)]

        begun = {}  # sum -> the term that starts it, in the order of the steps

        def add(sum_, term, c=1.0):
            if begun.setdefault(sum_, term) == term:
                return (4, f"{sum_} = {'-' if c < 0 else ''}{term};")
            return (4, f"{sum_} {'-=' if c < 0 else '+='} {term};")

        def contract(n):
            a, i = steps[n]
            out = []
            for q in mine[a]:
                if q in folds:
                    out.append(add(f"acc{it(q)}[0]", f"sign * P{n}_{q.index}"))
                    continue
                names = {self.lit(1.0): f"P{n}_{q.index}"}
                for (i1, j, k, c) in q.p.nnz:
                    if (i1 if fwd else k) != i:
                        continue
                    key = self.lit(q.ratio(c))
                    if key not in names:
                        names[key] = f"m{n}_{q.index}_{len(names)}"
                        out.append((4, f"const v4t {names[key]} = {key} * P{n}_{q.index};"))
                    yj = self.yat(q, j)
                    out.append(add(f"acc{it(q)}[{k if fwd else i1}]", f"y[{yj}] * {names[key]}", c))
                    if not fwd:
                        out.append(add(f"dy[{yj}]", f"x{it(q)}[{i1}] * {names[key]}", c))
            return out

        for n in range(N):
            contract(n)

        def store(row0, end):
            """Rows past the batch repeat its last one, in what was read and so in the results, and write it again: no
            store hangs on a lane's row."""
            out = []
            for t in used_t:
                for r in range(4):
                    text = f"float* op = oeq_at({dst} + {row0} * {LT} + {T[t].off}, {row_at(r, end)} + ch{t}); " + \
                        " ".join(f"__builtin_nontemporal_store((float)acc{t}[{k}][{r}], op + {k});" for k in range(T[t].d))
                    out.append((6, (f"if (16 * wave + l16 < {T[t].mul}) " if T[t].mul < 64 else "") + "{ " + text + " }"))
            return out

        def lead(n):
            a, i = steps[n]
            out = []
            for ca, cb in TERMS:
                for st in range(slots[a]):
                    for q in mine[a]:
                        out.append(f"P{n}_{q.index} = oeq_mfma_bf(f{n}[{st}][{ca}], w{q.index}[{st}][{cb}], P{n}_{q.index}, 0, 0, 0);")
            return out

        for n, (a, i) in enumerate(steps):
            if n in (0, N - 1):
                for q in mine[a]:
                    s(f"v4t P{n}_{q.index} = v4t{{}};")
        s(f"oeq_bf8 f0[{slots[steps[0][0]]}][3];")
        s(f"v4t y[{L2}];")
        for j in range(L2):
            s(f"y[{j}] = v4t{{}};")
        for t in used_t:
            s(f"v4t acc{t}[{T[t].d}];")
            for k in range(T[t].d):
                s(f"acc{t}[{k}] = v4t{{}};")
            if not fwd:
                s(f"v4t x{t}[{T[t].d}];")
                for k in range(T[t].d):
                    s(f"x{t}[{k}] = v4t{{}};")
        if not fwd:
            s(f"v4t dy[{L2}];")
            for j in range(L2):
                s(f"dy[{j}] = v4t{{}};")

            # dY of a tile: the waves' shares, in wave order, on top of what an earlier kernel has left there. Read beside
            # one step and added up beside a later one, each element by one thread: accesses of the threads past the
            # tile are out of the buffer's range, and no branch cuts a step in two. Without a tile to finish, as at first,
            # the block's own first tile is written as it is, or with what its sums replace when they are there.
            def finish(buf):
                s("const int fend = (int)min((i64)15, num_batch - 1 - frow0);")
                s(f"const __amdgpu_buffer_rsrc_t dyr = __builtin_amdgcn_make_buffer_rsrc(L2_grad + frow0 * {L2}, 0, (fend + 1) * {4 * L2}, 0x00027000);")
                s(f"float sdy[{ny}][4], ody[{ny}];")
                take, give = [], []
                for n in range(ny):
                    v = f"(tid + {256 * n})"
                    take.append((8, " ".join(f"sdy[{n}][{q}] = s_dy[{buf}][{q}][min({v}, {16 * L2 - 1})];" for q in range(4))
                                 + (f" ody[{n}] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(dyr, 4 * {v}, 0, 0));" if number else "")))
                    tot = f"sign * (((sdy[{n}][0] + sdy[{n}][1]) + sdy[{n}][2]) + sdy[{n}][3])"
                    if number:
                        tot = f"ody[{n}] + (ready ? {tot} : 0.0f)"
                    give.append((8, f"__builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, {tot}), dyr, 4 * {v}, 0, 0);"))
                return take, give
        s("int cur = 0;")
        s("i64 prow0 = (i64)blockIdx.x * 16;  // first row of the tile whose results are still to be stored")
        s("oeq_block_sync();")
        self.put(s, fetch(0))
        s.open("for (i64 tile = blockIdx.x; tile < ntiles; tile += gridDim.x, cur ^= 1)")
        s("const i64 row0 = tile * 16;")
        # the tile whose rows are requested during this one
        where("(tile + 2 * (i64)gridDim.x)", "const i64 ")
        s(f"const float* rows = {src} + first * {LA};")
        s(f"const unsigned own = (unsigned)min(tid >> 4, end) * {4 * LA}u;")
        s("const int pend = (int)min((i64)15, num_batch - 1 - prow0);")
        take = give = []
        if not fwd:
            # (two tiles back: its shares were written beside the first component of the tile before)
            s("const bool ready = tile >= (i64)blockIdx.x + 2 * (i64)gridDim.x;")
            s("const i64 frow0 = (ready ? tile - 2 * (i64)gridDim.x : (i64)blockIdx.x) * 16;")
            take, give = finish("cur")
        # the step that writes an operand of the next tile: not the first, which has the rows of the tile before to store,
        # nor the last, which reads them
        writer = lambda m: min(1 + m * max(1, N - 4) // len(units), N - 2) if N > 2 else 0
        for n, (a, i) in enumerate(steps):
            tasks, reads = [], []
            if n + 1 < N:
                s(f"oeq_bf8 f{n + 1}[{slots[steps[n + 1][0]]}][3];")
                reads = fetch(n + 1)
            # a share of the next tile's operands, and of the requests for the one after
            for ua, ust in (units[m] for m in range(len(units)) if writer(m) == n):
                tasks += write(ua, ust, "s_a[cur ^ 1]")
                tasks.append((1, "redo |= oeq_too_large(top) ? next : 0u; top = 0.0f;"))
                tasks += request(ua, ust)
            tasks += contract((n or N) - 1)
            if n == min(1, N - 2):
                # (before the tile's barrier: the next tile's first step writes these shares over)
                tasks += take
            if n == min(1, N - 1):
                if not fwd:
                    # X of the next tile, whose registers this tile's has left beside the step before
                    s("const i64 xfirst = min((tile + gridDim.x) * 16, num_batch - 1);")
                    s("const int xend = (int)min((i64)15, num_batch - 1 - xfirst);")
                    tasks += [v for t in used_t for v in request_x(t)]
            if n == N - 1:
                tasks += give
            if n == N - 1:
                s("oeq_block_sync();  // the next tile's operands are written, this tile's are read")
                reads = fetch(0, "cur ^ 1")
            tasks = self.spread_reads(reads, tasks)
            if n not in (0, N - 1):
                for q in mine[a]:
                    s(f"v4t P{n}_{q.index};")
            pre = [f"P{n}_{q.index} = v4t{{}};" for q in mine[a]]
            for line in pre:
                s(line)
            s("__builtin_amdgcn_sched_barrier(0);")
            if n == 0:
                half = lead(0)
                cut = len(half) // 2
                self.interleave(s, half[:cut], tasks)
                tasks = store("prow0", "pend")
                tasks += [(1, f"y[{j}] = *(const v4t*)&s_y[cur][{j}][4 * lq];") for j in range(L2)]
                if not fwd:
                    tasks += self.reduce_dy("s_dy[cur ^ 1]")
                self.interleave(s, half[cut:], tasks)
                if not fwd:
                    for t in used_t:
                        for k in range(T[t].d):
                            s(f"x{t}[{k}] = xn{t}[{k}];")
                write_y("cur ^ 1")
                request_y()
            else:
                self.interleave(s, lead(n), tasks)
        s("next = (next << 1) | (next >> 31);")
        s("prow0 = row0;")
        if number == 0:
            for t in range(len(T)):
                if not any(it(q) == t for q in self.subs):
                    s.open(f"for (int z = tid; z < {16 * T[t].mul * T[t].d}; z += 256)")
                    s(f"const i64 row = row0 + z / {T[t].mul * T[t].d};")
                    s(f"if (row < num_batch) {dst}[row * {LT} + {T[t].off} + z % {T[t].mul * T[t].d}] = 0.0f;")
                    s.close()
        s.close()
        s("const int pend = (int)min((i64)15, num_batch - 1 - prow0);")
        self.put(s, contract(N - 1))
        self.put(s, store("prow0", "pend"))
        if not fwd:
            self.put(s, self.reduce_dy("s_dy[cur ^ 1]"))
            s("const i64 tiles_here = (ntiles - 1 - blockIdx.x) / gridDim.x + 1;")
            s("oeq_block_sync();")
            s("const bool ready = true;")
            for back, buf in ((2, "cur"), (1, "cur ^ 1")):
                s.open(f"if (tiles_here >= {back})")
                s(f"const i64 frow0 = ((i64)blockIdx.x + (tiles_here - {back}) * gridDim.x) * 16;")
                for part in finish(buf):
                    self.put(s, part)
                s.close()
        self.emit_redo(s, kind, subs, number, folds, where)
        s.close()

    def emit_redo(self, s: Src, kind: str, subs, number: int, folds, where):
        """Rows with an operand that three bf16 parts do not hold, all rows of the block if a weight is one: once more with fp32
        matrix instructions, after the last tile, on operands straight from memory. dY of such a row is formed anew from the
        sub-paths of the kernels before this one too, whose sums the first pass has written over."""
        low = self.low
        A, T, ia, it = self.sides(kind)
        L2, fwd = low.L2, kind == "forward"
        src, LA = ("L1_in", low.L1) if fwd else ("L3_grad", low.L3)
        dst, LT = ("L3_out", low.L3) if fwd else ("L1_grad", low.L1)
        used_a = sorted({ia(q) for q in subs})
        mine = sorted(subs, key=it)
        every = mine if fwd else [q for k in self.plan(kind)[:number] for q in sorted(k, key=it)] + mine
        s("__shared__ unsigned s_redo[8];")
        s("s_redo[wave] = redo, s_redo[4 + wave] = wrows;")
        s("oeq_block_sync();")
        s("redo = __builtin_amdgcn_readfirstlane(s_redo[0] | s_redo[1] | s_redo[2] | s_redo[3]);")
        s("const unsigned whole = __builtin_amdgcn_readfirstlane(s_redo[4] | s_redo[5] | s_redo[6] | s_redo[7]);")
        s("if (!redo) return;")
        s("oeq_block_sync_all();  // (behind the stores of the rows that are written once more)")
        # (lane numbers anew: kept, they would take registers in the loop above)
        s.open("")
        s("const int id = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));")
        s("const int tid = 64 * wave + id, l16 = id & 15, lq = id >> 4;")
        s("unsigned turn = 0;")
        s.open("for (i64 tile = blockIdx.x; tile < ntiles; tile += gridDim.x, ++turn)")
        s("if (!(redo >> (turn & 31) & 1)) continue;")
        where("tile", "const i64 ")
        s(f"const float* rows = {src} + first * {LA};")
        # which rows: the splits again (tiles 32 turns apart share a bit)
        s("float gone = 0.0f;")
        s.open("")
        s(f"const float* ap = rows + min(tid >> 4, end) * {LA};")
        for a in used_a:
            s(f"for (int z = tid & 15; z < {A[a].mul * A[a].d}; z += 16) gone = oeq_top(gone, {self.lit(SCALE)} * ap[{A[a].off} + z], 0.0f);")
        for q in folds:
            b, b2 = A[ia(q)], low.in2[q.p.i2]
            s(f"const float* yp{q.index} = L2_in + (first + min(tid >> 4, end)) * {L2} + {self.yat(q, 0)};")
            s(f"const float yt{q.index}[{b2.d}] = {{{', '.join(f'yp{q.index}[{j}]' for j in range(b2.d))}}};")
            s.open(f"for (int z = tid & 15; z < {b.mul}; z += 16)")
            for line in self.fold_terms(q, "v", lambda i: f"ap[{b.off} + {b.d} * z + {i}]"):
                s(line)
            s(f"gone = oeq_top(gone, {self.lit(SCALE)} * v, 0.0f);")
            s.close()
        s.close()
        s("const unsigned long long rows_gone = __builtin_amdgcn_ballot_w64(gone >= 3.39e38f);")
        s("unsigned four = 0;")
        s("for (int r = 0; r < 4; ++r) four |= (rows_gone >> (16 * r) & 0xffff) ? 1u << r : 0u;")
        s("oeq_block_sync();  // (the words of the tile before are read)")
        s("s_redo[wave] = four << (4 * wave);")
        s("oeq_block_sync();")
        s("const unsigned bad = whole | __builtin_amdgcn_readfirstlane(s_redo[0] | s_redo[1] | s_redo[2] | s_redo[3]);")
        s("if (!bad) continue;")
        s("int col = 16 * wave + l16;")
        s(f"const float* ap = rows + min(l16, end) * {LA};")
        opaque = "asm volatile(\"\" : \"+v\"(col));  // (no address is worked out ahead: registers)"
        if not fwd:
            # (Y as it is met: its components together with those of dY would be too many registers)
            s("unsigned yr[4];")
            s(f"for (int r = 0; r < 4; ++r) yr[r] = {4 * L2}u * min(4 * lq + r, end);")
            s(f"const float* yp = L2_in + first * {L2};")
            s(f"v4t dy[{L2}];")
            s(" ".join(f"dy[{j}] = v4t{{}};" for j in range(L2)))
        at = 0
        while at < len(every):
            t, own = it(every[at]), any(every[at] is q for q in mine)
            group = []
            while at < len(every) and it(every[at]) == t:
                group.append(every[at])
                at += 1
            b = T[t]
            s.open("")
            if own:
                s(f"v4t acc[{b.d}];")
                s(" ".join(f"acc[{k}] = v4t{{}};" for k in range(b.d)))
            if not fwd:
                s(f"v4t x[{b.d}];")
                for i in range(b.d):
                    s(f"for (int r = 0; r < 4; ++r) x[{i}][r] = oeq_sel(col < {b.mul}, "
                      f"L1_in[(first + min(4 * lq + r, end)) * {low.L1} + {b.off + i} + min(col, {b.mul - 1}) * {b.d}]);")
                s("__builtin_amdgcn_sched_barrier(0);")
            for q in group:
                a = A[ia(q)]
                ld = low.in2[q.p.i2].mul * low.out[q.p.io].mul
                cu, ct = (ld, 1) if fwd else (1, ld)
                base = q.p.woff + q.v * low.out[q.p.io].mul
                if fwd:
                    # contracted first, as the fp32 kernels do: what a small Y brings back into range stays in it
                    b2 = low.in2[q.p.i2]
                    s.open("")
                    s(f"const float* yp = L2_in + (first + min(l16, end)) * {L2} + {self.yat(q, 0)};")
                    s(f"const float y[{b2.d}] = {{{', '.join(f'yp[{j}]' for j in range(b2.d))}}};")
                    for kk in sorted({k for _, _, k, _ in q.p.nnz}):
                        s(opaque)
                        s("#pragma unroll 4")
                        s.open(f"for (int u0 = 0; u0 < {a.mul}; u0 += 4)")
                        s(f"const int u = min(u0 + lq, {a.mul - 1});")
                        s(f"const float* xp = ap + {a.off} + {a.d} * u;")
                        terms = " + ".join(f"{self.lit(c)} * y[{j}] * xp[{i}]" for i, j, k, c in q.p.nnz if k == kk)
                        s(f"const float av = oeq_sel(u0 + lq < {a.mul}, {terms});")
                        s(f"const float bv = oeq_sel(u0 + lq < {a.mul} && col < {b.mul}, W[{base} + u * {cu} + min(col, {b.mul - 1}) * {ct}]);")
                        s(f"acc[{kk}] = oeq_mfma(av, bv, acc[{kk}], 0, 0, 0);")
                        s.close()
                        s("__builtin_amdgcn_sched_barrier(0);")
                    s.close()
                    continue
                for i in sorted({k for _, _, k, _ in q.p.nnz}):
                    s.open("")
                    s("v4t P = v4t{};")
                    s(opaque)
                    s("#pragma unroll 4")
                    s.open(f"for (int u0 = 0; u0 < {a.mul}; u0 += 4)")
                    s(f"const int u = min(u0 + lq, {a.mul - 1});")
                    s(f"const float av = oeq_sel(u0 + lq < {a.mul}, ap[{a.off + i} + {a.d} * u]);")
                    s(f"const float bv = oeq_sel(u0 + lq < {a.mul} && col < {b.mul}, W[{base} + u * {cu} + min(col, {b.mul - 1}) * {ct}]);")
                    s("P = oeq_mfma(av, bv, P, 0, 0, 0);")
                    s.close()
                    for (i1, j, k, c) in q.p.nnz:
                        if k != i:
                            continue
                        if own:
                            s(f"acc[{i1}] += {self.lit(c)} * oeq_rows4(yp + {self.yat(q, j)}, yr) * P;")
                        s(f"dy[{self.yat(q, j)}] += {self.lit(c)} * x[{i1}] * P;")
                    s("__builtin_amdgcn_sched_barrier(0);")
                    s.close()
            if own:
                s.open("for (int r = 0; r < 4; ++r)")
                s(f"float* op = {dst} + (first + 4 * lq + r) * {LT} + {b.off} + {b.d} * col;")
                s(f"if (4 * lq + r <= end && (bad >> (4 * lq + r) & 1) && col < {b.mul}) {{ "
                  + " ".join(f"op[{k}] = acc[{k}][r];" for k in range(b.d)) + " }")
                s.close()
            s.close()
        if not fwd:
            for j in range(L2):
                s.open("for (int r = 0; r < 4; ++r)")
                s(f"float v = dy[{j}][r];")
                for ctrl in ("0x140", "0x141", "0x1B", "0xB1"):
                    s(f"v += oeq_dpp<{ctrl}>(v);")
                s(f"if (l16 == 0) s_dy[0][wave][(4 * lq + r) * {L2} + {j}] = v;")
                s.close()
            s("oeq_block_sync();")
            s.open(f"for (int z = tid; z < {16 * L2}; z += 256)")
            s(f"const float v = ((s_dy[0][0][z] + s_dy[0][1][z]) + s_dy[0][2][z]) + s_dy[0][3][z];")
            s(f"if (z / {L2} <= end && (bad >> (z / {L2}) & 1)) L2_grad[first * {L2} + z] = v;")
            s.close()
            s("oeq_block_sync();")
        s.close()
        s.close()

    def reduce_dy(self, into: str):
        """Sum over the 16 lanes that hold a row's channels. A step adds the lanes of a mirrored half to the ones of the other
        and leaves half as many values: a lane keeps those of the half it lies in. n / 16 consecutive ones of the 4 x L2
        values of its group of lanes, which lie one after the other in memory, too, are a lane's in the end."""
        L2 = self.low.L2
        n = 4 * L2
        cur = (n + 15) // 16 * 16
        val = [f"dy[{o % L2}][{o // L2}]" if o < n else "0.0f" for o in range(cur)]
        out = [(0, f"float rv[{cur // 2 + 2}]; int at = 0;")]
        for ctrl, bit, upper in (("row_mirror", 8, "0xc"), ("row_half_mirror", 4, "0xa"), ("0x1B", 2, None), ("0xB1", 1, None)):
            half = cur // 2
            for j in range(0, half, 1 if upper is None else 3):
                if upper is None:
                    out.append((3, f"{{ const bool hi = (l16 & {bit}) != 0; const float keep = hi ? {val[j + half]} : {val[j]}, send = hi ? {val[j]} : {val[j + half]}; "
                                   f"rv[{j}] = keep + oeq_dpp<{ctrl}>(send); }}"))
                    continue
                # (three at a time; past the last pair: it once more)
                at = [min(j + m, half - 1) for m in range(3)]
                into_ = [f"rv[{j + m}]" if j + m < half else f"rv[{cur // 2}]" for m in range(3)]
                out.append((7, f"OEQ_FOLD_LANES({', '.join(into_ + [val[m] for m in at] + [val[m + half] for m in at])}, \"{ctrl}\", \"{upper}\")"))
            out.append((1, f"at += (l16 & {bit}) ? {half} : 0;"))
            val, cur = [f"rv[{j}]" for j in range(half)], half
        return out + [(1, f"if (at + {t} < {n}) {into}[wave][4 * lq * {L2} + at + {t}] = rv[{t}];") for t in range(cur)]

    # ------------------------------------------------------------------------ dW
    def split_dw(self, subs):
        """(waves along the input channels, waves along the output channels, 16-channel tiles of a sub-path's outputs
        that a wave sums)"""
        most = max(c16(self.low.in1[q.p.i1].mul) for q in subs)
        wu = 4 if most > 2 else most
        return wu, 4 // wu, lambda q: (c16(self.low.out[q.p.io].mul) + 4 // wu - 1) // (4 // wu)

    def registers_dw(self, subs) -> int:
        low = self.low
        _, _, per = self.split_dw(subs)
        into = max(sum(4 * per(q) for q in subs if q.p.io == o) for o in {q.p.io for q in subs})
        x = 8 * sum(low.in1[a].d for a in {q.p.i1 for q in subs})
        g = 8 * sum(low.out[o].d for o in {q.p.io for q in subs})
        return 4 * sum(per(q) for q in subs) + into + x + 16 + max(x, g) + 18 * max(per(q) for q in subs) + 32 + 32

    def table_dw(self, subs):
        """(component of Y, ratio of a coefficient to its path's unit), each once."""
        return sorted({(self.yat(q, j), q.ratio(c)) for q in subs for _, j, _, c in q.p.nnz})

    def lds_dw(self, subs) -> int:
        low = self.low
        return 2 * (3072 * sum(low.out[o].d * c16(low.out[o].mul) for o in {q.p.io for q in subs}) + 192 * len(self.table_dw(subs)))

    def folds_dw(self, subs):
        """Sub-paths whose input has one component and whose output has more (0 x l -> l): Y and dZ are contracted by the
        threads that split dZ, and one component is multiplied, not 2 l + 1. As many as the LDS has room for, and three more
        products remain."""
        low, out, room = self.low, [], LDS_BUDGET // self.waves("dw") - self.lds_dw(subs)
        for q in sorted(subs, key=lambda q: -low.out[q.p.io].d):
            if low.in1[q.p.i1].d == 1 and low.out[q.p.io].d > 1:
                room -= 2 * 3072 * c16(low.out[q.p.io].mul)
                if room >= 0 and len(self.stages_dw([p for p in subs if p not in out and p is not q])) >= 3:
                    out.append(q)
        return out

    def stages_dw(self, subs, folds=()):
        """(output block, component, sub-path), in the order in which they are multiplied; first those that are folded."""
        out = self.low.out
        return [(q.p.io, q.key, q) for q in folds] + \
            [(o, k, q) for o in sorted({q.p.io for q in subs}, key=lambda o: -out[o].d) for k in range(out[o].d)
             for q in subs if q.p.io == o and q not in folds and any(kk == k for _, _, kk, _ in q.p.nnz)]

    def emit_dw(self, s: Src, name: str, sig: str):
        """One kernel, in which a block goes through the parts of ``plan_dw`` one after the other: the steps of 32 rows seldom
        divide evenly among the blocks, and those that have one more of a part have one fewer of the next. Small batches have blocks to
        spare, and their parts run side by side. 64x{0e,1o,2e}, forward and backward, a launch per part / one: 2 000 rows 85 /
        72 - 81 us, 4 500 99 / 90, 20 000 187 / 171, 60 000 408 / 391, 100 003 and 131 072 the same."""
        parts = self.plan_dw()
        tables = [self.table_dw(subs) for subs in parts]
        words = []
        for n, (subs, table) in enumerate(zip(parts, tables)):
            s(f"static __constant__ const float {name}_c{n}[{len(table)}] = {{{', '.join(self.lit(r) for _, r in table)}}};")
            s(f"static __constant__ const int {name}_j{n}[{len(table)}] = {{{', '.join(str(j) for j, _ in table)}}};")
            words.append(2 * sum(768 * c16(self.low.out[o].mul) for o, _ in self.operands_dw(subs)) + 96 * len(table))
        self.open_kernel(s, name, sig, self.waves("dw"))
        s("const int tid = (int)threadIdx.x;")
        s(f"__shared__ __attribute__((aligned(16))) unsigned s_lds[{max(words)}];")
        s("const i64 nsteps = (num_batch + 31) / 32;")
        s("const int more = (int)(nsteps % gridDim.x);  // blocks with one step more")
        for n, subs in enumerate(parts):
            s.open("")
            s(f"const i64 begin = (blockIdx.x + {n} * (gridDim.x - more)) % gridDim.x;  // the block's first step")
            if n:
                s("oeq_block_sync();")
            self.emit_dw_part(s, f"{name}_c{n}", f"{name}_j{n}", subs, tables[n])
            s.close()
        s.close()
        return [name]

    def operands_dw(self, subs):
        """(output block, component or folded sub-path) whose operands are in LDS."""
        return list(dict.fromkeys((o, k) for o, k, _ in self.stages_dw(subs, self.folds_dw(subs))))

    def emit_dw_part(self, s: Src, coefficients: str, components: str, subs, table):
        low = self.low
        L2 = low.L2
        WU, WW, per = self.split_dw(subs)
        used_a, used_o = sorted({q.p.i1 for q in subs}), sorted({q.p.io for q in subs}, key=lambda o: -low.out[o].d)
        folds = self.folds_dw(subs)
        stages = self.stages_dw(subs, folds)
        where, total = {}, 0
        for o, k in self.operands_dw(subs):
            where[(o, k)] = total
            total += 768 * c16(low.out[o].mul)
        # dZ's operands, and components of Y times the coefficients they are met with
        s(f"unsigned (* const s_g)[{total}] = (unsigned (*)[{total}])s_lds;")
        s(f"float (* const s_y)[{len(table)}][32] = (float (*)[{len(table)}][32])(s_lds + {2 * total});")
        s(f"const int wu = wave % {WU}, ww = wave / {WU};")
        s("(void)ww;")
        s("const float sign = (blockIdx.x & 1) ? -1.0f : 1.0f;")
        for q in subs:
            s(f"v4t dw{q.index}[{per(q)}];")
            for j in range(per(q)):
                s(f"dw{q.index}[{j}] = v4t{{}};")
        for o in used_o:
            s(f"float g{o}[{8 * low.out[o].d}];")
            s(f"const int gc{o} = min(16 * wave + l16, {low.out[o].mul - 1});")
        for a in used_a:
            s(f"float x{a}[8][{low.in1[a].d}], xn{a}[8][{low.in1[a].d}];")
            s(f"const int xc{a} = min(16 * wu + l16, {low.in1[a].mul - 1});")
        s(f"v4t yv[{AHEAD + 1}][2];  // a component of Y for the lane's eight rows, and the next ones")
        # (a thread's elements: row tid / 32 + 8 n of the table, row tid % 32 of the tile; past the table its last row again)
        ny = (len(table) + 7) // 8
        s(f"float ry[{ny}], yc[{ny}];")
        s(f"int yj[{ny}];")
        s("#pragma unroll")
        s.open(f"for (int n = 0; n < {ny}; ++n)")
        s(f"const int at = min((tid >> 5) + 8 * n, {len(table) - 1});")
        s(f"yc[n] = {self.lit(SCALE)} * sign * {coefficients}[at], yj[n] = {components}[at];")
        s.close()

        def rows_of(step):
            s(f"const i64 first = min((i64)({step}) * 32, num_batch - 1);")
            s("const int end = (int)min((i64)31, num_batch - 1 - first);")

        def request_g(o, e):
            b = low.out[o]
            return [(4, f"{{ const float* gp = oeq_at(L3_grad + first * {low.L3} + {b.off}, 4u * (unsigned)(min(8 * lq + {e}, end) * {low.L3} + gc{o} * {b.d})); "
                     + " ".join(f"g{o}[{e * b.d + k}] = gp[{k}];" for k in range(b.d)) + " }")]

        def request_x(a, e):
            b = low.in1[a]
            return [(4, f"{{ const float* xp = oeq_at(L1_in + first * {low.L1} + {b.off}, 4u * (unsigned)(min(8 * lq + {e}, end) * {low.L1} + xc{a} * {b.d})); "
                     + " ".join(f"xn{a}[{e}][{i}] = xp[{i}];" for i in range(b.d)) + " }")]

        # (Y is a step ahead of dZ, with which it is contracted on the way to LDS, and so has three copies)
        def request_y(step):
            s(f"const i64 yfirst = min((i64)({step}) * 32, num_batch - 1);")
            s("const int yend = (int)min((i64)31, num_batch - 1 - yfirst);")
            s(f"const int yrows = (int)max((i64)0, min((i64)32, num_batch - (i64)({step}) * 32));")
            return [(4, f"ry[{n}] = *oeq_at(L2_in + yfirst * {L2}, 4u * (unsigned)(min(tid & 31, yend) * {L2} + yj[{n}]));")
                    for n in range(ny)]

        def write_y(buf):
            """Zeros for the rows past the batch, which repeat its last one otherwise."""
            return [(5, f"s_y[{buf}][min((tid >> 5) + {8 * n}, {len(table) - 1})][tid & 31] = oeq_sel((tid & 31) < yrows, yc[{n}] * ry[{n}]);")
                    for n in range(ny)]

        def fold(q, v, buf):
            """dZ and Y of a folded sub-path, for the lane's column and eight rows."""
            o, terms, y = q.p.io, q.p.nnz, f"yf{q.index}"
            get = lambda m: [(2, f"{y}[{m & 1}][{h}] = *(const v4t*)&{buf}[{at_of(q, terms[m][1], terms[m][3])}][8 * lq + {4 * h}];") for h in (0, 1)]
            out = [(0, f"float {v}[8]; v4t {y}[2][2];")] + get(0)
            for m, (_, j, k, c) in enumerate(terms):
                out += get(m + 1) if m + 1 < len(terms) else []
                op = ("= -" if c < 0 else "= ") if m == 0 else "-= " if c < 0 else "+= "
                out += [(4, " ".join(f"{v}[{4 * h + r}] {op}{y}[{m & 1}][{h}][{r}] * g{o}[{(4 * h + r) * low.out[o].d + k}];" for r in range(4)))
                        for h in (0, 1)]
            return out

        def write_g(o, buf, ynext):
            """dZ of the wave's columns of a block as operands."""
            b = low.out[o]
            out = []
            for k in [k for oo, k in where if oo == o]:
                only = f"if (16 * wave < {16 * c16(b.mul)}) " if b.mul <= 48 else ""
                q = next((q for q in folds if q.key == k), None)
                v = f"v{o}_{k}" if q is None else f"vf{q.index}"
                if q is None:
                    out.append((0, f"float {v}[8];"))
                    out += [(4, " ".join(f"{v}[{e}] = {self.lit(SCALE)} * g{o}[{e * b.d + k}];" for e in range(h, h + 4))) for h in (0, 4)]
                else:
                    out += fold(q, v, ynext)
                out += self.split_tasks(v, "tg")
                out += [(1, only + f"*(oeq_u4*)({buf} + {where[(o, k)] + 256 * c} + 768 * wave + 4 * lane) = oeq_u4{{tg[{c}][0], tg[{c}][1], tg[{c}][2], tg[{c}][3]}};")
                        for c in range(3)]
            return out

        places = {q.index: [n for n, (_, _, p) in enumerate(stages) if p is q] for q in subs}
        N = len(stages)
        at_of = lambda q, j, c: table.index((self.yat(q, j), q.ratio(c)))

        # (stage, row of the table) in the order in which stages 1 .. N - 1 are contracted, and the first one's
        js_of = lambda n: sorted({at_of(stages[n % N][2], j, c) for (_, j, kk, c) in stages[n % N][2].p.nnz if kk == stages[n % N][1]})
        later = [(n, j) for n in range(1, N) for j in js_of(n)]

        def read_y(units, u, buf):
            if u >= len(units):
                return []
            n, j = units[u]
            row = f"{buf}[{j}]"
            return [(2, f"yv[{u % (AHEAD + 1)}][0] = *(const v4t*)&{row}[8 * lq]; "
                        f"yv[{u % (AHEAD + 1)}][1] = *(const v4t*)&{row}[8 * lq + 4];")]

        def t_tasks(n):
            """The contraction of X and Y for stage n, eight rows a lane, as operands. Y comes from LDS, component by
            component, AHEAD of the sums."""
            o, k, q = stages[n % N]
            if q in folds:
                return [(4, " ".join(f"t[{4 * h + r}] = {self.lit(SCALE)} * x{q.p.i1}[{4 * h + r}][0];" for r in range(4))) for h in (0, 1)] + \
                    self.split_tasks("t", f"ta[{n % 2}]")
            buf = "s_y[ycur]" if n < N else "s_y[ynext]"
            units = later if n % N else [(0, j) for j in js_of(0)]
            out, first = [], True
            for u, (m, j) in enumerate(units):
                if m != n % N:
                    continue
                if u == 0:
                    for v in range(AHEAD):
                        out += read_y(units, v, buf)
                out += read_y(units, u + AHEAD, buf)
                for i, jj, kk, c in q.p.nnz:
                    if kk != k or at_of(q, jj, c) != j:
                        continue
                    op = ("= -" if c < 0 else "= ") if first else "-= " if c < 0 else "+= "
                    for h in range(2):
                        out.append((4, " ".join(f"t[{4 * h + r}] {op}yv[{u % (AHEAD + 1)}][{h}][{r}] * x{q.p.i1}[{4 * h + r}][{i}];"
                                                for r in range(4))))
                    first = False
            return out + self.split_tasks("t", f"ta[{n % 2}]")

        operand = lambda q: f"__builtin_bit_cast(oeq_bf8, oeq_u4{{{', '.join(f'{q}[{m}]' for m in range(4))}}})"

        def read_bg(n, pair, buf):
            o, k, q = stages[n % N]
            out = []
            for j in pair:
                nt = f"{j}" if WW == 1 else f"min(ww + {j * WW}, {c16(low.out[o].mul) - 1})"
                for c in range(3):
                    out.append((1, f"bg[{j}][{c}] = __builtin_bit_cast(oeq_bf8, *(const oeq_u4*)({buf} + {where[(o, k)] + 256 * c} + 768 * ({nt}) + 4 * lane));"))
            return out

        most = max(per(q) for q in subs)
        pairs = lambda q: [list(range(j, min(j + 2, per(q)))) for j in range(0, per(q), 2)]

        # A step's products into the running sums. By fp32 matrix instructions with the identity, which spare the moves out of the
        # accumulation registers but keep the vector unit for 32 cycles a value where an addition and its moves take 14: dW
        # 298 us, 281 by additions (64x{0e,1o,2e}, 100 003 rows; the pass 642 -> 630, 20 000 rows 165 -> 159).
        flush = lambda p, j: " ".join(f"dw{p.index}[{j}][{i}] += sign * tm{p.index}[{j}][{i}];" for i in range(4))

        def lead(n, pair):
            o, k, q = stages[n]
            return [f"tm{q.index}[{j}] = oeq_mfma_bf({operand(f'ta[{n % 2}][{ca}]')}, bg[{j}][{cb}], tm{q.index}[{j}], 0, 0, 0);"
                    for ca, cb in TERMS for j in pair]

        # ---- the first step's operands
        s.open("if (begin < nsteps)")
        s("float t[8];")
        s("unsigned ta[2][3][4], tg[3][4];")
        s(f"oeq_bf8 bg[{most}][3];")
        for q in subs:
            s(f"v4t tm{q.index}[{per(q)}];")
        s.open("")
        rows_of("begin")
        for o in used_o:
            for e in range(8):
                self.put(s, request_g(o, e))
        for a in used_a:
            for e in range(8):
                self.put(s, request_x(a, e))
        for n, step in enumerate(("begin", "begin + gridDim.x")):
            s.open("")
            self.put(s, request_y(step))
            self.put(s, write_y(n))
            s.close()
        s("oeq_block_sync();")
        for o in used_o:
            self.put(s, write_g(o, "s_g[0]", "s_y[0]"))
        s.close()
        for a in used_a:
            for e in range(8):
                for i in range(low.in1[a].d):
                    s(f"x{a}[{e}][{i}] = xn{a}[{e}][{i}];")
        s("int cur = 0, ycur = 0;")
        s("oeq_block_sync();")
        self.put(s, t_tasks(0))
        self.put(s, read_bg(0, pairs(stages[0][2])[0], "s_g[0]"))
        s.open("for (i64 step = begin; step < nsteps; step += gridDim.x, cur ^= 1)")
        # the step whose rows are requested, and written to LDS, during this one
        rows_of("step + gridDim.x")
        s("const int ynext = ycur == 2 ? 0 : ycur + 1, yput = ynext == 2 ? 0 : ynext + 1;")
        pending = []   # sums to be flushed beside a later stage's products
        g_req = [t for o in used_o for e in range(8) for t in request_g(o, e)] + request_y("step + 2 * (i64)gridDim.x")
        g_put = [t for o in used_o for t in write_g(o, "s_g[cur ^ 1]", "s_y[ynext]")] + write_y("yput")
        x_req = [t for a in used_a for e in range(8) for t in request_x(a, e)]
        # (stages over which these are spread: X is requested when dZ has left the registers)
        spread = lambda items, n, lo, hi: items[max(0, n - lo) * len(items) // (hi - lo):(n + 1 - lo) * len(items) // (hi - lo)] \
            if lo <= n < hi else []
        req_end = max(1, 3 * N // 20)
        put_from = min(max(req_end, 3 * N // 5), N - 2)
        put_end = min(max(put_from + 1, 9 * N // 10), N - 1)
        for n, (o, k, q) in enumerate(stages):
            tasks = []
            tasks += spread(g_req, n, 0, req_end) + spread(g_put, n, put_from, put_end) + spread(x_req, n, put_from, put_end)
            if n == places[q.index][0]:
                for j in range(per(q)):
                    s(f"tm{q.index}[{j}] = v4t{{}};")
            new_group = n + 1 == N or stages[n + 1][:2] != stages[n][:2]
            group_start = n == 0 or stages[n - 1][:2] != stages[n][:2]
            ps = pairs(q)
            buf, nbuf = "s_g[cur]", "s_g[cur]" if n + 1 < N else "s_g[cur ^ 1]"
            if n + 1 == N:
                if group_start:
                    # (read before the barrier: past it, other waves write over this step's operands)
                    for pair in ps[1:]:
                        self.put(s, read_bg(n, pair, buf))
                s("oeq_block_sync();  // the next step's operands are written, this one's are read")
                tasks += [(1, " ".join(f"x{a}[{e}][{i}] = xn{a}[{e}][{i}];" for i in range(low.in1[a].d)))
                          for a in used_a for e in range(8)]
            tasks += t_tasks(n + 1)
            tasks = [(4, flush(p, j)) for p in pending for j in range(per(p))] + tasks
            pending = [q] if n == places[q.index][-1] else []
            seq = [lead(n, pair) for pair in ps]
            # operands of this group that are not there yet (its second half), and the next group's first half once
            # this stage is done with its own
            weight = sum(w for w, _ in tasks)
            cut = [[] for _ in seq]
            at = 0
            for m in range(len(seq)):
                acc = 0
                while at < len(tasks) and (m + 1 == len(seq) or acc + tasks[at][0] / 2 < weight / len(seq)):
                    cut[m].append(tasks[at])
                    acc += tasks[at][0]
                    at += 1
            for m in range(len(seq)):
                extra = []
                if group_start and m + 1 < len(ps) and n + 1 < N:
                    extra = read_bg(n, ps[m + 1], buf)
                if new_group and m > 0 and m == len(ps) - 1:
                    extra = extra + read_bg(n + 1, pairs(stages[(n + 1) % N][2])[0], nbuf)
                self.interleave(s, seq[m], extra + cut[m])
            if new_group and len(ps) == 1:
                self.put(s, read_bg(n + 1, pairs(stages[(n + 1) % N][2])[0], nbuf))
            if n + 1 == N:
                for p in pending:
                    for j in range(per(p)):
                        s(flush(p, j))
                s("ycur = ynext;")
                if N % 2:
                    s("for (int c = 0; c < 3; ++c) for (int m = 0; m < 4; ++m) ta[0][c][m] = ta[1][c][m];")
        s.close()
        s.close()
        # Operands above the range that three parts hold, and infinities, have made NaN of the sums they met.
        s("float off = 0.0f;")
        for q in subs:
            s("#pragma unroll")
            s(f"for (int j = 0; j < {per(q)}; ++j) for (int i = 0; i < 4; ++i) off += 0.0f * dw{q.index}[j][i];")
        s("const bool again = __builtin_amdgcn_ballot_w64(off != off) != 0;")
        s.open("if (again)")
        self.emit_redo_dw(s, subs)
        s.close()
        s(f"float* prow = wpartial + (i64)blockIdx.x * {low.WN};")
        for q in subs:
            U, Wn = low.in1[q.p.i1].mul, low.out[q.p.io].mul
            for j in range(per(q)):
                s("#pragma unroll")
                s.open("for (int i = 0; i < 4; ++i)")
                nt = f"{j}" if WW == 1 else f"(ww + {j * WW})"
                s(f"const int u = 16 * wu + 4 * lq + i, w = 16 * {nt} + l16;")
                s(f"if (u < {U} && w < {Wn}) prow[{self.wpos(q, 'u', 'w')}] = (again ? 1.0f : {self.lit(q.unit / SCALE ** 2)}) * dw{q.index}[{j}][i];")
                s.close()

    def emit_redo_dw(self, s: Src, subs):
        """The wave's sums once more with fp32 matrix instructions, on operands straight from memory; no other wave is waited
        for."""
        low = self.low
        _, WW, per = self.split_dw(subs)
        for q in subs:
            a, b2, o = low.in1[q.p.i1], low.in2[q.p.i2], low.out[q.p.io]
            s(" ".join(f"dw{q.index}[{j}] = v4t{{}};" for j in range(per(q))))
            s.open("for (i64 step = begin; step < nsteps; step += gridDim.x)")
            s("#pragma unroll 1")
            s.open("for (int r0 = 0; r0 < 32; r0 += 4)")
            s("const i64 row = min(step * 32 + r0 + lq, num_batch - 1);")
            s(f"const bool there = step * 32 + r0 + lq < num_batch, in = there && 16 * wu + l16 < {a.mul};")
            s(f"const float* xp = L1_in + row * {low.L1} + {a.off} + {a.d} * min(16 * wu + l16, {a.mul - 1});")
            s(f"const float* yp = L2_in + row * {low.L2} + {self.yat(q, 0)};")
            s(f"const float* gp = L3_grad + row * {low.L3} + {o.off};")
            for kk in sorted({k for _, _, k, _ in q.p.nnz}):
                s.open("")
                terms = " + ".join(f"{self.lit(c)} * yp[{j}] * xp[{i}]" for i, j, k, c in q.p.nnz if k == kk)
                s(f"const float av = oeq_sel(in, {terms});")
                for j in range(per(q)):
                    w = f"16 * (ww + {j * WW}) + l16"
                    s(f"dw{q.index}[{j}] = oeq_mfma(av, oeq_sel(there && {w} < {o.mul}, gp[{o.d} * min({w}, {o.mul - 1}) + {kk}]), dw{q.index}[{j}], 0, 0, 0);")
                s.close()
            s.close()
            s.close()
