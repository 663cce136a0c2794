// stencil_ns.hpp -- K2, FP64 null-space path: batched local RBF-FD solves for
// conditionally positive definite splines, 16 or 32 lanes per stencil.
//
// Replaces the same hot loops as stencil_lu.hpp (src/generate_operator.jl:55-65,
// :89-166, method 3 at :388-467; src/hyperviscosity_operator.jl:66-161).
//
// The system  [Phi P; P^T 0] [w; lambda] = [b; p]  needs only w.  Gauss-Jordan
// on the n x NP block P alone, with row pivoting, picks NP nodes (positions
// 0..NP-1 from here on, the others follow) and leaves
//     T = P2 P1^-1   (the other nodes' rows against the picked ones)
// and P1^-1.  The weights with P^T w = p are w = (w0 - T^T y, y) with
// w0 = P1^-T p, and with Z = [-T^T; I] the y solve the N2 x N2 system
//     S y = Z^T (b - Phi w0),   S = Z^T Phi Z,   N2 = n - NP.
// For r^m with m odd and degree >= (m-1)/2, S is definite, so it is inverted
// without pivoting.  One step of refinement on the full residual b - Phi w
// follows; the weights are then as accurate as an LU solve of the whole
// system (both sit at the rounding of Phi itself: median 7.6e-13 against
// 7.6e-13 at n = 31, maximum 2.6e-11 against 2.7e-11, over 1,224 stencils
// against a 113-bit solve; without the step 1.5 to 3 times that).  Where Phi is
// so well conditioned that the residual's own rounding shows, its large part is
// summed exactly (SPLIT).
//
// Why: the solve is bound by VALU issue.  Elimination of the whole system
// takes n + NP dependent steps of pivot search, row publication through LDS
// and broadcasts around its FMAs.  Here only the NP panel steps search and
// publish (rows of NP entries); everything after them is products of small
// matrices whose broadcasts are fused into the FMA (v_fmac_f64_dpp with
// row_newbcast: one instruction per multiply-add, no LDS), since lane k of a
// group holds row k.  About half the multiply-adds remain.
//
// Measured, whole weights calls on 1M stencils, three operators, against the
// Gauss-Jordan kernel: n = 31 3.34 against 7.03 ms, n = 21 2.26 against 4.07 ms;
// six operators at n = 20 2.69 against 4.52 ms (m = 3, SPLIT: 3.34); 262,144
// stencils of n = 31 with 1M output rows 2.08 against 4.51 ms.  A wavefront of four
// stencils issues 4,961 VALU instructions at n = 31 (8,440 there), on 70% of its
// SIMD's cycles; the rest are waits on the panel's LDS round trips and on dependent
// steps of S^-1 that two wavefronts per SIMD do not cover.  n = 13 stays with the
// elimination: 1.16 against 1.17 ms with three operators, 1.66 against 1.33 ms with
// six (its seven unpicked nodes fill less than half of the 16 lanes).
//
// GEN: n at run time, up to the compiled size, with the missing nodes' rows of
// S zero and its pivots not taken; against the eliminations padded to 16, 32, 48
// .. equations 1.4 to 6.5 times as fast (ns_upto in stencil.hip).
//
// What it cannot solve it hands back: a stencil with a panel pivot below
// kNsPanelTol of its column's size (nodes on which the monomials are dependent
// up to rounding), a pivot of S of the wrong sign or below kNsPivotTol of the
// largest, or weights that are not finite goes to a list that the pivoting
// Gauss-Jordan kernel solves afterwards (which also reports singular systems).
//
// A task is one stencil with the output rows that use it (one row, or the
// grouped rows of an X node): after the factorisation each row's right-hand
// sides are solved in chunks of RC operators.  A column sees the same
// operations wherever it sits, so grouped and single rows get the same bits.
#pragma once
#include "stencil_lu.hpp"

namespace rbffd {

// A pivot of S below this share of the largest pivot (or of the wrong sign)
// sends the stencil to the pivoting kernel.  Against a 113-bit solve of 14,472
// stencils of clustered nodes, by that share: above 1e-4 the weights' error is
// 0.87 of an LU solve's of the whole system (geometric mean), 1e-5 to 1e-4
// 0.42, 1e-7 to 1e-6 0.05, below 1e-8 0.01; the refinement step contracts the
// error by 1e-2 or better down to 1e-9 and no longer at 1e-10.  Jittered grids
// reach down to 1e-4 (n = 57) and 7e-3 (n = 13), uniform random nodes to 2e-7.
constexpr double kNsPivotTol = 9.313225746154785e-10;  // 2^-30

// A panel pivot below this share of the bounding box's value of its monomial
// sends the stencil to the pivoting kernel.  Monomials that are dependent on a
// stencil's nodes (as many straight rows of nodes as the degree, along an axis
// or a diagonal) leave a pivot of rounding instead of zero, at most 3.6e-14 over
// degrees 2 to 6; T is noise then, and Dx, which such nodes do determine, comes
// out 8% off in the worst tenth of the rows (four rows of nodes, n = 39, degree
// 4) where the elimination keeps 4e-11.  From pivots of 1e-13 on the weights are
// closer to a 113-bit solve than an LU solve's of the whole system (1e-3 against
// 0.2 there, 1e-6 against 0.1 at 1e-10, level at 1e-3).
constexpr double kNsPanelTol = 9.094947017729282e-13;  // 2^-40

// ---- multiply-adds with a fused broadcast: lane L of each 16-lane DPP row.
// A DPP read needs two wait states after a VALU write of its source; the
// compiler does not see inside the asm, so every block starts with them.
#define RBFFD_FB(d, s, m, l) "v_fmac_f64_dpp %" #d ", %" #s ", %" #m " row_newbcast:%" #l " row_mask:0xf bank_mask:0xf\n\t"

// a_i += s_i(lane L) * m
template <int L>
__device__ __forceinline__ void fb_row(double &a0, double &a1, double &a2, double &a3, double &a4, double &a5,
        double &a6, double &a7, double s0, double s1, double s2, double s3, double s4, double s5, double s6,
        double s7, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 8, 16, 17) RBFFD_FB(1, 9, 16, 17) RBFFD_FB(2, 10, 16, 17) RBFFD_FB(3, 11, 16,
            17) RBFFD_FB(4, 12, 16, 17) RBFFD_FB(5, 13, 16, 17) RBFFD_FB(6, 14, 16, 17) RBFFD_FB(7, 15, 16, 17)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5), "+v"(a6), "+v"(a7)
        : "v"(s0), "v"(s1), "v"(s2), "v"(s3), "v"(s4), "v"(s5), "v"(s6), "v"(s7), "v"(m), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_row(double &a0, double &a1, double &a2, double &a3, double &a4, double &a5,
        double &a6, double s0, double s1, double s2, double s3, double s4, double s5, double s6, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 7, 14, 15) RBFFD_FB(1, 8, 14, 15) RBFFD_FB(2, 9, 14, 15) RBFFD_FB(3, 10, 14, 15)
            RBFFD_FB(4, 11, 14, 15) RBFFD_FB(5, 12, 14, 15) RBFFD_FB(6, 13, 14, 15)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5), "+v"(a6)
        : "v"(s0), "v"(s1), "v"(s2), "v"(s3), "v"(s4), "v"(s5), "v"(s6), "v"(m), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_row(double &a0, double &a1, double &a2, double &a3, double &a4, double &a5,
        double s0, double s1, double s2, double s3, double s4, double s5, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 6, 12, 13) RBFFD_FB(1, 7, 12, 13) RBFFD_FB(2, 8, 12, 13) RBFFD_FB(3, 9, 12, 13)
            RBFFD_FB(4, 10, 12, 13) RBFFD_FB(5, 11, 12, 13)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5)
        : "v"(s0), "v"(s1), "v"(s2), "v"(s3), "v"(s4), "v"(s5), "v"(m), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_row(double &a0, double &a1, double &a2, double &a3, double &a4, double s0,
        double s1, double s2, double s3, double s4, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 5, 10, 11) RBFFD_FB(1, 6, 10, 11) RBFFD_FB(2, 7, 10, 11) RBFFD_FB(3, 8, 10, 11)
            RBFFD_FB(4, 9, 10, 11)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4)
        : "v"(s0), "v"(s1), "v"(s2), "v"(s3), "v"(s4), "v"(m), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_row(double &a0, double &a1, double &a2, double &a3, double s0, double s1,
        double s2, double s3, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 4, 8, 9) RBFFD_FB(1, 5, 8, 9) RBFFD_FB(2, 6, 8, 9) RBFFD_FB(3, 7, 8, 9)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
        : "v"(s0), "v"(s1), "v"(s2), "v"(s3), "v"(m), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_row(double &a0, double &a1, double &a2, double s0, double s1, double s2, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 7) RBFFD_FB(1, 4, 6, 7) RBFFD_FB(2, 5, 6, 7)
        : "+v"(a0), "+v"(a1), "+v"(a2)
        : "v"(s0), "v"(s1), "v"(s2), "v"(m), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_row(double &a0, double &a1, double s0, double s1, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 5) RBFFD_FB(1, 3, 4, 5)
        : "+v"(a0), "+v"(a1)
        : "v"(s0), "v"(s1), "v"(m), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_row(double &a0, double s0, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 3)
        : "+v"(a0)
        : "v"(s0), "v"(m), "i"(L));
}
// a_i += s(lane L_i) * m
template <int L0, int L1, int L2, int L3, int L4, int L5, int L6, int L7>
__device__ __forceinline__ void fb_lane(double &a0, double &a1, double &a2, double &a3, double &a4, double &a5,
        double &a6, double &a7, double s, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 8, 9, 10) RBFFD_FB(1, 8, 9, 11) RBFFD_FB(2, 8, 9, 12) RBFFD_FB(3, 8, 9, 13)
            RBFFD_FB(4, 8, 9, 14) RBFFD_FB(5, 8, 9, 15) RBFFD_FB(6, 8, 9, 16) RBFFD_FB(7, 8, 9, 17)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5), "+v"(a6), "+v"(a7)
        : "v"(s), "v"(m), "i"(L0), "i"(L1), "i"(L2), "i"(L3), "i"(L4), "i"(L5), "i"(L6), "i"(L7));
}
template <int L0, int L1, int L2, int L3, int L4, int L5, int L6>
__device__ __forceinline__ void fb_lane(double &a0, double &a1, double &a2, double &a3, double &a4, double &a5,
        double &a6, double s, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 7, 8, 9) RBFFD_FB(1, 7, 8, 10) RBFFD_FB(2, 7, 8, 11) RBFFD_FB(3, 7, 8, 12)
            RBFFD_FB(4, 7, 8, 13) RBFFD_FB(5, 7, 8, 14) RBFFD_FB(6, 7, 8, 15)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5), "+v"(a6)
        : "v"(s), "v"(m), "i"(L0), "i"(L1), "i"(L2), "i"(L3), "i"(L4), "i"(L5), "i"(L6));
}
template <int L0, int L1, int L2, int L3, int L4, int L5>
__device__ __forceinline__ void fb_lane(double &a0, double &a1, double &a2, double &a3, double &a4, double &a5,
        double s, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 6, 7, 8) RBFFD_FB(1, 6, 7, 9) RBFFD_FB(2, 6, 7, 10) RBFFD_FB(3, 6, 7, 11)
            RBFFD_FB(4, 6, 7, 12) RBFFD_FB(5, 6, 7, 13)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5)
        : "v"(s), "v"(m), "i"(L0), "i"(L1), "i"(L2), "i"(L3), "i"(L4), "i"(L5));
}
template <int L0, int L1, int L2, int L3, int L4>
__device__ __forceinline__ void fb_lane(double &a0, double &a1, double &a2, double &a3, double &a4, double s,
        double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 5, 6, 7) RBFFD_FB(1, 5, 6, 8) RBFFD_FB(2, 5, 6, 9) RBFFD_FB(3, 5, 6, 10)
            RBFFD_FB(4, 5, 6, 11)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4)
        : "v"(s), "v"(m), "i"(L0), "i"(L1), "i"(L2), "i"(L3), "i"(L4));
}
template <int L0, int L1, int L2, int L3>
__device__ __forceinline__ void fb_lane(double &a0, double &a1, double &a2, double &a3, double s, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 4, 5, 6) RBFFD_FB(1, 4, 5, 7) RBFFD_FB(2, 4, 5, 8) RBFFD_FB(3, 4, 5, 9)
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
        : "v"(s), "v"(m), "i"(L0), "i"(L1), "i"(L2), "i"(L3));
}
template <int L0, int L1, int L2>
__device__ __forceinline__ void fb_lane(double &a0, double &a1, double &a2, double s, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 4, 5) RBFFD_FB(1, 3, 4, 6) RBFFD_FB(2, 3, 4, 7)
        : "+v"(a0), "+v"(a1), "+v"(a2)
        : "v"(s), "v"(m), "i"(L0), "i"(L1), "i"(L2));
}
template <int L0, int L1>
__device__ __forceinline__ void fb_lane(double &a0, double &a1, double s, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 3, 4) RBFFD_FB(1, 2, 3, 5)
        : "+v"(a0), "+v"(a1)
        : "v"(s), "v"(m), "i"(L0), "i"(L1));
}
template <int L0>
__device__ __forceinline__ void fb_lane(double &a0, double s, double m)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 3)
        : "+v"(a0)
        : "v"(s), "v"(m), "i"(L0));
}
// a_o += sum over i of s_o(lane L + i) * m_i, the columns interleaved
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[1], const double (&s)[1], double m0, double m1, double m2,
        double m3, double m4, double m5, double m6, double m7)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 10) RBFFD_FB(0, 1, 3, 11) RBFFD_FB(0, 1, 4, 12) RBFFD_FB(0, 1, 5, 13)
            RBFFD_FB(0, 1, 6, 14) RBFFD_FB(0, 1, 7, 15) RBFFD_FB(0, 1, 8, 16) RBFFD_FB(0, 1, 9, 17)
        : "+v"(a[0])
        : "v"(s[0]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "v"(m6), "v"(m7), "i"(L), "i"(L + 1),
                "i"(L + 2), "i"(L + 3), "i"(L + 4), "i"(L + 5), "i"(L + 6), "i"(L + 7));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[1], const double (&s)[1], double m0, double m1, double m2,
        double m3, double m4, double m5, double m6)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 9) RBFFD_FB(0, 1, 3, 10) RBFFD_FB(0, 1, 4, 11) RBFFD_FB(0, 1, 5, 12)
            RBFFD_FB(0, 1, 6, 13) RBFFD_FB(0, 1, 7, 14) RBFFD_FB(0, 1, 8, 15)
        : "+v"(a[0])
        : "v"(s[0]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "v"(m6), "i"(L), "i"(L + 1), "i"(L + 2),
                "i"(L + 3), "i"(L + 4), "i"(L + 5), "i"(L + 6));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[1], const double (&s)[1], double m0, double m1, double m2,
        double m3, double m4, double m5)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 8) RBFFD_FB(0, 1, 3, 9) RBFFD_FB(0, 1, 4, 10) RBFFD_FB(0, 1, 5, 11)
            RBFFD_FB(0, 1, 6, 12) RBFFD_FB(0, 1, 7, 13)
        : "+v"(a[0])
        : "v"(s[0]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "i"(L), "i"(L + 1), "i"(L + 2),
                "i"(L + 3), "i"(L + 4), "i"(L + 5));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[1], const double (&s)[1], double m0, double m1, double m2,
        double m3, double m4)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 7) RBFFD_FB(0, 1, 3, 8) RBFFD_FB(0, 1, 4, 9) RBFFD_FB(0, 1, 5, 10)
            RBFFD_FB(0, 1, 6, 11)
        : "+v"(a[0])
        : "v"(s[0]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "i"(L), "i"(L + 1), "i"(L + 2), "i"(L + 3),
                "i"(L + 4));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[1], const double (&s)[1], double m0, double m1, double m2,
        double m3)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 6) RBFFD_FB(0, 1, 3, 7) RBFFD_FB(0, 1, 4, 8) RBFFD_FB(0, 1, 5, 9)
        : "+v"(a[0])
        : "v"(s[0]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "i"(L), "i"(L + 1), "i"(L + 2), "i"(L + 3));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[1], const double (&s)[1], double m0, double m1, double m2)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 5) RBFFD_FB(0, 1, 3, 6) RBFFD_FB(0, 1, 4, 7)
        : "+v"(a[0])
        : "v"(s[0]), "v"(m0), "v"(m1), "v"(m2), "i"(L), "i"(L + 1), "i"(L + 2));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[1], const double (&s)[1], double m0, double m1)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 4) RBFFD_FB(0, 1, 3, 5)
        : "+v"(a[0])
        : "v"(s[0]), "v"(m0), "v"(m1), "i"(L), "i"(L + 1));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[1], const double (&s)[1], double m0)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 1, 2, 3)
        : "+v"(a[0])
        : "v"(s[0]), "v"(m0), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[2], const double (&s)[2], double m0, double m1, double m2,
        double m3, double m4, double m5, double m6, double m7)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 12) RBFFD_FB(1, 3, 4, 12) RBFFD_FB(0, 2, 5, 13) RBFFD_FB(1, 3, 5, 13)
            RBFFD_FB(0, 2, 6, 14) RBFFD_FB(1, 3, 6, 14) RBFFD_FB(0, 2, 7, 15) RBFFD_FB(1, 3, 7, 15) RBFFD_FB(0, 2,
            8, 16) RBFFD_FB(1, 3, 8, 16) RBFFD_FB(0, 2, 9, 17) RBFFD_FB(1, 3, 9, 17) RBFFD_FB(0, 2, 10, 18)
            RBFFD_FB(1, 3, 10, 18) RBFFD_FB(0, 2, 11, 19) RBFFD_FB(1, 3, 11, 19)
        : "+v"(a[0]), "+v"(a[1])
        : "v"(s[0]), "v"(s[1]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "v"(m6), "v"(m7), "i"(L),
                "i"(L + 1), "i"(L + 2), "i"(L + 3), "i"(L + 4), "i"(L + 5), "i"(L + 6), "i"(L + 7));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[2], const double (&s)[2], double m0, double m1, double m2,
        double m3, double m4, double m5, double m6)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 11) RBFFD_FB(1, 3, 4, 11) RBFFD_FB(0, 2, 5, 12) RBFFD_FB(1, 3, 5, 12)
            RBFFD_FB(0, 2, 6, 13) RBFFD_FB(1, 3, 6, 13) RBFFD_FB(0, 2, 7, 14) RBFFD_FB(1, 3, 7, 14) RBFFD_FB(0, 2,
            8, 15) RBFFD_FB(1, 3, 8, 15) RBFFD_FB(0, 2, 9, 16) RBFFD_FB(1, 3, 9, 16) RBFFD_FB(0, 2, 10, 17)
            RBFFD_FB(1, 3, 10, 17)
        : "+v"(a[0]), "+v"(a[1])
        : "v"(s[0]), "v"(s[1]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "v"(m6), "i"(L), "i"(L + 1),
                "i"(L + 2), "i"(L + 3), "i"(L + 4), "i"(L + 5), "i"(L + 6));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[2], const double (&s)[2], double m0, double m1, double m2,
        double m3, double m4, double m5)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 10) RBFFD_FB(1, 3, 4, 10) RBFFD_FB(0, 2, 5, 11) RBFFD_FB(1, 3, 5, 11)
            RBFFD_FB(0, 2, 6, 12) RBFFD_FB(1, 3, 6, 12) RBFFD_FB(0, 2, 7, 13) RBFFD_FB(1, 3, 7, 13) RBFFD_FB(0, 2,
            8, 14) RBFFD_FB(1, 3, 8, 14) RBFFD_FB(0, 2, 9, 15) RBFFD_FB(1, 3, 9, 15)
        : "+v"(a[0]), "+v"(a[1])
        : "v"(s[0]), "v"(s[1]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "i"(L), "i"(L + 1),
                "i"(L + 2), "i"(L + 3), "i"(L + 4), "i"(L + 5));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[2], const double (&s)[2], double m0, double m1, double m2,
        double m3, double m4)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 9) RBFFD_FB(1, 3, 4, 9) RBFFD_FB(0, 2, 5, 10) RBFFD_FB(1, 3, 5, 10)
            RBFFD_FB(0, 2, 6, 11) RBFFD_FB(1, 3, 6, 11) RBFFD_FB(0, 2, 7, 12) RBFFD_FB(1, 3, 7, 12) RBFFD_FB(0, 2,
            8, 13) RBFFD_FB(1, 3, 8, 13)
        : "+v"(a[0]), "+v"(a[1])
        : "v"(s[0]), "v"(s[1]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "i"(L), "i"(L + 1), "i"(L + 2),
                "i"(L + 3), "i"(L + 4));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[2], const double (&s)[2], double m0, double m1, double m2,
        double m3)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 8) RBFFD_FB(1, 3, 4, 8) RBFFD_FB(0, 2, 5, 9) RBFFD_FB(1, 3, 5, 9)
            RBFFD_FB(0, 2, 6, 10) RBFFD_FB(1, 3, 6, 10) RBFFD_FB(0, 2, 7, 11) RBFFD_FB(1, 3, 7, 11)
        : "+v"(a[0]), "+v"(a[1])
        : "v"(s[0]), "v"(s[1]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "i"(L), "i"(L + 1), "i"(L + 2), "i"(L + 3));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[2], const double (&s)[2], double m0, double m1, double m2)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 7) RBFFD_FB(1, 3, 4, 7) RBFFD_FB(0, 2, 5, 8) RBFFD_FB(1, 3, 5, 8)
            RBFFD_FB(0, 2, 6, 9) RBFFD_FB(1, 3, 6, 9)
        : "+v"(a[0]), "+v"(a[1])
        : "v"(s[0]), "v"(s[1]), "v"(m0), "v"(m1), "v"(m2), "i"(L), "i"(L + 1), "i"(L + 2));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[2], const double (&s)[2], double m0, double m1)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 6) RBFFD_FB(1, 3, 4, 6) RBFFD_FB(0, 2, 5, 7) RBFFD_FB(1, 3, 5, 7)
        : "+v"(a[0]), "+v"(a[1])
        : "v"(s[0]), "v"(s[1]), "v"(m0), "v"(m1), "i"(L), "i"(L + 1));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[2], const double (&s)[2], double m0)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 2, 4, 5) RBFFD_FB(1, 3, 4, 5)
        : "+v"(a[0]), "+v"(a[1])
        : "v"(s[0]), "v"(s[1]), "v"(m0), "i"(L));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[3], const double (&s)[3], double m0, double m1, double m2,
        double m3, double m4, double m5, double m6, double m7)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 14) RBFFD_FB(1, 4, 6, 14) RBFFD_FB(2, 5, 6, 14) RBFFD_FB(0, 3, 7, 15)
            RBFFD_FB(1, 4, 7, 15) RBFFD_FB(2, 5, 7, 15) RBFFD_FB(0, 3, 8, 16) RBFFD_FB(1, 4, 8, 16) RBFFD_FB(2, 5,
            8, 16) RBFFD_FB(0, 3, 9, 17) RBFFD_FB(1, 4, 9, 17) RBFFD_FB(2, 5, 9, 17) RBFFD_FB(0, 3, 10, 18)
            RBFFD_FB(1, 4, 10, 18) RBFFD_FB(2, 5, 10, 18) RBFFD_FB(0, 3, 11, 19) RBFFD_FB(1, 4, 11, 19) RBFFD_FB(2,
            5, 11, 19) RBFFD_FB(0, 3, 12, 20) RBFFD_FB(1, 4, 12, 20) RBFFD_FB(2, 5, 12, 20) RBFFD_FB(0, 3, 13, 21)
            RBFFD_FB(1, 4, 13, 21) RBFFD_FB(2, 5, 13, 21)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "v"(m6), "v"(m7),
                "i"(L), "i"(L + 1), "i"(L + 2), "i"(L + 3), "i"(L + 4), "i"(L + 5), "i"(L + 6), "i"(L + 7));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[3], const double (&s)[3], double m0, double m1, double m2,
        double m3, double m4, double m5, double m6)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 13) RBFFD_FB(1, 4, 6, 13) RBFFD_FB(2, 5, 6, 13) RBFFD_FB(0, 3, 7, 14)
            RBFFD_FB(1, 4, 7, 14) RBFFD_FB(2, 5, 7, 14) RBFFD_FB(0, 3, 8, 15) RBFFD_FB(1, 4, 8, 15) RBFFD_FB(2, 5,
            8, 15) RBFFD_FB(0, 3, 9, 16) RBFFD_FB(1, 4, 9, 16) RBFFD_FB(2, 5, 9, 16) RBFFD_FB(0, 3, 10, 17)
            RBFFD_FB(1, 4, 10, 17) RBFFD_FB(2, 5, 10, 17) RBFFD_FB(0, 3, 11, 18) RBFFD_FB(1, 4, 11, 18) RBFFD_FB(2,
            5, 11, 18) RBFFD_FB(0, 3, 12, 19) RBFFD_FB(1, 4, 12, 19) RBFFD_FB(2, 5, 12, 19)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "v"(m6), "i"(L),
                "i"(L + 1), "i"(L + 2), "i"(L + 3), "i"(L + 4), "i"(L + 5), "i"(L + 6));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[3], const double (&s)[3], double m0, double m1, double m2,
        double m3, double m4, double m5)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 12) RBFFD_FB(1, 4, 6, 12) RBFFD_FB(2, 5, 6, 12) RBFFD_FB(0, 3, 7, 13)
            RBFFD_FB(1, 4, 7, 13) RBFFD_FB(2, 5, 7, 13) RBFFD_FB(0, 3, 8, 14) RBFFD_FB(1, 4, 8, 14) RBFFD_FB(2, 5,
            8, 14) RBFFD_FB(0, 3, 9, 15) RBFFD_FB(1, 4, 9, 15) RBFFD_FB(2, 5, 9, 15) RBFFD_FB(0, 3, 10, 16)
            RBFFD_FB(1, 4, 10, 16) RBFFD_FB(2, 5, 10, 16) RBFFD_FB(0, 3, 11, 17) RBFFD_FB(1, 4, 11, 17) RBFFD_FB(2,
            5, 11, 17)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "v"(m5), "i"(L), "i"(L + 1),
                "i"(L + 2), "i"(L + 3), "i"(L + 4), "i"(L + 5));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[3], const double (&s)[3], double m0, double m1, double m2,
        double m3, double m4)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 11) RBFFD_FB(1, 4, 6, 11) RBFFD_FB(2, 5, 6, 11) RBFFD_FB(0, 3, 7, 12)
            RBFFD_FB(1, 4, 7, 12) RBFFD_FB(2, 5, 7, 12) RBFFD_FB(0, 3, 8, 13) RBFFD_FB(1, 4, 8, 13) RBFFD_FB(2, 5,
            8, 13) RBFFD_FB(0, 3, 9, 14) RBFFD_FB(1, 4, 9, 14) RBFFD_FB(2, 5, 9, 14) RBFFD_FB(0, 3, 10, 15)
            RBFFD_FB(1, 4, 10, 15) RBFFD_FB(2, 5, 10, 15)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "v"(m4), "i"(L), "i"(L + 1),
                "i"(L + 2), "i"(L + 3), "i"(L + 4));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[3], const double (&s)[3], double m0, double m1, double m2,
        double m3)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 10) RBFFD_FB(1, 4, 6, 10) RBFFD_FB(2, 5, 6, 10) RBFFD_FB(0, 3, 7, 11)
            RBFFD_FB(1, 4, 7, 11) RBFFD_FB(2, 5, 7, 11) RBFFD_FB(0, 3, 8, 12) RBFFD_FB(1, 4, 8, 12) RBFFD_FB(2, 5,
            8, 12) RBFFD_FB(0, 3, 9, 13) RBFFD_FB(1, 4, 9, 13) RBFFD_FB(2, 5, 9, 13)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(m0), "v"(m1), "v"(m2), "v"(m3), "i"(L), "i"(L + 1), "i"(L + 2),
                "i"(L + 3));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[3], const double (&s)[3], double m0, double m1, double m2)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 9) RBFFD_FB(1, 4, 6, 9) RBFFD_FB(2, 5, 6, 9) RBFFD_FB(0, 3, 7, 10)
            RBFFD_FB(1, 4, 7, 10) RBFFD_FB(2, 5, 7, 10) RBFFD_FB(0, 3, 8, 11) RBFFD_FB(1, 4, 8, 11) RBFFD_FB(2, 5,
            8, 11)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(m0), "v"(m1), "v"(m2), "i"(L), "i"(L + 1), "i"(L + 2));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[3], const double (&s)[3], double m0, double m1)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 8) RBFFD_FB(1, 4, 6, 8) RBFFD_FB(2, 5, 6, 8) RBFFD_FB(0, 3, 7, 9)
            RBFFD_FB(1, 4, 7, 9) RBFFD_FB(2, 5, 7, 9)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(m0), "v"(m1), "i"(L), "i"(L + 1));
}
template <int L>
__device__ __forceinline__ void fb_dot(double (&a)[3], const double (&s)[3], double m0)
{
    asm("s_nop 1\n\t" RBFFD_FB(0, 3, 6, 7) RBFFD_FB(1, 4, 6, 7) RBFFD_FB(2, 5, 6, 7)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
        : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(m0), "i"(L));
}

// a[j] += s[j](lane L) * m for CNT columns j = J, J + 1, ... (mod W)
template <int L, int J, int CNT, int W>
__device__ __forceinline__ void fb_cols(double (&a)[W], const double (&s)[W], double m)
{
    if constexpr (CNT > 8) {
        fb_cols<L, J, 8>(a, s, m);
        fb_cols<L, J + 8, CNT - 8>(a, s, m);
    } else if constexpr (CNT == 8)
        fb_row<L>(a[(J + 0) % W], a[(J + 1) % W], a[(J + 2) % W], a[(J + 3) % W], a[(J + 4) % W], a[(J + 5) % W],
                a[(J + 6) % W], a[(J + 7) % W], s[(J + 0) % W], s[(J + 1) % W], s[(J + 2) % W], s[(J + 3) % W],
                s[(J + 4) % W], s[(J + 5) % W], s[(J + 6) % W], s[(J + 7) % W], m);
    else if constexpr (CNT == 7)
        fb_row<L>(a[(J + 0) % W], a[(J + 1) % W], a[(J + 2) % W], a[(J + 3) % W], a[(J + 4) % W], a[(J + 5) % W],
                a[(J + 6) % W], s[(J + 0) % W], s[(J + 1) % W], s[(J + 2) % W], s[(J + 3) % W], s[(J + 4) % W],
                s[(J + 5) % W], s[(J + 6) % W], m);
    else if constexpr (CNT == 6)
        fb_row<L>(a[(J + 0) % W], a[(J + 1) % W], a[(J + 2) % W], a[(J + 3) % W], a[(J + 4) % W], a[(J + 5) % W],
                s[(J + 0) % W], s[(J + 1) % W], s[(J + 2) % W], s[(J + 3) % W], s[(J + 4) % W], s[(J + 5) % W], m);
    else if constexpr (CNT == 5)
        fb_row<L>(a[(J + 0) % W], a[(J + 1) % W], a[(J + 2) % W], a[(J + 3) % W], a[(J + 4) % W], s[(J + 0) % W],
                s[(J + 1) % W], s[(J + 2) % W], s[(J + 3) % W], s[(J + 4) % W], m);
    else if constexpr (CNT == 4)
        fb_row<L>(a[(J + 0) % W], a[(J + 1) % W], a[(J + 2) % W], a[(J + 3) % W], s[(J + 0) % W], s[(J + 1) % W],
                s[(J + 2) % W], s[(J + 3) % W], m);
    else if constexpr (CNT == 3)
        fb_row<L>(a[(J + 0) % W], a[(J + 1) % W], a[(J + 2) % W], s[(J + 0) % W], s[(J + 1) % W], s[(J + 2) % W], m);
    else if constexpr (CNT == 2)
        fb_row<L>(a[(J + 0) % W], a[(J + 1) % W], s[(J + 0) % W], s[(J + 1) % W], m);
    else if constexpr (CNT == 1)
        fb_row<L>(a[(J + 0) % W], s[(J + 0) % W], m);
}
// a[JA + i] += s[JS + i](lane L) * m for i < CNT
template <int L, int JA, int JS, int CNT, int WA, int WS>
__device__ __forceinline__ void fb_sub(double (&a)[WA], const double (&s)[WS], double m)
{
    if constexpr (CNT > 8) {
        fb_sub<L, JA, JS, 8>(a, s, m);
        fb_sub<L, JA + 8, JS + 8, CNT - 8>(a, s, m);
    } else if constexpr (CNT == 8)
        fb_row<L>(a[JA + 0], a[JA + 1], a[JA + 2], a[JA + 3], a[JA + 4], a[JA + 5], a[JA + 6], a[JA + 7], s[JS + 0],
                s[JS + 1], s[JS + 2], s[JS + 3], s[JS + 4], s[JS + 5], s[JS + 6], s[JS + 7], m);
    else if constexpr (CNT == 7)
        fb_row<L>(a[JA + 0], a[JA + 1], a[JA + 2], a[JA + 3], a[JA + 4], a[JA + 5], a[JA + 6], s[JS + 0], s[JS + 1],
                s[JS + 2], s[JS + 3], s[JS + 4], s[JS + 5], s[JS + 6], m);
    else if constexpr (CNT == 6)
        fb_row<L>(a[JA + 0], a[JA + 1], a[JA + 2], a[JA + 3], a[JA + 4], a[JA + 5], s[JS + 0], s[JS + 1], s[JS + 2],
                s[JS + 3], s[JS + 4], s[JS + 5], m);
    else if constexpr (CNT == 5)
        fb_row<L>(a[JA + 0], a[JA + 1], a[JA + 2], a[JA + 3], a[JA + 4], s[JS + 0], s[JS + 1], s[JS + 2], s[JS + 3],
                s[JS + 4], m);
    else if constexpr (CNT == 4)
        fb_row<L>(a[JA + 0], a[JA + 1], a[JA + 2], a[JA + 3], s[JS + 0], s[JS + 1], s[JS + 2], s[JS + 3], m);
    else if constexpr (CNT == 3)
        fb_row<L>(a[JA + 0], a[JA + 1], a[JA + 2], s[JS + 0], s[JS + 1], s[JS + 2], m);
    else if constexpr (CNT == 2)
        fb_row<L>(a[JA + 0], a[JA + 1], s[JS + 0], s[JS + 1], m);
    else if constexpr (CNT == 1)
        fb_row<L>(a[JA + 0], s[JS + 0], m);
}
// a[j] += s[j / 16](lane j % 16) * m for CNT columns j = J, J + 1, ... (mod W);
// one asm block stays inside one 16-column slot of s
template <int J, int CNT, int W, int NB>
__device__ __forceinline__ void fb_lanes(double (&a)[W], const double (&s)[NB], double m)
{
    if constexpr (CNT > 0) {
        constexpr int j0 = J % W, sl = j0 / 16;
        // columns up to the next slot or the wrap (with one slot the wrap may sit inside a block)
        constexpr int room = NB == 1 ? CNT : ((16 * sl + 16 < W ? 16 * sl + 16 : W) - j0);
        constexpr int run = CNT < room ? CNT : room;
        constexpr int n = run < 8 ? run : 8;
#define RBFFD_L(i) (((J + i) % W) % 16)
#define RBFFD_A(i) a[(J + i) % W]
        if constexpr (n == 8)
            fb_lane<RBFFD_L(0), RBFFD_L(1), RBFFD_L(2), RBFFD_L(3), RBFFD_L(4), RBFFD_L(5), RBFFD_L(6),
                    RBFFD_L(7)>(RBFFD_A(0), RBFFD_A(1), RBFFD_A(2), RBFFD_A(3), RBFFD_A(4), RBFFD_A(5), RBFFD_A(6),
                    RBFFD_A(7), s[sl], m);
        else if constexpr (n == 7)
            fb_lane<RBFFD_L(0), RBFFD_L(1), RBFFD_L(2), RBFFD_L(3), RBFFD_L(4), RBFFD_L(5), RBFFD_L(6)>(RBFFD_A(0),
                    RBFFD_A(1), RBFFD_A(2), RBFFD_A(3), RBFFD_A(4), RBFFD_A(5), RBFFD_A(6), s[sl], m);
        else if constexpr (n == 6)
            fb_lane<RBFFD_L(0), RBFFD_L(1), RBFFD_L(2), RBFFD_L(3), RBFFD_L(4), RBFFD_L(5)>(RBFFD_A(0), RBFFD_A(1),
                    RBFFD_A(2), RBFFD_A(3), RBFFD_A(4), RBFFD_A(5), s[sl], m);
        else if constexpr (n == 5)
            fb_lane<RBFFD_L(0), RBFFD_L(1), RBFFD_L(2), RBFFD_L(3), RBFFD_L(4)>(RBFFD_A(0), RBFFD_A(1), RBFFD_A(2),
                    RBFFD_A(3), RBFFD_A(4), s[sl], m);
        else if constexpr (n == 4)
            fb_lane<RBFFD_L(0), RBFFD_L(1), RBFFD_L(2), RBFFD_L(3)>(RBFFD_A(0), RBFFD_A(1), RBFFD_A(2), RBFFD_A(3),
                    s[sl], m);
        else if constexpr (n == 3)
            fb_lane<RBFFD_L(0), RBFFD_L(1), RBFFD_L(2)>(RBFFD_A(0), RBFFD_A(1), RBFFD_A(2), s[sl], m);
        else if constexpr (n == 2)
            fb_lane<RBFFD_L(0), RBFFD_L(1)>(RBFFD_A(0), RBFFD_A(1), s[sl], m);
        else if constexpr (n == 1)
            fb_lane<RBFFD_L(0)>(RBFFD_A(0), s[sl], m);
#undef RBFFD_L
#undef RBFFD_A
        fb_lanes<J + n, CNT - n>(a, s, m);
    }
}
// a[o] += sum over k in K0..K1-1 of s[k / 16][o](lane k % 16) * m[k]
template <int K0, int K1, int RC, int NB, int W>
__device__ __forceinline__ void fb_sum(double (&a)[RC], const double (&s)[NB][RC], const double (&m)[W])
{
    if constexpr (K1 > K0) {
        constexpr int sl = K0 / 16, l = K0 % 16;
        constexpr int run = K1 - K0 < 16 - l ? K1 - K0 : 16 - l;
        constexpr int n = run < 8 ? run : 8;
        if constexpr (n == 8)
            fb_dot<l>(a, s[sl], m[K0], m[K0 + 1], m[K0 + 2], m[K0 + 3], m[K0 + 4], m[K0 + 5], m[K0 + 6], m[K0 + 7]);
        else if constexpr (n == 7)
            fb_dot<l>(a, s[sl], m[K0], m[K0 + 1], m[K0 + 2], m[K0 + 3], m[K0 + 4], m[K0 + 5], m[K0 + 6]);
        else if constexpr (n == 6)
            fb_dot<l>(a, s[sl], m[K0], m[K0 + 1], m[K0 + 2], m[K0 + 3], m[K0 + 4], m[K0 + 5]);
        else if constexpr (n == 5)
            fb_dot<l>(a, s[sl], m[K0], m[K0 + 1], m[K0 + 2], m[K0 + 3], m[K0 + 4]);
        else if constexpr (n == 4)
            fb_dot<l>(a, s[sl], m[K0], m[K0 + 1], m[K0 + 2], m[K0 + 3]);
        else if constexpr (n == 3)
            fb_dot<l>(a, s[sl], m[K0], m[K0 + 1], m[K0 + 2]);
        else if constexpr (n == 2)
            fb_dot<l>(a, s[sl], m[K0], m[K0 + 1]);
        else if constexpr (n == 1)
            fb_dot<l>(a, s[sl], m[K0]);
        fb_sum<K0 + n, K1>(a, s, m);
    }
}

// The same sum in two chains: the residual's rounding shows in the weights
template <int K1, int RC, int NB, int W>
__device__ __forceinline__ void fb_sum2(double (&a)[RC], const double (&s)[NB][RC], const double (&m)[W])
{
    double h[2][RC];
#pragma unroll
    for (int o = 0; o < RC; ++o) h[0][o] = h[1][o] = 0.0;
    fb_sum<0, K1 / 2>(h[0], s, m);
    fb_sum<K1 / 2, K1>(h[1], s, m);
#pragma unroll
    for (int o = 0; o < RC; ++o) a[o] += h[0][o] + h[1][o];
}

// a[o] += sum over i < n of s[o](lane L + i) * m[i]
template <int L, int RC, int n>
__device__ __forceinline__ void fb_run(double (&a)[RC], const double (&s)[RC], const double (&m)[n])
{
    static_assert(n <= 8, "run");
    if constexpr (n == 8) fb_dot<L>(a, s, m[0], m[1], m[2], m[3], m[4], m[5], m[6], m[7]);
    else if constexpr (n == 7) fb_dot<L>(a, s, m[0], m[1], m[2], m[3], m[4], m[5], m[6]);
    else if constexpr (n == 6) fb_dot<L>(a, s, m[0], m[1], m[2], m[3], m[4], m[5]);
    else if constexpr (n == 5) fb_dot<L>(a, s, m[0], m[1], m[2], m[3], m[4]);
    else if constexpr (n == 4) fb_dot<L>(a, s, m[0], m[1], m[2], m[3]);
    else if constexpr (n == 3) fb_dot<L>(a, s, m[0], m[1], m[2]);
    else if constexpr (n == 2) fb_dot<L>(a, s, m[0], m[1]);
    else fb_dot<L>(a, s, m[0]);
}

// sum over k in K0..K1-1 of (sh + sl)[k / 16][o](lane k % 16) * load(k) in two
// parts: the products of the upper halves, which a1 adds up without rounding,
// and the others, 2^-23 of them, in a2.  c splits the loaded factors (split_at).
template <int K0, int K1, int RC, int NB, class Load>
__device__ __forceinline__ void fb_sum_split(double (&a1)[RC], double (&a2)[RC], const double (&sh)[NB][RC],
                                             const double (&sl)[NB][RC], double c, Load &&load)
{
    if constexpr (K1 > K0) {
        constexpr int l = K0 % 16, left = K1 - K0 < 16 - l ? K1 - K0 : 16 - l, n = left < 8 ? left : 8;
        double f[n], h[n];
        for_blocks<0, n>([&](auto ic) { f[decltype(ic)::value] = load(std::integral_constant<int, K0 + decltype(ic)::value>{}); });
        fb_run<l>(a2, sl[K0 / 16], f);
#pragma unroll
        for (int i = 0; i < n; ++i) {
            h[i] = (f[i] + c) - c;
            f[i] -= h[i];
        }
        fb_run<l>(a1, sh[K0 / 16], h);
        fb_run<l>(a2, sh[K0 / 16], f);
        fb_sum_split<K0 + n, K1>(a1, a2, sh, sl, c, load);
    }
}

// (v + split_at(e)) - split_at(e) is v rounded to a multiple of 2^(e - 23), for
// |v| <= 2^e.  Products of two such halves are multiples of 2^(e + e' - 46) of at
// most 2^(e + e'), so sums of up to 64 of them are exact in 53 bits.
__device__ __forceinline__ double split_at(int e)
{
    return __longlong_as_double((long long)((uint64_t)(uint32_t)(1023 + 29 + e) << 52 | 0x0008000000000000ull));
}

__device__ __forceinline__ uint32_t lds_address(const void *p)
{
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

// Two doubles to slots I and J of a row in LDS.  Written out because the
// compiler makes ds_write_b128 of neighbouring stores, whose data must first be
// moved into four consecutive registers (382 moves in the panel at n = 31);
// this takes each from where it is.  A store needs no wait of its own: LDS
// serves a wavefront in order, and the compiler's counts for the reads behind
// it only get more cautious.
template <int I, int J>
__device__ __forceinline__ void lds_write2(uint32_t a, double x, double y)
{
    asm volatile("ds_write2_b64 %0, %1, %2 offset0:%3 offset1:%4" ::"v"(a), "v"(x), "v"(y), "i"(I), "i"(J) : "memory");
}

// v with its high word replaced by hi where c holds
__device__ __forceinline__ double hi_if(double v, bool c, uint32_t hi)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t h = c ? hi : (uint32_t)(b >> 32);
    return __longlong_as_double((long long)(((uint64_t)h << 32) | (uint32_t)b));
}

// whether row S of this lane, (lane mod G) + G S, is at most c: a lane mask known
// at compile time
template <int G, int S>
__device__ __forceinline__ bool upto(int c)
{
    const int e = c - G * S;
    const uint64_t m = e < 0 ? 0ull : (2ull << (e >= G ? G - 1 : e)) - 1ull;
    return __builtin_amdgcn_inverse_ballot_w64(m * (G == 16 ? 0x0001000100010001ull : 0x0000000100000001ull));
}

// A lane swap needs two wait states after a VALU write of its sources, which the
// compiler provides for its own writes only: a value that may come from an asm
// block passes through here first.
__device__ __forceinline__ double settled(double v)
{
    asm("s_nop 1" : "+v"(v));
    return v;
}

// Per-lane rows as broadcast sources: src[b] holds, in every 16-lane DPP row of
// a group, rows 16 b .. 16 b + 15.  With 16 lanes these are the lane's own row
// slots; with 32, v_permlane16_swap gives both halves to both DPP rows.
template <int G, int S, int R>
__device__ __forceinline__ void spread(const double (&own)[S], double (&src)[R])
{
    if constexpr (G == 16) {
        static_assert(S == R, "row slots");
#pragma unroll
        for (int b = 0; b < R; ++b) src[b] = own[b];
    } else {
        static_assert(S == 1 && R <= 2, "row slots");
        const uint64_t v = (uint64_t)__double_as_longlong(settled(own[0]));
        const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
#pragma unroll
        for (int b = 0; b < R; ++b)
            src[b] = __longlong_as_double((long long)(((uint64_t)(uint32_t)hi[b] << 32) | (uint32_t)lo[b]));
    }
}
// x's odd 16-lane rows exchanged with y's even ones (v_permlane16_swap)
__device__ __forceinline__ void swap_rows(double x, double y, double &p, double &q)
{
    asm("s_nop 1" : "+v"(x), "+v"(y));  // as settled
    const uint64_t a = (uint64_t)__double_as_longlong(x), b = (uint64_t)__double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)a, (uint32_t)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(a >> 32), (uint32_t)(b >> 32), false, false);
    p = __longlong_as_double((long long)(((uint64_t)(uint32_t)hi[0] << 32) | (uint32_t)lo[0]));
    q = __longlong_as_double((long long)(((uint64_t)(uint32_t)hi[1] << 32) | (uint32_t)lo[1]));
}
template <int G, int S, int R, int RC>
__device__ __forceinline__ void spread(const double (&own)[S][RC], double (&src)[R][RC])
{
#pragma unroll
    for (int o = 0; o < RC; ++o) {
        double a[S], b[R];
#pragma unroll
        for (int i = 0; i < S; ++i) a[i] = own[i][o];
        spread<G>(a, b);
#pragma unroll
        for (int i = 0; i < R; ++i) src[i][o] = b[i];
    }
}

// the high word of |v|
__device__ __forceinline__ uint32_t high_abs(double v)
{
    return (uint32_t)((uint64_t)__double_as_longlong(v) >> 32) & 0x7FFFFFFFu;
}

// 1 / x to within an ulp (x finite and not zero): the instruction gives 23
// bits, one cubic step the rest
__device__ __forceinline__ double rcp_nr(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// sqrt(x) for x >= 2^-700: Goldschmidt's coupled iteration from the 1 / sqrt(x)
// estimate (g -> sqrt(x), h -> 1 / (2 sqrt(x))), then two steps on the residual
// x - g^2.  Smaller arguments are not scaled first (7 instructions fewer); x = 0
// gives NaN, so a duplicated node fails the finiteness check
__device__ __forceinline__ double ns_sqrt(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(g, r, g);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// Powers of r = |v| at one point for the closed-form operators.
struct NsPhsAt {
    double r2, r, rm2, rm4;  // r^2, r, r^(m-2), r^(m-4)
};

__device__ __forceinline__ NsPhsAt ns_phs_at(int m, double vx, double vy)
{
    NsPhsAt q;
    q.r2 = sq_sum(vx, vy);
    q.r = ns_sqrt(q.r2);
    if (m >= 5) {  // uniform
        q.rm4 = upow(q.r2, (m - 5) >> 1) * q.r;
        q.rm2 = q.rm4 * q.r2;
    } else {
        q.rm2 = m == 3 ? q.r : q.r / q.r2;
        q.rm4 = q.rm2 / q.r2;
    }
    return q;
}

// Operator applied to the PHS (m odd): closed forms; for the pure k-th
// derivatives the chain rule over t -> t^2 + const,
//   t^(k mod 2) r^(m-2k) sum_i c[i] (t^2)^(h-i) (r^2)^i,   h = k / 2,
// with the constants c precomputed by the host.
template <class C>
__device__ __forceinline__ double ns_op_phs(int op, int k, int m, const C &c, double vx, double vy, double sx,
                                            double sy, const NsPhsAt &q)
{
    // no contraction: a column's bits do not depend on the code around it
#pragma clang fp contract(off)
    if (op == OP_E) return upow(q.r2, m >> 1) * q.r;
    const double dm = (double)m;
    switch (op) {
    case OP_DX:  return dm * vx * q.rm2;
    case OP_DY:  return dm * vy * q.rm2;
    case OP_DXX: return dm * q.rm2 + dm * (dm - 2.0) * vx * vx * q.rm4;
    case OP_DYY: return dm * q.rm2 + dm * (dm - 2.0) * vy * vy * q.rm4;
    case OP_DXY: return dm * (dm - 2.0) * vx * vy * q.rm4;
    case OP_LAP: {
        const double fxx = dm * q.rm2 + dm * (dm - 2.0) * vx * vx * q.rm4;
        const double fyy = dm * q.rm2 + dm * (dm - 2.0) * vy * vy * q.rm4;
        return sx * sx * fxx + sy * sy * fyy;
    }
    default: {  // OP_XK, OP_YK
        const double t = op == OP_XK ? vx : vy;
        const double t2 = t * t;
        double s = c[0], rp = 1.0;
        for (int i = 1; i <= (k >> 1); ++i) {
            rp *= q.r2;
            s = s * t2 + c[i] * rp;
        }
        if (k & 1) s *= t;
        const int e = m - 2 * k;  // odd
        return e > 0 ? s * (upow(q.r2, e >> 1) * q.r) : s * (q.r / upow(q.r2, (1 - e) >> 1));
    }
    }
}

// x^e for a per-lane exponent 0 <= e < 8
__device__ __forceinline__ double lpow(double x, int e)
{
    double p = e & 1 ? x : 1.0;
    x *= x;
    p = e & 2 ? p * x : p;
    x *= x;
    return e & 4 ? p * x : p;
}

// degree of monomial q < 28, per lane (mono_deg's order)
__device__ __forceinline__ int mono_degree(int q)
{
    return (q >= 1) + (q >= 3) + (q >= 6) + (q >= 10) + (q >= 15) + (q >= 21);
}

// d^a/dx^a d^b/dy^b of x^ea y^eb (a, b uniform, the exponents per lane)
__device__ __forceinline__ double ns_mono(int ea, int eb, int a, int b, double x, double y)
{
#pragma clang fp contract(off)
    double c = 1.0;
    for (int t = 0; t < a; ++t) c *= (double)(ea - t);  // zero once a > ea
    for (int t = 0; t < b; ++t) c *= (double)(eb - t);
    return c * (lpow(x, max(ea - a, 0)) * lpow(y, max(eb - b, 0)));
}

__device__ __forceinline__ double ns_op_mono(int op, int k, int ea, int eb, double x, double y, double sx, double sy)
{
#pragma clang fp contract(off)
    if (op == OP_LAP) return sx * sx * ns_mono(ea, eb, 2, 0, x, y) + sy * sy * ns_mono(ea, eb, 0, 2, x, y);
    int a = 0, b = 0;
    switch (op) {
    case OP_DX: a = 1; break;
    case OP_DY: b = 1; break;
    case OP_DXX: a = 2; break;
    case OP_DYY: b = 2; break;
    case OP_DXY: a = 1; b = 1; break;
    case OP_XK: a = k; break;
    case OP_YK: b = k; break;
    default: break;
    }
    return ns_mono(ea, eb, a, b, x, y);
}

// Fixed sizes that take the split residual (fb_sum_split): low powers with
// polynomials more than one degree above what definiteness asks for.  Errors
// against a 113-bit solve relative to the elimination's (geometric mean of a
// row's, second derivatives): with the plain residual 1.2 at (m, degree) = (3, 4),
// 1.1 at (3, 5), 1.05 at (5, 4) and (5, 5), at most 0.99 from m = 7 on and at
// (5, 3); with the split one 0.87, 0.74 at m = 3.  It takes 4% (n = 57) to 29%
// (n = 20) of the solve.  The kernels with n at run time always take it: 1.05
// without, 0.97 with it, for 2 to 8% of their time.
constexpr bool ns_split(int polydeg, int m) { return m <= 5 && polydeg > (m + 1) / 2; }

template <int NN, int NP, int G>
struct NsShape {
    static constexpr int N2 = NN - NP;
    static constexpr int S = 64 / G;                                      // stencils per wavefront
    static constexpr int S1 = (NP + G - 1) / G, S2 = (N2 + G - 1) / G;    // row slots per lane of the two node sets
    static constexpr int B1 = (NP + 15) / 16, B2 = (N2 + 15) / 16;        // their 16-row broadcast sources
    static constexpr int NODES = (NN + G - 1) / G;
    static constexpr int TS = NP | 1;  // row stride of the panel's result: odd, so a column read has no bank conflicts
    // Phi by position: the picked nodes' upper triangle, the NP x N2 block, the others' upper triangle
    // (rows of the block an odd stride apart: its rows are read across lanes too)
    static constexpr int WS = N2 | 1;
    static constexpr int F11 = 0, F12 = NP * (NP + 1) / 2, F22 = F12 + NP * WS;
    static constexpr int PHI = F22 + N2 * (N2 + 1) / 2;
    static constexpr int RPS = cmax_<PHI, NN * TS>::v;  // reciprocal pivots of S, behind Phi
    // per group; with 16 lanes 16 modulo 32 doubles, so two groups' odd-stride reads fall on all 64 banks
    static constexpr int U = G == 16 ? (RPS + N2 + 15) / 32 * 32 + 16 : (RPS + N2 + 1) & ~1;
    static constexpr __host__ __device__ int tri(int w, int a) { return a * (2 * w - a + 1) / 2 - a; }
};

template <int NN, int NP, int G>
struct alignas(16) NsLDS {
    using T = NsShape<NN, NP, G>;
    double u[T::S][T::U];       // the panel's pivot row, then P1^-1 and T, then Phi
    double xi[T::S][2 * NN];    // scaled coordinates by position
    double frame[T::S][5];      // centre and scales, the splitting constant of Phi (split_at)
    int g[T::S][NN], rank[T::S][NN];  // global index and output column by position
};

// Wavefronts per SIMD the kernel is compiled for.  n = 31: LDS (20 KB a
// wavefront) and the row registers hold it to two.  n = 20 and 21: three, with
// 26 and 35 registers spilled, take 2.00 ms per 1M stencils of n = 21 where two
// without spills take 2.29 ms; with the split residual, which spills 102 there,
// two take 0.40 against 0.48 ms per 160,000 stencils of n = 20.  n = 42 and 43:
// two, with 75 and 70 registers spilled at three operators (127 and 134 split), one
// without spills 2.79 against 2.06 ms split; the kernel for up to 42 nodes and 10
// monomials spills 135 and takes 1.72 ms at n = 35 where one wavefront takes 2.29.
// n = 31 spills 39 with the split residual, the kernels with n at run time for up to
// 26 and 31 nodes 15 and 42; the others none.
template <int NN, int NP, int G, bool SPLIT>
constexpr int ns_min_waves()
{
    if (G == 32) return NN <= 43 ? 2 : 1;
    return NN <= 21 && !SPLIT ? 3 : 2;
}

// NN nodes (GEN: at most NN, a.n of them), NP monomials, G lanes per stencil,
// RC operators at a time, SPLIT: the refinement's residual without rounding in
// its large part
template <int NN, int NP, int G, int RC, bool GEN, bool SPLIT>
__global__ __launch_bounds__(64, (ns_min_waves<NN, NP, G, SPLIT>())) void solve_ns_kernel(const NsArgs a)
{
    using T = NsShape<NN, NP, G>;
    constexpr int N2 = T::N2, S1 = T::S1, S2 = T::S2, B1 = T::B1, B2 = T::B2, NODES = T::NODES;
    constexpr int DEG = mono_deg(NP - 1);
    constexpr uint64_t kLane0 = G == 16 ? 0x0001000100010001ull : 0x0000000100000001ull;  // lane 0 of each group
    constexpr uint32_t kGroup = (uint32_t)((1ull << G) - 1);
    __shared__ NsLDS<NN, NP, G> L;
    const int lane = threadIdx.x & 63, grp = lane / G, t = lane % G;
    double *const U = L.u[grp];
    const int n = GEN ? a.n : NN, n2 = n - NP;
    const bool grouped = a.grp_x != nullptr;
    long ntasks = a.ntasks;
    if (a.ntasks_dev) ntasks = min(ntasks, (long)*a.ntasks_dev);
    const long task0 = (long)blockIdx.x * T::S;
    if (task0 >= ntasks) return;  // whole wavefront
    // a group without a task works on a copy of the first and stores nothing
    const bool live = task0 + grp < ntasks;
    const long task = live ? task0 + grp : task0;
    long xs;
    int yk, ybase = 0, ny = 1;
    if (grouped) {
        xs = a.grp_x[task];
        ybase = a.grp_start[task];
        ny = a.grp_count[task];
        yk = a.ylist[ybase];
    } else {
        yk = a.rows ? a.rows[task] : (int)task;
        xs = a.y2x ? a.y2x[yk] : yk;
    }
    const int m = a.m;
    const bool m3 = a.method == 3;

    // ---- stencil frame (src/scalestencil.jl:10-21, src/generate_operator.jl:100-134)
    double C[NODES][NP];  // this lane's rows of P: nodes t + G r
    uint32_t alive[NODES];
    double sx = 1.0, sy = 1.0, cx, cy;
    double nx[NODES], nyy[NODES];
    int gid[NODES], rk[NODES];
    {
#pragma clang fp contract(off)
        const int c = max(a.stencils[xs * n], 0);  // a failed search leaves -1: every read stays in X
        cx = a.X[2 * (long)c];
        cy = a.X[2 * (long)c + 1];
        double mx = 0.0, my = 0.0;
        int *gl = reinterpret_cast<int *>(U);
#pragma unroll
        for (int r = 0; r < NODES; ++r) {
            const int i = t + G * r;
            gid[r] = i < n ? max(a.stencils[xs * n + i], 0) : c;
            if (i < NN) gl[i] = i < n ? gid[r] : 0x7FFFFFFF;
            nx[r] = a.X[2 * (long)gid[r]] - cx;
            nyy[r] = a.X[2 * (long)gid[r] + 1] - cy;
            mx = fmax(mx, __builtin_fabs(nx[r]));
            my = fmax(my, __builtin_fabs(nyy[r]));
        }
        if (!m3) {
            mx = group_max_nonneg_f64<G>(mx);
            my = group_max_nonneg_f64<G>(my);
            sx = 1.0 / mx;
            sy = 1.0 / my;
        }
#pragma unroll
        for (int r = 0; r < NODES; ++r) {
            // method 3 leaves the frame unscaled, its centre at (eps, eps) (src/generate_operator.jl:393-410)
            nx[r] = m3 ? (t + G * r == 0 ? kEps : nx[r]) : nx[r] * sx;
            nyy[r] = m3 ? (t + G * r == 0 ? kEps : nyy[r]) : nyy[r] * sy;
        }
        __builtin_amdgcn_wave_barrier();
        // the output column of each node: the rank of its global index inside the stencil
#pragma unroll
        for (int r = 0; r < NODES; ++r) rk[r] = 0;
#pragma unroll
        for (int j = 0; j < NN; ++j) {
            const int gj = gl[j];
#pragma unroll
            for (int r = 0; r < NODES; ++r) rk[r] += gj < gid[r] ? 1 : 0;
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (t == 0) {
        L.frame[grp][0] = cx;
        L.frame[grp][1] = cy;
        L.frame[grp][2] = sx;
        L.frame[grp][3] = sy;
    }

    // ---- the panel: in-place Gauss-Jordan of P with row pivoting.  Rows keep
    // their scale (a picked row is multiplied by its reciprocal pivot at the
    // end); column k becomes the inverse's once step k is done.
#pragma unroll
    for (int r = 0; r < NODES; ++r) {
        double px[DEG + 1], py[DEG + 1];
        px[0] = py[0] = 1.0;
#pragma unroll
        for (int d = 1; d <= DEG; ++d) { px[d] = px[d - 1] * nx[r]; py[d] = py[d - 1] * nyy[r]; }
        alive[r] = t + G * r < n ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int q = 0; q < NP; ++q) C[r][q] = px[mono_ea(q)] * py[mono_eb(q)];
    }
    int pos[NODES];
    double fin[NODES];
#pragma unroll
    for (int r = 0; r < NODES; ++r) { pos[r] = 0; fin[r] = 1.0; }
    const uint32_t ua = lds_address(U);
    for_blocks<0, NP>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        // pivot search: the largest |C[.][k]| among rows not yet picked, as a
        // key whose low 7 bits name the node
        uint32_t key = 0;
        double cv = C[0][k];
#pragma unroll
        for (int r = 0; r < NODES; ++r) {
            const uint32_t kr = ((__float_as_uint((float)C[r][k]) & 0x7FFFFF00u) |
                                 (0x80u | (uint32_t)(127 - (t + G * r)))) & alive[r];
            if (r == 0) {
                key = kr;
            } else if (kr > key) {
                key = kr;
                cv = C[r][k];
            }
        }
        const double crp = rcp_nr(cv);
        key = group_max_u32<G>(key);
        const int v = 127 - (int)(key & 127u);
        const bool iam = t == v % G;
        // the picked row goes to the group, its reciprocal pivot in the pivot's place
#pragma unroll
        for (int r = 0; r < NODES; ++r) {
            if (iam && v / G == r) {
                for_blocks<0, NP / 2>([&](auto jc) {
                    constexpr int j = 2 * decltype(jc)::value;
                    lds_write2<j, j + 1>(ua, j == k ? crp : C[r][j], j + 1 == k ? crp : C[r][j + 1]);
                });
                if constexpr (NP % 2) U[NP - 1] = NP - 1 == k ? crp : C[r][NP - 1];
                alive[r] = 0u;
                pos[r] = k;
                fin[r] = crp;
            }
        }
        __builtin_amdgcn_wave_barrier();
        double pr[B1];
#pragma unroll
        for (int b = 0; b < B1; ++b) pr[b] = U[t % 16 + 16 * b];
        const double rp = row_bcast64<k % 16>(pr[k / 16]);
        double l[NODES];
#pragma unroll
        for (int r = 0; r < NODES; ++r) {
            const bool me = iam && v / G == r;
            // the picked row's multiplier: its high word zeroed leaves a value below 2^-1022, which the additions lose
            l[r] = hi_if(-(C[r][k] * rp), me, 0u);
            C[r][k] = me ? 1.0 : l[r];
            // the next step's column first
            if constexpr (k + 1 < NP) fb_lanes<k + 1, 1>(C[r], pr, l[r]);
        }
#pragma unroll
        for (int r = 0; r < NODES; ++r)
            fb_lanes<(k + 1 < NP ? k + 2 : k + 1) % NP, NP - 1 - (k + 1 < NP)>(C[r], pr, l[r]);
        __builtin_amdgcn_wave_barrier();
    });
    // a panel pivot at the rounding of its column (rows not picked hold 1 and pass):
    // a monomial's value on the bounding box is 1 where the frame is scaled
    bool bad = false;
    if (!m3) {  // uniform
        if (SPLIT && t == 0) L.frame[grp][4] = split_at((3 * m + 1) / 2);  // r^2 at most 8
#pragma unroll
        for (int r = 0; r < NODES; ++r) bad |= !(__builtin_fabs(fin[r]) * kNsPanelTol < 1.0);
    } else {
        double mx = 0.0, my = 0.0;
#pragma unroll
        for (int r = 0; r < NODES; ++r) {
            mx = fmax(mx, __builtin_fabs(nx[r]));
            my = fmax(my, __builtin_fabs(nyy[r]));
        }
        mx = group_max_nonneg_f64<G>(mx);
        my = group_max_nonneg_f64<G>(my);
        if (SPLIT && t == 0) {
            const int q = (int)((uint64_t)__double_as_longlong(4.0 * sq_sum(mx, my)) >> 52) - 1022;  // r^2 < 2^q
            L.frame[grp][4] = split_at(min(max((q * m + 1) >> 1, -1000), 900));
        }
#pragma unroll
        for (int r = 0; r < NODES; ++r) {
            const int d = mono_degree(pos[r]), ea = pos[r] - d * (d + 1) / 2;
            const double f = __builtin_fabs(fin[r]);
            // below 2^-120 the float keys of the pivot search lose bits
            bad |= !(f * (lpow(mx, ea) * lpow(my, d - ea)) * kNsPanelTol < 1.0) || !(f < 0x1p120);
        }
    }
    // positions of the rows that were not picked: slot by slot, lane by lane
    {
        int base = NP;
#pragma unroll
        for (int r = 0; r < NODES; ++r) {
            const bool fr = alive[r] != 0u;
            const uint64_t bal = __builtin_amdgcn_ballot_w64(fr);
            const uint32_t gm = (uint32_t)(bal >> (grp * G)) & kGroup;
            if (fr) pos[r] = base + __builtin_popcount(gm & ((1u << t) - 1u));
            base += __builtin_popcount(gm);
        }
    }
#pragma unroll
    for (int r = 0; r < NODES; ++r) {
        if (t + G * r < n) {
#pragma unroll
            for (int j = 0; j < NP; ++j) U[pos[r] * T::TS + j] = C[r][j] * fin[r];
            L.xi[grp][2 * pos[r]] = nx[r];
            L.xi[grp][2 * pos[r] + 1] = nyy[r];
            L.g[grp][pos[r]] = gid[r];
            L.rank[grp][pos[r]] = rk[r];
        }
    }
    __builtin_amdgcn_wave_barrier();
    // this lane's rows from here on: picked nodes kb[s] = t + G s, others
    // qa[s] = t + G s (lanes past the end repeat the last row and store nothing)
    int kb[S1], qa[S2];
    double nT[S2][NP];   // -T, row qa
    double nTt[S1][N2];  // -T, column kb
    double Pit[S1][NP];  // P1^-1, column kb
#pragma unroll
    for (int s = 0; s < S1; ++s) {
        kb[s] = min(t + G * s, NP - 1);
#pragma unroll
        for (int k = 0; k < NP; ++k) Pit[s][k] = U[k * T::TS + kb[s]];
#pragma unroll
        for (int i = 0; i < N2; ++i) nTt[s][i] = !GEN || i < n2 ? U[(NP + i) * T::TS + kb[s]] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < S2; ++s) {
        qa[s] = min(t + G * s, n2 - 1);
#pragma unroll
        for (int k = 0; k < NP; ++k) nT[s][k] = U[(NP + qa[s]) * T::TS + k];
    }
    __builtin_amdgcn_wave_barrier();

    __builtin_amdgcn_sched_barrier(0);
    // ---- Phi by position, each pair once
    if constexpr (GEN) {  // columns past the last node stay zero
        for (int i = t; i < T::PHI; i += G) U[i] = 0.0;
        __builtin_amdgcn_wave_barrier();
    }
    {
        auto pairs = [&](auto mc) {
            constexpr int MC = decltype(mc)::value;
            const int mm = MC > 0 ? MC : m;
            auto phs = [&](double x0, double y0, int p) {
                const double dx = x0 - L.xi[grp][2 * p], dy = y0 - L.xi[grp][2 * p + 1];
                const double r2 = sq_sum(dx, dy);
                return upow(r2, mm >> 1) * ns_sqrt(r2);
            };
#pragma unroll
            for (int s = 0; s < S2; ++s) {
                if (t + G * s < n2) {
                    const double x = L.xi[grp][2 * (NP + qa[s])], y = L.xi[grp][2 * (NP + qa[s]) + 1];
#pragma unroll 3
                    for (int k = 0; k < NP; ++k) U[T::F12 + k * T::WS + qa[s]] = phs(x, y, k);
                    U[T::F22 + T::tri(N2, qa[s]) + qa[s]] = 0.0;
#pragma unroll 2
                    for (int d = 1; d <= n2 / 2; ++d) {
                        int j = qa[s] + d;
                        if (j >= n2) j -= n2;
                        U[T::F22 + T::tri(N2, min(qa[s], j)) + max(qa[s], j)] = phs(x, y, NP + j);
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < S1; ++s) {
                if (t + G * s < NP) {
                    const double x = L.xi[grp][2 * kb[s]], y = L.xi[grp][2 * kb[s] + 1];
                    U[T::F11 + T::tri(NP, kb[s]) + kb[s]] = 0.0;
#pragma unroll 2
                    for (int d = 1; d <= NP / 2; ++d) {
                        int j = kb[s] + d;
                        if (j >= NP) j -= NP;
                        U[T::F11 + T::tri(NP, min(kb[s], j)) + max(kb[s], j)] = phs(x, y, j);
                    }
                }
            }
        };
        switch (m) {
        case 3: pairs(std::integral_constant<int, 3>{}); break;
        case 5: pairs(std::integral_constant<int, 5>{}); break;
        case 7: pairs(std::integral_constant<int, 7>{}); break;
        case 9: pairs(std::integral_constant<int, 9>{}); break;
        default: pairs(std::integral_constant<int, 0>{}); break;
        }
    }
    __builtin_amdgcn_wave_barrier();
    // Phi(picked row k, picked column c), Phi(k, other j), Phi(other row q, picked c), Phi(q, other j);
    // the two triangles: one addition and a select per entry, the mask by the row's slot (GG lanes apart)
    auto f11 = [&](auto gg, int k, auto sc, auto cc) {
        constexpr int GG = decltype(gg)::value, s = decltype(sc)::value, c = decltype(cc)::value;
        const int up = T::F11 + T::tri(NP, k), lo = k + (T::F11 + T::tri(NP, c) - c);
        return U[(upto<GG, s>(c) ? up : lo) + c];
    };
    auto f12 = [&](int k, int j) { return U[T::F12 + k * T::WS + j]; };
    auto f21 = [&](int q, int c) { return U[T::F12 + c * T::WS + q]; };
    auto f22 = [&](int q, auto sc, auto jc) {
        constexpr int s = decltype(sc)::value, j = decltype(jc)::value;
        const int up = T::F22 + T::tri(N2, q), lo = q + (T::F22 + T::tri(N2, j) - j);
        return U[(upto<G, s>(j) ? up : lo) + j];
    };
    using LanesG = std::integral_constant<int, G>;
    using Lanes16 = std::integral_constant<int, 16>;

    __builtin_amdgcn_sched_barrier(0);
    // ---- S = Phi22 - T Phi12 - (Phi21 - T Phi11) T^T, one row per lane slot.
    // Columns go in blocks of 16, to bound the registers; the picked nodes' rows
    // are loaded as broadcast sources (every DPP row of a group holds them all).
    double S[S2][N2];
    int ks[B1];
#pragma unroll
    for (int b = 0; b < B1; ++b) ks[b] = min(t % 16 + 16 * b, NP - 1);
    for_blocks<0, S2>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        for_blocks<0, N2>([&](auto jc) { S[s][decltype(jc)::value] = f22(qa[s], sc, jc); });
    });
    for_blocks<0, (NP + 15) / 16>([&](auto blk) {
        constexpr int c0 = 16 * decltype(blk)::value, W = NP - c0 < 16 ? NP - c0 : 16;
        double V[S2][W], B[B1][W];
        for_blocks<0, B1>([&](auto bc) {
            constexpr int b = decltype(bc)::value;
            for_blocks<0, W>([&](auto cc) {
                B[b][decltype(cc)::value] =
                    f11(Lanes16{}, ks[b], bc, std::integral_constant<int, c0 + decltype(cc)::value>{});
            });
        });
#pragma unroll
        for (int s = 0; s < S2; ++s) {
#pragma unroll
            for (int c = 0; c < W; ++c) V[s][c] = f21(qa[s], c0 + c);
            for_blocks<0, NP>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                fb_sub<k % 16, 0, 0, W>(V[s], B[k / 16], nT[s][k]);
            });
        }
        // + V (-T)^T: column c of -T, over the lanes of the other nodes
        for_blocks<0, W>([&](auto cc) {
            constexpr int c = decltype(cc)::value;
            double own[S2], tc[B2];
#pragma unroll
            for (int s = 0; s < S2; ++s) own[s] = nT[s][c0 + c];
            spread<G>(own, tc);
#pragma unroll
            for (int s = 0; s < S2; ++s) fb_lanes<0, N2>(S[s], tc, V[s][c]);
        });
        __builtin_amdgcn_sched_barrier(0);
    });
    for_blocks<0, (N2 + 15) / 16>([&](auto blk) {
        constexpr int j0 = 16 * decltype(blk)::value, W = N2 - j0 < 16 ? N2 - j0 : 16;
        double B[B1][W];
#pragma unroll
        for (int b = 0; b < B1; ++b)
#pragma unroll
            for (int j = 0; j < W; ++j) B[b][j] = f12(ks[b], j0 + j);
#pragma unroll
        for (int s = 0; s < S2; ++s)
            for_blocks<0, NP>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                fb_sub<k % 16, j0, 0, W>(S[s], B[k / 16], nT[s][k]);
            });
        __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (GEN) {
#pragma unroll
        for (int s = 0; s < S2; ++s)
#pragma unroll
            for (int j = 0; j < N2; ++j) S[s][j] = j < n2 ? S[s][j] : 0.0;
    }

    // ---- S^-1 in place without pivoting (S is definite); row q stays scaled by
    // its pivot, whose reciprocal (rps) multiplies the products
    if constexpr (G == 16) {
        for_blocks<0, N2>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            if (GEN && k >= n2) return;  // uniform
            const double rp = rcp_nr(row_bcast64<k % 16>(S[k / 16][k]));
            U[T::RPS + k] = rp;  // the same value from every lane of the group
            double l[S2];
#pragma unroll
            for (int s = 0; s < S2; ++s) {
                const bool me = s == k / 16 && __builtin_amdgcn_inverse_ballot_w64(kLane0 << (k % 16));
                l[s] = hi_if(-(S[s][k] * rp), me, 0u);
                S[s][k] = me ? 1.0 : l[s];
            }
#pragma unroll
            for (int s = 0; s < S2; ++s)
                if constexpr (k + 1 < N2) fb_cols<k % 16, k + 1, 1>(S[s], S[k / 16], l[s]);
#pragma unroll
            for (int s = 0; s < S2; ++s)
                fb_cols<k % 16, (k + 1 < N2 ? k + 2 : k + 1) % N2, N2 - 1 - (k + 1 < N2)>(S[s], S[k / 16], l[s]);
        });
    } else {
        // 32 lanes: a lane holds row t, and a pivot row would have to cross the
        // group's two DPP rows entry by entry.  One lane swap per register pair
        // turns that into two rows a lane, t % 16 and t % 16 + 16, with one half
        // of the columns in each DPP row: the pivot row then broadcasts inside
        // each, and only the multipliers cross (the pivot row's transpose, one
        // value a lane, would cross as cheaply and do in exact arithmetic, but on
        // uniform random nodes at n = 57 it left weights 1e-2 off).
        constexpr int H = (N2 + 1) / 2;
        double R[2][H];
#pragma unroll
        for (int j = 0; j < H; ++j) swap_rows(S[0][j], H + j < N2 ? S[0][H + j] : 0.0, R[0][j], R[1][j]);
        for_blocks<0, N2>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            if (GEN && k >= n2) return;              // uniform
            constexpr int hk = k / H, kk = k % H;    // its column's DPP row and register
            constexpr uint64_t half = 0x0000FFFF0000FFFFull << (16 * hk);
            double c[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const double own[1] = {R[s][kk]};
                double both[2];
                spread<G>(own, both);
                c[s] = both[hk];
            }
            const double rp = rcp_nr(row_bcast64<k % 16>(c[k / 16]));
            U[T::RPS + k] = rp;
            // the column becomes -c rp (1 in the pivot row): zero plus the
            // multiplier times the pivot row's entry, set to 1
            double l[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const bool me = s == k / 16 && __builtin_amdgcn_inverse_ballot_w64(0x0001000100010001ull << (k % 16));
                const bool col = __builtin_amdgcn_inverse_ballot_w64(half);
                l[s] = hi_if(-(c[s] * rp), me, 0u);
                R[s][kk] = col ? 0.0 : R[s][kk];
                if (s == k / 16)
                    R[s][kk] = hi_if(R[s][kk], __builtin_amdgcn_inverse_ballot_w64(
                                                   half & (0x0001000100010001ull << (k % 16))), 0x3FF00000u);
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) fb_cols<k % 16, (kk + 1) % H, 1>(R[s], R[k / 16], l[s]);
#pragma unroll
            for (int s = 0; s < 2; ++s) fb_cols<k % 16, (kk + 2) % H, H - 1>(R[s], R[k / 16], l[s]);
        });
#pragma unroll
        for (int j = 0; j < H; ++j) {
            double a, b;
            swap_rows(R[0][j], R[1][j], a, b);
            S[0][j] = a;
            if (H + j < N2) S[0][H + j] = b;
        }
    }
    // pivots: the reciprocals' extremes over the group
    double rps[S2], rmin = 1e300, rmax = -1e300;
    const double sgn = ((m + 1) >> 1) & 1 ? -1.0 : 1.0;  // sign of the definite form, (-1)^((m+1)/2)
#pragma unroll
    for (int s = 0; s < S2; ++s) {
        rps[s] = U[T::RPS + qa[s]];
        rmin = fmin(rmin, sgn * rps[s]);
        rmax = fmax(rmax, sgn * rps[s]);
    }
    // a wrong sign makes rmin negative, a NaN fails the finiteness check of the weights
    const bool definite = !(rmin <= 0.0);
    rmax = group_max_nonneg_f64<G>(fmax(rmax, 0.0));
    const double imax = group_max_nonneg_f64<G>(definite ? 1.0 / rmin : 1e300);
    __builtin_amdgcn_sched_barrier(0);
    // the smallest pivot is 1 / rmax, the largest imax
    bad |= !definite || !(kNsPivotTol * imax * rmax < 1.0);

    // ---- the rows' right-hand sides, RC operators at a time
    double gx = a.Y[2 * (long)yk], gy = a.Y[2 * (long)yk + 1];
    for (int sub = 0;; ++sub) {
        const bool on = live && sub < ny;
        if (!__builtin_amdgcn_ballot_w64(sub < ny)) break;
        const long row = yk;
        // the arguments are read again for each row: held over the loop they
        // outgrow the scalar registers
        auto *ap = (const __attribute__((address_space(4))) NsArgs *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(ap));
        int fo = 0;
        asm volatile("" : "+v"(fo));  // read back from LDS here, not held in registers
        const double hx = L.frame[grp][2 + fo], hy = L.frame[grp][3 + fo];
        double px, py;
        {
#pragma clang fp contract(off)
            px = m3 ? kEps : (gx - L.frame[grp][fo]) * hx;
            py = m3 ? kEps : (gy - L.frame[grp][1 + fo]) * hy;
        }
        if (sub + 1 < ny) {  // the next row's point
            yk = ap->ylist[ybase + sub + 1];
            gx = ap->Y[2 * (long)yk];
            gy = ap->Y[2 * (long)yk + 1];
        }
        // u = Y - xi with exact zeros -> eps (src/generate_operator.jl:125-154)
        auto u_at = [&](double x, double y, double &ux, double &uy) {
            ux = m3 ? x : px - x;
            uy = m3 ? y : py - y;
            if (!m3 && ux == 0.0) ux = kEps;
            if (!m3 && uy == 0.0) uy = kEps;
        };
        for (int o0 = 0; o0 < ap->nops; o0 += RC) {
            double ba[S2][RC], bb[S1][RC], np[S1][RC];
            // kept inside the row loop: hoisted out of it, what depends on the
            // operators costs more registers than it saves work
            int kind[RC], ord[RC];
            int mh = m;
            asm volatile("" : "+s"(mh));
#pragma unroll
            for (int o = 0; o < RC; ++o) {
                kind[o] = ap->op_kind[min(o0 + o, ap->nops - 1)];
                ord[o] = ap->op_k[min(o0 + o, ap->nops - 1)];
                asm volatile("" : "+s"(kind[o]), "+s"(ord[o]));
            }
            auto rhs_at = [&](int p, double (&b)[RC]) {
                double ux, uy;
                u_at(L.xi[grp][2 * p], L.xi[grp][2 * p + 1], ux, uy);
                const NsPhsAt q = ns_phs_at(mh, ux, uy);
#pragma unroll
                for (int o = 0; o < RC; ++o)
                    b[o] = ns_op_phs(kind[o], ord[o], mh, ap->xk_c[min(o0 + o, ap->nops - 1)], ux, uy, hx, hy, q);
                __builtin_amdgcn_sched_barrier(0);
            };
#pragma unroll
            for (int s = 0; s < S2; ++s) rhs_at(NP + qa[s], ba[s]);
#pragma unroll
            for (int s = 0; s < S1; ++s) {
                rhs_at(kb[s], bb[s]);
                int q = kb[s];  // the exponents of monomial kb
                asm volatile("" : "+v"(q));
                const int d = mono_degree(q), ea = q - d * (d + 1) / 2, eb = d - ea;
#pragma unroll
                for (int o = 0; o < RC; ++o) np[s][o] = -ns_op_mono(kind[o], ord[o], ea, eb, px, py, hx, hy);
            }
            __builtin_amdgcn_sched_barrier(0);
            // the negated weights: w1n = -w0 first, w2n = 0
            double w1n[S1][RC], w2n[S2][RC];
            {
                double src[B1][RC];
                spread<G>(np, src);
#pragma unroll
                for (int s = 0; s < S1; ++s) {
#pragma unroll
                    for (int o = 0; o < RC; ++o) w1n[s][o] = 0.0;
                    fb_sum<0, NP>(w1n[s], src, Pit[s]);
                }
            }
#pragma unroll
            for (int s = 0; s < S2; ++s)
#pragma unroll
                for (int o = 0; o < RC; ++o) w2n[s][o] = 0.0;
            // the solve, then one step of refinement: residual b - Phi w,
            // projected on the null space, through S^-1
#pragma nounroll
            for (int it = 0; it < 2; ++it) {
                double ra[S2][RC], rb[S1][RC];
                int kh[S1], qh[S2];  // addresses formed here each time, not held in registers
#pragma unroll
                for (int s = 0; s < S1; ++s) {
                    kh[s] = kb[s];
                    asm volatile("" : "+v"(kh[s]));
                }
#pragma unroll
                for (int s = 0; s < S2; ++s) {
                    qh[s] = qa[s];
                    asm volatile("" : "+v"(qh[s]));
                }
                if (!SPLIT || !it) {
                    double src[B1][RC];
                    spread<G>(w1n, src);
#pragma unroll
                    for (int s = 0; s < S2; ++s) {
                        double f[NP];
#pragma unroll
                        for (int c = 0; c < NP; ++c) f[c] = f21(qh[s], c);
#pragma unroll
                        for (int o = 0; o < RC; ++o) ra[s][o] = ba[s][o];
                        fb_sum2<NP>(ra[s], src, f);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    for_blocks<0, S1>([&](auto sc) {
                        constexpr int s = decltype(sc)::value;
                        double f[NP];
                        for_blocks<0, NP>([&](auto cc) { f[decltype(cc)::value] = f11(LanesG{}, kh[s], sc, cc); });
#pragma unroll
                        for (int o = 0; o < RC; ++o) rb[s][o] = bb[s][o];
                        fb_sum2<NP>(rb[s], src, f);
                        __builtin_amdgcn_sched_barrier(0);
                    });
                }
                if constexpr (!SPLIT) {
                    if (it) {
                        double src[B2][RC];
                        spread<G>(w2n, src);
                        for_blocks<0, S2>([&](auto sc) {
                            constexpr int s = decltype(sc)::value;
                            double f[N2];
                            for_blocks<0, N2>([&](auto jc) { f[decltype(jc)::value] = f22(qh[s], sc, jc); });
                            fb_sum2<N2>(ra[s], src, f);
                            __builtin_amdgcn_sched_barrier(0);
                        });
#pragma unroll
                        for (int s = 0; s < S1; ++s) {
                            double f[N2];
#pragma unroll
                            for (int j = 0; j < N2; ++j) f[j] = f12(kh[s], j);
                            fb_sum2<N2>(rb[s], src, f);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                } else if (it) {
                    // b - Phi w in halves: the upper ones' products sum exactly
                    double a1[S2][RC], a2[S2][RC], b1[S1][RC], b2[S1][RC], cw[RC];
#pragma unroll
                    for (int o = 0; o < RC; ++o) {
                        uint32_t h = 0;
#pragma unroll
                        for (int s = 0; s < S1; ++s) h = max(h, high_abs(w1n[s][o]));
#pragma unroll
                        for (int s = 0; s < S2; ++s) h = max(h, high_abs(w2n[s][o]));
                        h = group_max_u32<G>(h);
                        // split_at of the largest weight's exponent
                        cw[o] = __longlong_as_double((long long)((uint64_t)((h & 0x7FF00000u) + 0x01E80000u) << 32));
#pragma unroll
                        for (int s = 0; s < S2; ++s) a1[s][o] = a2[s][o] = 0.0;
#pragma unroll
                        for (int s = 0; s < S1; ++s) b1[s][o] = b2[s][o] = 0.0;
                    }
                    int fp = 0;
                    asm volatile("" : "+v"(fp));
                    const double cp = L.frame[grp][4 + fp];
                    {
                        double hi[S1][RC], lo[S1][RC], sh[B1][RC], sl[B1][RC];
#pragma unroll
                        for (int s = 0; s < S1; ++s)
#pragma unroll
                            for (int o = 0; o < RC; ++o) {
                                hi[s][o] = (w1n[s][o] + cw[o]) - cw[o];
                                lo[s][o] = w1n[s][o] - hi[s][o];
                            }
                        spread<G>(hi, sh);
                        spread<G>(lo, sl);
#pragma unroll
                        for (int s = 0; s < S2; ++s) {
                            fb_sum_split<0, NP>(a1[s], a2[s], sh, sl, cp, [&](auto cc) { return f21(qh[s], decltype(cc)::value); });
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        for_blocks<0, S1>([&](auto sc) {
                            constexpr int s = decltype(sc)::value;
                            fb_sum_split<0, NP>(b1[s], b2[s], sh, sl, cp, [&](auto cc) { return f11(LanesG{}, kh[s], sc, cc); });
                            __builtin_amdgcn_sched_barrier(0);
                        });
                    }
                    {
                        double hi[S2][RC], lo[S2][RC], sh[B2][RC], sl[B2][RC];
#pragma unroll
                        for (int s = 0; s < S2; ++s)
#pragma unroll
                            for (int o = 0; o < RC; ++o) {
                                hi[s][o] = (w2n[s][o] + cw[o]) - cw[o];
                                lo[s][o] = w2n[s][o] - hi[s][o];
                            }
                        spread<G>(hi, sh);
                        spread<G>(lo, sl);
                        for_blocks<0, S2>([&](auto sc) {
                            constexpr int s = decltype(sc)::value;
                            fb_sum_split<0, N2>(a1[s], a2[s], sh, sl, cp, [&](auto jc) { return f22(qh[s], sc, jc); });
                            __builtin_amdgcn_sched_barrier(0);
                        });
#pragma unroll
                        for (int s = 0; s < S1; ++s) {
                            fb_sum_split<0, N2>(b1[s], b2[s], sh, sl, cp, [&](auto jc) { return f12(kh[s], decltype(jc)::value); });
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
#pragma unroll
                    for (int o = 0; o < RC; ++o) {
#pragma unroll
                        for (int s = 0; s < S2; ++s) ra[s][o] = (ba[s][o] + a1[s][o]) + a2[s][o];
#pragma unroll
                        for (int s = 0; s < S1; ++s) rb[s][o] = (bb[s][o] + b1[s][o]) + b2[s][o];
                    }
                }
                {
                    double src[B1][RC];
                    spread<G>(rb, src);
#pragma unroll
                    for (int s = 0; s < S2; ++s) fb_sum2<NP>(ra[s], src, nT[s]);
                }
                double dn[S2][RC], src[B2][RC];
                spread<G>(ra, src);
#pragma unroll
                for (int s = 0; s < S2; ++s) {
                    double y[RC];
#pragma unroll
                    for (int o = 0; o < RC; ++o) y[o] = 0.0;
                    fb_sum<0, N2>(y, src, S[s]);
#pragma unroll
                    for (int o = 0; o < RC; ++o) {
                        dn[s][o] = -rps[s] * y[o];
                        w2n[s][o] += dn[s][o];
                    }
                }
                spread<G>(dn, src);
#pragma unroll
                for (int s = 0; s < S1; ++s) fb_sum<0, N2>(w1n[s], src, nTt[s]);
            }
            // ---- CSR output, columns sorted by global index
#pragma unroll
            for (int o = 0; o < RC; ++o) {
                if (o0 + o < ap->nops) {
                    const double f = m3 ? -1.0 : -op_post_scale(kind[o], ord[o], hx, hy);
                    double *out = ap->vals[o0 + o] + row * n;
#pragma unroll
                    for (int s = 0; s < S2; ++s) {
                        if (t + G * s < n2) {
                            const double wv = f * w2n[s][o];
                            bad |= !__builtin_isfinite(wv);
                            if (on) out[L.rank[grp][NP + qa[s]]] = wv;
                        }
                    }
#pragma unroll
                    for (int s = 0; s < S1; ++s) {
                        if (t + G * s < NP) {
                            const double wv = f * w1n[s][o];
                            bad |= !__builtin_isfinite(wv);
                            if (on) out[L.rank[grp][kb[s]]] = wv;
                        }
                    }
                }
            }
        }
        if (ap->colidx && on) {
#pragma unroll
            for (int s = 0; s < S2; ++s)
                if (t + G * s < n2) ap->colidx[row * n + L.rank[grp][NP + qa[s]]] = L.g[grp][NP + qa[s]];
#pragma unroll
            for (int s = 0; s < S1; ++s)
                if (t + G * s < NP) ap->colidx[row * n + L.rank[grp][kb[s]]] = L.g[grp][kb[s]];
        }
        if (ap->status && on && t == 0 && !ap->status_accumulate) ap->status[row] = 0;
    }
    // rows for the pivoting kernel
    const uint64_t bm = __builtin_amdgcn_ballot_w64(bad);
    if (((bm >> (grp * G)) & kGroup) && live) {
        for (int q = t; q < ny; q += G) a.redo[1 + atomicAdd(a.redo, 1)] = grouped ? a.ylist[ybase + q] : yk;
    }
}

// One wavefront per block.
template <int NN, int NP, int RC, bool GEN, bool SPLIT>
void launch_ns_rc(const NsArgs &a, hipStream_t s)
{
    constexpr int G = ns_lanes(NN, NP);
    const unsigned nb = (unsigned)((a.ntasks + 64 / G - 1) / (64 / G));
    solve_ns_kernel<NN, NP, G, RC, GEN, SPLIT><<<nb, 64, 0, s>>>(a);
}

template <int NN, int NP, bool GEN, bool SPLIT>
void launch_ns_shape(const NsArgs &a, hipStream_t s)
{
    if (a.nops == 1) launch_ns_rc<NN, NP, 1, GEN, SPLIT>(a, s);
    else if (a.nops == 2) launch_ns_rc<NN, NP, 2, GEN, SPLIT>(a, s);
    else launch_ns_rc<NN, NP, 3, GEN, SPLIT>(a, s);
}

}  // namespace rbffd

#define RBFFD_DEFINE_NS_UPTO(nn, pp) \
    namespace rbffd {                \
    void launch_ns_upto_##nn##_##pp(const NsArgs &a, hipStream_t s) { launch_ns_shape<nn, pp, true, true>(a, s); } \
    }
#define RBFFD_DEFINE_NS(nn, pp) \
    namespace rbffd {           \
    void launch_ns_##nn##_##pp(const NsArgs &a, hipStream_t s)              \
    {                                                                       \
        if (ns_split(mono_deg(pp - 1), a.m)) launch_ns_shape<nn, pp, false, true>(a, s); \
        else launch_ns_shape<nn, pp, false, false>(a, s);                   \
    }                                                                       \
    }
