// fg_mg.hip -- multigrid V-cycle preconditioner of the pressure PCG.
//
// The reference preconditions its PCG with the inverse-Poisson
// preconditioner (inversepoissonpreconditioner.h:45-79), whose iteration
// count grows linearly with the grid side (about 140 / 280 / 565 iterations
// to 1e-6 on dam-break systems of 128^2 / 256^2 / 512^2 cells).  This V-cycle
// is a fixed symmetric positive definite linear operator, so PCG converges
// to the same solution of the same system; it takes 9 / 11 / 14.
//
// Hierarchy (rebuilt for every solve, since the fluid region changes):
//   level 0      the pressure matrix A' itself: 5-point, integer
//                coefficients, from SceneDev::stencil;
//   level l+1    cells of 2x2 level-l cells, active where any of the four
//                is; operator A_{l+1} = R A_l P (Galerkin), P the bilinear
//                cell-centred prolongation restricted to active cells
//                (weights 9/16, 3/16, 3/16, 1/16 from the four nearest
//                coarse cells), R = P^T / 4.  The coarse operators have 5x5
//                stencils; their entries are summed in FP64 and mirrored so
//                that each stored operator is exactly symmetric.
//   bottom       the first level with at most kMgBottomMax cells per side
//                (at least level 1).
// Smoother: one L1-Jacobi sweep before and after the coarse correction,
// x += w (r - A x) / sum_k |a_k| with w = kMgOmega = 1.5.  The L1 diagonal
// dominates A, so the eigenvalues of A / sum_k |a_k| lie in (0, 1] and the
// sweep converges for every symmetric positive definite A and every w < 2
// (a damped plain Jacobi sweep does not on all of these Galerkin
// operators).  Over-relaxed weights take fewer PCG iterations: from zero
// on dam-break systems of 128^2 / 256^2 / 512^2 cells 11 / 13 / 17 with
// w = 1, 9 / 11 / 14 with 1.5 or 1.6, more again from 1.8; on the
// warm-started solves of 256 mixed scenes 6.2 a solve on average with 1.5
// (1.3: 6.6, 1.4: 6.4, 1.6: 6.5, 1.7: 7.7).  The bottom
// level gets kMgBottomSweeps sweeps from zero.  Every step is the same
// before and after, so the cycle is symmetric.
//
// Non-fluid rows of A' are identity rows: z = r there, as in the IPP.
// Level 0 as the V-cycle sees it is A' without the row-wrapping couplings
// the reference's linear offsets create at j = 0 and j = J-1 (a fluid cell
// on the grid edge, see k_stencil); the smoother's L1 diagonal still counts
// them, which only enlarges it.  The cycle stays symmetric; PCG itself
// multiplies by the full A'.
#include <type_traits>
#include <utility>

#include "fg_kernels.h"

namespace fg {

namespace {

// Both stop flags are read unconditionally (scalar loads issued together
// with the caller's other uniform loads, no branch between them).
__device__ __forceinline__ bool mg_iterating(const SceneDev& s)
{
    cptr<SceneScalars> sc = cst(s.sc);
    const int od = sc->outer_done, id = sc->inner_done;
    return (s.active != 0) & (s.precond == kPrecondMG) & (od == 0) & (id == 0);
}

// L1 diagonal of a level-0 row: n + (number of fluid neighbours)
__device__ __forceinline__ float l1_diag0(uint8_t code)
{
    return (float)(((code >> 4) & 7) + __popc(code & 15u));
}

// 1-D restriction weights of the fine cells 2c-1 .. 2c+2 (times 4)
__device__ __forceinline__ float w1(int a) { return (a == 1 || a == 2) ? 0.75f : 0.25f; }

// Coarse correction at fine cell (fi, fj) from the coarser level's y (I x J):
// the (up to) four nearest coarse cells, weights 9/16, 3/16, 3/16, 1/16.
// The four loads are unconditional (clamped index, weight 0 outside), so
// they issue together.  Inactive coarse cells hold y = 0.
template <typename P>
__device__ __forceinline__ float prolong_at(P y, int I, int J, int fi, int fj)
{
    const int p0 = fi >> 1, q0 = fj >> 1;
    const int p1 = (fi & 1) ? p0 + 1 : p0 - 1, q1 = (fj & 1) ? q0 + 1 : q0 - 1;
    const int pi[2] = {p0, p1}, qj[2] = {q0, q1};
    const float wi[2] = {0.75f, 0.25f};
    float v[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int i = min(max(pi[a], 0), I - 1), j = min(max(qj[b], 0), J - 1);
            v[a][b] = y[i * J + j];
        }
    float acc = 0.f;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const bool ok = pi[a] >= 0 && pi[a] < I && qj[b] >= 0 && qj[b] < J;
            acc += ((wi[a] * wi[b]) * v[a][b]) * mask01(ok);
        }
    return acc;
}

// The 25 stored coefficients of row c: one 128-byte line (the row's
// kMgRowStride floats), seven 16-byte loads issued together.
typedef float coef4 __attribute__((ext_vector_type(4)));   // a builtin vector: loads from any address space
__device__ __forceinline__ void load_coef_row(gptr<const float> coef, int c, float (&a)[kMgStencil])
{
    gptr<const coef4> r4 = (gptr<const coef4>)(coef + (size_t)c * kMgRowStride);
    coef4 q[7];
#pragma unroll
    for (int u = 0; u < 7; u++) q[u] = r4[u];
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) a[k] = q[k >> 2][k & 3];
}

// The 25 entries of an active level-l row (dinv != 0): the canonical stencil
// on canonical rows (dinv < 0), else the stored coefficients, loaded only by
// the lanes whose rows need them; and their sum over v.  Two steps, so that a
// kernel can issue the loads early.
template <typename MT>
__device__ __forceinline__ void row_load(const MT& M, int l, gptr<const float> coef, int c, float dinv_c,
                                         float (&a)[kMgStencil])
{
    const auto& cn = M.canon[l];
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) a[k] = cn[k];
    if (dinv_c > 0.f) load_coef_row(coef, c, a);
}
__device__ __forceinline__ float row_sum(const float (&a)[kMgStencil], const float (&v)[kMgStencil])
{
    float ax = 0.f;
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) ax += a[k] * v[k];
    return ax;
}
template <typename MT>
__device__ __forceinline__ float row_dot(const MT& M, int l, gptr<const float> coef, int c, float dinv_c,
                                         const float (&v)[kMgStencil])
{
    float a[kMgStencil];
    row_load(M, l, coef, c, dinv_c, a);
    return row_sum(a, v);
}

// r at coarse cell (ci, cj) from the finer level's y (FI x FJ): 1-D weights
// 1/4, 3/4, 3/4, 1/4 over fine cells 2c-1 .. 2c+2, times 1/4.  Inactive fine
// cells hold y = 0; the loads are unconditional (clamped index, weight 0
// outside the grid).
template <typename P>
__device__ __forceinline__ float restrict_at(P fy, int FI, int FJ, int ci, int cj)
{
    float v[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int fi = min(max(2 * ci - 1 + a, 0), FI - 1), fj = min(max(2 * cj - 1 + b, 0), FJ - 1);
            v[a][b] = fy[fi * FJ + fj];
        }
    float acc = 0.f;
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int fi = 2 * ci - 1 + a, fj = 2 * cj - 1 + b;
            const bool ok = fi >= 0 && fi < FI && fj >= 0 && fj < FJ;
            acc += ((w1(a) * w1(b)) * v[a][b]) * mask01(ok);
        }
    return 0.25f * acc;
}

// The 5x5 neighbourhood of (ci, cj) in x (LI x LJ), 0 outside the grid
// (clamped loads times a 0/1 factor, so every load issues).
template <typename P>
__device__ __forceinline__ void gather25(P x, int LI, int LJ, int ci, int cj, float (&xv)[kMgStencil])
{
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) {
        const int ni = ci + k / 5 - 2, nj = cj + k % 5 - 2;
        const bool ok = ni >= 0 && ni < LI && nj >= 0 && nj < LJ;
        const float v = x[min(max(ni, 0), LI - 1) * LJ + min(max(nj, 0), LJ - 1)];
        xv[k] = v * mask01(ok);
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// set-up, per level l >= 1 in increasing order (one launch per level for all
// scenes of the group; a thread per level-l cell)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void mg_mark_block(const SceneDev& s, int l, int bx)
{
    if (!s.active || s.precond != kPrecondMG) return;
    const auto& M = *cst(s.mg);
    if (l >= M.n) return;
    const auto& L = M.lv[l];
    const int c = bx * kBlock + threadIdx.x;
    if (c >= L.I * L.J) return;
    const int ci = c / L.J, cj = c - ci * L.J;
    const int FI = l == 1 ? s.I : M.lv[l - 1].I, FJ = l == 1 ? s.J : M.lv[l - 1].J;
    gptr<const uint8_t> fact = gbl<const uint8_t>(l == 1 ? s.stencil : M.lv[l - 1].act);
    uint8_t act = 0;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int fi = 2 * ci + a, fj = 2 * cj + b;
            const bool ok = fi < FI && fj < FJ;
            const uint8_t v = fact[ok ? fi * FJ + fj : 0];
            if (ok) act |= l == 1 ? (uint8_t)(v >> 7) : v;
        }
    gbl(L.act)[c] = act;
}

__global__ void __launch_bounds__(kBlock) k_mg_mark(const SceneDev* scenes, int l)
{
    mg_mark_block(scenes[blockIdx.y], l, blockIdx.x);
}

// floor(t / 2) for small t of either sign
__device__ __forceinline__ constexpr int half_floor(int t) { return t >= 0 ? t / 2 : -((1 - t) / 2); }
__device__ __forceinline__ constexpr double w1c(int a) { return (a == 1 || a == 2) ? 0.75 : 0.25; }

// compile-time loop: f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>)
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int DI, int DJ>
__device__ __forceinline__ void galerkin_add(double (&acc)[kMgStencil], double w, double v)
{
    if constexpr (DI >= -2 && DI <= 2 && DJ >= -2 && DJ <= 2) {
        constexpr int k = (DI + 2) * 5 + (DJ + 2);
        acc[k] = __builtin_fma(w, v, acc[k]);
    }
}

// One entry (value v) of fine row f = (2ci-1+A, 2cj-1+B) coupling it to
// g = f + (EI, EJ): spread R_f v P_g over g's coarse parents.  A weight has
// 7 significant bits and v 24 (a float), so each product is exact in FP64
// and the fused multiply-add rounds as the product and the sum would.
template <int A, int B, int EI, int EJ>
__device__ __forceinline__ void galerkin_spread(double (&acc)[kMgStencil], double v)
{
    constexpr int ti = -1 + A + EI, tj = -1 + B + EJ;   // g - 2C
    constexpr int pi0 = half_floor(ti), pj0 = half_floor(tj);
    constexpr int pi1 = (ti & 1) ? pi0 + 1 : pi0 - 1, pj1 = (tj & 1) ? pj0 + 1 : pj0 - 1;
    constexpr double wc = w1c(A) * w1c(B);
    galerkin_add<pi0, pj0>(acc, wc * 0.5625, v);
    galerkin_add<pi0, pj1>(acc, wc * 0.1875, v);
    galerkin_add<pi1, pj0>(acc, wc * 0.1875, v);
    galerkin_add<pi1, pj1>(acc, wc * 0.0625, v);
}

// The fine row A's (2ci - 1 + A) part of coarse row C = (ci, cj): its four
// fine cells, their stencil entries and those entries' coarse parents sit at
// compile-time offsets from C, so the 25 FP64 accumulators stay in registers.
// Every load is unconditional (clamped fine index; a fine cell outside the
// grid contributes zero).  Inactive fine rows hold all-zero coefficients
// (level >= 1) or a non-fluid code (level 0): they add nothing.
template <bool FINE0, int A, typename MT>
__device__ __forceinline__ void galerkin_part(const SceneDev& s, const MT& M, int l, int ci, int cj,
                                              double (&acc)[kMgStencil])
{
    const int FI = FINE0 ? s.I : M.lv[l - 1].I, FJ = FINE0 ? s.J : M.lv[l - 1].J;
    const int fi = 2 * ci - 1 + A;
    const bool row = fi >= 0 && fi < FI;
    const int fr = min(max(fi, 0), FI - 1) * FJ;
    if constexpr (FINE0) {
        gptr<const uint8_t> code = gbl<const uint8_t>(s.stencil);
        uint8_t cd[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int fj = 2 * cj - 1 + b;
            const uint8_t k = code[fr + min(max(fj, 0), FJ - 1)];
            cd[b] = row && fj >= 0 && fj < FJ ? k : 0;
        }
        static_for<4>([&](auto bb) {
            constexpr int b = decltype(bb)::value;
            const int fj = 2 * cj - 1 + b;
            const uint8_t k = cd[b];
            const double on = (k & 0x80) ? 1.0 : 0.0;
            galerkin_spread<A, b, 0, 0>(acc, on * (double)((k >> 4) & 7));
            galerkin_spread<A, b, -1, 0>(acc, (k & 1) ? -on : 0.0);
            galerkin_spread<A, b, 1, 0>(acc, (k & 2) ? -on : 0.0);
            galerkin_spread<A, b, 0, -1>(acc, ((k & 4) && fj > 0) ? -on : 0.0);   // not the row-wrapping coupling
            galerkin_spread<A, b, 0, 1>(acc, ((k & 8) && fj < FJ - 1) ? -on : 0.0);
        });
    } else {
        gptr<const float> fc = gbl<const float>(M.lv[l - 1].coef);
        float v[4][kMgStencil];
        float in[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int fj = 2 * cj - 1 + b;
            in[b] = mask01(row && fj >= 0 && fj < FJ);
            load_coef_row(fc, fr + min(max(fj, 0), FJ - 1), v[b]);
        }
        static_for<4>([&](auto bb) {
            constexpr int b = decltype(bb)::value;
            static_for<kMgStencil>([&](auto ee) {
                constexpr int e = decltype(ee)::value;
                galerkin_spread<A, b, e / 5 - 2, e % 5 - 2>(acc, (double)(v[b][e] * in[b]));
            });
        });
    }
}

// A_l = R A_{l-1} P: kGalCells coarse rows a block, wave a summing fine row
// a's part of each (lane = coarse row), the four parts added in LDS, entries
// of inactive coarse neighbours dropped, and the row written as 16-byte
// stores.  The parts are sums of products of few bits, exact in FP64 on the
// upper levels, so where the order of the sums changed, they hardly do.
// Bound by instruction issue: 1,600 multiply-adds and 400 conversions a row
// (a wave a quarter of them, since the small levels have a few waves for the
// whole chip).  A thread a row, with the activity selected at every addition
// (10 us at any size below 128^2), took 11.1 us a launch at 128^2 and 100 us
// at 4096^2; this form 7.7 and 105 us (the large one is the coefficients' traffic: 1.4 GB
// over its eight levels), 14.4 and 12.6 us at 1024^2.
// An inactive row must hold zeros; its dinv, not yet rewritten for this
// hierarchy, says whether it held any: +0 (bit pattern 0) only on a row that
// was inactive before (or never set: the arena starts zeroed), whose
// coefficients are zero already -- most of the level, and most of its writes.
__global__ void __launch_bounds__(kBlock) k_mg_galerkin(const SceneDev* scenes, int l)
{
    static_assert(kGalCells == 64 && kBlock == 256, "a coarse row a lane, a fine row a wave");
    __shared__ double part[4][kMgStencil][kGalCells];
    const SceneDev& s = scenes[blockIdx.y];
    if (!s.active || s.precond != kPrecondMG) return;
    const auto& M = *cst(s.mg);
    if (l >= M.n) return;
    const auto& L = M.lv[l];
    const int CL = L.I * L.J, lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if ((int)blockIdx.x * kGalCells >= CL) return;
    const int c0 = blockIdx.x * kGalCells + lane, c = min(c0, CL - 1);
    gptr<const uint8_t> act = gbl<const uint8_t>(L.act);
    const bool on = c0 < CL && act[c] != 0;
    const bool clear = c0 < CL && !on && __float_as_uint(gbl<const float>(L.dinv)[c]) != 0u;
    const int ci = c / L.J, cj = c - ci * L.J;
    const bool any = __any(on);   // the block's rows: the same in every wave
    if (any) {
        double acc[kMgStencil];
#pragma unroll
        for (int k = 0; k < kMgStencil; k++) acc[k] = 0.0;
        if (l == 1) {
            if (w == 0) galerkin_part<true, 0>(s, M, l, ci, cj, acc);
            else if (w == 1) galerkin_part<true, 1>(s, M, l, ci, cj, acc);
            else if (w == 2) galerkin_part<true, 2>(s, M, l, ci, cj, acc);
            else galerkin_part<true, 3>(s, M, l, ci, cj, acc);
        } else {
            if (w == 0) galerkin_part<false, 0>(s, M, l, ci, cj, acc);
            else if (w == 1) galerkin_part<false, 1>(s, M, l, ci, cj, acc);
            else if (w == 2) galerkin_part<false, 2>(s, M, l, ci, cj, acc);
            else galerkin_part<false, 3>(s, M, l, ci, cj, acc);
        }
#pragma unroll
        for (int k = 0; k < kMgStencil; k++) part[w][k][lane] = acc[k];
    }
    __syncthreads();
    if (!on && !clear) return;
    // wave w: entries 4w .. 4w+3 and 16+4w .. 19+4w (the row has 25)
    typedef float v4 __attribute__((ext_vector_type(4)));
    gptr<float> out = gbl(L.coef) + (size_t)c * kMgRowStride;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int k0 = 16 * h + 4 * w;
        if (k0 >= kMgStencil) break;
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = min(k0 + e, kMgStencil - 1), ni = ci + k / 5 - 2, nj = cj + k % 5 - 2;
            const bool in = ni >= 0 && ni < L.I && nj >= 0 && nj < L.J;
            const bool use = act[min(max(ni, 0), L.I - 1) * L.J + min(max(nj, 0), L.J - 1)] != 0 && in && on;
            double t = 0.0;
            if (any) t = ((part[0][k][lane] + part[1][k][lane]) + part[2][k][lane]) + part[3][k][lane];
            x[e] = use ? (float)(0.25 * t) : 0.f;
        }
        if (k0 + 4 <= kMgStencil) *(gptr<v4>)(out + k0) = v4{x[0], x[1], x[2], x[3]};
        else out[k0] = x[0];   // entry 24
    }
}

// Mirror the upper entries into the lower ones (exact symmetry) and form the
// L1 diagonal.  Reads only entries k > 12, writes only k < 12 of its own row.
// Rows equal to the level's canonical interior stencil (every entry within
// 1e-5 of the canonical diagonal; other rows differ by more than 1 %) are
// flagged by a negative dinv and read the canonical stencil later.
// A block takes a 16 x 16 tile of rows: the upper entries (13..24) of the
// tile's rows and of its two-row halo are staged in LDS with row-contiguous
// loads (a row's entries share one line), so the mirrored reads, which
// touch twelve neighbouring rows each, come from LDS.
constexpr int kSymTile = 16, kSymR = kSymTile + 4, kSymUp = 13;   // 12 entries, padded to an odd stride
__device__ __forceinline__ int sym_tiles(int LI, int LJ)
{
    return ((LI + kSymTile - 1) / kSymTile) * ((LJ + kSymTile - 1) / kSymTile);
}

__device__ __forceinline__ void mg_sym_block(const SceneDev& s, int l, int bx)
{
    static_assert(kBlock == kSymTile * kSymTile, "one tile row per thread");
    if (!s.active || s.precond != kPrecondMG) return;
    const auto& M = *cst(s.mg);
    if (l >= M.n) return;
    const auto& L = M.lv[l];
    const int LI = L.I, LJ = L.J;
    if (bx >= sym_tiles(LI, LJ)) return;   // the whole block is past the level
    __shared__ float up[kSymR * kSymR][kSymUp];   // entries 13..24 of the region's rows
    const int tilesJ = (LJ + kSymTile - 1) / kSymTile;
    const int ti = bx / tilesJ, tj = bx - ti * tilesJ;
    const int ri0 = ti * kSymTile - 2, rj0 = tj * kSymTile - 2;
    gptr<float> coef = gbl(L.coef);
    typedef float v4 __attribute__((ext_vector_type(4)));
    // stage: region row q's floats 12..27 as four 16-byte loads, entries 13..24 kept
    for (int w = threadIdx.x; w < kSymR * kSymR * 4; w += kBlock) {
        const int q = w >> 2, part = w & 3;
        const int gi = ri0 + q / kSymR, gj = rj0 + q % kSymR;
        const bool in = gi >= 0 && gi < LI && gj >= 0 && gj < LJ;
        const int n = min(max(gi, 0), LI - 1) * LJ + min(max(gj, 0), LJ - 1);
        const v4 x = *(gptr<const v4>)(coef + (size_t)n * kMgRowStride + 12 + 4 * part);
        const float m = mask01(in);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = 12 + 4 * part + e;
            if (k >= 13 && k <= 24) up[q][k - 13] = x[e] * m;
        }
    }
    __syncthreads();
    const int li = threadIdx.x / kSymTile, lj = threadIdx.x % kSymTile;
    const int ci0 = ti * kSymTile + li, cj0 = tj * kSymTile + lj;
    const bool valid = ci0 < LI && cj0 < LJ;
    const int ci = min(ci0, LI - 1), cj = min(cj0, LJ - 1), c = ci * LJ + cj;
    float v[kMgStencil];
    {   // own row: entries 12..24 (and the next three floats) in four loads
        v4 o[4];
#pragma unroll
        for (int u = 0; u < 4; u++) o[u] = *(gptr<const v4>)(coef + (size_t)c * kMgRowStride + 12 + 4 * u);
#pragma unroll
        for (int k = 12; k < kMgStencil; k++) v[k] = o[(k - 12) >> 2][(k - 12) & 3];
    }
    const uint8_t av = gbl<const uint8_t>(L.act)[c];
    // lower entries: the mirrored upper entry 24 - k of neighbour k (outside
    // the level: 0, as staged)
#pragma unroll
    for (int k = 0; k < 12; k++) {
        const int q = (li + 2 + k / 5 - 2) * kSymR + (lj + 2 + k % 5 - 2);
        v[k] = up[q][(24 - k) - 13];
    }
    float cn[kMgStencil];
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) cn[k] = M.canon[l][k];
    const float tol = 1e-5f * cn[12];
    float sum = 0.f;
    bool canon_row = true;
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) {
        sum += fabsf(v[k]);
        canon_row = canon_row && fabsf(v[k] - cn[k]) <= tol;
    }
    const bool act = av != 0;
    // an inactive row is all zero already (k_mg_galerkin), mirrored entries
    // included; the lower entries go out as three 16-byte stores
    if (valid && act) {
#pragma unroll
        for (int u = 0; u < 3; u++) {
            const v4 x = {v[4 * u], v[4 * u + 1], v[4 * u + 2], v[4 * u + 3]};
            *(gptr<v4>)(coef + (size_t)c * kMgRowStride + 4 * u) = x;
        }
    }
    const float di = (act && sum > 0.f) ? kMgOmega / sum : 0.f;
    if (valid) gbl(L.dinv)[c] = (canon_row && di > 0.f) ? -di : (act && di == 0.f ? -0.f : di);
    // active rows that will read their stored coefficients (for the kernels'
    // byte counts): one atomic per block, once per solve
    const int stored = __syncthreads_count(valid && di > 0.f && !canon_row);
    if (threadIdx.x == 0 && stored) atomicAdd(&s.sc->mg_stored[l], stored);
}

__global__ void __launch_bounds__(kBlock) k_mg_sym(const SceneDev* scenes, int l)
{
    mg_sym_block(scenes[blockIdx.y], l, blockIdx.x);
}

// k_mg_sym of level l (blocks [0, nsym)) and k_mg_mark of level l+1 (the
// rest) in one launch: they touch different arrays, and both must be done
// before the Galerkin product of level l+1.
__global__ void __launch_bounds__(kBlock) k_mg_symmark(const SceneDev* scenes, int l, int nsym)
{
    const SceneDev& s = scenes[blockIdx.y];
    if ((int)blockIdx.x < nsym) mg_sym_block(s, l, blockIdx.x);
    else mg_mark_block(s, l + 1, blockIdx.x - nsym);
}

// ---------------------------------------------------------------------------
// the V-cycle: z = M r, r the current PCG residual (which: 0 = cr, 1 = cr2).
// Each kernel takes its scenes and blocks from a block map (flat launch over
// the packed iterating scenes) or from a (blocks, scenes) grid.  All loads
// of a thread are unconditional (clamped indices, masked afterwards) so they
// issue together; the kernels are latency-bound.
// ---------------------------------------------------------------------------

// Level 0 -> 1: x0 = w r / D1 on the fine level, res0 = r - A' x0, and
// r1 = R res0 over each level-1 cell's 4x4 fine support.  A block owns a
// kD0Tile x kD0Tile tile of level-1 cells (mg_d0_tiles blocks a scene) and
// stages its fine patch (the supports with the stencil's reach, kD0R cells
// a side) in LDS: code and r, then x0 once per fine cell, then res0 once
// per fine cell of the supports, then each thread sums its cell's 16
// weighted res0.  Each value is formed by the same expression as it would
// be per coarse cell, so r1 does not depend on the tiling.
// kStep: the PCG step that makes r, fused: alpha from the partials of p.q,
// r = r_old - alpha q over the patch (its halo formed again by each of the
// tiles that need it, from the same values), r and x += alpha p (FP64)
// written for the tile's own 2 kD0Tile x 2 kD0Tile fine cells.  On its own
// that step is a launch that moves 32 B a cell and whose r this one reads
// back; together 33 B, 27 % more of r_old, q and the code for the halo, and
// one launch of an iteration's latency chain less: 9.4 -> 6.5 us at 128^2,
// 94 -> 83 us at 4096^2 (the two kernels, this one).
constexpr int kD0R = 2 * kD0Tile + 4;
template <bool kStep>
__device__ __forceinline__ void mg_down0_tile(const SceneDev* scenes, const int2* map, int arg)
{
    static_assert(kD0Tile * kD0Tile == kBlock, "one level-1 cell per thread");
    __shared__ float xs[kD0R][kD0R + 1];   // x0
    __shared__ float rs[kD0R][kD0R + 1];   // r, then res0 (own cell only)
    __shared__ uint8_t cs[kD0R][kD0R + 4];
    const SceneBlock sb = scene_block(map, true);
    const SceneDev& s = scenes[sb.scene];
    cptr<SceneScalars> scr = cst(s.sc);
    const auto& L1 = cst(s.mg)->lv[1];
    const int I1 = L1.I, J1 = L1.J;
    const int tjn = (J1 + kD0Tile - 1) / kD0Tile;
    // one test after the uniform loads, so that they issue together; the
    // whole block takes it
    if (!mg_iterating(s) | (sb.block >= mg_d0_tiles(I1, J1))) return;
    const int ti = sb.block / tjn, tj = sb.block - ti * tjn;
    const int I = s.I, J = s.J;
    const int fi0 = 2 * kD0Tile * ti - 2, fj0 = 2 * kD0Tile * tj - 2;   // the patch's first fine cell
    const int it = arg;
    gptr<const float> r = gbl<const float>(kStep ? ((it & 1) ? s.cr2 : s.cr) : (arg ? s.cr2 : s.cr));
    gptr<float> rnew = gbl((it & 1) ? s.cr : s.cr2);
    gptr<const float> q = gbl<const float>(s.cw);
    gptr<const float> p = gbl<const float>((it & 1) ? s.cs1 : s.cp);
    gptr<double> x = gbl(s.x64);
    gptr<const uint8_t> code = gbl<const uint8_t>(s.stencil);
    {   // code, r and x0 of the patch (outside the grid: code 0, r 0)
        constexpr int Q = (kD0R * kD0R + kBlock - 1) / kBlock;
        uint8_t kq[Q];
        float vq[Q], qq[Q], pq[Q];
        double xq[Q];
#pragma unroll
        for (int u = 0; u < Q; u++) {
            const int k = min((int)threadIdx.x + u * kBlock, kD0R * kD0R - 1);
            const int a = k / kD0R, b = k % kD0R;
            const int f = min(max(fi0 + a, 0), I - 1) * J + min(max(fj0 + b, 0), J - 1);   // clamped, not selected
            kq[u] = code[f];
            vq[u] = r[f];
            if constexpr (kStep) {
                qq[u] = q[f];
                // x and p are the own cells' alone: a halo lane loads an own cell's
                const int g = min(max(fi0 + min(max(a, 2), kD0R - 3), 0), I - 1) * J +
                              min(max(fj0 + min(max(b, 2), kD0R - 3), 0), J - 1);
                xq[u] = x[g];
                pq[u] = p[g];
            }
        }
        float alpha = 0.f;
        if constexpr (kStep) {
            double t[1];
            sum_partials<1>(s, kSlotPQ, s.up_blocks, t);   // k_pcg_dir's
            const bool lead = sb.block == 0 && threadIdx.x == 0;
            if (!(t[0] > 0.0) || !finite_d(t[0])) {   // breakdown: end this sweep (every block sees it)
                if (lead) s.sc->inner_done = 1;
                return;
            }
            alpha = (float)(scr->gamma[it & 1] / t[0]);
            if (lead) {
                s.sc->inner_iters = it + 1;
                s.sc->total_iters += 1;
            }
        }
#pragma unroll
        for (int u = 0; u < Q; u++) {
            const int k0 = threadIdx.x + u * kBlock;
            if (k0 >= kD0R * kD0R) break;
            const int a = k0 / kD0R, b = k0 % kD0R;
            const int fi = fi0 + a, fj = fj0 + b;
            const bool in = fi >= 0 && fi < I && fj >= 0 && fj < J;
            const uint8_t k = in ? kq[u] : 0;
            float rv = vq[u];
            if constexpr (kStep) {
                rv = rv - alpha * qq[u];
                if (in && a >= 2 && a < kD0R - 2 && b >= 2 && b < kD0R - 2) {
                    const int f = fi * J + fj;
                    rnew[f] = rv;
                    x[f] = xq[u] + (double)alpha * (double)pq[u];
                }
            }
            rv = rv * mask01(in);
            const float d = l1_diag0(k);
            xs[a][b] = ((k & 0x80) && d > 0.f) ? kMgOmega * rv / d : 0.f;
            rs[a][b] = rv;
            cs[a][b] = k;
        }
    }
    __syncthreads();
    // res0 on the supports (patch cells 1 .. kD0R-2 each way); 0 off fluid rows
    for (int q = threadIdx.x; q < (kD0R - 2) * (kD0R - 2); q += kBlock) {
        const int a = 1 + q / (kD0R - 2), b = 1 + q % (kD0R - 2);
        const uint8_t k = cs[a][b];
        float ax = (float)((k >> 4) & 7) * xs[a][b];
        ax -= (k & 1) ? xs[a - 1][b] : 0.f;
        ax -= (k & 2) ? xs[a + 1][b] : 0.f;
        ax -= (k & 4) ? xs[a][b - 1] : 0.f;
        ax -= (k & 8) ? xs[a][b + 1] : 0.f;
        rs[a][b] = (k & 0x80) ? rs[a][b] - ax : 0.f;
    }
    __syncthreads();
    const int li = threadIdx.x / kD0Tile, lj = threadIdx.x % kD0Tile;
    const int ci = ti * kD0Tile + li, cj = tj * kD0Tile + lj;
    if ((ci >= I1) | (cj >= J1)) return;
    const int c = ci * J1 + cj;
    if (!gbl<const uint8_t>(L1.act)[c]) {   // inactive coarse cell: nothing to restrict
        gbl(L1.r)[c] = 0.f;
        return;
    }
    float acc = 0.f;
#pragma unroll
    for (int a = 1; a < 5; a++)
#pragma unroll
        for (int b = 1; b < 5; b++) {
            const uint8_t k = cs[2 * li + a][2 * lj + b];
            acc += (k & 0x80) ? (w1(a - 1) * w1(b - 1)) * rs[2 * li + a][2 * lj + b] : 0.f;
        }
    gbl(L1.r)[c] = 0.25f * acc;
}

// r as it is (which: 0 = cr, 1 = cr2): the V-cycle that starts a sweep
__global__ void __launch_bounds__(kBlock) k_mg_down0(const SceneDev* scenes, const int2* map, int which)
{
    mg_down0_tile<false>(scenes, map, which);
}

// the step of PCG iteration it, then its V-cycle's first part
__global__ void __launch_bounds__(kBlock) k_mg_step0(const SceneDev* scenes, const int2* map, int it)
{
    mg_down0_tile<true>(scenes, map, it);
}

// Level l (1 <= l < t): x = r * dinv, y = res = r - A_l x.
__global__ void __launch_bounds__(kBlock) k_mg_resid(const SceneDev* scenes, const int2* map, int l)
{
    const SceneBlock sb = scene_block(map, true);
    const SceneDev& s = scenes[sb.scene];
    const auto& M = *cst(s.mg);
    const auto& L = M.lv[l];
    const int LI = L.I, LJ = L.J, CL = LI * LJ;
    const int c = sb.block * kBlock + threadIdx.x;
    if (!mg_iterating(s) | (l >= M.t) | (c >= CL)) return;   // l >= t: in k_mg_coarse
    gptr<const float> r = gbl<const float>(L.r), dinv = gbl<const float>(L.dinv);
    const float dc = dinv[c];
    if (dc == 0.f) {   // inactive row: r = 0 and no coefficients
        gbl(L.y)[c] = 0.f;
        return;
    }
    const int ci = c / LJ, cj = c - ci * LJ;
    float xv[kMgStencil];
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) {
        const int ni = ci + k / 5 - 2, nj = cj + k % 5 - 2;
        const bool ok = ni >= 0 && ni < LI && nj >= 0 && nj < LJ;
        const int n = min(max(ni, 0), LI - 1) * LJ + min(max(nj, 0), LJ - 1);   // clamped, not selected
        const float rn = r[n], dn = dinv[n];
        xv[k] = (rn * fabsf(dn)) * mask01(ok);   // a 0/1 factor, not a select: the load stays unconditional
    }
    const float rc = r[c];
    const float ax = row_dot(M, l, gbl<const float>(L.coef), c, dc, xv);
    gbl(L.y)[c] = rc - ax;
}

// Level l-1 -> l (2 <= l < t): r_l = R y_{l-1}.
__global__ void __launch_bounds__(kBlock) k_mg_restrict(const SceneDev* scenes, const int2* map, int l)
{
    const SceneBlock sb = scene_block(map, true);
    const SceneDev& s = scenes[sb.scene];
    const auto& M = *cst(s.mg);
    const auto& L = M.lv[l];
    const auto& F = M.lv[l - 1];
    const int LJ = L.J, FI = F.I, FJ = F.J;
    const int c = sb.block * kBlock + threadIdx.x;
    if (!mg_iterating(s) | (l >= M.t) | (c >= L.I * LJ)) return;   // l >= t: in k_mg_coarse
    gptr<const float> fy = gbl<const float>(F.y);
    if (!gbl<const uint8_t>(L.act)[c]) {
        gbl(L.r)[c] = 0.f;
        return;
    }
    const int ci = c / LJ, cj = c - ci * LJ;
    gbl(L.r)[c] = restrict_at(fy, FI, FJ, ci, cj);
}

// Levels t .. n-1 of one scene in one block (t = MgLevels::t, chosen so
// that level t has at most kMgCoarseTop = kMgCoarseThreads cells and levels
// t .. n-1 at most kMgCoarseCells together): r_t = R y_{t-1} (r_1 comes
// from k_mg_down0 when t = 1), the down steps of k_mg_resid and
// k_mg_restrict to the bottom, kMgBottomSweeps L1-Jacobi sweeps from zero
// there, then the up steps of k_mg_prolong and k_mg_post back to level t,
// whose y it writes for the level above.  The arithmetic and its order are
// those of the per-level kernels, so where t falls does not change z.
// Thread c owns cell c of every level.  One CU runs the whole block, so it
// is bound by instruction issue (16 waves on four SIMDs) and by latency:
//   - global loads come in two rounds, every level's dinv with level t's
//     input (its 4x4 patch of y_{t-1}) and the bottom's rows, then the
//     stored coefficient rows of the thread's level-t cell; a level's 25
//     coefficients stay in registers for the way down and the way up;
//   - every level's x and y lie in LDS with a two-cell halo of zeros
//     (dynamic LDS, MgLevels::thalo floats each, cleared while the first
//     loads are in flight), so a stencil, a restriction and a prolongation
//     read at fixed offsets from the cell, with no bounds tests or masks (a
//     halo zero adds what the masked clamped value did);
//   - the bottom's sweeps alternate between its x and y, the first from
//     zero without its stencil.
// Masked and clamped addresses for each of the 25 terms, and the bottom's
// coefficients read from LDS in every sweep, took 13.8 us a launch at
// 32 x 32 over 16 x 16 cells; this form 9.7 us (the 128^2 dam break).
__device__ __forceinline__ bool mg_active(float dinv) { return __float_as_uint(dinv) != 0u; }

// sum_k a_k x_k over the 5x5 neighbourhood of x[home], rows w floats apart
__device__ __forceinline__ float coarse_dot(const float (&a)[kMgStencil], const float* x, int home, int w)
{
    float ax = 0.f;
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) ax += a[k] * x[home + (k / 5 - 2) * w + (k % 5 - 2)];
    return ax;
}

__global__ void __launch_bounds__(kMgCoarseThreads) k_mg_coarse(const SceneDev* scenes)
{
    constexpr int NT = kMgCoarseThreads;
    static_assert(kMgBottomMax * kMgBottomMax <= NT, "one bottom cell per thread");
    static_assert(kMgCoarseTop <= NT, "one level-t cell per thread");
    static_assert(kMgBottomSweeps % 2 == 0, "the bottom's last sweep writes its y");
    __shared__ float rs[kMgCoarseCells], ds[kMgCoarseCells];
    extern __shared__ float4 halo4[];
    const SceneDev& s = scenes[blockIdx.y];
    const auto& M = *cst(s.mg);
    const int t = M.t, nb = M.n - 1;
    if (!mg_iterating(s)) return;
    const int tid = threadIdx.x;
    const int HT = M.thalo;   // a multiple of 4
    float* const hx = reinterpret_cast<float*>(halo4);
    float* const hy = hx + HT;
    const auto& T = M.lv[t];
    const auto& B = M.lv[nb];
    const int TI = T.I, TJ = T.J, CT = TI * TJ;   // roff[t] = 0
    const bool tin = tid < CT;
    const int tc = tin ? tid : CT - 1;
    const int tci = tc / TJ, tcj = tc - tci * TJ;
    const int CB = B.I * B.J, ob = M.roff[nb];   // CB <= kMgBottomMax^2 (the hierarchy stops there)
    const bool bin = tid < CB;
    // round 1: dinv of levels t .. n-1 (contiguous), level t's input, and the
    // bottom's rows, whose sweeps read the stored coefficients of every row
    float dt, cb[kMgStencil];
    {
        gptr<const float> dg = gbl<const float>(T.dinv);
        const int TC = M.tcells;
        constexpr int Q = (kMgCoarseCells + NT - 1) / NT;
        float dv[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) dv[q] = dg[min(tid + q * NT, TC - 1)];
        float rt;
        if (t > 1) {   // r_t = R y_{t-1} from the launch before
            const auto& F = M.lv[t - 1];
            rt = restrict_at(gbl<const float>(F.y), F.I, F.J, tci, tcj);
        } else {
            rt = gbl<const float>(M.lv[1].r)[tc];
        }
#pragma unroll
        for (int k = 0; k < kMgStencil; k++) cb[k] = 0.f;
        if (bin) load_coef_row(gbl<const float>(B.coef), tid, cb);
        for (int k = tid; k < HT / 2; k += NT) halo4[k] = make_float4(0.f, 0.f, 0.f, 0.f);   // hx and hy
        __syncthreads();
        dt = dv[0];   // level t's dinv of cell tc
#pragma unroll
        for (int q = 0; q < Q; q++)
            if (tid + q * NT < TC) ds[tid + q * NT] = dv[q];
        if (tin) {
            const float r = (t == 1 || mg_active(dt)) ? rt : 0.f;
            rs[tc] = r;
            if (t < nb) hx[(tci + 2) * (TJ + 4) + tcj + 2] = r * fabsf(dt);   // x = r dinv
        }
    }
    // round 2: this thread's level-t row
    float ct[kMgStencil];
    if (t < nb) row_load(M, t, gbl<const float>(T.coef), tc, tin ? dt : 0.f, ct);
    __syncthreads();
    int ho = 0;   // level l's place in hx and hy
    for (int l = t; l < nb; l++) {   // down: y = r - A x, r_{l+1} = R y, x_{l+1} = r_{l+1} dinv
        const auto& L = M.lv[l];
        const int LJ = L.J, CL = L.I * LJ, o = M.roff[l], w = LJ + 4;
        if (tid < CL) {
            const float dc = ds[o + tid];
            const int ci = tid / LJ, cj = tid - ci * LJ, home = ho + (ci + 2) * w + cj + 2;
            float y = 0.f;   // inactive row: r = 0 and no coefficients
            if (dc != 0.f) {
                float ax;
                if (l == t) {
                    ax = coarse_dot(ct, hx, home, w);
                } else {
                    float a[kMgStencil];
                    row_load(M, l, gbl<const float>(L.coef), tid, dc, a);
                    ax = coarse_dot(a, hx, home, w);
                }
                y = rs[o + tid] - ax;
            }
            hy[home] = y;
        }
        __syncthreads();
        const auto& N = M.lv[l + 1];
        const int NJ = N.J, NC = N.I * NJ, on = M.roff[l + 1], hn = ho + (L.I + 4) * w;
        if (tid < NC) {   // restrict_at on the halo
            const int ci = tid / NJ, cj = tid - ci * NJ;
            const float dn = ds[on + tid];
            const float* const f = hy + ho + (2 * ci + 1) * w + 2 * cj + 1;   // fine cell (2 ci - 1, 2 cj - 1)
            float acc = 0.f;
#pragma unroll
            for (int a = 0; a < 4; a++)
#pragma unroll
                for (int b = 0; b < 4; b++) acc += (w1(a) * w1(b)) * f[a * w + b];
            const float r = mg_active(dn) ? 0.25f * acc : 0.f;
            rs[on + tid] = r;
            if (l + 1 < nb) hx[hn + (ci + 2) * (NJ + 4) + cj + 2] = r * fabsf(dn);
        }
        ho = hn;
        __syncthreads();
    }
    {   // bottom: y = kMgBottomSweeps sweeps of x += dinv (r - A x) from 0
        const int w = B.J + 4, ci = tid / B.J, cj = tid - ci * B.J, home = ho + (ci + 2) * w + cj + 2;
        const float dv = bin ? fabsf(ds[ob + tid]) : 0.f, rv = bin ? rs[ob + tid] : 0.f;
        float x = 0.f + dv * (rv - 0.f);
        if (bin) hx[home] = x;
        __syncthreads();
#pragma unroll 1
        for (int sw = 1; sw < kMgBottomSweeps; sw++) {
            const float* const from = (sw & 1) ? hx : hy;
            float* const to = (sw & 1) ? hy : hx;
            if (bin) {
                x = x + dv * (rv - coarse_dot(cb, from, home, w));
                to[home] = x;
            }
            __syncthreads();
        }
        if (bin && nb == t) gbl(B.y)[tid] = x;
    }
    for (int l = nb - 1; l >= t; l--) {   // up: x = r dinv + P y_{l+1}, y = x + dinv (r - A x)
        const auto& L = M.lv[l];
        const auto& N = M.lv[l + 1];
        const int LJ = L.J, CL = L.I * LJ, o = M.roff[l], w = LJ + 4, wn = N.J + 4;
        const int hn = ho;
        ho -= (L.I + 4) * w;
        const int ci = tid / LJ, cj = tid - ci * LJ, home = ho + (ci + 2) * w + cj + 2;
        const float dc = tid < CL ? ds[o + tid] : 0.f, rc = tid < CL ? rs[o + tid] : 0.f;
        float x = 0.f;
        if (tid < CL) {
            if (mg_active(dc)) {   // prolong_at on the halo
                const int p0 = (ci >> 1) + 2, q0 = (cj >> 1) + 2;
                const int p1 = (ci & 1) ? p0 + 1 : p0 - 1, q1 = (cj & 1) ? q0 + 1 : q0 - 1;
                const float* const f = hy + hn;
                float acc = 0.f;
                acc += (0.75f * 0.75f) * f[p0 * wn + q0];
                acc += (0.75f * 0.25f) * f[p0 * wn + q1];
                acc += (0.25f * 0.75f) * f[p1 * wn + q0];
                acc += (0.25f * 0.25f) * f[p1 * wn + q1];
                x = rc * fabsf(dc) + acc;
            }
            hx[home] = x;
        }
        __syncthreads();
        if (tid < CL) {
            float y = 0.f;   // inactive row: x = 0
            if (dc != 0.f) {
                float ax;
                if (l == t) {
                    ax = coarse_dot(ct, hx, home, w);
                } else {
                    float a[kMgStencil];
                    row_load(M, l, gbl<const float>(L.coef), tid, dc, a);
                    ax = coarse_dot(a, hx, home, w);
                }
                y = x + fabsf(dc) * (rc - ax);
            }
            hy[home] = y;
            if (l == t) gbl(L.y)[tid] = y;
        }
        if (l > t) __syncthreads();
    }
}

// The fused V-cycle levels (the default; the per-level kernels above and
// below stay for comparison, fg_ctx_set_vcycle_fused).  A block owns a
// kTile x kTile tile of cells and stages what its cells' stencils reach in
// LDS, so a level's two steps take one launch instead of two.  Every value
// is formed by the expression the per-level kernels use, at the same clamped
// coordinates and with the same 0/1 masks, so z keeps its bits.
static_assert(kVcTile * kVcTile == kBlock, "one cell of the tile per thread");
// Each is one short chain of memory round trips (launches of 64 to 1,400
// blocks; the arithmetic is a microsecond), so a thread issues everything it
// can name at once -- its patch positions, its own row's r and dinv -- before
// the stop flags are looked at, and its stored coefficients as soon as dinv
// says that it has some, ahead of the staging and its barrier.
// Launches over a block map (several scenes) look at the flags first: between
// two polls part of the scenes have stopped, and without the test ahead of
// them the early loads moved 4.2 bytes per algorithmic byte of k_mg_rr, 3.5 of
// k_mg_pp and 3.1 of k_pcg_dir on the 256 mixed scenes (1.4, 1.1 and 1.1 with
// it), 8.2, 6.3 and 15.9 us a launch against 7.9, 6.0 and 15.4.
constexpr int kRRY = 2 * kRRTile + 2;   // fine cells a side whose residual the restriction reads
constexpr int kRRX = kRRY + 4;          // and the x their stencils read
static_assert(kRRY * kRRY == kBlock, "one fine residual per thread: a second round would be a second chain");
constexpr int kPPX = kVcTile + 4;       // level-l cells a side whose x the post-smoothing reads

// Level l (1 <= l < t), down: x = r dinv and y = r - A_l x over the fine
// patch of a kRRTile x kRRTile tile of level-(l+1) cells, then r_{l+1} = R y
// for the tile's cells (l + 1 < t) or y written out for k_mg_coarse to
// restrict (l + 1 = t).  The tile is smaller than k_mg_pp's: each fine
// residual is a 25-term row with its own coefficient loads, and the tile of 7
// gives each thread exactly one (8 x 8 had a second round for 68 of 324).
// x outside level l is staged as 0 (the per-level kernels mask it); y there
// holds the value of its clamped cell and is masked.
// Averages over levels 1-4 of the 1024^2 dam break: 5.1 us a launch with the
// 8 x 8 tile and the loads after the flags, 4.1 us so; k_mg_pp 4.2 and 4.0 us.
__global__ void __launch_bounds__(kBlock) k_mg_rr(const SceneDev* scenes, const int2* map, int l)
{
    __shared__ float xs[kRRX][kRRX + 1];
    __shared__ float ys[kRRY][kRRY + 1];
    const SceneBlock sb = scene_block(map, true);
    const SceneDev& s = scenes[sb.scene];
    const auto& M = *cst(s.mg);
    // a level the scene does not launch (another one of the group does)
    if ((s.active == 0) | (s.precond != kPrecondMG) | (l + 1 > M.t)) return;
    if (map && !mg_iterating(s)) return;   // of several scenes: see kRRY
    const auto& L = M.lv[l];
    const auto& N = M.lv[l + 1];
    const int LI = L.I, LJ = L.J, NI = N.I, NJ = N.J;
    const int tjn = (NJ + kRRTile - 1) / kRRTile;
    if (sb.block >= ((NI + kRRTile - 1) / kRRTile) * tjn) return;
    const int ti = sb.block / tjn, tj = sb.block - ti * tjn;
    const int yi0 = 2 * kRRTile * ti - 1, yj0 = 2 * kRRTile * tj - 1;   // the residual patch's first fine cell
    const int xi0 = yi0 - 2, xj0 = yj0 - 2;
    gptr<const float> r = gbl<const float>(L.r), dinv = gbl<const float>(L.dinv);
    constexpr int Q = (kRRX * kRRX + kBlock - 1) / kBlock;
    float rq[Q], dq[Q];
#pragma unroll
    for (int u = 0; u < Q; u++) {
        const int q = min((int)threadIdx.x + u * kBlock, kRRX * kRRX - 1);
        const int fi = min(max(xi0 + q / kRRX, 0), LI - 1), fj = min(max(xj0 + q % kRRX, 0), LJ - 1);
        rq[u] = r[fi * LJ + fj];
        dq[u] = dinv[fi * LJ + fj];
    }
    // this thread's residual (at the clamped cell of its position) and its
    // coarse cell's activity
    const int ya = threadIdx.x / kRRY, yb = threadIdx.x % kRRY;
    const int ci = min(max(yi0 + ya, 0), LI - 1), cj = min(max(yj0 + yb, 0), LJ - 1), c = ci * LJ + cj;
    float dc = dinv[c], rc = r[c];
    const int ni = kRRTile * ti + (int)threadIdx.x / kRRTile, nj = kRRTile * tj + (int)threadIdx.x % kRRTile;
    const bool coarse = (int)threadIdx.x < kRRTile * kRRTile && ni < NI && nj < NJ;
    int na = gbl<const uint8_t>(N.act)[coarse ? ni * NJ + nj : 0];
#pragma unroll
    for (int u = 0; u < Q; u++) asm volatile("" : "+v"(rq[u]), "+v"(dq[u]));
    asm volatile("" : "+v"(dc), "+v"(rc), "+v"(na));
    if (!mg_iterating(s)) return;
    float a[kMgStencil];
    row_load(M, l, gbl<const float>(L.coef), c, dc, a);
#pragma unroll
    for (int u = 0; u < Q; u++) {
        const int q = threadIdx.x + u * kBlock, fi = xi0 + q / kRRX, fj = xj0 + q % kRRX;
        const bool ok = fi >= 0 && fi < LI && fj >= 0 && fj < LJ;
        if (q < kRRX * kRRX) xs[q / kRRX][q % kRRX] = ok ? rq[u] * fabsf(dq[u]) : 0.f;
    }
    __syncthreads();
    {
        float y = 0.f;   // inactive row: r = 0 and no coefficients
        if (dc != 0.f) {
            float xv[kMgStencil];
#pragma unroll
            for (int k = 0; k < kMgStencil; k++) xv[k] = xs[ci - xi0 + k / 5 - 2][cj - xj0 + k % 5 - 2];
            y = rc - row_sum(a, xv);
        }
        ys[ya][yb] = y;
    }
    __syncthreads();
    if (l + 1 < M.t) {   // r_{l+1} = R y (restrict_at on the patch)
        if (!coarse) return;
        const int n = ni * NJ + nj, li = threadIdx.x / kRRTile, lj = threadIdx.x % kRRTile;
        if (!na) {
            gbl(N.r)[n] = 0.f;
            return;
        }
        float acc = 0.f;
#pragma unroll
        for (int p = 0; p < 4; p++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int fi = 2 * ni - 1 + p, fj = 2 * nj - 1 + q;
                const bool ok = fi >= 0 && fi < LI && fj >= 0 && fj < LJ;
                acc += ((w1(p) * w1(q)) * ys[2 * li + p][2 * lj + q]) * mask01(ok);
            }
        gbl(N.r)[n] = 0.25f * acc;
    } else {   // level t's input: y of the tile's own fine cells
        const int q = threadIdx.x;
        if (q >= 4 * kRRTile * kRRTile) return;
        const int p = q / (2 * kRRTile), b = q % (2 * kRRTile);
        const int fi = 2 * kRRTile * ti + p, fj = 2 * kRRTile * tj + b;
        if ((fi < LI) & (fj < LJ)) gbl(L.y)[fi * LJ + fj] = ys[p + 1][b + 1];
    }
}

// Level l (1 <= l < t), up: x = r dinv + P y_{l+1} over a tile of level-l
// cells and its two-cell halo (0 outside the level), then y = x + dinv (r -
// A_l x) for the tile.
__global__ void __launch_bounds__(kBlock) k_mg_pp(const SceneDev* scenes, const int2* map, int l)
{
    __shared__ float xs[kPPX][kPPX + 1];
    const SceneBlock sb = scene_block(map, true);
    const SceneDev& s = scenes[sb.scene];
    const auto& M = *cst(s.mg);
    if ((s.active == 0) | (s.precond != kPrecondMG) | (l >= M.t)) return;
    if (map && !mg_iterating(s)) return;   // of several scenes: see kRRY
    const auto& L = M.lv[l];
    const auto& Cl = M.lv[l + 1];
    const int LI = L.I, LJ = L.J;
    const int tjn = (LJ + kVcTile - 1) / kVcTile;
    if (sb.block >= ((LI + kVcTile - 1) / kVcTile) * tjn) return;
    const int ti = sb.block / tjn, tj = sb.block - ti * tjn;
    const int xi0 = kVcTile * ti - 2, xj0 = kVcTile * tj - 2;
    gptr<const float> r = gbl<const float>(L.r), dinv = gbl<const float>(L.dinv);
    gptr<const uint8_t> act = gbl<const uint8_t>(L.act);
    gptr<const float> yc = gbl<const float>(Cl.y);
    const int li = threadIdx.x / kVcTile, lj = threadIdx.x % kVcTile;
    const int ci = kVcTile * ti + li, cj = kVcTile * tj + lj;
    const bool in = (ci < LI) & (cj < LJ);
    const int c = min(ci, LI - 1) * LJ + min(cj, LJ - 1);
    float dc = dinv[c], rc = r[c];
    constexpr int Q = (kPPX * kPPX + kBlock - 1) / kBlock;
    float rq[Q], dq[Q], pq[Q];
    int aq[Q];
#pragma unroll
    for (int u = 0; u < Q; u++) {
        const int q = min((int)threadIdx.x + u * kBlock, kPPX * kPPX - 1);
        const int fi = min(max(xi0 + q / kPPX, 0), LI - 1), fj = min(max(xj0 + q % kPPX, 0), LJ - 1);
        aq[u] = act[fi * LJ + fj];
        rq[u] = r[fi * LJ + fj];
        dq[u] = dinv[fi * LJ + fj];
        pq[u] = prolong_at(yc, Cl.I, Cl.J, fi, fj);
    }
    asm volatile("" : "+v"(dc), "+v"(rc));
    if (!mg_iterating(s)) return;
    float a[kMgStencil];
    row_load(M, l, gbl<const float>(L.coef), c, in ? dc : 0.f, a);
#pragma unroll
    for (int u = 0; u < Q; u++) {
        const int q = threadIdx.x + u * kBlock, fi = xi0 + q / kPPX, fj = xj0 + q % kPPX;
        const bool ok = fi >= 0 && fi < LI && fj >= 0 && fj < LJ;
        if (q < kPPX * kPPX) xs[q / kPPX][q % kPPX] = ok && aq[u] ? rq[u] * fabsf(dq[u]) + pq[u] : 0.f;
    }
    __syncthreads();
    if (!in) return;
    if (dc == 0.f) {   // inactive row: x = 0
        gbl(L.y)[c] = 0.f;
        return;
    }
    float xv[kMgStencil];
#pragma unroll
    for (int k = 0; k < kMgStencil; k++) xv[k] = xs[li + k / 5][lj + k % 5];
    gbl(L.y)[c] = xv[12] + fabsf(dc) * (rc - row_sum(a, xv));
}

// Level l (1 <= l < t), up: x = r * dinv + P y_{l+1}.
__global__ void __launch_bounds__(kBlock) k_mg_prolong(const SceneDev* scenes, const int2* map, int l)
{
    const SceneBlock sb = scene_block(map, true);
    const SceneDev& s = scenes[sb.scene];
    const auto& M = *cst(s.mg);
    const auto& L = M.lv[l];
    const auto& Cl = M.lv[l + 1];
    const int LJ = L.J;
    const int c = sb.block * kBlock + threadIdx.x;
    if (!mg_iterating(s) | (l >= M.t) | (c >= L.I * LJ)) return;   // l >= t: in k_mg_coarse
    if (!gbl<const uint8_t>(L.act)[c]) {
        gbl(L.x)[c] = 0.f;
        return;
    }
    const int ci = c / LJ, cj = c - ci * LJ;
    const float rc = gbl<const float>(L.r)[c], dc = gbl<const float>(L.dinv)[c];
    const float pc = prolong_at(gbl<const float>(Cl.y), Cl.I, Cl.J, ci, cj);
    gbl(L.x)[c] = rc * fabsf(dc) + pc;
}

// Level l (1 <= l < t), up: y = x + dinv (r - A_l x).
__global__ void __launch_bounds__(kBlock) k_mg_post(const SceneDev* scenes, const int2* map, int l)
{
    const SceneBlock sb = scene_block(map, true);
    const SceneDev& s = scenes[sb.scene];
    const auto& M = *cst(s.mg);
    const auto& L = M.lv[l];
    const int LI = L.I, LJ = L.J, CL = LI * LJ;
    const int c = sb.block * kBlock + threadIdx.x;
    if (!mg_iterating(s) | (l >= M.t) | (c >= CL)) return;   // l >= t: in k_mg_coarse
    gptr<const float> x = gbl<const float>(L.x);
    const float dc = gbl<const float>(L.dinv)[c];
    if (dc == 0.f) {   // inactive row: x = 0
        gbl(L.y)[c] = 0.f;
        return;
    }
    const int ci = c / LJ, cj = c - ci * LJ;
    float xv[kMgStencil];
    gather25(x, LI, LJ, ci, cj, xv);
    const float rc = gbl<const float>(L.r)[c];
    const float ax = row_dot(M, l, gbl<const float>(L.coef), c, dc, xv);
    gbl(L.y)[c] = xv[12] + fabsf(dc) * (rc - ax);
}

// Level 0, up: z0 = w r / D1 + P y1 at the cell and its fluid neighbours, then
// z = z0 + w (r - A' z0) / D1; z = r on non-fluid rows.  Writes z and the
// partials of r.z and r.r the next PCG iteration reduces.
// A block owns kUpTile x kUpTile tiles of the grid (one, or a run of
// consecutive ones: SceneDev::up_blocks blocks a scene, a partial each) and
// stages in LDS the tile with a one-cell halo, code and r, and the level-1
// patch under it, so z0 is formed once per cell (and once more per halo
// cell) from LDS instead of five times from 30 global loads, which bound
// the per-cell form by instruction issue.  The quotients by D1, an integer up
// to kMaxD1, are a product with its reciprocal and one step with the exact
// remainder: the division's result, but for a remainder that is subnormal
// (an ulp of it) and an infinite residual (NaN; the solve ends as it does
// for infinity).  A tile is the fine side of
// k_mg_step0's and k_pcg_dir's, in their order, so what one writes the
// other reads through the same XCD's L2.  Per-cell form (each cell its
// neighbours' z0) 8.3 us at 128^2, 10.1 us at 1024^2; an LDS window of whole
// rows over linear chunks 97 us at 4096^2; this form 4.8, 7.3 and 36 us.
constexpr int kMaxD1 = 11;               // a code's count (three bits; 4 where materials made it) and four neighbours
static_assert(kUpTile % 2 == 0 && kUpTile * kUpTile % kBlock == 0 && kBlock % kUpTile == 0, "whole rows of a tile a pass");

__global__ void __launch_bounds__(kBlock) k_mg_up0(const SceneDev* scenes, const int2* map, int which)
{
    __shared__ float zs[kUpR][kUpR + 1];     // z0
    __shared__ float rs[kUpR][kUpR + 1];
    __shared__ uint8_t cs[kUpR][kUpR + 2];
    __shared__ float ys[kUpY][kUpY + 1];
    __shared__ float inv[kMaxD1 + 1];        // 1 / D1
    const SceneBlock sb = scene_block(map, true);
    const SceneDev& s = scenes[sb.scene];
    const auto& L1 = cst(s.mg)->lv[1];
    if (!mg_iterating(s) | (sb.block >= s.up_blocks)) return;
    const int I = s.I, J = s.J, I1 = L1.I, J1 = L1.J;
    gptr<const float> y1 = gbl<const float>(L1.y);
    gptr<const float> r = gbl<const float>(which ? s.cr2 : s.cr);
    gptr<const uint8_t> code = gbl<const uint8_t>(s.stencil);
    gptr<float> z = gbl(s.cu);
    const int tilesJ = up_tiles_j(J);
    const TileRun run = up_run(up_tiles(I, J), s.up_blocks, sb.block);
    if (threadIdx.x <= kMaxD1) inv[threadIdx.x] = threadIdx.x ? 1.0f / (float)threadIdx.x : 0.f;
    // w x / D1 (0 where D1 is)
    auto over_d = [&](float x, int d) {
        const float n = kMgOmega * x, rd = inv[d], q = n * rd;
        return d > 0 ? __builtin_fmaf(__builtin_fmaf(-(float)d, q, n), rd, q) : 0.f;
    };
    auto l1 = [](uint8_t k) { return ((k >> 4) & 7) + __popc(k & 15u); };
    double rz = 0.0, rr = 0.0;
    for (int tile = run.first; tile < run.end; tile++) {
        const TileAt at = up_tile(tile, tilesJ);
        constexpr int Q = (kUpR * kUpR + kBlock - 1) / kBlock, QY = (kUpY * kUpY + kBlock - 1) / kBlock;
        uint8_t kq[Q];
        float vq[Q], yq[QY];
#pragma unroll
        for (int u = 0; u < Q; u++) {
            const int k = min((int)threadIdx.x + u * kBlock, kUpR * kUpR - 1);
            const int f = up_halo(at, k, I, J);
            kq[u] = code[f];
            vq[u] = r[f];
        }
#pragma unroll
        for (int u = 0; u < QY; u++) {
            const int k = min((int)threadIdx.x + u * kBlock, kUpY * kUpY - 1);
            const TileAt y = up_patch(at, k);
            const int ci = y.i, cj = y.j;
            const bool ok = ci >= 0 && ci < I1 && cj >= 0 && cj < J1;
            yq[u] = y1[min(max(ci, 0), I1 - 1) * J1 + min(max(cj, 0), J1 - 1)] * mask01(ok);
        }
        __syncthreads();   // the tile before is done with the LDS
#pragma unroll
        for (int u = 0; u < Q; u++) {
            const int k = threadIdx.x + u * kBlock;
            if (k >= kUpR * kUpR) break;
            cs[k / kUpR][k % kUpR] = kq[u];
            rs[k / kUpR][k % kUpR] = vq[u];
        }
#pragma unroll
        for (int u = 0; u < QY; u++) {
            const int k = threadIdx.x + u * kBlock;
            if (k < kUpY * kUpY) ys[k / kUpY][k % kUpY] = yq[u];
        }
        __syncthreads();
        // z0 of the tile and its halo (outside the grid: not used)
#pragma unroll
        for (int u = 0; u < Q; u++) {
            const int k = threadIdx.x + u * kBlock;
            if (k >= kUpR * kUpR) break;
            const int a = k / kUpR, b = k % kUpR;
            const int p0 = up_near(a), q0 = up_near(b), p1 = up_far(a), q1 = up_far(b);   // prolong_at on the patch
            float acc = 0.f;
            acc += (0.75f * 0.75f) * ys[p0][q0];
            acc += (0.75f * 0.25f) * ys[p0][q1];
            acc += (0.25f * 0.75f) * ys[p1][q0];
            acc += (0.25f * 0.25f) * ys[p1][q1];
            zs[a][b] = over_d(vq[u], l1(kq[u])) + acc;
        }
        __syncthreads();
        const int b = 1 + (int)threadIdx.x % kUpTile, j = at.j + b - 1;
#pragma unroll
        for (int u = 0; u < kUpTile * kUpTile / kBlock; u++) {
            const int a = 1 + (int)threadIdx.x / kUpTile + u * (kBlock / kUpTile), i = at.i + a - 1;
            if (i >= I || j >= J) continue;
            const uint8_t k = cs[a][b];
            const float rc = rs[a][b];
            // the fluid neighbours that enter A' (not the row-wrapping coupling)
            const float z0 = zs[a][b];
            float ax = (float)((k >> 4) & 7) * z0;
            ax -= (k & 1) ? zs[a - 1][b] : 0.f;
            ax -= (k & 2) ? zs[a + 1][b] : 0.f;
            ax -= ((k & 4) && j > 0) ? zs[a][b - 1] : 0.f;
            ax -= ((k & 8) && j < J - 1) ? zs[a][b + 1] : 0.f;
            const int d = l1(k);
            const float zc = ((k & 0x80) && d > 0) ? z0 + over_d(rc - ax, d) : rc;
            z[i * J + j] = zc;
            rz += (double)rc * (double)zc;
            rr += (double)rc * (double)rc;
        }
    }
    double v[2] = {rz, rr};
    put_partials<2>(s, kSlotCG, v, sb.block);
}

}  // namespace fg

namespace fg {
#define FG_MG_LAUNCH1(name, T, a) \
    void launch_##name(dim3 g, hipStream_t st, const SceneDev* sc, T a) { fg_launch(k_##name, g, dim3(kBlock), st, sc, a); }
#define FG_MG_LAUNCH_MAP(name, T, a) \
    void launch_##name(dim3 g, hipStream_t st, const SceneDev* sc, const int2* map, T a) \
    { \
        fg_launch(k_##name, g, dim3(kBlock), st, sc, map, a); \
    }
FG_MG_LAUNCH1(mg_mark, int, l)
FG_MG_LAUNCH1(mg_galerkin, int, l)
FG_MG_LAUNCH1(mg_sym, int, l)
void launch_mg_symmark(dim3 g, hipStream_t st, const SceneDev* sc, int l, int nsym)
{
    fg_launch(k_mg_symmark, g, dim3(kBlock), st, sc, l, nsym);
}
FG_MG_LAUNCH_MAP(mg_down0, int, which)
FG_MG_LAUNCH_MAP(mg_step0, int, it)
FG_MG_LAUNCH_MAP(mg_up0, int, which)
FG_MG_LAUNCH_MAP(mg_resid, int, l)
FG_MG_LAUNCH_MAP(mg_restrict, int, l)
FG_MG_LAUNCH_MAP(mg_prolong, int, l)
FG_MG_LAUNCH_MAP(mg_post, int, l)
FG_MG_LAUNCH_MAP(mg_rr, int, l)
FG_MG_LAUNCH_MAP(mg_pp, int, l)
void launch_mg_coarse(dim3 g, hipStream_t st, const SceneDev* sc, int max_halo)
{
    fg_launch_shm(k_mg_coarse, g, dim3(kMgCoarseThreads), 2 * sizeof(float) * max_halo, st, sc);
}
}  // namespace fg
