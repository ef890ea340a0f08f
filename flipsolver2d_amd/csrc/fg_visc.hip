// fg_visc.hip -- viscosity: LightViscosityModel (FlipSolver2dLib/
// viscositymodel.cpp:4-140) and the viscosity part of centeredParamsToGrid
// (flipsolver2d.cpp:1379-1431).
//
// k_visc_grid: a cell's viscosity is the quadratic-B-spline average of the
//   particles' viscosity over the cells i-2 .. i+1, j-2 .. j+1 (where the
//   spline at (x - i, y - j) is nonzero), summed in (cell, id) order; a
//   SOURCE cell takes its emitter's (afterTransfer, 396-397).
// The model (after the projection and updateVelocityFromSolids): one matrix
//   over the cells -- diagonal 1 on solid rows, 1 + 4 nu dt elsewhere;
//   symmetric couplings to (i+1, j) and (i, j+1) as the reference's
//   assembly leaves them, i.e. the later writer's value: nu of the far end
//   times dt unless that end is solid (then the near end's) -- solved twice,
//   for rho U and rho V on the cells' faces (i, j), by Jacobi-preconditioned
//   CG in FP64 from zero (Eigen's ConjugateGradient with its diagonal
//   preconditioner), both systems in the same launches:
//     k_visc_setup    matrix, b, x = 0, r = b; partials bb, rz
//     k_visc_p        the sums of the kernel before: the stop test
//                     ||r||^2 < tol^2 ||b||^2 and beta; p = r / d + beta p_old;
//                     q = A p; partials p.q
//     k_visc_x        the sums of p.q: alpha; x += alpha p, r -= alpha q;
//                     partials r.r, r.z
//     k_visc_apply    U = x / rho, V likewise (faces i < I, j < J)
// Two launches an iteration: every block sums the partials of the kernel
// before it, in the same order, and p is formed where it is multiplied (in
// LDS, once a cell and halo cell) and alternates between two buffers.  With
// the sums in one-block launches and p in one of its own an iteration of
// eight 256^2 scenes was five launches and 42 us; this form 29 us (k_visc_p 17,
// k_visc_x 10).
// The second projection (flipsolver2d.cpp:450-453) reuses the solve.
#include "fg_kernels.h"

namespace fg {

__device__ __forceinline__ int visc_blocks(const SceneDev& s) { return (s.I * s.J + kBlock - 1) / kBlock; }

__global__ void __launch_bounds__(kBlock) k_visc_grid(const SceneDev* scenes)
{
    const SceneDev& s = scenes[blockIdx.y];
    if (!s.active || !s.visc_on) return;
    const int I = s.I, J = s.J;
    const int c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= I * J) return;
    const int i = c / J, j = c - (c / J) * J;
    float wt = 1e-10f, vv = 0.0f;
    bool known = false;
    const int j0 = max(0, j - 2), j1 = min(J - 1, j + 1);
    // the four rows' bounds at once, then kVgItems particles a step whose
    // loads issue together (clamped; summed in order): with a load, its test
    // and the next particle in turn the loop ran at a load's latency a
    // particle, 95 us at eight 256^2 scenes; this 56
    constexpr int kVgItems = 4;
    int kb[4], ke[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int a = i - 2 + q;
        const bool row = a >= 0 && a < I;
        const int ac = min(max(a, 0), I - 1);
        kb[q] = gbl(s.cellStart)[ac * J + j0];
        ke[q] = row ? gbl(s.cellStart)[ac * J + j1 + 1] : kb[q];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        for (int k = kb[q]; k < ke[q]; k += kVgItems) {
            float2 p[kVgItems];
            float nu[kVgItems];
#pragma unroll
            for (int u = 0; u < kVgItems; u++) {
                const int ku = min(k + u, ke[q] - 1);
                p[u] = ldg2(s.pos, ku);
                nu[u] = gbl(s.pvisc)[ku];
            }
#pragma unroll
            for (int u = 0; u < kVgItems; u++) {
                if (k + u >= ke[q]) continue;
                const float w = qbspline(p[u].x - (float)i, p[u].y - (float)j);
                // NBFlipSolver's own (nbflipsolver.cpp:441-504): |w| > 1e-6, and
                // the sum divided only where some weight counted
                if (s.nb ? fabsf(w) > 1e-6f : w > 1e-9f) {
                    wt += w;
                    vv += w * nu[u];
                    known = true;
                }
            }
        }
    }
    if (s.nb) {   // its SOURCE cells are set in the combination (k_nb_combine_vel)
        s.cvisc[c] = known ? vv / wt : vv;
        return;
    }
    float v = vv / wt;
    if (s.mat[c] == M_SOURCE) {
        const int e = s.eid[c];
        if (e >= 0 && e < s.n_emitters) v = s.emitters[e].w;
    }
    s.cvisc[c] = v;
}

// vsc: bb 0-1, rz of even iterations 2-3 and of odd ones 4-5, done 12-13,
// iterations 14-15 (system 0 U, 1 V).
__device__ __forceinline__ int visc_tiles_j(const SceneDev& s) { return (s.J + kViscTile - 1) / kViscTile; }
__device__ __forceinline__ int visc_tiles(const SceneDev& s) { return ((s.I + kViscTile - 1) / kViscTile) * visc_tiles_j(s); }
// The direction of system q at iteration it.  The second buffers are arrays
// that the pressure solves before and after the viscosity solve leave free
// (b; the residuals cr and cr2, one after the other: 8 bytes a cell), the
// partials of p.q those of its z and direction (8 bytes a cell).
__device__ __forceinline__ gptr<double> visc_p(const SceneDev& s, int q, int it)
{
    if ((it & 1) == 0) return gbl(s.vp + (size_t)q * s.I * s.J);
    return gbl(q == 0 ? s.b : reinterpret_cast<double*>(s.cr));
}
__device__ __forceinline__ double* visc_pq(const SceneDev& s) { return reinterpret_cast<double*>(s.cu); }

__global__ void __launch_bounds__(kBlock) k_visc_setup(const SceneDev* scenes)
{
    const SceneDev& s = scenes[blockIdx.y];
    if (!s.active || !s.visc_on || (int)blockIdx.x >= visc_blocks(s)) return;
    const int I = s.I, J = s.J, C = I * J;
    const int c = blockIdx.x * kBlock + threadIdx.x;
    double bbu = 0, bbv = 0, rzu = 0, rzv = 0;
    if (c < C) {
        const int i = c / J, j = c - (c / J) * J;
        const double scale = s.dt;
        const bool sc = is_solid(s.mat[c]);
        const float vc = s.cvisc[c];
        const double d = sc ? 1.0 : 4.0 * (vc * scale) + 1.0;
        double e = 0.0, n = 0.0;
        if (i + 1 < I) {
            const bool sb = is_solid(s.mat[c + J]);
            if (!(sc && sb)) e = (sc ? s.cvisc[c + J] : vc) * scale;
        }
        if (j + 1 < J) {
            const bool sb = is_solid(s.mat[c + 1]);
            if (!(sc && sb)) n = (sc ? s.cvisc[c + 1] : vc) * scale;
        }
        s.vd[c] = d;
        s.ve[c] = e;
        s.vn[c] = n;
        const float rho = (float)s.rho;
        const double bu = rho * s.u[(size_t)i * J + j];        // fillRhs: float product
        const double bv = rho * s.v[(size_t)i * (J + 1) + j];
        s.vx[c] = 0.0;
        s.vx[C + c] = 0.0;
        s.vr[c] = bu;
        s.vr[C + c] = bv;
        const double zu = bu / d, zv = bv / d;
        bbu = bu * bu;
        bbv = bv * bv;
        rzu = bu * zu;
        rzv = bv * zv;
    }
    double v[4] = {bbu, bbv, rzu, rzv};
    put_sums<4>(s.vpart, visc_blocks(s), blockIdx.x, v);
}

__global__ void __launch_bounds__(kBlock) k_visc_p(const SceneDev* scenes, int it, double tol2)
{
    constexpr int R = kViscTile + 2, Q = (R * R + kBlock - 1) / kBlock;
    static_assert(kViscTile * kViscTile == kBlock, "one cell of the tile per thread");
    __shared__ double ps[2][R][R + 1];
    const SceneDev& s = scenes[blockIdx.y];
    if (!s.active || !s.visc_on || (int)blockIdx.x >= visc_tiles(s)) return;
    const int I = s.I, J = s.J, C = I * J;
    const int tj = visc_tiles_j(s), i0 = kViscTile * (int)(blockIdx.x / tj), j0 = kViscTile * (int)(blockIdx.x % tj);
    // loads first (clamped; positions outside the grid are not used)
    double dq[Q], rq[2][Q], oq[2][Q];
#pragma unroll
    for (int u = 0; u < Q; u++) {
        const int k = min((int)threadIdx.x + u * kBlock, R * R - 1);
        const int c = min(max(i0 - 1 + k / R, 0), I - 1) * J + min(max(j0 - 1 + k % R, 0), J - 1);
        dq[u] = gbl(s.vd)[c];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            rq[q][u] = gbl(s.vr)[(size_t)q * C + c];
            oq[q][u] = it > 0 ? visc_p(s, q, it - 1)[c] : 0.0;
        }
    }
    const int a = 1 + threadIdx.x / kViscTile, b = 1 + threadIdx.x % kViscTile, i = i0 + a - 1, j = j0 + b - 1;
    const bool in = i < I && j < J;
    const int c = min(i, I - 1) * J + min(j, J - 1);
    const double e = gbl(s.ve)[c], n = gbl(s.vn)[c], ew = gbl(s.ve)[max(c - J, 0)], ns = gbl(s.vn)[max(c - 1, 0)];
    // the sums of k_visc_setup (bb, rz) or of the iteration before (rr, rz)
    double sum[4];
    sum_rows<4>(s.vpart, visc_blocks(s), visc_blocks(s), sum);
    double* const v = s.vsc;
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    bool go[2];
    double beta[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        // a block that sees the lead's flag of this very launch stops as its own sums would have it
        const bool done = it > 0 && gbl(v)[12 + q] != 0.0;
        const bool stop = it == 0 ? sum[q] == 0.0 : sum[q] < tol2 * gbl(v)[q];   // a zero right-hand side: x = 0
        go[q] = !done && !stop;
        beta[q] = it == 0 ? 0.0 : sum[2 + q] / gbl(v)[2 + 2 * ((it - 1) & 1) + q];
        if (lead && !done) {
            if (it == 0) v[q] = sum[q];
            v[2 + 2 * (it & 1) + q] = sum[2 + q];
            v[12 + q] = stop ? 1.0 : 0.0;
            v[14 + q] = it == 0 ? 0.0 : gbl(v)[14 + q] + 1.0;
        }
    }
    if (!go[0] && !go[1]) return;
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int u = 0; u < Q; u++) {
            const int k = threadIdx.x + u * kBlock;
            if (k < R * R) ps[q][k / R][k % R] = it == 0 ? rq[q][u] / dq[u] : rq[q][u] / dq[u] + beta[q] * oq[q][u];
        }
    __syncthreads();
    const double d = gbl(s.vd)[c];
    double pq[2] = {0.0, 0.0};
    if (in) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (!go[q]) continue;
            const double p = ps[q][a][b];
            double t = d * p;
            if (i + 1 < I) t += e * ps[q][a + 1][b];
            if (i > 0) t += ew * ps[q][a - 1][b];
            if (j + 1 < J) t += n * ps[q][a][b + 1];
            if (j > 0) t += ns * ps[q][a][b - 1];
            visc_p(s, q, it)[c] = p;
            gbl(s.vq)[(size_t)q * C + c] = t;
            pq[q] = p * t;
        }
    }
    put_sums<2>(visc_pq(s), visc_tiles(s), blockIdx.x, pq);
}

__global__ void __launch_bounds__(kBlock) k_visc_x(const SceneDev* scenes, int it)
{
    const SceneDev& s = scenes[blockIdx.y];
    if (!s.active || !s.visc_on || (int)blockIdx.x >= visc_blocks(s)) return;
    const int C = s.I * s.J;
    const int c = blockIdx.x * kBlock + threadIdx.x, cc = min(c, C - 1);
    const double d = gbl(s.vd)[cc];
    double p[2], x[2], r[2], t[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const size_t k = (size_t)q * C + cc;
        p[q] = visc_p(s, q, it)[cc];
        x[q] = gbl(s.vx)[k];
        r[q] = gbl(s.vr)[k];
        t[q] = gbl(s.vq)[k];
    }
    cptr<double> v = cst(s.vsc);   // k_visc_p's
    const bool go[2] = {v[12] == 0.0, v[13] == 0.0};
    if (!go[0] && !go[1]) return;
    double pq[2];
    sum_rows<2>(visc_pq(s), visc_tiles(s), visc_tiles(s), pq);
    double sum[4] = {0.0, 0.0, 0.0, 0.0};   // rr, rz
    if (c < C) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (!go[q]) continue;
            const double alpha = v[2 + 2 * (it & 1) + q] / pq[q];
            const size_t k = (size_t)q * C + c;
            gbl(s.vx)[k] = x[q] + alpha * p[q];
            const double rn = r[q] - alpha * t[q];
            gbl(s.vr)[k] = rn;
            sum[q] = rn * rn;
            sum[2 + q] = rn * (rn / d);
        }
    }
    put_sums<4>(s.vpart, visc_blocks(s), blockIdx.x, sum);
}

__global__ void __launch_bounds__(kBlock) k_visc_apply(const SceneDev* scenes)
{
    const SceneDev& s = scenes[blockIdx.y];
    if (!s.active || !s.visc_on) return;
    const int I = s.I, J = s.J, C = I * J;
    const int c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= C) return;
    const int i = c / J, j = c - (c / J) * J;
    if (c == 0) {
        s.sc->visc_iters = (int32_t)fmax(s.vsc[14], s.vsc[15]);
        s.sc->visc_done = s.vsc[12] != 0.0 && s.vsc[13] != 0.0;
    }
    const float rho = (float)s.rho;
    s.u[(size_t)i * J + j] = (float)(s.vx[c] / rho);          // applyResult
    s.v[(size_t)i * (J + 1) + j] = (float)(s.vx[C + c] / rho);
}

// how many scenes of the launch still iterate (either system)
__global__ void k_visc_flags(const SceneDev* scenes, int n, int32_t* out)
{
    int open = 0;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        const SceneDev& s = scenes[k];
        if (s.active && s.visc_on && (s.vsc[12] == 0.0 || s.vsc[13] == 0.0)) open++;
    }
    for (int o = 32; o > 0; o >>= 1) open += __shfl_down(open, o, 64);
    if (threadIdx.x == 0) out[0] = open;
}

}  // namespace fg

namespace fg {
#define FG_VLAUNCH(name) \
    void launch_##name(dim3 g, hipStream_t st, const SceneDev* sc) { fg_launch(k_##name, g, dim3(kBlock), st, sc); }
FG_VLAUNCH(visc_grid)
FG_VLAUNCH(visc_setup)
FG_VLAUNCH(visc_apply)
void launch_visc_p(dim3 g, hipStream_t st, const SceneDev* sc, int it, double tol2)
{
    fg_launch(k_visc_p, g, dim3(kBlock), st, sc, it, tol2);
}
void launch_visc_x(dim3 g, hipStream_t st, const SceneDev* sc, int it) { fg_launch(k_visc_x, g, dim3(kBlock), st, sc, it); }
void launch_visc_flags(hipStream_t st, const SceneDev* sc, int n, int32_t* out)
{
    hipLaunchKernelGGL(k_visc_flags, dim3(1), dim3(64), 0, st, sc, n, out);
}
}  // namespace fg
