// HIP kernels for gfx950 (MI355X) of the Laplace-solve-per-RK4-stage path.
//
// Layout (as the reference, BuildLinearSystem.f90:117): sigma-fastest columns,
//   q = k + nzg*(i + nxg*j);  plane fields p = i + nxg*j.
// The high-order matvec keeps whole sigma columns of a 2D tile (plus an alpha+1 halo) in LDS;
// every interior column's x-, y-, sigma- and mixed derivatives are formed from that tile, so
// phi is read from HBM once per matvec (halo re-reads hit L2 / MALL) and y written once.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>
#include <cstdint>

namespace ow3d {

__host__ __device__ constexpr int cmin(int a, int b) { return a < b ? a : b; }
__host__ __device__ constexpr int cmax(int a, int b) { return a > b ? a : b; }
__host__ __device__ constexpr int cclamp(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// a b + c with one rounding.  The smoother's column code writes its roundings out (contraction off): FP32 V
// cycles are only linear to rounding, so that a product fused in one form of a kernel and not in another would
// move a mixed-precision solution by up to 1e-8.
__device__ __forceinline__ float fma1(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma1(double a, double b, double c) { return __builtin_fma(a, b, c); }

// c ? a : b of two values (a conditional on array elements would select their address and put the array in scratch)
template <typename T>
__device__ __forceinline__ T pick(bool c, T a, T b) { return c ? a : b; }

// Barrier that orders the block's LDS accesses only.  __syncthreads() also waits for every HBM load and store in
// flight; here loads issued early stay in flight across it, and nothing waits for stores that no thread of the
// block reads back.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Kernels launched inside a device-driven Laplace solve take the solve's "done" flag and return at once
// when it is set, so a fixed launch sequence (a captured graph) costs almost nothing after convergence.
// nullptr: always run.
__device__ __forceinline__ bool solve_done(const int *skip) { return skip != nullptr && *skip != 0; }

// Columns between HBM and registers, two values per load or store where every column starts on an even element.
template <typename S>
struct alignas(2 * sizeof(S)) ColPair { S a, b; };
template <int NZ, typename S, typename T>
__device__ __forceinline__ void load_column(const S *__restrict__ p, T (&v)[NZ]) {
    if constexpr (NZ % 2 == 0) {
        const ColPair<S> *q = reinterpret_cast<const ColPair<S> *>(p);
#pragma unroll
        for (int k = 0; k < NZ / 2; k++) { const ColPair<S> w = q[k]; v[2 * k] = (T)w.a; v[2 * k + 1] = (T)w.b; }
    } else {
#pragma unroll
        for (int k = 0; k < NZ; k++) v[k] = (T)p[k];
    }
}
// N values (a multiple of 16 bytes) from a 16-byte aligned address.
template <int N, typename T>
__device__ __forceinline__ void load_record(const T *__restrict__ p, T (&v)[N]) {
    constexpr int W = 16 / sizeof(T);
    struct alignas(16) Quad { T e[W]; };
    static_assert(N % W == 0, "whole 16-byte loads");
#pragma unroll
    for (int q = 0; q < N / W; q++) {
        const Quad w = reinterpret_cast<const Quad *>(p)[q];
#pragma unroll
        for (int e = 0; e < W; e++) v[q * W + e] = w.e[e];
    }
}
template <int NZ, typename T, typename O>
__device__ __forceinline__ void store_column(O *__restrict__ p, const T (&v)[NZ]) {
    if constexpr (NZ % 2 == 0) {
        ColPair<O> *q = reinterpret_cast<ColPair<O> *>(p);
#pragma unroll
        for (int k = 0; k < NZ / 2; k++) q[k] = ColPair<O>{(O)v[2 * k], (O)v[2 * k + 1]};
    } else {
#pragma unroll
        for (int k = 0; k < NZ; k++) p[k] = (O)v[k];
    }
}

// ---------------------------------------------------------------------------------------------
// High-order matvec  (BuildLinearSystem.f90:1-290)
// ---------------------------------------------------------------------------------------------
// Two values of the matvec's result as one store.  A device-pointer caller's y is only 8-byte aligned
// (ow3d_laplace_apply_device); global memory takes 16-byte stores at any multiple of 4.
struct OutPair { double a, b; };
static_assert(alignof(OutPair) == 8, "y's alignment");

struct MvArgs {
    int nxg, nyg, nxy;
    const double *sx, *sy, *sz;  // stencil rows [N][2][2A+1]
    const double *zs;            // sigma of each level (0 on the ghost level)
    const double *cf;            // 7 planes: sigma coefficients affine in sigma, s2 = A2 + sigma*B2, s4 = A4 + sigma*B4,
                                 // s3 = A3 + sigma*B3, s5 = S5; planes (A2, B2, A4, B4, A3, B3, S5)
    const int *skip;             // solve_done flag (nullptr: always run)
};

// Per-column coefficient planes from the surface and the bottom: DetermineTransformationConstantsArray.f90
// (lines 190-201) written as functions affine in sigma, evaluated once per column and stage.
__device__ __forceinline__ void column_coefs(double d, double Ex, double Ey, double Es, double hx, double hy, double hs,
                                             double *cf, int nxy, int p) {
    const double id = 1.0 / d, id2 = id * id;
    const double H2 = hx * hx + hy * hy, C = Ex * hx + Ey * hy, E2 = Ex * Ex + Ey * Ey;
    cf[p] = hx * id;
    cf[nxy + p] = -(hx + Ex) * id;
    cf[2 * nxy + p] = hy * id;
    cf[3 * nxy + p] = -(hy + Ey) * id;
    cf[4 * nxy + p] = (-2.0 * H2 - 2.0 * C) * id2 + hs * id;
    cf[5 * nxy + p] = (2.0 * H2 + 4.0 * C + 2.0 * E2) * id2 - (hs + Es) * id;
    cf[6 * nxy + p] = id;
}

// Copies a window of rows x cols sigma-columns (NZ values each) of a field in HBM into LDS: window row r
// starts at src + r * pitch; LDS holds element (r, c, k) at (r * RS + c) * NZP + k.  All loads of a thread
// are issued before its first LDS store, so a block waits for HBM once, not once per row.
// The two halves are also available separately (WindowRegs: load into registers, store to LDS) so that a
// kernel can issue the loads of several windows before it waits for any of them.
// FP32 windows of columns with an even NZ move two values per load (8 bytes): callers pass src at an even
// element offset with an even pitch, so every pair is 8-byte aligned and stays inside one window row.
template <typename T, int NZ, int MR, int MC, int NT>
struct WindowRegs {
    static constexpr int RL = MC * NZ, TOT = MR * RL;
    static constexpr bool PAIRS = NZ % 2 == 0 && sizeof(T) == 4;
    static constexpr int W = PAIRS ? 2 : 1, PER = (TOT / W + NT - 1) / NT;
    T v[PER * W];
    __device__ __forceinline__ void load(const T *__restrict__ src, size_t pitch, int rows, int cols) {
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int e = ((int)threadIdx.x + q * NT) * W;
            const int r = e / RL, c = e - r * RL;
            const bool ok = e < TOT && r < rows && c < cols * NZ;
            if constexpr (PAIRS) {
                float2 w = make_float2(0.0f, 0.0f);
                if (ok) w = *reinterpret_cast<const float2 *>(src + (size_t)r * pitch + c);
                v[2 * q] = w.x;
                v[2 * q + 1] = w.y;
            } else {
                v[q] = ok ? src[(size_t)r * pitch + c] : T(0);
            }
        }
    }
    template <int NZP, int RS, typename U>
    __device__ __forceinline__ void store(U *lds, int rows, int cols) const {
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int e = ((int)threadIdx.x + q * NT) * W;
            const int r = e / RL, c = e - r * RL;
            if (e < TOT && r < rows && c < cols * NZ) {
                const int cc = c / NZ, k = c - cc * NZ;
                const int a = (r * RS + cc) * NZP + k;
                if constexpr (PAIRS) {
                    lds[a] = (U)v[2 * q];
                    lds[k + 1 < NZ ? a + 1 : a + NZP - NZ + 1] = (U)v[2 * q + 1];   // next level or next column
                } else {
                    lds[a] = (U)v[q];
                }
            }
        }
    }
};
// Copies one tile row of ncol columns from LDS (column c's NZ values at src + c * NZP) to dst (NZ values
// per column, contiguous), converting to O.  For an even NZ two values go per store: dst is then at an even
// element offset (a row of columns of an even depth), so every pair is aligned.
template <int NZ, int NZP, int NT, typename T, typename O>
__device__ __forceinline__ void store_row(O *__restrict__ dst, const T *src, int ncol) {
    if constexpr (NZ % 2 == 0 && (sizeof(O) == 4 || sizeof(O) == 8)) {
        using O2 = typename std::conditional<sizeof(O) == 4, float2, double2>::type;
        for (int e = 2 * (int)threadIdx.x; e < ncol * NZ; e += 2 * NT) {
            const int c = e / NZ, k = e - c * NZ, a = c * NZP + k;
            O2 w;
            w.x = (O)src[a];
            w.y = (O)src[k + 1 < NZ ? a + 1 : a + NZP - NZ + 1];   // next level or next column
            *reinterpret_cast<O2 *>(dst + e) = w;
        }
    } else {
        for (int e = (int)threadIdx.x; e < ncol * NZ; e += NT) {
            const int c = e / NZ, k = e - c * NZ;
            dst[e] = (O)src[c * NZP + k];
        }
    }
}
template <typename T, int NZ, int NZP, int MR, int MC, int RS, int NT>
__device__ __forceinline__ void stage_window(T *lds, const T *__restrict__ src, size_t pitch, int rows, int cols) {
    WindowRegs<T, NZ, MR, MC, NT> w;
    w.load(src, pitch, rows, cols);
    w.template store<NZP, RS>(lds, rows, cols);
}

// Block index -> tile index such that each of the 8 XCDs (which receive blocks round-robin) works on a
// contiguous range of tiles, so halo columns shared by neighbouring tiles are re-read from the same L2.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
    const int q = nb / 8, rem = nb % 8, xcd = b % 8, slot = b / 8;
    return (xcd < rem ? xcd * (q + 1) : rem * (q + 1) + (xcd - rem) * q) + slot;
}

// 3D, one thread per grid point: block = 16 x TY columns x NZ levels, NT threads.  The tile is
// stored k-fastest in LDS exactly as in HBM (row segments are straight copies), and threads are mapped
// k-fastest too, so every LDS access of a wave and every global load / store is contiguous.
// Phase 1 forms the x- and y-derivatives of every tile point (the first passes of the mixed
// derivatives go to LDS); phase 2 the sigma derivatives, the mixed derivatives and the row.
template <int NZ, int A, int TY, int NT>
__global__ __launch_bounds__(NT) void k_matvec3p(MvArgs g, const double *__restrict__ phi, double *__restrict__ out) {
    if (solve_done(g.skip)) return;
    constexpr int TX = 16, RA = 2 * A + 1, R = A + 1, WX = TX + 2 * R, WY = TY + 2 * R, NC = TX * TY, NP = NC * NZ;
    constexpr int PER = (NP + NT - 1) / NT;
    __shared__ double sP[WX * WY * NZ];
    __shared__ double sDx[NP];
    __shared__ double sDy[NP];
    __shared__ double sSX[(TX + 2) * 2 * RA];
    __shared__ double sSY[(TY + 2) * 2 * RA];
    __shared__ double sSZ[NZ * 2 * RA];
    __shared__ double sZS[NZ];
    __shared__ double sCF[7 * NC];
    const int nxg = g.nxg, nyg = g.nyg, nxy = g.nxy;
    const int gxt = (nxg + TX - 1) / TX;
    const int tile = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const int i0 = (tile % gxt) * TX, j0 = (tile / gxt) * TY;
    const int lox = cmax(cmin(i0 - R, nxg - 2 - 2 * A), 0);
    const int loy = cmax(cmin(j0 - R, nyg - 2 - 2 * A), 0);
    const int wx = cmin(WX, nxg - lox), wy = cmin(WY, nyg - loy);
    {
        // coefficient planes of the tile's columns, loaded together with the phi window
        constexpr int CPT = (7 * NC + NT - 1) / NT;
        double cv[CPT];
#pragma unroll
        for (int q = 0; q < CPT; q++) {
            const int e = (int)threadIdx.x + q * NT;
            const int pl = e / NC, c = e - pl * NC, ii = i0 + c % TX, jj = j0 + c / TX;
            cv[q] = (e < 7 * NC && ii < nxg && jj < nyg) ? g.cf[(size_t)pl * nxy + ii + (size_t)nxg * jj] : 0.0;
        }
        stage_window<double, NZ, NZ, WY, WX, WX, NT>(sP, phi + ((size_t)loy * nxg + lox) * NZ, (size_t)nxg * NZ, wy, wx);
#pragma unroll
        for (int q = 0; q < CPT; q++) {
            const int e = (int)threadIdx.x + q * NT;
            if (e < 7 * NC) sCF[e] = cv[q];
        }
    }
    for (int e = threadIdx.x; e < (TX + 2) * 2 * RA; e += NT) {
        const int r = e / (2 * RA), ii = i0 - 1 + r;
        if (ii >= 0 && ii < nxg) sSX[e] = g.sx[(size_t)ii * 2 * RA + (e - r * 2 * RA)];
    }
    for (int e = threadIdx.x; e < (TY + 2) * 2 * RA; e += NT) {
        const int r = e / (2 * RA), jj = j0 - 1 + r;
        if (jj >= 0 && jj < nyg) sSY[e] = g.sy[(size_t)jj * 2 * RA + (e - r * 2 * RA)];
    }
    for (int e = threadIdx.x; e < NZ * 2 * RA; e += NT) sSZ[e] = g.sz[e];
    if (threadIdx.x < NZ) sZS[threadIdx.x] = g.zs[threadIdx.x];
    __syncthreads();
    auto P = [&](int k, int ii, int jj) -> double { return sP[((jj - loy) * WX + (ii - lox)) * NZ + k]; };
    auto SX = [&](int ii) -> const double * { return sSX + (ii - (i0 - 1)) * 2 * RA; };
    auto SY = [&](int jj) -> const double * { return sSY + (jj - (j0 - 1)) * 2 * RA; };
    double acc[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
        acc[r] = 0.0;
        const int pt = threadIdx.x + r * NT;
        if (pt >= NP) break;
        const int col = pt / NZ, k = pt - col * NZ;
        const int i = i0 + col % TX, j = j0 + col / TX;
        if (i >= nxg || j >= nyg || i == 0 || i == nxg - 1 || j == 0 || j == nyg - 1) continue;
        const int wsx = cclamp(i - A, 0, nxg - RA), wsy = cclamp(j - A, 0, nyg - RA);
        double d1 = 0.0, d2 = 0.0, e1 = 0.0, e2 = 0.0;
        {
            const double *S1 = SX(i), *S2 = S1 + RA;
#pragma unroll
            for (int m = 0; m < RA; m++) { const double v = P(k, wsx + m, j); d1 += S1[m] * v; d2 += S2[m] * v; }
        }
        {
            const double *S1 = SY(j), *S2 = S1 + RA;
#pragma unroll
            for (int m = 0; m < RA; m++) { const double v = P(k, i, wsy + m); e1 += S1[m] * v; e2 += S2[m] * v; }
        }
        if (k == 0) {  // corner-corrected first pass on the sigma ghost level (ConstructTableCrossDerivatives.f90:173-186)
            int sh = 0;
            if (wsx == 0) sh = 1;
            if (wsx + RA - 1 == nxg - 1) sh = -1;
            if (sh != 0) {
                const double *S = SX(i - sh);
                double t = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) t += S[m] * P(0, wsx + sh + m, j);
                d1 = t;
            }
            sh = 0;
            if (wsy == 0) sh = 1;
            if (wsy + RA - 1 == nyg - 1) sh = -1;
            if (sh != 0) {
                const double *S = SY(j - sh);
                double t = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) t += S[m] * P(0, i, wsy + sh + m);
                e1 = t;
            }
        }
        sDx[pt] = d1;
        sDy[pt] = e1;
        acc[r] = d2 + e2;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int pt = threadIdx.x + r * NT;
        if (pt >= NP) break;
        const int col = pt / NZ, k = pt - col * NZ;
        const int i = i0 + col % TX, j = j0 + col / TX;
        if (i >= nxg || j >= nyg) continue;
        const bool wxl = (i == 0 || i == nxg - 1), wyl = (j == 0 || j == nyg - 1);
        double o;
        if ((wxl && wyl) || ((wxl || wyl) && k == 0) || (!wxl && !wyl && k == NZ - 1)) {
            o = P(k, i, j);
        } else if (wxl) {
            const int ib = (i == 0) ? 1 : nxg - 2, ws = cclamp(ib - A, 0, nxg - RA);
            const double *S = SX(ib);
            o = 0.0;
#pragma unroll
            for (int m = 0; m < RA; m++) o += S[m] * P(k, ws + m, j);
        } else if (wyl) {
            const int jb = (j == 0) ? 1 : nyg - 2, ws = cclamp(jb - A, 0, nyg - RA);
            const double *S = SY(jb);
            o = 0.0;
#pragma unroll
            for (int m = 0; m < RA; m++) o += S[m] * P(k, i, ws + m);
        } else {
            const double A2 = sCF[col], B2 = sCF[NC + col], A4 = sCF[2 * NC + col], B4 = sCF[3 * NC + col];
            const double S5 = sCF[6 * NC + col];
            const double *dxc = sDx + col * NZ, *dyc = sDy + col * NZ;
            if (k == 0) {
                const int wz = cclamp(1 - A, 0, NZ - RA);
                const double *Z1 = sSZ + (1 * 2) * RA;
                double dz = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) dz += Z1[m] * P(wz + m, i, j);
                // h_x = A2 * d and h_y = A4 * d with d = 1 / S5: no bottom-slope planes are read
                const double sg = sZS[1], d = 1.0 / S5, hx = A2 * d, hy = A4 * d;
                o = (S5 + hx * (A2 + sg * B2) + hy * (A4 + sg * B4)) * dz + hx * dxc[1] + hy * dyc[1];
            } else {
                const double A3 = sCF[4 * NC + col], B3 = sCF[5 * NC + col];
                const int wz = cclamp(k - A, 0, NZ - RA);
                const double *Z1 = sSZ + (k * 2) * RA, *Z2 = Z1 + RA;
                double dz = 0.0, dzz = 0.0, dxz = 0.0, dyz = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) {
                    const double z1 = Z1[m], cv = P(wz + m, i, j);
                    dz += z1 * cv;
                    dzz += Z2[m] * cv;
                    dxz += z1 * dxc[wz + m];
                    dyz += z1 * dyc[wz + m];
                }
                const double sg = sZS[k];
                const double s2 = A2 + sg * B2, s4 = A4 + sg * B4, s3 = A3 + sg * B3;
                o = acc[r] + s3 * dz + 2.0 * (s2 * dxz + s4 * dyz) + (s2 * s2 + s4 * s4 + S5 * S5) * dzz;
            }
        }
        out[((size_t)j * nxg + i) * NZ + k] = o;
    }
}

// The column matvec with the work of each column split between two waves: a block of TX x TY columns
// has 2 TX TY threads; the first TX TY take the x-side of column t (d/dx, d2/dx2, the first sigma
// derivative of phi and the mixed x-sigma term, the bottom row), the others the y-side of column
// t - TX TY (d/dy, d2/dy2, the mixed y-sigma term).  The y-side leaves its part of every row in LDS; the x-side
// adds it.  Each thread holds half the live values of a one-thread-per-column kernel and a block has
// twice the waves.  ORDER 0: a row is summed as d2x + d2y, then s3 dz, 2 (s2 dxz + s4 dyz) and the second sigma
// derivative's term, which the x-side forms; 1: the y-side forms its whole part, with the second sigma derivative,
// and the x-side adds it last (both are rounding of the same sum; solves that amplify rounding keep the one they use).
// The live values of a column take about 220 VGPRs (two waves per SIMD), so two blocks share a CU and one block's loads
// overlap the other's arithmetic; with registers for three it spills (46-56 us where it takes 30).  Bound by the chain of
// one tile (loads, LDS, four stencils per level, LDS, stores: 8.5 us), four and a half times in a row at 513^2.  With
// 10 levels, 6th order, at 33^2, 97 x 161, 257^2, 513^2: one thread per column and 16 x 16 tiles 15.5, 14.2, 21.9 and
// 47.7 us; ORDER 0 10.1, 8.6, 14.3 and 31.6 us; ORDER 1 with the test of the done flag before the loads, the planes
// loaded where they are used and row-by-row stores 10.7, 8.9, 15.7 and 33.0 us, now 10.0, 8.3, 14.1 and 30.4 us.
template <int NZ, int A, int TX, int TY, int ORDER>
struct MvSplit {
    static constexpr int NC = TX * TY, NT = 2 * NC, RA = 2 * A + 1, R = A + 1, WX = TX + 2 * R, WY = TY + 2 * R, PS = (WX * WY) | 1;
    static constexpr int YP = ORDER == 0 ? 2 : 1;   // values per row that the y-side passes on
    static constexpr int ROWS = (TX + 2 + TY + 2) * 2 * RA, LDS = NZ * PS + ROWS + YP * NZ * NC;   // in doubles
};
template <int NZ, int A, int TX, int TY, int ORDER>
__global__ __launch_bounds__(2 * TX * TY) void k_matvec3s(MvArgs g, const double *__restrict__ phi, double *__restrict__ out) {
    using G = MvSplit<NZ, A, TX, TY, ORDER>;
    constexpr int NC = G::NC, NT = G::NT, RA = G::RA, R = G::R, WX = G::WX, WY = G::WY, PS = G::PS;
    __shared__ double lds[G::LDS];
    double *const sP = lds, *const sSX = lds + NZ * PS, *const sSY = sSX + (TX + 2) * 2 * RA, *const sYp = lds + NZ * PS + G::ROWS;
    const int nxg = g.nxg, nyg = g.nyg, nxy = g.nxy;
    const int gxt = (nxg + TX - 1) / TX;
    const int tile = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const int i0 = (tile % gxt) * TX, j0 = (tile / gxt) * TY;
    const int lox = cmax(cmin(i0 - R, nxg - 2 - 2 * A), 0);
    const int loy = cmax(cmin(j0 - R, nyg - 2 - 2 * A), 0);
    const int wx = cmin(WX, nxg - lox), wy = cmin(WY, nyg - loy);
    const bool yside = threadIdx.x >= NC;
    const int col = yside ? (int)threadIdx.x - NC : (int)threadIdx.x;
    const int tx = col % TX, ty = col / TX;
    const int i = i0 + tx, j = j0 + ty;
    const bool active = (i < nxg) && (j < nyg);
    double cf[7];   // the column's planes A2, B2, A4, B4, A3, B3, S5
    {
        // every HBM load of the block first, and before the test of the done flag: the phi window (stored level-major;
        // two values at a time for an even NZ: rows of columns start at even offsets, so every pair is aligned and
        // stays inside one window row), the stencil rows of its columns and rows, the planes
        constexpr bool PAIRS = NZ % 2 == 0;
        constexpr int W = PAIRS ? 2 : 1;
        constexpr int RL = WX * NZ, TOT = WY * RL, PER = (TOT / W + NT - 1) / NT;
        double v[PER * W];
        const double *src = phi + ((size_t)loy * nxg + lox) * NZ;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int e = ((int)threadIdx.x + q * NT) * W, r = e / RL, c = e - r * RL;
            const bool ok = e < TOT && r < wy && c < wx * NZ;
            if constexpr (PAIRS) {
                double2 w = make_double2(0.0, 0.0);
                if (ok) w = *reinterpret_cast<const double2 *>(src + (size_t)r * nxg * NZ + c);
                v[2 * q] = w.x;
                v[2 * q + 1] = w.y;
            } else {
                v[q] = ok ? src[(size_t)r * nxg * NZ + c] : 0.0;
            }
        }
        const double *cfp = g.cf + (active ? i + (size_t)nxg * j : 0);
#pragma unroll
        for (int q = 0; q < 7; q++) cf[q] = cfp[(size_t)q * nxy];
        constexpr int SXN = (TX + 2) * 2 * RA, SYN = (TY + 2) * 2 * RA, SPER = (SXN + SYN + NT - 1) / NT;
        double sv[SPER];
#pragma unroll
        for (int q = 0; q < SPER; q++) {
            const int e = (int)threadIdx.x + q * NT, f = e < SXN ? e : e - SXN, r = f / (2 * RA), m = f - r * 2 * RA;
            const int ii = cclamp((e < SXN ? i0 : j0) - 1 + r, 0, (e < SXN ? nxg : nyg) - 1);
            sv[q] = e < SXN + SYN ? (e < SXN ? g.sx : g.sy)[(size_t)ii * 2 * RA + m] : 0.0;
        }
        if (solve_done(g.skip)) return;
#pragma unroll
        for (int q = 0; q < SPER; q++) {
            const int e = (int)threadIdx.x + q * NT;
            if (e < SXN + SYN) sSX[e] = sv[q];
        }
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int e = ((int)threadIdx.x + q * NT) * W, r = e / RL, c = e - r * RL;
            if (e < TOT && r < wy && c < wx * NZ) {
                const int cc = c / NZ, k = c - cc * NZ;
                double *d = sP + k * PS + r * WX + cc;
                if constexpr (PAIRS) {   // an even NZ: k is even, so k + 1 is the same column's
                    d[0] = v[2 * q];
                    d[PS] = v[2 * q + 1];
                } else {
                    d[0] = v[q];
                }
            }
        }
    }
    lds_barrier();
    auto P = [&](int k, int ii, int jj) -> double { return sP[k * PS + (jj - loy) * WX + (ii - lox)]; };
    auto SX = [&](int ii) -> const double * { return sSX + (ii - (i0 - 1)) * 2 * RA; };
    auto SY = [&](int jj) -> const double * { return sSY + (jj - (j0 - 1)) * 2 * RA; };
    const bool wxl = (i == 0 || i == nxg - 1), wyl = (j == 0 || j == nyg - 1);
    const bool interior = active && !wxl && !wyl;
    const double A2 = cf[0], B2 = cf[1], A4 = cf[2], B4 = cf[3], A3 = cf[4], B3 = cf[5], S5 = cf[6];
    double o[NZ];
    double dzk[NZ], zz[NZ], xz[NZ], dz0 = 0.0, dx1 = 0.0;   // ORDER 0: the x-side's derivatives of each row, summed once the y-side's part is there
    if (yside) {
        if (interior) {
            const int wsy = cclamp(j - A, 0, nyg - RA);
            double dy[NZ];
            const double *S1 = SY(j), *S2 = S1 + RA;
#pragma unroll
            for (int k = 0; k < NZ; k++) {
                double d1 = 0.0, d2 = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) { const double v = P(k, i, wsy + m); d1 += S1[m] * v; d2 += S2[m] * v; }
                dy[k] = d1; o[k] = d2;
            }
            double dyc0 = dy[0];
            {
                int sh = 0;
                if (wsy == 0) sh = 1;
                if (wsy + RA - 1 == nyg - 1) sh = -1;
                if (sh != 0) {
                    const double *S = SY(j - sh);
                    double t = 0.0;
#pragma unroll
                    for (int m = 0; m < RA; m++) t += S[m] * P(0, i, wsy + sh + m);
                    dyc0 = t;
                }
            }
            // ORDER 1: the second sigma derivative is this side's share of the column's own terms (the x side takes
            // the first), so that both halves of a column do the same work
            double pc[NZ];
            if constexpr (ORDER == 1) {
#pragma unroll
                for (int k = 0; k < NZ; k++) pc[k] = P(k, i, j);
            }
#pragma unroll
            for (int k = 1; k < NZ - 1; k++) {
                const int wz = cclamp(k - A, 0, NZ - RA);
                const double *Z1 = g.sz + (k * 2) * RA, *Z2 = Z1 + RA;
                double dyz = 0.0, dzz = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) {
                    dyz += Z1[m] * ((wz + m == 0) ? dyc0 : dy[wz + m]);
                    if constexpr (ORDER == 1) dzz += Z2[m] * pc[wz + m];
                }
                const double sg = g.zs[k];
                const double s4 = A4 + sg * B4;
                if constexpr (ORDER == 1) {
                    const double s2 = A2 + sg * B2;
                    o[k] = o[k] + 2.0 * (s4 * dyz) + (s2 * s2 + s4 * s4 + S5 * S5) * dzz;
                } else {
                    sYp[(NZ + k) * NC + col] = s4 * dyz;
                }
            }
            if constexpr (ORDER == 1) {
                const double d = 1.0 / S5;
                o[0] = (A4 * d) * dy[1];   // h_y dy at the bottom row (h_y = A4 d, d = 1 / S5)
            } else {
                o[0] = dy[1];
            }
#pragma unroll
            for (int k = 0; k < NZ - 1; k++) sYp[k * NC + col] = o[k];
        }
    } else if (active) {
        if (wxl && wyl) {
#pragma unroll
            for (int k = 0; k < NZ; k++) o[k] = P(k, i, j);
        } else if (wxl || wyl) {
            const int ib = wxl ? ((i == 0) ? 1 : nxg - 2) : ((j == 0) ? 1 : nyg - 2);
            const int ws = wxl ? cclamp(ib - A, 0, nxg - RA) : cclamp(ib - A, 0, nyg - RA);
            const double *S = wxl ? SX(ib) : SY(ib);
            o[0] = P(0, i, j);
#pragma unroll
            for (int k = 1; k < NZ; k++) {
                double s = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) s += S[m] * (wxl ? P(k, ws + m, j) : P(k, i, ws + m));
                o[k] = s;
            }
        } else {
            double dx[NZ], pc[NZ];
            const int wsx = cclamp(i - A, 0, nxg - RA);
            {
                const double *S1 = SX(i), *S2 = S1 + RA;
#pragma unroll
                for (int k = 0; k < NZ; k++) {
                    double d1 = 0.0, d2 = 0.0;
#pragma unroll
                    for (int m = 0; m < RA; m++) { const double v = P(k, wsx + m, j); d1 += S1[m] * v; d2 += S2[m] * v; }
                    dx[k] = d1; o[k] = d2;
                }
            }
#pragma unroll
            for (int k = 0; k < NZ; k++) pc[k] = P(k, i, j);
            double dxc0 = dx[0];
            {
                int sh = 0;
                if (wsx == 0) sh = 1;
                if (wsx + RA - 1 == nxg - 1) sh = -1;
                if (sh != 0) {
                    const double *S = SX(i - sh);
                    double t = 0.0;
#pragma unroll
                    for (int m = 0; m < RA; m++) t += S[m] * P(0, wsx + sh + m, j);
                    dxc0 = t;
                }
            }
            {
                constexpr int wz = (1 - A) < 0 ? 0 : (1 - A);
                const double *Z1 = g.sz + (1 * 2) * RA;
                double dz = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) dz += Z1[m] * pc[wz + m];
                if constexpr (ORDER == 1) {
                    const double sg = g.zs[1], d = 1.0 / S5, hx = A2 * d, hy = A4 * d;
                    o[0] = (S5 + hx * (A2 + sg * B2) + hy * (A4 + sg * B4)) * dz + hx * dx[1];
                } else { dz0 = dz; dx1 = dx[1]; }
            }
#pragma unroll
            for (int k = 1; k < NZ - 1; k++) {
                const int wz = cclamp(k - A, 0, NZ - RA);
                const double *Z1 = g.sz + (k * 2) * RA, *Z2 = Z1 + RA;
                double dz = 0.0, dxz = 0.0, dzz = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) {
                    const double z1 = Z1[m];
                    dz += z1 * pc[wz + m];
                    if constexpr (ORDER == 0) dzz += Z2[m] * pc[wz + m];
                    dxz += z1 * ((wz + m == 0) ? dxc0 : dx[wz + m]);
                }
                const double sg = g.zs[k];
                const double s2 = A2 + sg * B2, s3 = A3 + sg * B3;
                if constexpr (ORDER == 1) o[k] = o[k] + s3 * dz + 2.0 * (s2 * dxz);
                else { xz[k] = dxz; dzk[k] = dz; zz[k] = dzz; }
            }
            o[NZ - 1] = pc[NZ - 1];
        }
    }
    lds_barrier();   // every y-side part is there
    if (!yside && interior) {
        if constexpr (ORDER == 1) {
#pragma unroll
            for (int k = 0; k < NZ - 1; k++) o[k] += sYp[k * NC + col];
        } else {
            const double d = 1.0 / S5, hx = A2 * d, hy = A4 * d, sb = g.zs[1];
            o[0] = (S5 + hx * (A2 + sb * B2) + hy * (A4 + sb * B4)) * dz0 + hx * dx1 + hy * sYp[col];
#pragma unroll
            for (int k = 1; k < NZ - 1; k++) {
                const double d2y = sYp[k * NC + col], yz = sYp[(NZ + k) * NC + col], sg = g.zs[k];
                const double s2 = A2 + sg * B2, s4 = A4 + sg * B4, s3 = A3 + sg * B3;
                o[k] = (o[k] + d2y) + s3 * dzk[k] + 2.0 * (s2 * xz[k] + yz) + (s2 * s2 + s4 * s4 + S5 * S5) * zz[k];
            }
        }
    }
    if (!yside && active) {
#pragma unroll
        for (int k = 0; k < NZ; k++) sP[col * (NZ | 1) + k] = o[k];
    }
    lds_barrier();
    {
        constexpr int E = NZ % 2 == 0 ? 2 : 1, CH = TX * NZ / E, PER = (TY * CH + NT - 1) / NT;
        const int ie = cmin(i0 + TX, nxg), je = cmin(j0 + TY, nyg);
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int e = (int)threadIdx.x + q * NT, r = e / CH, c = (e - r * CH) * E, ii = c / NZ, k = c - ii * NZ;
            if (r < je - j0 && i0 + ii < ie) {
                const double *d = sP + (r * TX + ii) * (NZ | 1) + k;
                double *g2 = out + ((size_t)(j0 + r) * nxg + i0 + ii) * NZ + k;
                if constexpr (E == 2) *reinterpret_cast<OutPair *>(g2) = OutPair{d[0], d[1]};
                else *g2 = *d;
            }
        }
    }
}

// x-z problems (Ny == 1), one thread per grid point: block = 64 columns x NZ levels.
template <int NZ, int A>
__global__ __launch_bounds__(256) void k_matvec2p(MvArgs g, const double *__restrict__ phi, double *__restrict__ out) {
    if (solve_done(g.skip)) return;
    constexpr int NT = 256, TX = 64, RA = 2 * A + 1, R = A + 1, WX = TX + 2 * R, NP = TX * NZ, PER = (NP + NT - 1) / NT;
    __shared__ double sP[WX * NZ];
    __shared__ double sDx[NP];
    const int nxg = g.nxg, nxy = g.nxy;
    const int i0 = blockIdx.x * TX;
    const int lox = cmax(cmin(i0 - R, nxg - 2 - 2 * A), 0);
    const int wx = cmin(WX, nxg - lox);
    stage_window<double, NZ, NZ, 1, WX, WX, NT>(sP, phi + (size_t)lox * NZ, 0, 1, wx);
    __syncthreads();
    auto P = [&](int k, int ii) -> double { return sP[(ii - lox) * NZ + k]; };
    double acc[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
        acc[r] = 0.0;
        const int pt = threadIdx.x + r * NT;
        if (pt >= NP) break;
        const int col = pt / NZ, k = pt - col * NZ;
        const int i = i0 + col;
        if (i >= nxg || i == 0 || i == nxg - 1) continue;
        const int wsx = cclamp(i - A, 0, nxg - RA);
        const double *S1 = g.sx + (size_t)(i * 2) * RA, *S2 = S1 + RA;
        double d1 = 0.0, d2 = 0.0;
#pragma unroll
        for (int m = 0; m < RA; m++) { const double v = P(k, wsx + m); d1 += S1[m] * v; d2 += S2[m] * v; }
        if (k == 0) {
            int sh = 0;
            if (wsx == 0) sh = 1;
            if (wsx + RA - 1 == nxg - 1) sh = -1;
            if (sh != 0) {
                const double *S = g.sx + (size_t)((i - sh) * 2) * RA;
                double t = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) t += S[m] * P(0, wsx + sh + m);
                d1 = t;
            }
        }
        sDx[pt] = d1;
        acc[r] = d2;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int pt = threadIdx.x + r * NT;
        if (pt >= NP) break;
        const int col = pt / NZ, k = pt - col * NZ;
        const int i = i0 + col;
        if (i >= nxg) continue;
        double o;
        if (i == 0 || i == nxg - 1) {
            if (k == 0) o = P(0, i);
            else {
                const int ib = (i == 0) ? 1 : nxg - 2, ws = cclamp(ib - A, 0, nxg - RA);
                const double *S = g.sx + (size_t)(ib * 2) * RA;
                o = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) o += S[m] * P(k, ws + m);
            }
        } else if (k == NZ - 1) {
            o = P(k, i);
        } else {
            const int p = i;
            const double A2 = g.cf[p], B2 = g.cf[nxy + p], S5 = g.cf[6 * nxy + p];
            const double *dxc = sDx + col * NZ;
            if (k == 0) {
                const int wz = cclamp(1 - A, 0, NZ - RA);
                const double *Z1 = g.sz + (size_t)(1 * 2) * RA;
                double dz = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) dz += Z1[m] * P(wz + m, i);
                const double hx = A2 * (1.0 / S5), sg = g.zs[1];
                o = hx * dxc[1] + (S5 + hx * (A2 + sg * B2)) * dz;
            } else {
                const double A3 = g.cf[4 * nxy + p], B3 = g.cf[5 * nxy + p];
                const int wz = cclamp(k - A, 0, NZ - RA);
                const double *Z1 = g.sz + (size_t)(k * 2) * RA, *Z2 = Z1 + RA;
                double dz = 0.0, dzz = 0.0, dxz = 0.0;
#pragma unroll
                for (int m = 0; m < RA; m++) {
                    const double z1 = Z1[m], cv = P(wz + m, i);
                    dz += z1 * cv;
                    dzz += Z2[m] * cv;
                    dxz += z1 * dxc[wz + m];
                }
                const double sg = g.zs[k];
                const double s2 = A2 + sg * B2, s3 = A3 + sg * B3;
                o = acc[r] + 2.0 * s2 * dxz + (s2 * s2 + S5 * S5) * dzz + s3 * dz;
            }
        }
        out[(size_t)i * NZ + k] = o;
    }
}

// ---------------------------------------------------------------------------------------------
// Free-surface plane: ghost update + derivatives  (DifferentiationsFreeSurfacePlane.f90:12-32,
// UpdateGhostLayerX.f90, UpdateGhostLayerY.f90), sigma-coefficient fields for the matvec.
// ---------------------------------------------------------------------------------------------
struct PlaneArgs {
    int nxg, nyg, nxy, gx, gy, a, b, nonlinear;
    const double *sx, *sy, *h;
    const double *bath;   // 3 planes: h_x, h_y, h_xx+h_yy
    double *E, *P, *Ex, *Exx, *Ey, *Eyy, *Px, *Py, *cf;
};

// one block per row j: x ghost values of E and P (rows with j in [gy, nyg-gy)), then x derivatives.
// RA: the stencil width 2a + 1 when known at compile time (loads of all taps issued together), 0: g.a's.
template <int RA>
static __global__ __launch_bounds__(256) void k_surface_x(PlaneArgs g) {
    const int j = blockIdx.x, nxg = g.nxg, ra = RA > 0 ? RA : 2 * g.a + 1;
    double *E = g.E + (size_t)j * nxg, *P = g.P + (size_t)j * nxg;
    if (j >= g.gy && j < g.nyg - g.gy && threadIdx.x < 4) {
        double *v = (threadIdx.x & 1) ? P : E;
        if (threadIdx.x < 2) {
            const double *st = g.sx + (size_t)(1 * 2) * ra;
            double s = 0.0;
#pragma unroll
            for (int m = 1; m < (RA > 0 ? RA : ra); m++) s += st[m] * v[m];
            v[0] = (0.0 - s) / st[0];
        } else {
            const double *st = g.sx + (size_t)((nxg - 2) * 2) * ra;
            double s = 0.0;
#pragma unroll
            for (int m = 0; m < (RA > 0 ? RA : ra) - 1; m++) s += st[m] * v[nxg - ra + m];
            v[nxg - 1] = (0.0 - s) / st[ra - 1];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nxg; i += blockDim.x) {
        const int ws = cclamp(i - g.a, 0, nxg - ra);
        const double *S1 = g.sx + (size_t)(i * 2) * ra, *S2 = S1 + ra;
        double e1 = 0.0, e2 = 0.0, p1 = 0.0;
#pragma unroll
        for (int m = 0; m < (RA > 0 ? RA : ra); m++) { e1 += S1[m] * E[ws + m]; e2 += S2[m] * E[ws + m]; p1 += S1[m] * P[ws + m]; }
        const size_t q = (size_t)j * nxg + i;
        g.Ex[q] = e1; g.Exx[q] = e2; g.Px[q] = p1;
        if (g.nyg == 1) {  // x-z problem: coefficient fields complete here
            const double d = g.nonlinear ? E[i] + g.h[q] : g.h[q];
            column_coefs(d, g.nonlinear ? e1 : 0.0, 0.0, g.nonlinear ? e2 : 0.0, g.bath[q], 0.0, g.bath[2 * g.nxy + q], g.cf, g.nxy, (int)q);
        }
    }
}

// y ghost values (columns with i in [gx, nxg-gx)), y derivatives and coefficients: one thread per plane
// point, 64 consecutive columns x 4 rows per block so that every load and store of a wave is contiguous.
// A ghost value depends only on interior values of its column, so each thread whose stencil reaches a
// ghost row evaluates it itself; the threads of the ghost rows also write it back.
template <int RB>
static __global__ __launch_bounds__(256) void k_surface_y(PlaneArgs g) {
    const int nxg = g.nxg, nyg = g.nyg, rb = RB > 0 ? RB : 2 * g.b + 1;
    const int i = (int)blockIdx.x * 64 + (int)(threadIdx.x & 63), j = (int)blockIdx.y * 4 + (int)(threadIdx.x >> 6);
    if (i >= nxg || j >= nyg) return;
    const bool gcol = i >= g.gx && i < nxg - g.gx;
    auto val = [&](const double *v, int jj) -> double {
        if (gcol && jj == 0) {
            const double *st = g.sy + (size_t)(1 * 2) * rb;
            double s = 0.0;
#pragma unroll
            for (int m = 1; m < (RB > 0 ? RB : rb); m++) s += st[m] * v[i + (size_t)nxg * m];
            return (0.0 - s) / st[0];
        }
        if (gcol && jj == nyg - 1) {
            const double *st = g.sy + (size_t)((nyg - 2) * 2) * rb;
            double s = 0.0;
#pragma unroll
            for (int m = 0; m < (RB > 0 ? RB : rb) - 1; m++) s += st[m] * v[i + (size_t)nxg * (nyg - rb + m)];
            return (0.0 - s) / st[rb - 1];
        }
        return v[i + (size_t)nxg * jj];
    };
    const int ws = cclamp(j - g.b, 0, nyg - rb);
    const double *S1 = g.sy + (size_t)(j * 2) * rb, *S2 = S1 + rb;
    double e1 = 0.0, e2 = 0.0, p1 = 0.0;
#pragma unroll
    for (int m = 0; m < (RB > 0 ? RB : rb); m++) {
        const double ev = val(g.E, ws + m), pv = val(g.P, ws + m);
        e1 += S1[m] * ev; e2 += S2[m] * ev; p1 += S1[m] * pv;
    }
    const size_t q = i + (size_t)nxg * j;
    const double eq = val(g.E, j);
    g.Ey[q] = e1; g.Eyy[q] = e2; g.Py[q] = p1;
    if (g.nonlinear)
        column_coefs(eq + g.h[q], g.Ex[q], e1, g.Exx[q] + e2, g.bath[q], g.bath[g.nxy + q], g.bath[2 * g.nxy + q], g.cf, g.nxy, (int)q);
    else
        column_coefs(g.h[q], 0.0, 0.0, 0.0, g.bath[q], g.bath[g.nxy + q], g.bath[2 * g.nxy + q], g.cf, g.nxy, (int)q);
    if (gcol && (j == 0 || j == nyg - 1)) {   // every reader above evaluated the ghost value itself
        const double pq = val(g.P, j);
        g.E[q] = eq; g.P[q] = pq;
    }
}

// W = dsigma/dz * one-sided sigma derivative at the surface (VerticalFreeSurfaceVelocity.f90:17).
// RC: the stencil width when known at compile time, 0: rc.
template <int RC>
static __global__ void k_vertical_velocity(int nxy, int nzg, int rc, const double *__restrict__ szTop,
                                    const double *__restrict__ cf, const double *__restrict__ phi, double *__restrict__ W) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nxy) return;
    if (RC > 0) rc = RC;
    const double *col = phi + (size_t)p * nzg + (nzg - rc);
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < (RC > 0 ? RC : rc); m++) s += szTop[m] * col[m];
    W[p] = cf[6 * nxy + p] * s;   // dsigma/dz = 1/d
}

// Free-surface right-hand side (rhsFreeSurface3D.f90:13-28, rhsLinearFreeSurface3D.f90:11-12) fused with
// the RK4 stage combination (Runge_Kutta_4.f90:38-48, 102-113, 159-170, 230-256), corner zeroing
// (Zero_Corners.f90) and damping zones (RelaxationModule_new.f90).
struct Zone { int axis, i0, i1, j0, j1, off; };
struct StageArgs {
    int nxg, nyg, nxy, dim3, nonlinear, stage, nzones, zero_corners;
    double g, dt;
    const double *E, *P;            // state at t_n
    const double *Es;               // stage surface elevation (for the rhs)
    const double *W, *Ex, *Ey, *Px, *Py;
    double *KE, *KP;                // accumulated k1 + 2 k2 + 2 k3
    double *Eo, *Po;                // output: next stage state, or the new state at stage 4
    const Zone *zones; const double *gam;
};
static __global__ void k_stage(StageArgs a) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.nxy) return;
    const int i = p % a.nxg, j = p / a.nxg;
    double kE, kP;
    const double w = a.W[p], e = a.Es[p];
    if (!a.nonlinear) { kE = w; kP = -a.g * e; }
    else if (!a.dim3) {
        const double ex = a.Ex[p], px = a.Px[p];
        kE = -ex * px + w * (1.0 + ex * ex);
        kP = -a.g * e - 0.5 * (px * px - w * w * (1.0 + ex * ex));
    } else {
        const double ex = a.Ex[p], ey = a.Ey[p], px = a.Px[p], py = a.Py[p];
        kE = -ex * px - ey * py + w * (1.0 + ex * ex + ey * ey);
        kP = -a.g * e - 0.5 * (px * px + py * py - w * w * (1.0 + ex * ex + ey * ey));
    }
    if (a.zero_corners && a.dim3 && (i == 0 || i == a.nxg - 1) && (j == 0 || j == a.nyg - 1)) { kE = 0.0; kP = 0.0; }
    double ne, np_;
    if (a.stage == 1) { a.KE[p] = kE; a.KP[p] = kP; ne = a.E[p] + 0.5 * a.dt * kE; np_ = a.P[p] + 0.5 * a.dt * kP; }
    else if (a.stage == 2) { a.KE[p] += 2.0 * kE; a.KP[p] += 2.0 * kP; ne = a.E[p] + 0.5 * a.dt * kE; np_ = a.P[p] + 0.5 * a.dt * kP; }
    else if (a.stage == 3) { a.KE[p] += 2.0 * kE; a.KP[p] += 2.0 * kP; ne = a.E[p] + a.dt * kE; np_ = a.P[p] + a.dt * kP; }
    else { ne = a.E[p] + a.dt / 6.0 * (a.KE[p] + kE); np_ = a.P[p] + a.dt / 6.0 * (a.KP[p] + kP); }
    for (int z = 0; z < a.nzones; z++) {
        const Zone Z = a.zones[z];
        if (i >= Z.i0 && i <= Z.i1 && j >= Z.j0 && j <= Z.j1) {
            const double gm = a.gam[Z.off + (Z.axis == 0 ? i - Z.i0 : j - Z.j0)];
            ne = ne * gm; np_ = np_ * gm;
        }
    }
    a.Eo[p] = ne; a.Po[p] = np_;
}

// Fluid velocities at every grid point from phi (StoreKinematicData.f90:266-326): W = dphi/dsigma, U =
// dphi/dx and V = dphi/dy with the path's first-derivative stencil rows (off-centred near the ends as
// DiffZArbitrary / DiffXEven / DiffYEven), in nonlinear mode plus the chain-rule terms
// ((1 - z)/d h_x - z/d eta_x) W and ((1 - z)/d h_y - z/d eta_y) W (z: the level's sigma coordinate, the
// ghost level's included; d = h + eta); the vertical velocity is W / d.  One thread per point.
struct KinArgs {
    int nxg, nyg, nzg, a, b, c, nonlinear;
    const double *sx, *sy, *sz;    // stencil rows [N][2][2a+1] (first derivative first)
    const double *z;               // sigma coordinate of each level, ghost level included
    const double *h, *bath;        // depth; bath planes h_x, h_y
    const double *E, *Ex, *Ey;     // surface and its derivatives
};
static __global__ __launch_bounds__(256) void k_kinematics(KinArgs a, const double *__restrict__ phi, double *__restrict__ U,
                                                           double *__restrict__ V, double *__restrict__ Wv,
                                                           double *__restrict__ Ws = nullptr) {
    const size_t nxy = (size_t)a.nxg * a.nyg, n = nxy * a.nzg;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        const int k = (int)(q % a.nzg);
        const size_t p = q / a.nzg;
        const int i = (int)(p % a.nxg), j = (int)(p / a.nxg);
        const int rz = 2 * a.c + 1, wz = cclamp(k - a.c, 0, a.nzg - rz);
        const double *Sz = a.sz + (size_t)(k * 2) * rz;
        double w = 0.0;
        for (int m = 0; m < rz; m++) w += Sz[m] * phi[p * a.nzg + wz + m];
        double u = 0.0, v = 0.0;
        if (a.nxg > 1) {
            const int rx = 2 * a.a + 1, wx = cclamp(i - a.a, 0, a.nxg - rx);
            const double *Sx = a.sx + (size_t)(i * 2) * rx;
            for (int m = 0; m < rx; m++) u += Sx[m] * phi[((size_t)j * a.nxg + wx + m) * a.nzg + k];
        }
        if (a.nyg > 1) {
            const int ry = 2 * a.b + 1, wy = cclamp(j - a.b, 0, a.nyg - ry);
            const double *Sy = a.sy + (size_t)(j * 2) * ry;
            for (int m = 0; m < ry; m++) v += Sy[m] * phi[((size_t)(wy + m) * a.nxg + i) * a.nzg + k];
        }
        const double d = a.h[p] + a.E[p], z = a.z[k];
        if (a.nonlinear) {
            if (a.nxg > 1) u = u + ((1 - z) / d * a.bath[p] - z / d * a.Ex[p]) * w;
            if (a.nyg > 1) v = v + ((1 - z) / d * a.bath[nxy + p] - z / d * a.Ey[p]) * w;
        }
        U[q] = u; V[q] = v; Wv[q] = w / d;
        if (Ws) Ws[q] = w;
    }
}

// The velocity gradients StoreKinematicData.f90:327-478 writes after u, v, w, from F = (W, U, V) with
// W = dphi/dsigma (not divided by d) and U, V the velocities above: for each field, G = Dsigma(F) / d,
// Dx(F) + cx Dsigma(F), Dy(F) + cy Dsigma(F) with the chain-rule factors cx = (1 - z)/d h_x - z/d eta_x,
// cy likewise (nonlinear mode only), x (y) derivatives zero when the grid has one column (row).  G holds
// the 9 fields of n points in that order (for W: d w_z, (d w)_x, (d w)_y).  One thread per point.
static __global__ __launch_bounds__(256) void k_kinematics_grad(KinArgs a, const double *__restrict__ W,
                                                                const double *__restrict__ U, const double *__restrict__ V,
                                                                double *__restrict__ G) {
    const size_t nxy = (size_t)a.nxg * a.nyg, n = nxy * a.nzg;
    const double *F[3] = {W, U, V};
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        const int k = (int)(q % a.nzg);
        const size_t p = q / a.nzg;
        const int i = (int)(p % a.nxg), j = (int)(p / a.nxg);
        const int rz = 2 * a.c + 1, wz = cclamp(k - a.c, 0, a.nzg - rz);
        const double *Sz = a.sz + (size_t)(k * 2) * rz;
        const double d = a.h[p] + a.E[p], z = a.z[k];
        const double cx = ((1 - z) / d * a.bath[p] - z / d * a.Ex[p]);
        const double cy = ((1 - z) / d * a.bath[nxy + p] - z / d * a.Ey[p]);
        for (int f = 0; f < 3; f++) {
            const double *Fv = F[f];
            double fz = 0.0;
            for (int m = 0; m < rz; m++) fz += Sz[m] * Fv[p * a.nzg + wz + m];
            double fx = 0.0, fy = 0.0;
            if (a.nxg > 1) {
                const int rx = 2 * a.a + 1, wx = cclamp(i - a.a, 0, a.nxg - rx);
                const double *Sx = a.sx + (size_t)(i * 2) * rx;
                for (int m = 0; m < rx; m++) fx += Sx[m] * Fv[((size_t)j * a.nxg + wx + m) * a.nzg + k];
                if (a.nonlinear) fx = fx + cx * fz;
            }
            if (a.nyg > 1) {
                const int ry = 2 * a.b + 1, wy = cclamp(j - a.b, 0, a.nyg - ry);
                const double *Sy = a.sy + (size_t)(j * 2) * ry;
                for (int m = 0; m < ry; m++) fy += Sy[m] * Fv[((size_t)(wy + m) * a.nxg + i) * a.nzg + k];
                if (a.nonlinear) fy = fy + cy * fz;
            }
            G[(size_t)(3 * f) * n + q] = fz / d;
            G[(size_t)(3 * f + 1) * n + q] = fx;
            G[(size_t)(3 * f + 2) * n + q] = fy;
        }
    }
}

// Laplace right-hand side: Dirichlet data P on the free surface of non-ghost columns, zero elsewhere
// (Runge_Kutta_4.f90:65-69 with no wall flux).
static __global__ void k_fill_rhs(int nxg, int nyg, int nzg, int gx, int gy, const double *__restrict__ P, double *__restrict__ b) {
    const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t n = (size_t)nxg * nyg * nzg;
    if (q >= n) return;
    const int k = (int)(q % nzg);
    const size_t col = q / nzg;
    const int i = (int)(col % nxg), j = (int)(col / nxg);
    double v = 0.0;
    if (k == nzg - 1 && i >= gx && i < nxg - gx && j >= gy && j < nyg - gy) v = P[col];
    b[q] = v;
}

// ---------------------------------------------------------------------------------------------
// Vector kernels (grid-stride)
// ---------------------------------------------------------------------------------------------
// y = a*x + b*y
static __global__ void k_axpby(size_t n, double a, const double *__restrict__ x, double b, double *__restrict__ y,
                               const int *skip = nullptr) {
    if (solve_done(skip)) return;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        y[q] = a * x[q] + b * y[q];
}
// y = b - y
static __global__ void k_bminus(size_t n, const double *__restrict__ b, double *__restrict__ y, const int *skip) {
    if (solve_done(skip)) return;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        y[q] = b[q] - y[q];
}
template <typename S, typename D>
__global__ void k_convert(size_t n, const S *__restrict__ x, D *__restrict__ y, const int *skip) {
    if (solve_done(skip)) return;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        y[q] = (D)x[q];
}
// Preconditioner input: b = (T) r and the iterate x = 0 in one pass.
template <typename T>
__global__ void k_precond_in(size_t n, const double *__restrict__ r, T *__restrict__ b, T *__restrict__ x, const int *skip) {
    if (solve_done(skip)) return;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        b[q] = (T)r[q];
        x[q] = T(0);
    }
}
template <typename T>
__global__ void k_fill(size_t n, T v, T *__restrict__ y, const int *skip) {
    if (solve_done(skip)) return;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        y[q] = v;
}

// Block sum of NA per-thread accumulators, stored at part[blockIdx.x * PSTRIDE + i] (fixed order: lanes by halves, then the
// waves).  At each of the first steps over the lanes half of the accumulators go to the other half of the lanes, which
// sums the same pairs: about NA exchanges for all of them where a reduction of each takes 6 NA.  k_dcgs_a with 18 vectors
// at 513 x 513 x 10 86.7 us before, 83.9 after (bound by the basis it reads); a 33 x 33 x 9 RK4 step, where the
// exchanges were a third of the kernel, 8.99 and 8.78 ms.
template <int NA, int PSTRIDE>
__device__ __forceinline__ void block_reduce_store(const double (&acc)[NA], double *part) {
    static_assert(NA <= 64, "one accumulator or more per lane");
    constexpr int NP = NA <= 1 ? 1 : NA <= 2 ? 2 : NA <= 4 ? 4 : NA <= 8 ? 8 : NA <= 16 ? 16 : NA <= 32 ? 32 : 64;
    __shared__ double red[NA][4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double v[NA];
#pragma unroll
    for (int i = 0; i < NA; i++) v[i] = acc[i];
    int mine = 0;   // the lane's accumulator
#pragma unroll
    for (int h = NP / 2, off = 32; h > 0; h >>= 1, off >>= 1) {
        const bool hi = (lane & off) != 0;
#pragma unroll
        for (int q = 0; q < h; q++) {
            if (q >= NA) continue;
            const bool two = q + h < NA;
            const double give = two ? (hi ? v[q] : v[q + h < NA ? q + h : q]) : v[q], keep = two ? (hi ? v[q + h < NA ? q + h : q] : v[q]) : v[q];
            v[q] = keep + __shfl_xor(give, off, 64);
        }
        mine += hi ? h : 0;
    }
#pragma unroll
    for (int off = 32 / NP; off > 0; off >>= 1) v[0] += __shfl_xor(v[0], off, 64);
    if (lane % (64 / NP) == 0 && mine < NA) red[mine][wv] = v[0];
    __syncthreads();
    if (threadIdx.x < NA) {
        const int i = threadIdx.x;
        part[(size_t)blockIdx.x * PSTRIDE + i] = ((red[i][0] + red[i][1]) + red[i][2]) + red[i][3];
    }
}

// The Krylov kernels below take the number of basis vectors K as a template parameter: every load of a
// grid point is issued before the first use (no predicated loads, no waits between them).

// part[b][i] = sum over block b's range of V_i . w for i < K (V_i = V + i*n); NORM adds w . w at index K.
template <int K, int NORM, int PSTRIDE>
__global__ __launch_bounds__(256) void k_mdot(size_t n, const double *__restrict__ V, const double *__restrict__ w,
                                               double *__restrict__ part, const int *skip) {
    if (solve_done(skip)) return;
    double acc[K + NORM];
#pragma unroll
    for (int i = 0; i < K + NORM; i++) acc[i] = 0.0;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        double v[K];
#pragma unroll
        for (int i = 0; i < K; i++) v[i] = V[(size_t)i * n + q];
        const double wq = w[q];
#pragma unroll
        for (int i = 0; i < K; i++) acc[i] += v[i] * wq;
        if (NORM) acc[K + NORM - 1] += wq * wq;
    }
    block_reduce_store<K + NORM, PSTRIDE>(acc, part);
}

// v <- v - sum_i h_i V_i; part gets the dots of the new v with V_i (i < K) and its squared norm (index K).
template <int K, int PSTRIDE>
__global__ __launch_bounds__(256) void k_gs_update_dot(size_t n, const double *__restrict__ V, const double *__restrict__ h,
                                                        double *__restrict__ v, double *__restrict__ part, const int *skip) {
    if (solve_done(skip)) return;
    double acc[K + 1], hh[K];
#pragma unroll
    for (int i = 0; i < K; i++) { acc[i] = 0.0; hh[i] = h[i]; }
    acc[K] = 0.0;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        double vv[K];
#pragma unroll
        for (int i = 0; i < K; i++) vv[i] = V[(size_t)i * n + q];
        double x = v[q];
#pragma unroll
        for (int i = 0; i < K; i++) x -= hh[i] * vv[i];
        v[q] = x;
#pragma unroll
        for (int i = 0; i < K; i++) acc[i] += vv[i] * x;
        acc[K] += x * x;
    }
    block_reduce_store<K + 1, PSTRIDE>(acc, part);
}

// v <- (v + sign * sum_i h_i V_i) * scale  (sign -1: orthogonalisation; +1, scale 1: solution update);
// scale_dev, when given, holds the scale in device memory.
template <int K>
__global__ __launch_bounds__(256) void k_gs_update(size_t n, const double *__restrict__ V, const double *__restrict__ h,
                                                    double sign, double scale, const double *scale_dev, double *__restrict__ v,
                                                    const int *skip) {
    if (solve_done(skip)) return;
    if (scale_dev) scale = *scale_dev;
    double hh[K];
#pragma unroll
    for (int i = 0; i < K; i++) hh[i] = sign * h[i];
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        double vv[K];
#pragma unroll
        for (int i = 0; i < K; i++) vv[i] = V[(size_t)i * n + q];
        double x = v[q];
#pragma unroll
        for (int i = 0; i < K; i++) x += hh[i] * vv[i];
        v[q] = x * scale;
    }
}

// out[i] = sum_b part[b][i]; one block per entry, fixed summation order (deterministic).
template <int MAXK>
__global__ __launch_bounds__(256) void k_reduce_parts(int nblk, int k, const double *part, double *out, const int *skip) {
    if (solve_done(skip)) return;
    const int i = blockIdx.x;
    if (i >= k) return;
    double s = 0.0;
    for (int b = threadIdx.x; b < nblk; b += 256) s += part[(size_t)b * MAXK + i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    __shared__ double w[4];
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[i] = ((w[0] + w[1]) + w[2]) + w[3];
}

// ---------------------------------------------------------------------------------------------
// Device-driven Krylov solves: the scalar work of GMRES(m) (Hessenberg column, Givens rotations,
// stopping test, back substitution) and of defect correction runs in one-thread kernels on the solve's
// stream, so a whole solve is a fixed launch sequence with no host round trip.  After convergence the
// solve's kernels see `done` and return at once.
// ---------------------------------------------------------------------------------------------
constexpr int KRYLOV_MAXK = 32;   // basis limit: GMRESmaxiterations <= KRYLOV_MAXK - 1

struct KrylovState {
    int done;       // solve finished (converged, breakdown or out of iterations)
    int skip2;      // 0 only between the two passes of an Arnoldi step that needs the DGKS second pass
    int k;          // Arnoldi steps taken
    int kk;         // basis vectors combined into the solution
    int matvecs;    // operator applications of this solve
    int status;     // 0 converged, 1 not converged
    double beta, tol, est, scale;
    double H[KRYLOV_MAXK * KRYLOV_MAXK];   // Hessenberg entry (i, j) at H[i * KRYLOV_MAXK + j]
    double cs[KRYLOV_MAXK], sn[KRYLOV_MAXK], g[KRYLOV_MAXK + 1], h1[KRYLOV_MAXK], y[KRYLOV_MAXK];
    // over all solves of the handle
    long long it_total, it_solves;
    int it_min, it_max, status_any;
    // speculative RK4 steps: a solve enqueued with fewer iteration slots than its budget that used them all
    // without stopping sets overflow; amax[stage] = most slots a solve of that stage used in this step
    int overflow, amax[4];
    long long sv_total, sv_solves;   // statistics at the start of the step (restored when it is replayed)
    int sv_min, sv_max, sv_status;
    // one-reduction CGS2 (left preconditioning): the Hessenberg columns before rotation, and the pending
    // basis vector's second-pass projections cv and inverse norm ib (the vector is normalised in the next
    // step's first pass)
    double Hr[KRYLOV_MAXK * KRYLOV_MAXK];
    double cv[KRYLOV_MAXK], ib;
};

// Start of a speculative RK4 step: clear the per-step report, keep the statistics for a replay.
static __global__ void k_step_begin(KrylovState *S) {
    if (threadIdx.x != 0) return;
    S->overflow = 0;
    for (int i = 0; i < 4; i++) S->amax[i] = 0;
    S->sv_total = S->it_total; S->sv_solves = S->it_solves; S->sv_min = S->it_min; S->sv_max = S->it_max;
    S->sv_status = S->status_any;
}
// Replay of a step: statistics as they were before it.
static __global__ void k_step_restore(KrylovState *S) {
    if (threadIdx.x != 0) return;
    S->it_total = S->sv_total; S->it_solves = S->sv_solves; S->it_min = S->sv_min; S->it_max = S->sv_max;
    S->status_any = S->sv_status;
}
// End of a step: overflow flag and per-stage slot use to host-visible memory.
static __global__ void k_step_report(const KrylovState *S, int *out) {
    if (threadIdx.x != 0) return;
    out[0] = S->overflow;
    for (int i = 0; i < 4; i++) out[1 + i] = S->amax[i];
}

// Start of a solve (before its first operator application).
static __global__ void k_solve_begin(KrylovState *S) {
    if (threadIdx.x != 0) return;
    S->done = 0; S->skip2 = 1; S->k = 0; S->kk = 0; S->matvecs = 1; S->status = 1;
}

// GMRES: hv[0] = |M^-1 (b - A x0)|^2.  Sets the stopping tolerance (rtol * beta + atol) and the scale of
// the first basis vector.
static __global__ void k_gmres_start(KrylovState *S, const double *hv, double rtol, double atol) {
    if (threadIdx.x != 0) return;
    const double beta = sqrt(hv[0]);
    S->beta = beta; S->tol = rtol * beta + atol; S->est = beta;
    if (beta <= S->tol) { S->done = 1; S->status = 0; return; }
    S->scale = 1.0 / beta;
    S->ib = 1.0;
    S->g[0] = beta;
}

// Value of lane i (uniform) of a wave, in every lane.
__device__ __forceinline__ double lane_value(double v, int i) {
    union { double d; int w[2]; } u;
    u.d = v;
    u.w[0] = __builtin_amdgcn_readlane(u.w[0], i);
    u.w[1] = __builtin_amdgcn_readlane(u.w[1], i);
    return u.d;
}
// Hessenberg column k (1-based step) of one wave: lane i holds col[i] (col[0..k-1] projections, col[k] = hn the new vector's
// norm) and the previous rotations cs[i], sn[i].  Applies the previous rotations and the new one, updates the residual
// estimate and the stopping test, and returns the rotated column, which the caller writes as column k - 1 of H.  The
// chain over the rotations reads the lanes' registers: from LDS each of its k steps waited for the store before it.
// g0 = S->g[k - 1], tol = S->tol, matvecs = S->matvecs.
__device__ __forceinline__ double gmres_column(KrylovState *S, int k, double col, double cs, double sn, int m, double g0, double tol, int matvecs) {
    constexpr int M = KRYLOV_MAXK;
    const int t = threadIdx.x;
    const double hn = lane_value(col, k);
    double a = lane_value(col, 0), out = col;
    for (int i = 0; i < k - 1; i++) {
        const double b = lane_value(col, i + 1), c = lane_value(cs, i), s = lane_value(sn, i);
        const double top = c * a + s * b;
        a = c * b - s * a;
        if (t == i) out = top;
    }
    const double b = hn;
    const double rr = sqrt(a * a + b * b);
    double c = 1.0, sv = 0.0;
    if (rr > 0.0) { c = a / rr; sv = b / rr; }
    if (t == k - 1) out = rr;
    if (t == k) out = hn;
    if (t == 0) {
        S->cs[k - 1] = c; S->sn[k - 1] = sv;
        S->g[k] = -sv * g0;
        S->g[k - 1] = c * g0;
        const double est = fabs(-sv * g0);
        S->est = est; S->k = k;
        S->scale = hn > 0.0 ? 1.0 / hn : 1.0;
        if (!(k < m && !(est <= tol) && matvecs < m) || hn == 0.0 || k + 1 >= M) S->done = 1;
    }
    return out;
}

// Arnoldi step k, first pass: hv[0..k-1] = V_i . w, hv[k] = w . w (classical Gram-Schmidt).  Keeps the
// column when the projection removed at most half of the squared norm, else asks for the second pass.
// One wave: lane i holds entry i.
static __global__ __launch_bounds__(64) void k_gmres_pass1(KrylovState *S, const double *hv, int k, int m) {
    constexpr int M = KRYLOV_MAXK;
    const int t = threadIdx.x;
    double col = t <= k ? hv[t] : 0.0;
    const double cs = t < k - 1 ? S->cs[t] : 0.0, sn = t < k - 1 ? S->sn[t] : 0.0, g0 = S->g[k - 1], tol = S->tol;
    const int matvecs = S->matvecs + 1;
    if (S->done) return;
    const double nrm2 = lane_value(col, k);
    double nn = nrm2;
    for (int i = 0; i < k; i++) { const double c = lane_value(col, i); nn -= c * c; }
    const bool second = !(nn > 0.5 * nrm2);
    if (t == 0) { S->matvecs = matvecs; S->skip2 = second ? 0 : 1; }
    if (second) {
        if (t < k) S->h1[t] = col;
    } else {
        if (t == k) col = sqrt(nn);
        col = gmres_column(S, k, col, cs, sn, m, g0, tol, matvecs);
        if (t <= k) S->H[t * M + (k - 1)] = col;
    }
}

// Arnoldi step k, second (DGKS) pass: hv holds the projections of the once-orthogonalised vector.
static __global__ __launch_bounds__(64) void k_gmres_pass2(KrylovState *S, const double *hv, int k, int m) {
    constexpr int M = KRYLOV_MAXK;
    const int t = threadIdx.x;
    const double h2 = t <= k ? hv[t] : 0.0, h1 = t < k ? S->h1[t] : 0.0;
    const double cs = t < k - 1 ? S->cs[t] : 0.0, sn = t < k - 1 ? S->sn[t] : 0.0, g0 = S->g[k - 1], tol = S->tol;
    const int matvecs = S->matvecs;
    if (S->skip2) return;
    double n2 = lane_value(h2, k);
    for (int i = 0; i < k; i++) { const double c = lane_value(h2, i); n2 -= c * c; }
    double col = h1 + h2;
    if (t == k) col = sqrt(fmax(n2, 0.0));
    col = gmres_column(S, k, col, cs, sn, m, g0, tol, matvecs);
    if (t == 0) S->skip2 = 1;
    if (t <= k) S->H[t * M + (k - 1)] = col;
}

// One-reduction classical Gram-Schmidt with reorthogonalisation (DCGS2: Swirydowicz, Langou, Ananthan,
// Yang and Thomas, Numer. Linear Algebra Appl. 28 (2021) e2343; Bielich et al., Parallel Comput. 112
// (2022) 102940) for left-preconditioned GMRES.  Step k (1-based) applies the operator to the candidate u
// in slot k-1 -- the once-orthogonalised, unnormalised vector of step k-1 -- rather than to the basis
// vector V_{k-1} = (u - sum_{i<k-1} c_i V_i) ib, whose second-pass projections c and inverse norm ib were
// found in step k-1.  By linearity z = M^-1 A u = (1/ib) M^-1 A V_{k-1} + V H c (H the unrotated
// Hessenberg columns 0..k-2), so with d = V^T z over V_0..V_{k-1}:
//   first pass: V_{k-1} normalised in place and d in one read of the basis (k_dcgs_a),
//   second pass: u' = (z - V d) ib and its projections c' = V^T u', |u'|^2 in one more read (k_dcgs_b),
//   column k-1: h = (d - H c) ib, H(0..k-1, k-1) = h + c', H(k, k-1) = sqrt(|u'|^2 - |c'|^2).
// Two reads of the basis per step instead of three (projection, second projection, update).

// Step k >= 2, first pass: slot K-1 holds u; V_{K-1} = (u - sum_{i<K-1} c_i V_i) ib is written back, and
// part gets the dots of z (slot K) with V_0 .. V_{K-1}.
template <int K, int PSTRIDE>
__global__ __launch_bounds__(256) void k_dcgs_a(size_t n, double *__restrict__ V, const KrylovState *S,
                                                 double *__restrict__ part, const int *skip) {
    static_assert(K >= 2, "the first step has no pending vector");
    if (solve_done(skip)) return;
    double c[K - 1], acc[K];
#pragma unroll
    for (int i = 0; i < K - 1; i++) c[i] = S->cv[i];
    const double ib = S->ib;
#pragma unroll
    for (int i = 0; i < K; i++) acc[i] = 0.0;
    double *__restrict__ u = V + (size_t)(K - 1) * n;
    const double *__restrict__ z = V + (size_t)K * n;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        double vv[K - 1];
#pragma unroll
        for (int i = 0; i < K - 1; i++) vv[i] = V[(size_t)i * n + q];
        double x = u[q];
        const double zq = z[q];
#pragma unroll
        for (int i = 0; i < K - 1; i++) x -= c[i] * vv[i];
        x *= ib;
        u[q] = x;
#pragma unroll
        for (int i = 0; i < K - 1; i++) acc[i] += vv[i] * zq;
        acc[K - 1] += x * zq;
    }
    block_reduce_store<K, PSTRIDE>(acc, part);
}

// Step k, second pass: v <- (v - sum_{i<K} h_i V_i) ib (h the first pass's dots); part gets the dots of the
// new v with V_i (i < K) and its squared norm (index K).
template <int K, int PSTRIDE>
__global__ __launch_bounds__(256) void k_dcgs_b(size_t n, const double *__restrict__ V, const double *__restrict__ h,
                                                 const KrylovState *S, double *__restrict__ v, double *__restrict__ part,
                                                 const int *skip) {
    if (solve_done(skip)) return;
    double acc[K + 1], hh[K];
#pragma unroll
    for (int i = 0; i < K; i++) { acc[i] = 0.0; hh[i] = h[i]; }
    acc[K] = 0.0;
    const double ib = S->ib;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        double vv[K];
#pragma unroll
        for (int i = 0; i < K; i++) vv[i] = V[(size_t)i * n + q];
        double x = v[q];
#pragma unroll
        for (int i = 0; i < K; i++) x -= hh[i] * vv[i];
        x *= ib;
        v[q] = x;
#pragma unroll
        for (int i = 0; i < K; i++) acc[i] += vv[i] * x;
        acc[K] += x * x;
    }
    block_reduce_store<K + 1, PSTRIDE>(acc, part);
}

// The two passes on pairs of grid points (16-byte loads and stores), for an even n: the basis vectors then
// start 16-byte aligned.  Each lane sums its pair's products in order (first point, then second).
template <int K, int PSTRIDE>
__global__ __launch_bounds__(256) void k_dcgs_a2(size_t n, double *__restrict__ V, const KrylovState *S,
                                                  double *__restrict__ part, const int *skip) {
    static_assert(K >= 2, "the first step has no pending vector");
    if (solve_done(skip)) return;
    double c[K - 1], acc[K];
#pragma unroll
    for (int i = 0; i < K - 1; i++) c[i] = S->cv[i];
    const double ib = S->ib;
#pragma unroll
    for (int i = 0; i < K; i++) acc[i] = 0.0;
    double2 *__restrict__ u = reinterpret_cast<double2 *>(V + (size_t)(K - 1) * n);
    const double2 *__restrict__ z = reinterpret_cast<const double2 *>(V + (size_t)K * n);
    const size_t n2 = n / 2;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n2; q += (size_t)gridDim.x * blockDim.x) {
        double2 vv[K - 1];
#pragma unroll
        for (int i = 0; i < K - 1; i++) vv[i] = reinterpret_cast<const double2 *>(V + (size_t)i * n)[q];
        double2 x = u[q];
        const double2 zq = z[q];
#pragma unroll
        for (int i = 0; i < K - 1; i++) { x.x -= c[i] * vv[i].x; x.y -= c[i] * vv[i].y; }
        x.x *= ib; x.y *= ib;
        u[q] = x;
#pragma unroll
        for (int i = 0; i < K - 1; i++) { acc[i] += vv[i].x * zq.x; acc[i] += vv[i].y * zq.y; }
        acc[K - 1] += x.x * zq.x; acc[K - 1] += x.y * zq.y;
    }
    block_reduce_store<K, PSTRIDE>(acc, part);
}
template <int K, int PSTRIDE>
__global__ __launch_bounds__(256) void k_dcgs_b2(size_t n, const double *__restrict__ V, const double *__restrict__ h,
                                                  const KrylovState *S, double *__restrict__ v, double *__restrict__ part,
                                                  const int *skip) {
    if (solve_done(skip)) return;
    double acc[K + 1], hh[K];
#pragma unroll
    for (int i = 0; i < K; i++) { acc[i] = 0.0; hh[i] = h[i]; }
    acc[K] = 0.0;
    const double ib = S->ib;
    double2 *__restrict__ v2 = reinterpret_cast<double2 *>(v);
    const size_t n2 = n / 2;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n2; q += (size_t)gridDim.x * blockDim.x) {
        double2 vv[K];
#pragma unroll
        for (int i = 0; i < K; i++) vv[i] = reinterpret_cast<const double2 *>(V + (size_t)i * n)[q];
        double2 x = v2[q];
#pragma unroll
        for (int i = 0; i < K; i++) { x.x -= hh[i] * vv[i].x; x.y -= hh[i] * vv[i].y; }
        x.x *= ib; x.y *= ib;
        v2[q] = x;
#pragma unroll
        for (int i = 0; i < K; i++) { acc[i] += vv[i].x * x.x; acc[i] += vv[i].y * x.y; }
        acc[K] += x.x * x.x; acc[K] += x.y * x.y;
    }
    block_reduce_store<K + 1, PSTRIDE>(acc, part);
}

// Step k: d = the first pass's dots (k), e = the second pass's dots and squared norm (k + 1).  Completes
// Hessenberg column k - 1, rotates it, updates the residual estimate and the stopping test, and keeps c'
// and the new inverse norm for the next step.
// One wave, a chain of latencies: everything is loaded before the first wait, the rows of H go to LDS (padded), the rest
// stays in the lanes' registers.  With one load per term of the sums and the rotations in LDS it took 6.8 us on average
// over a 513 x 513 solve and 5.1 us at 33 x 33, now 5.4 and 4.4.
static __global__ __launch_bounds__(64) void k_dcgs_column(KrylovState *S, const double *d, const double *e, int k, int m) {
    constexpr int M = KRYLOV_MAXK, PITCH = M + 1, PER = M * (M - 1) / 64;
    __shared__ double sH[(M - 1) * PITCH];
    const int t = threadIdx.x;
    double hr[PER + 1];
#pragma unroll
    for (int q = 0; q <= PER; q++) hr[q] = t + q * 64 < k * M ? S->Hr[t + q * 64] : 0.0;
    const double dv = t < k ? d[t] : 0.0, ev = t <= k ? e[t] : 0.0, cv = t < k - 1 ? S->cv[t] : 0.0;
    const double cs = t < k - 1 ? S->cs[t] : 0.0, sn = t < k - 1 ? S->sn[t] : 0.0, ib = S->ib, g0 = S->g[k - 1], tol = S->tol;
    const int matvecs = S->matvecs + 1;
    if (S->done) return;
#pragma unroll
    for (int q = 0; q <= PER; q++) {
        const int c = t + q * 64;
        if (c < k * M) sH[c / M * PITCH + c % M] = hr[q];
    }
    __syncthreads();
    // h_t = (d_t - sum_j H(t, j) c_j) ib over the columns j = t-1 .. k-2 that have row t
    double acc = dv;
    const double *row = sH + cmin(t, k - 1) * PITCH;
    for (int j = 0; j <= k - 2; j++) {
        const double c = lane_value(cv, j), h = row[j];
        if (j >= t - 1) acc -= h * c;
    }
    double col = acc * ib + ev;
    double n2 = lane_value(ev, k);
    for (int i = 0; i < k; i++) { const double c = lane_value(ev, i); n2 -= c * c; }
    const double hn = sqrt(fmax(n2, 0.0));
    if (t == k) col = hn;
    if (t <= k) S->Hr[t * M + (k - 1)] = col;
    if (t < k) S->cv[t] = ev;
    if (t == 0) {
        S->matvecs = matvecs;
        S->ib = hn > 0.0 ? 1.0 / hn : 1.0;
    }
    col = gmres_column(S, k, col, cs, sn, m, g0, tol, matvecs);
    if (t <= k) S->H[t * M + (k - 1)] = col;
}

__device__ inline void solve_stats(KrylovState *S) {
    S->it_total += S->matvecs; S->it_solves += 1;
    if (S->it_min < 0 || S->matvecs < S->it_min) S->it_min = S->matvecs;
    if (S->matvecs > S->it_max) S->it_max = S->matvecs;
    S->status_any |= S->status;
}

// End of a GMRES solve: back substitution H y = g on the kk leading columns (trailing zero pivots
// dropped), y to S->y; the solution update follows in k_basis_combine.  slots < full: the solve was
// enqueued with fewer Arnoldi steps than its budget (flags overflow when it used them all).
// (One wave stages the leading rows of H and g in LDS; lane 0 then substitutes.)
static __global__ __launch_bounds__(64) void k_gmres_finish(KrylovState *S, int slots, int full, int stage) {
    constexpr int M = KRYLOV_MAXK;
    __shared__ double sH[M * M], sg[M], sy[M];
    const int t = threadIdx.x, k = S->k;
    const bool solve = !(S->beta <= S->tol);
    if (solve) {
        for (int e = t; e < k * M; e += 64) sH[e] = S->H[e];
        if (t < k) sg[t] = S->g[t];
    }
    __syncthreads();
    if (t != 0) return;
    if (!S->done && slots < full) S->overflow = 1;
    if (k > S->amax[stage]) S->amax[stage] = k;
    int kk = 0;
    if (solve) {
        kk = k;
        while (kk > 0 && sH[(kk - 1) * M + (kk - 1)] == 0.0) kk--;
        for (int i = kk - 1; i >= 0; i--) {
            double acc = sg[i];
            for (int q = i + 1; q < kk; q++) acc -= sH[i * M + q] * sy[q];
            sy[i] = acc / sH[i * M + i];
            S->y[i] = sy[i];
        }
        S->status = (S->est <= S->tol) ? 0 : 1;
    }
    S->kk = kk;
    solve_stats(S);
}

// x += sum_{i < S->kk} S->y[i] V_i
static __global__ __launch_bounds__(256) void k_basis_combine(size_t n, const double *__restrict__ V, const KrylovState *S,
                                                              double *__restrict__ x) {
    const int kk = S->kk;
    if (kk == 0) return;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        double acc = x[q];
        for (int i0 = 0; i0 < kk; i0 += 8) {   // eight basis loads in flight per thread
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = (i0 + u < kk) ? V[(size_t)(i0 + u) * n + q] : 0.0;
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (i0 + u < kk) acc += S->y[i0 + u] * v[u];
        }
        x[q] = acc;
    }
}

// v *= S->scale
static __global__ void k_scale_state(size_t n, const KrylovState *S, double *__restrict__ v) {
    if (S->done) return;
    const double a = S->scale;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) v[q] *= a;
}

// Defect correction, iteration it (1-based): hv[0] = |z|^2 of the preconditioned defect z; the tolerance
// is set from the first one (dc.f:77-101).
static __global__ void k_dc_check(KrylovState *S, const double *hv, int it, double rtol, double atol) {
    if (threadIdx.x != 0 || S->done) return;
    const double alpha = sqrt(hv[0]);
    if (it == 1) { S->beta = alpha; S->tol = rtol * alpha + atol; }
    S->est = alpha; S->matvecs = it;
    if (alpha <= S->tol) { S->done = 1; S->status = 0; }
}

static __global__ void k_dc_finish(KrylovState *S, int slots, int full, int stage) {
    if (threadIdx.x != 0) return;
    if (!S->done && slots < full) S->overflow = 1;
    if (S->matvecs > S->amax[stage]) S->amax[stage] = S->matvecs;
    S->status = S->done ? S->status : 1;
    S->kk = 0;
    solve_stats(S);
}

// ---------------------------------------------------------------------------------------------
// Multigrid (low-order linearised operator, matrix-free; BuildLinearSystemMatrix.f90 row semantics)
// ---------------------------------------------------------------------------------------------
template <typename T>
struct LvArgs {
    int nxg, nyg, nzg, nxy, gx, gy, dim3;
    const T *sx, *sy, *sz;  // 3-point stencil rows [N][2][3]
    const T *zs;            // sigma of each level (0 on the ghost level)
    const T *col;           // 6 planes: 1/h, h_x, h_y, h_x/h, h_y/h, -2(h_x^2+h_y^2)/h^2 + (h_xx+h_yy)/h
    const int *skip;        // solve_done flag (nullptr: always run)
    int spec;               // 1: the kernels issue their loads before testing skip (small levels, where a
                            // launch is a chain of memory latencies); 0: skip is tested first
    // uniform horizontal grid (uni = 1): every interior column's centred 3-point x (y) rows are the same,
    // first derivative (-cx1, 0, cx1), second derivative (cx2, cxc, cx2)
    int uni;
    T cx1, cx2, cxc, cy1, cy2, cyc;
    const T *fac;           // records of the columns (LineRecord); nullptr: the sweep forms their line matrices
    int facq;               // 0: a record's values are contiguous; else its 16-byte chunk q is chunk q * facq + r of fac
};

// Level coefficients as the column kernels read them: 3-point stencil rows sx(i), sy(j), sz(k) (first then
// second derivative, 6 values), sigma levels zs(k), and the per-column planes col(plane, i, j).
// CoefG reads the level arrays in HBM; CoefS reads copies staged in LDS for a window of columns.
template <typename T>
struct CoefG {
    const LvArgs<T> &L;
    __device__ __forceinline__ const T *sx(int i) const { return L.sx + i * 6; }
    __device__ __forceinline__ const T *sy(int j) const { return L.sy + j * 6; }
    __device__ __forceinline__ const T *sz(int k) const { return L.sz + k * 6; }
    __device__ __forceinline__ T zs(int k) const { return L.zs[k]; }
    __device__ __forceinline__ T col(int pl, int i, int j) const { return L.col[(size_t)pl * L.nxy + i + (size_t)L.nxg * j]; }
};
template <typename T>
struct CoefS {
    const T *sx_, *sy_, *sz_, *zs_, *col_;
    int ib, jb, nx, np;   // window origin, row length and plane size of the staged column planes
    __device__ __forceinline__ const T *sx(int i) const { return sx_ + (i - ib) * 6; }
    __device__ __forceinline__ const T *sy(int j) const { return sy_ + (j - jb) * 6; }
    __device__ __forceinline__ const T *sz(int k) const { return sz_ + k * 6; }
    __device__ __forceinline__ T zs(int k) const { return zs_[k]; }
    __device__ __forceinline__ T col(int pl, int i, int j) const { return col_[pl * np + (j - jb) * nx + (i - ib)]; }
};

// LDS sizes (elements) of the staged coefficients of a window of MW x MH columns and NZ levels.
template <int MW, int MH, int NZ>
struct CoefLds {
    static constexpr int SX = MW * 6, SY = MH * 6, SZ = NZ * 6, ZS = NZ, COL = 6 * MW * MH;
    static constexpr int TOTAL = SX + SY + SZ + ZS + COL;
};

// Stages the coefficients of the window [lox, lox+wcols) x [loy, loy+wrows) (row length MW) into buf
// (CoefLds<MW, MH, NZ>::TOTAL elements) and returns the accessor.  Each segment is one predicated load per
// element with no branches around it, so all loads of a thread are in flight together.
template <typename T, int NZ, int MW, int MH, int NT>
struct CoefRegs {
    using S = CoefLds<MW, MH, NZ>;
    static constexpr int PX = (S::SX + NT - 1) / NT, PY = (S::SY + NT - 1) / NT, PZ = (S::SZ + S::ZS + NT - 1) / NT;
    static constexpr int PC = (S::COL + NT - 1) / NT;
    T vx[PX], vy[PY], vz[PZ], vc[PC];
    int lox, loy;
    __device__ __forceinline__ void load(const LvArgs<T> &L, int lox_, int loy_, int wcols, int wrows) {
        lox = lox_; loy = loy_;
        const int t = (int)threadIdx.x;
#pragma unroll
        for (int q = 0; q < PX; q++) {
            const int e = t + q * NT;
            vx[q] = (e < S::SX && e / 6 < wcols) ? L.sx[lox * 6 + e] : T(0);
        }
#pragma unroll
        for (int q = 0; q < PY; q++) {
            const int e = t + q * NT;
            vy[q] = (e < S::SY && e / 6 < wrows) ? L.sy[loy * 6 + e] : T(0);
        }
#pragma unroll
        for (int q = 0; q < PZ; q++) {
            const int e = t + q * NT;
            vz[q] = e < S::SZ ? L.sz[e] : (e < S::SZ + S::ZS ? L.zs[e - S::SZ] : T(0));
        }
#pragma unroll
        for (int q = 0; q < PC; q++) {
            const int e = t + q * NT;
            const int pl = e / (MW * MH), c = e - pl * (MW * MH), r = c / MW, cc = c - r * MW;
            vc[q] = (e < S::COL && r < wrows && cc < wcols) ? L.col[(size_t)pl * L.nxy + (size_t)(loy + r) * L.nxg + lox + cc] : T(0);
        }
    }
    __device__ __forceinline__ CoefS<T> store(T *buf) const {
        const int t = (int)threadIdx.x;
#pragma unroll
        for (int q = 0; q < PX; q++) { const int e = t + q * NT; if (e < S::SX) buf[e] = vx[q]; }
#pragma unroll
        for (int q = 0; q < PY; q++) { const int e = t + q * NT; if (e < S::SY) buf[S::SX + e] = vy[q]; }
#pragma unroll
        for (int q = 0; q < PZ; q++) { const int e = t + q * NT; if (e < S::SZ + S::ZS) buf[S::SX + S::SY + e] = vz[q]; }
#pragma unroll
        for (int q = 0; q < PC; q++) { const int e = t + q * NT; if (e < S::COL) buf[S::SX + S::SY + S::SZ + S::ZS + e] = vc[q]; }
        CoefS<T> C;
        C.sx_ = buf; C.sy_ = buf + S::SX; C.sz_ = buf + S::SX + S::SY; C.zs_ = buf + S::SX + S::SY + S::SZ;
        C.col_ = buf + S::SX + S::SY + S::SZ + S::ZS;
        C.ib = lox; C.jb = loy; C.nx = MW; C.np = MW * MH;
        return C;
    }
};
// Coefficients of the linearised (eta = 0) level operator at sigma level k: with eta = 0 the sigma
// coefficients (DetermineTransformationConstantsArray.f90:190-201) are (1 - sigma) times per-column
// constants, precomputed at set-up (planes 3, 4, 5 and 0 of col).
template <typename T, class CA>
__device__ __forceinline__ void low_coefs(const CA &C, int i, int j, int k, T &s2, T &s3, T &s4, T &s5) {
    const T om = T(1) - C.zs(k);
    s2 = om * C.col(3, i, j);
    s4 = om * C.col(4, i, j);
    s3 = om * C.col(5, i, j);
    s5 = C.col(0, i, j);
}

// Zebra z-line relaxation of column (i, j): exact tridiagonal solve in sigma of the level operator's
// rows with the neighbouring columns frozen (read through X(k, i, j)); the new column goes to out[0..NZ).
// Couplings to same-colour columns (|di| or |dj| = 2, from the corner-shifted first pass on the sigma
// ghost level) are left out, so that all columns of one colour can be relaxed at once.
// Tridiagonal solve of a zebra column given its rows (lo, di, up, rh; e2 = third entry of the bottom row): the
// elimination factors f[k] (f[0]: of row 1 from the bottom row) and reciprocal pivots of the matrix (up[0] is
// updated), then the substitution.  The surface row is the identity.
template <typename T, int NZ>
__device__ __forceinline__ void line_factor(T (&lo)[NZ], T (&di)[NZ], T (&up)[NZ], T e2, T (&f)[NZ], T (&inv)[NZ]) {
#pragma clang fp contract(off)
    f[0] = e2 != T(0) ? e2 / up[1] : T(0);   // no-op when the entry is zero
    di[0] = fma1(-f[0], lo[1], di[0]); up[0] = fma1(-f[0], di[1], up[0]);
    inv[0] = T(1) / di[0];
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) {
        f[k] = lo[k] * inv[k - 1];
        di[k] = fma1(-f[k], up[k - 1], di[k]);
        inv[k] = T(1) / di[k];
    }
}
template <typename T, int NZ>
__device__ __forceinline__ void line_solve(const T (&f)[NZ], const T (&up)[NZ], const T (&inv)[NZ], T (&rh)[NZ], T (&x)[NZ]) {
#pragma clang fp contract(off)
    rh[0] = fma1(-f[0], rh[1], rh[0]);
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) rh[k] = fma1(-f[k], rh[k - 1], rh[k]);
    x[NZ - 1] = rh[NZ - 1];
#pragma unroll
    for (int k = NZ - 2; k >= 0; k--) x[k] = fma1(-up[k], x[k + 1], rh[k]) * inv[k];
}
template <typename T, int NZ>
__device__ __forceinline__ void zebra_thomas(T (&lo)[NZ], T (&di)[NZ], T (&up)[NZ], T (&rh)[NZ], T e2, T *out) {
    T f[NZ], inv[NZ], x[NZ];
    line_factor<T, NZ>(lo, di, up, e2, f, inv);
    line_solve<T, NZ>(f, up, inv, rh, x);
#pragma unroll
    for (int k = 0; k < NZ; k++) out[k] = x[k];
}

// zebra_column for a column at least two columns away from every wall (2 <= i <= nxg-3, and the same in
// y): no clamped or shifted stencil windows, so every neighbour term is fixed at compile time.  Same
// terms in the same order as the general case.
template <typename T, int NZ, class XA, class CA>
__device__ __forceinline__ void zebra_column_interior(const LvArgs<T> &L, const CA &C, int i, int j, const XA &X, const T *bc, T *out) {
    const bool d3 = L.dim3;
    const T *SX1 = C.sx(i), *SX2 = SX1 + 3;
    const T *SY1 = C.sy(j), *SY2 = SY1 + 3;
    T lo[NZ], di[NZ], up[NZ], rh[NZ];
    T e2;
    {
        const T *Sz = C.sz(1);
        T s2, s3, s4, s5;
        low_coefs<T>(C, i, j, 1, s2, s3, s4, s5);
        const T hx = C.col(1, i, j), hy = d3 ? C.col(2, i, j) : T(0);
        const T cz = s5 + hx * s2 + hy * s4;
        T a1 = cz * Sz[1], off = T(0);
        off += hx * SX1[0] * X(1, i - 1, j);
        a1 += hx * SX1[1];
        off += hx * SX1[2] * X(1, i + 1, j);
        if (d3) {
            off += hy * SY1[0] * X(1, i, j - 1);
            a1 += hy * SY1[1];
            off += hy * SY1[2] * X(1, i, j + 1);
        }
        lo[0] = T(0); di[0] = cz * Sz[0]; up[0] = a1; e2 = cz * Sz[2];
        rh[0] = bc[0] - off;
    }
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) {
        const T *Z1 = C.sz(k), *Z2 = Z1 + 3;
        T s2, s3, s4, s5;
        low_coefs<T>(C, i, j, k, s2, s3, s4, s5);
        const T czz = s2 * s2 + s4 * s4 + s5 * s5;
        T a[3];
#pragma unroll
        for (int m = 0; m < 3; m++) a[m] = s3 * Z1[m] + czz * Z2[m];
        T off = T(0);
        off += SX2[0] * X(k, i - 1, j);
        a[1] += SX2[1];
        off += SX2[2] * X(k, i + 1, j);
#pragma unroll
        for (int mz = 0; mz < 3; mz++) {
            const int kk = k - 1 + mz;
            const T w0 = T(2) * s2 * Z1[mz] * SX1[0], w1 = T(2) * s2 * Z1[mz] * SX1[1], w2 = T(2) * s2 * Z1[mz] * SX1[2];
            off += w0 * X(kk, i - 1, j);
            a[mz] += w1;
            off += w2 * X(kk, i + 1, j);
        }
        if (d3) {
            off += SY2[0] * X(k, i, j - 1);
            a[1] += SY2[1];
            off += SY2[2] * X(k, i, j + 1);
#pragma unroll
            for (int mz = 0; mz < 3; mz++) {
                const int kk = k - 1 + mz;
                const T w0 = T(2) * s4 * Z1[mz] * SY1[0], w1 = T(2) * s4 * Z1[mz] * SY1[1], w2 = T(2) * s4 * Z1[mz] * SY1[2];
                off += w0 * X(kk, i, j - 1);
                a[mz] += w1;
                off += w2 * X(kk, i, j + 1);
            }
        }
        lo[k] = a[0]; di[k] = a[1]; up[k] = a[2];
        rh[k] = bc[k] - off;
    }
    lo[NZ - 1] = T(0); up[NZ - 1] = T(0); di[NZ - 1] = T(1); rh[NZ - 1] = bc[NZ - 1];
    zebra_thomas<T, NZ>(lo, di, up, rh, e2, out);
}

template <typename T, int NZ, class XA, class CA>
__device__ __forceinline__ void zebra_column(const LvArgs<T> &L, const CA &C, int i, int j, const XA &X, const T *bc, T *out) {
    const int nxg = L.nxg, nyg = L.nyg;
    if (i >= 2 && i <= nxg - 3 && (!L.dim3 || (j >= 2 && j <= nyg - 3))) {
        zebra_column_interior<T, NZ>(L, C, i, j, X, bc, out);
        return;
    }
    const int wsx = cclamp(i - 1, 0, nxg - 3), wsy = L.dim3 ? cclamp(j - 1, 0, nyg - 3) : 0;
    const T *SX1 = C.sx(i), *SX2 = SX1 + 3;
    const T *SY1 = C.sy(j), *SY2 = SY1 + 3;
    int shx = 0; if (wsx == 0) shx = 1; if (wsx + 2 == nxg - 1) shx = -1;
    int shy = 0;
    if (L.dim3) { if (wsy == 0) shy = 1; if (wsy + 2 == nyg - 1) shy = -1; }
    const T *SXc = C.sx(i - shx);
    const T *SYc = C.sy(j - shy);
    T lo[NZ], di[NZ], up[NZ], rh[NZ];
    T e2 = T(0);
#pragma unroll
    for (int k = 0; k < NZ; k++) { lo[k] = T(0); di[k] = T(0); up[k] = T(0); }
    // bottom ghost row
    {
        const T *Sz = C.sz(1);
        T s2, s3, s4, s5;
        low_coefs<T>(C, i, j, 1, s2, s3, s4, s5);
        const T hx = C.col(1, i, j), hy = L.dim3 ? C.col(2, i, j) : T(0);
        const T cz = s5 + hx * s2 + hy * s4;
        T a0 = cz * Sz[0], a1 = cz * Sz[1], a2 = cz * Sz[2], off = T(0);
        // branch-free: the own column's weight goes to the matrix, a neighbour's value times its weight
        // to the right-hand side (the own column is read in place of the neighbour where it is skipped)
#pragma unroll
        for (int m = 0; m < 3; m++) {
            const bool self = wsx + m == i;
            const T v = X(1, self ? i : wsx + m, j);
            a1 += self ? hx * SX1[m] : T(0);
            off += self ? T(0) : hx * SX1[m] * v;
        }
        if (L.dim3) {
#pragma unroll
            for (int m = 0; m < 3; m++) {
                const bool self = wsy + m == j;
                const T v = X(1, i, self ? j : wsy + m);
                a1 += self ? hy * SY1[m] : T(0);
                off += self ? T(0) : hy * SY1[m] * v;
            }
        }
        di[0] = a0; up[0] = a1; e2 = a2;
        rh[0] = bc[0] - off;
    }
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) {
        const T *Z1 = C.sz(k), *Z2 = Z1 + 3;
        T s2, s3, s4, s5;
        low_coefs<T>(C, i, j, k, s2, s3, s4, s5);
        const T czz = s2 * s2 + s4 * s4 + s5 * s5;
        T a[3];
#pragma unroll
        for (int m = 0; m < 3; m++) a[m] = s3 * Z1[m] + czz * Z2[m];
        T off = T(0);
#pragma unroll
        for (int m = 0; m < 3; m++) {
            const bool self = wsx + m == i;
            const T v = X(k, self ? i : wsx + m, j);
            a[1] += self ? SX2[m] : T(0);
            off += self ? T(0) : SX2[m] * v;
        }
#pragma unroll
        for (int mz = 0; mz < 3; mz++) {
            const int kk = k - 1 + mz;
            const int sh = (kk == 0) ? shx : 0;
            const T *S1 = (kk == 0) ? SXc : SX1;
#pragma unroll
            for (int m = 0; m < 3; m++) {
                const T w = T(2) * s2 * Z1[mz] * S1[m];
                const int ii = wsx + sh + m;
                const bool self = ii == i, skip = self || ii - i == 2 || i - ii == 2;
                const T v = X(kk, skip ? i : ii, j);
                a[mz] += self ? w : T(0);
                off += skip ? T(0) : w * v;
            }
        }
        if (L.dim3) {
#pragma unroll
            for (int m = 0; m < 3; m++) {
                const bool self = wsy + m == j;
                const T v = X(k, i, self ? j : wsy + m);
                a[1] += self ? SY2[m] : T(0);
                off += self ? T(0) : SY2[m] * v;
            }
#pragma unroll
            for (int mz = 0; mz < 3; mz++) {
                const int kk = k - 1 + mz;
                const int sh = (kk == 0) ? shy : 0;
                const T *S1 = (kk == 0) ? SYc : SY1;
#pragma unroll
                for (int m = 0; m < 3; m++) {
                    const T w = T(2) * s4 * Z1[mz] * S1[m];
                    const int jj = wsy + sh + m;
                    const bool self = jj == j, skip = self || jj - j == 2 || j - jj == 2;
                    const T v = X(kk, i, skip ? j : jj);
                    a[mz] += self ? w : T(0);
                    off += skip ? T(0) : w * v;
                }
            }
        }
        lo[k] = a[0]; di[k] = a[1]; up[k] = a[2];
        rh[k] = bc[k] - off;
    }
    di[NZ - 1] = T(1); rh[NZ - 1] = bc[NZ - 1];
    zebra_thomas<T, NZ>(lo, di, up, rh, e2, out);
}

// Residual o = b - L x of column (i, j) of a level (all row kinds: interior, bottom ghost, surface,
// wall ghost columns, corners), x read through X(k, i, j).
template <typename T, int NZ, class XA, class CA>
__device__ __forceinline__ void residual_column(const LvArgs<T> &L, const CA &C, int i, int j, const XA &X, const T *bc, T *o) {
    const int nxg = L.nxg, nyg = L.nyg, d3 = L.dim3;
    const bool wx = L.gx && (i == 0 || i == nxg - 1), wy = L.gy && (j == 0 || j == nyg - 1);
    if (wx && wy) {
#pragma unroll
        for (int k = 0; k < NZ; k++) o[k] = bc[k] - X(k, i, j);
    } else if (wx || wy) {
        o[0] = bc[0] - X(0, i, j);
        if (wx) {
            const int ib = i == 0 ? 1 : nxg - 2, ws = cclamp(ib - 1, 0, nxg - 3);
            const T *S = C.sx(ib);
#pragma unroll
            for (int k = 1; k < NZ; k++) o[k] = bc[k] - ((S[0] * X(k, ws, j) + S[1] * X(k, ws + 1, j)) + S[2] * X(k, ws + 2, j));
        } else {
            const int jb = j == 0 ? 1 : nyg - 2, ws = cclamp(jb - 1, 0, nyg - 3);
            const T *S = C.sy(jb);
#pragma unroll
            for (int k = 1; k < NZ; k++) o[k] = bc[k] - ((S[0] * X(k, i, ws) + S[1] * X(k, i, ws + 1)) + S[2] * X(k, i, ws + 2));
        }
    } else {
        const int wsx = cclamp(i - 1, 0, nxg - 3), wsy = d3 ? cclamp(j - 1, 0, nyg - 3) : 0;
        const T *SX1 = C.sx(i), *SX2 = SX1 + 3;
        const T *SY1 = C.sy(j), *SY2 = SY1 + 3;
        T xc[NZ], dxl[NZ], dyl[NZ];
#pragma unroll
        for (int k = 0; k < NZ; k++) {
            xc[k] = X(k, i, j);
            dxl[k] = (SX1[0] * X(k, wsx, j) + SX1[1] * X(k, wsx + 1, j)) + SX1[2] * X(k, wsx + 2, j);
            dyl[k] = d3 ? (SY1[0] * X(k, i, wsy) + SY1[1] * X(k, i, wsy + 1)) + SY1[2] * X(k, i, wsy + 2) : T(0);
        }
        {
            int sh = 0; if (wsx == 0) sh = 1; if (wsx + 2 == nxg - 1) sh = -1;
            if (sh) { const T *S = C.sx(i - sh); dxl[0] = (S[0] * X(0, wsx + sh, j) + S[1] * X(0, wsx + sh + 1, j)) + S[2] * X(0, wsx + sh + 2, j); }
            if (d3) {
                sh = 0; if (wsy == 0) sh = 1; if (wsy + 2 == nyg - 1) sh = -1;
                if (sh) { const T *S = C.sy(j - sh); dyl[0] = (S[0] * X(0, i, wsy + sh) + S[1] * X(0, i, wsy + sh + 1)) + S[2] * X(0, i, wsy + sh + 2); }
            }
        }
        o[NZ - 1] = bc[NZ - 1] - xc[NZ - 1];
#pragma unroll
        for (int k = 1; k < NZ - 1; k++) {
            const T *Z1 = C.sz(k), *Z2 = Z1 + 3;
            const T dz = (Z1[0] * xc[k - 1] + Z1[1] * xc[k]) + Z1[2] * xc[k + 1];
            const T dzz = (Z2[0] * xc[k - 1] + Z2[1] * xc[k]) + Z2[2] * xc[k + 1];
            const T dxx = (SX2[0] * X(k, wsx, j) + SX2[1] * X(k, wsx + 1, j)) + SX2[2] * X(k, wsx + 2, j);
            const T dyy = d3 ? (SY2[0] * X(k, i, wsy) + SY2[1] * X(k, i, wsy + 1)) + SY2[2] * X(k, i, wsy + 2) : T(0);
            const T dxz = (Z1[0] * dxl[k - 1] + Z1[1] * dxl[k]) + Z1[2] * dxl[k + 1];
            const T dyz = (Z1[0] * dyl[k - 1] + Z1[1] * dyl[k]) + Z1[2] * dyl[k + 1];
            T s2, s3, s4, s5;
            low_coefs<T>(C, i, j, k, s2, s3, s4, s5);
            o[k] = bc[k] - (dxx + dyy + s3 * dz + T(2) * (s2 * dxz + s4 * dyz) + (s2 * s2 + s4 * s4 + s5 * s5) * dzz);
        }
        {
            const T *Z1 = C.sz(1);
            const T dz = (Z1[0] * xc[0] + Z1[1] * xc[1]) + Z1[2] * xc[2];
            T s2, s3, s4, s5;
            low_coefs<T>(C, i, j, 1, s2, s3, s4, s5);
            const T hx = C.col(1, i, j), hy = d3 ? C.col(2, i, j) : T(0);
            o[0] = bc[0] - ((s5 + hx * s2 + hy * s4) * dz + hx * dxl[1] + hy * dyl[1]);
        }
    }
}

// Wall ghost point t of a level (t enumerates (ghost column, sigma level) pairs): Neumann rows relaxed
// pointwise, identity rows set to the right-hand side (the role of GaussSeidelSpecialPoints.f90).
template <typename T>
__device__ __forceinline__ void ghost_point(const LvArgs<T> &L, int t, T *__restrict__ x, const T *__restrict__ b) {
    const int nxg = L.nxg, nyg = L.nyg, nzg = L.nzg;
    const int col = t / nzg, k = t - col * nzg;
    int i, j;
    if (L.dim3) {
        const int nb = 2 * nxg + 2 * (nyg - 2);
        if (col >= nb) return;
        if (col < nxg) { i = col; j = 0; }
        else if (col < 2 * nxg) { i = col - nxg; j = nyg - 1; }
        else if (col < 2 * nxg + nyg - 2) { i = 0; j = 1 + col - 2 * nxg; }
        else { i = nxg - 1; j = 1 + col - 2 * nxg - (nyg - 2); }
    } else {
        if (col >= 2) return;
        i = col == 0 ? 0 : nxg - 1; j = 0;
    }
    const size_t q = ((size_t)j * nxg + i) * nzg + k;
    const bool wx = L.gx && (i == 0 || i == nxg - 1), wy = L.gy && (j == 0 || j == nyg - 1);
    if ((wx && wy) || k == 0) { x[q] = b[q]; return; }
    T s = T(0), dg = T(1);
    if (wx) {
        const int ib = i == 0 ? 1 : nxg - 2, ws = cclamp(ib - 1, 0, nxg - 3);
        const T *S = L.sx + (ib * 2) * 3;
        for (int m = 0; m < 3; m++) {
            if (ws + m == i) dg = S[m];
            else s += S[m] * x[((size_t)j * nxg + ws + m) * nzg + k];
        }
    } else {
        const int jb = j == 0 ? 1 : nyg - 2, ws = cclamp(jb - 1, 0, nyg - 3);
        const T *S = L.sy + (jb * 2) * 3;
        for (int m = 0; m < 3; m++) {
            if (ws + m == j) dg = S[m];
            else s += S[m] * x[((size_t)(ws + m) * nxg + i) * nzg + k];
        }
    }
    x[q] = (b[q] - s) / dg;
}

// Column index c of the sweep colour -> (i, j); false past the last column of that colour.
template <typename T>
__device__ __forceinline__ bool colour_column(const LvArgs<T> &L, int colour, int c, int &i, int &j) {
    const int nxi = L.nxg - 2 * L.gx, half = (nxi + 1) / 2;
    const int jr = c / half;
    j = L.dim3 ? jr + L.gy : 0;
    if (j >= (L.dim3 ? L.nyg - L.gy : 1)) return false;
    i = L.gx + (((L.gx + j) & 1) != colour ? 1 : 0) + 2 * (c - jr * half);
    return i < L.gx + nxi;
}

// Zebra sweep over the columns of one colour, one thread per column, x read and written in HBM.
template <typename T, int NZ>
__global__ __launch_bounds__(256) void k_mg_zebra(LvArgs<T> L, int colour, T *__restrict__ x, const T *__restrict__ b) {
    if (solve_done(L.skip)) return;
    int i, j;
    if (!colour_column(L, colour, (int)(blockIdx.x * blockDim.x + threadIdx.x), i, j)) return;
    const int nxg = L.nxg;
    auto X = [&](int k, int ii, int jj) -> T { return x[((size_t)jj * nxg + ii) * NZ + k]; };
    const size_t p = (size_t)i + (size_t)nxg * j;
    const CoefG<T> C{L};
    zebra_column<T, NZ>(L, C, i, j, X, b + p * NZ, x + p * NZ);
}

// LDS-tiled zebra z-line relaxation: a block stages a 32 x 8 tile of columns (plus a one-column
// halo) and the tile's right-hand sides, 128 threads each solve the sweep-colour column of one
// (even, odd) pair, and the whole tile is written back coalesced (columns of the other colour
// are rewritten unchanged; nothing else modifies them during the sweep).
template <typename T, int NZ>
__global__ __launch_bounds__(128) void k_mg_zebra_t(LvArgs<T> L, int colour, T *__restrict__ x, const T *__restrict__ b) {
    if (solve_done(L.skip)) return;
    constexpr int TX = 32, TY = 8, WX = TX + 2, WY = TY + 2, NZP = NZ | 1;
    __shared__ T sX[WX * WY * NZP];
    __shared__ T sB[TX * TY * NZP];
    const int nxg = L.nxg, nyg = L.nyg, d3 = L.dim3;
    const int i0 = L.gx + (int)blockIdx.x * TX, j0 = d3 ? L.gy + (int)blockIdx.y * TY : 0;
    const int ie = cmin(i0 + TX, nxg - L.gx), je = d3 ? cmin(j0 + TY, nyg - L.gy) : 1;
    const int lox = i0 - 1, loy = d3 ? j0 - 1 : 0;
    const int wcols = cmin(WX, nxg - lox), wrows = d3 ? cmin(WY, nyg - loy) : 1;
    stage_window<T, NZ, NZP, WY, WX, WX, 128>(sX, x + ((size_t)loy * nxg + lox) * NZ, (size_t)nxg * NZ, wrows, wcols);
    stage_window<T, NZ, NZP, TY, TX, TX, 128>(sB, b + ((size_t)j0 * nxg + i0) * NZ, (size_t)nxg * NZ, je - j0, ie - i0);
    __syncthreads();
    auto X = [&](int k, int ii, int jj) -> T { return sX[((jj - loy) * WX + (ii - lox)) * NZP + k]; };
    const int ty = threadIdx.x / 16, pr = threadIdx.x % 16;
    const int j = j0 + ty;
    int i = i0 + 2 * pr;
    if (((i + j) & 1) != colour) i++;
    if (j < je && i < ie)
        zebra_column<T, NZ>(L, CoefG<T>{L}, i, j, X, sB + ((j - j0) * TX + (i - i0)) * NZP, sX + ((j - loy) * WX + (i - lox)) * NZP);
    __syncthreads();
    for (int r = 0; r < je - j0; r++) {
        T *dst = x + ((size_t)(j0 + r) * nxg + i0) * NZ;
        for (int e = threadIdx.x; e < (ie - i0) * NZ; e += blockDim.x) {
            const int c = e / NZ, k = e - c * NZ;
            dst[e] = sX[((j0 + r - loy) * WX + (i0 + c - lox)) * NZP + k];
        }
    }
}

// A window of ROWS x COLS columns between HBM and LDS by rows: a thread takes the same piece (two values of a column
// where NZ is even) of every row (of every GR-th row with GR row groups), so that its addresses differ by a constant
// and each row is one contiguous segment.
template <typename S, int NZ, int ROWS, int COLS, int NT, int GR = 1>
struct RowWindow {
    static constexpr int E = NZ % 2 == 0 ? 2 : 1, CH = COLS * NZ / E, NG = NT / GR, PER = (CH + NG - 1) / NG, RG = (ROWS + GR - 1) / GR;
    S v[RG][PER][E];
    __device__ __forceinline__ void load(const S *__restrict__ src, size_t pitch, int rows, int cols) {
        const int t = GR == 1 ? (int)threadIdx.x : (int)threadIdx.x % NG, g = GR == 1 ? 0 : (int)threadIdx.x / NG;
#pragma unroll
        for (int p = 0; p < PER; p++) {
            const int e = (t + p * NG) * E;
            const bool in = e < cols * NZ;
#pragma unroll
            for (int q = 0; q < RG; q++) {
                const int r = q * GR + g;
                if (!in || r >= rows) continue;
                if constexpr (E == 2) {
                    const ColPair<S> w = *reinterpret_cast<const ColPair<S> *>(src + (size_t)r * pitch + e);
                    v[q][p][0] = w.a; v[q][p][1] = w.b;
                } else {
                    v[q][p][0] = src[(size_t)r * pitch + e];
                }
            }
        }
    }
    template <int NZP, int RS, typename T>
    __device__ __forceinline__ void store(T *lds, int rows, int cols) const {
        const int t = GR == 1 ? (int)threadIdx.x : (int)threadIdx.x % NG, g = GR == 1 ? 0 : (int)threadIdx.x / NG;
#pragma unroll
        for (int p = 0; p < PER; p++) {
            const int e = (t + p * NG) * E, c = e / NZ, k = e - c * NZ;
            if (e >= cols * NZ) continue;
            T *d = lds + c * NZP + k;
#pragma unroll
            for (int q = 0; q < RG; q++) {
                const int r = q * GR + g;
                if (r >= rows) continue;
#pragma unroll
                for (int m = 0; m < E; m++) d[r * RS * NZP + m] = (T)v[q][p][m];
            }
        }
    }
};

// Line system of an interior column (two columns or more from every wall) on a uniform horizontal grid: the
// matrix rows, and the right-hand side with the neighbours' terms.  Each mixed-derivative coupling is
// 2 s2 cx1 sum_m Z1[m] (x[i+1] - x[i-1]) on the three sigma levels around k (the centre weight of the first
// derivative is zero), and the differences and sums of the two neighbours are formed once per level, not once per
// row that uses them.  c: the column's level 0 in LDS, neighbours at +- SXS and +- SYS; cp: the column's six
// planes; S1x, S1y: its first-derivative rows (bottom row).
template <typename T, int NZ, bool D3>
__device__ __forceinline__ void line_matrix_uniform(const LvArgs<T> &L, const T (&cp)[6], const T (&S1x)[3], const T (&S1y)[3],
                                                    T (&lo)[NZ], T (&di)[NZ], T (&up)[NZ], T &e2) {
#pragma clang fp contract(off)
    {
        const T *Sz = L.sz + 6;
        const T om = T(1) - L.zs[1];
        const T s2 = om * cp[3], s4 = om * cp[4], s5 = cp[0];
        const T hx = cp[1], hy = D3 ? cp[2] : T(0);
        const T cz = fma1(hy, s4, fma1(hx, s2, s5));
        T a1 = fma1(cz, Sz[1], hx * S1x[1]);
        if constexpr (D3) a1 = fma1(hy, S1y[1], a1);
        lo[0] = T(0); di[0] = cz * Sz[0]; up[0] = a1; e2 = cz * Sz[2];
    }
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) {
        const T *Z1 = L.sz + k * 6, *Z2 = Z1 + 3;
        const T om = T(1) - L.zs[k];
        const T s2 = om * cp[3], s3 = om * cp[5], s5 = cp[0];
        T czz = fma1(s2, s2, s5 * s5), dc = L.cxc;
        if constexpr (D3) {
            const T s4 = om * cp[4];
            czz = fma1(s4, s4, czz);
            dc += L.cyc;
        }
        lo[k] = fma1(s3, Z1[0], czz * Z2[0]);
        di[k] = fma1(s3, Z1[1], czz * Z2[1]) + dc;
        up[k] = fma1(s3, Z1[2], czz * Z2[2]);
    }
}
// bw: the bottom row's weights of the west, east, south and north neighbour; c3, c4: h_x / h, h_y / h.
template <typename T, int NZ, bool D3, int SXS>
__device__ __forceinline__ void line_rhs_uniform(const LvArgs<T> &L, T c3, T c4, const T (&bw)[4], const T *c, int SYS, const T (&b)[NZ],
                                                 T (&rh)[NZ]) {
#pragma clang fp contract(off)
    T sx[NZ], gx[NZ], sy[NZ], gy[NZ];   // sums and differences of the x- and y-neighbours
#pragma unroll
    for (int k = 0; k < NZ; k++) {
        const T xm = c[k - SXS], xp = c[k + SXS];
        sx[k] = xm + xp; gx[k] = xp - xm;
        T ym = T(0), yp = T(0);
        if constexpr (D3) {
            ym = c[k - SYS]; yp = c[k + SYS];
            sy[k] = ym + yp; gy[k] = yp - ym;
        }
        if (k == 1) {
            T off = fma1(bw[1], xp, bw[0] * xm);
            if constexpr (D3) {
                off = fma1(bw[2], ym, off);
                off = fma1(bw[3], yp, off);
            }
            rh[0] = b[0] - off;
        }
    }
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) {
        const T *Z1 = L.sz + k * 6;
        const T om = T(1) - L.zs[k];
        const T s2 = om * c3;
        const T g = fma1(Z1[2], gx[k + 1], fma1(Z1[0], gx[k - 1], Z1[1] * gx[k]));
        T off = fma1(L.cx2, sx[k], ((T(2) * L.cx1) * s2) * g);
        if constexpr (D3) {
            const T s4 = om * c4;
            const T q = fma1(Z1[2], gy[k + 1], fma1(Z1[0], gy[k - 1], Z1[1] * gy[k]));
            off += fma1(L.cy2, sy[k], ((T(2) * L.cy1) * s4) * q);
        }
        rh[k] = b[k] - off;
    }
    rh[NZ - 1] = b[NZ - 1];
}

// Rows of a column's 3-point x and y windows (centred: beside a wall the ghost column is the outer neighbour), and
// the first row of the wall node beside it (of the high wall where there is none).
template <typename T, bool D3>
struct LineRows {
    T X1[3], X2[3], XW[3], Y1[3], Y2[3], YW[3];
    __device__ __forceinline__ void load(const LvArgs<T> &L, int i, int j) {
        const int iw = i == 1 ? 0 : L.nxg - 1, jw = j == 1 ? 0 : L.nyg - 1;
#pragma unroll
        for (int m = 0; m < 3; m++) {
            X1[m] = L.sx[i * 6 + m]; X2[m] = L.sx[i * 6 + 3 + m]; XW[m] = L.sx[iw * 6 + m];
            if constexpr (D3) { Y1[m] = L.sy[j * 6 + m]; Y2[m] = L.sy[j * 6 + 3 + m]; YW[m] = L.sy[jw * 6 + m]; }
        }
    }
    // Weights of the mixed derivative on the sigma ghost level: beside a wall its window is shifted one column
    // inwards and takes the wall node's row (ConstructTableCrossDerivatives.f90:173-186); the coupling to the
    // column two away is left out (all columns of a colour are relaxed at once).
    __device__ __forceinline__ static void ghost_level(const T (&S)[3], const T (&W)[3], int i, int n, T (&g)[3]) {
        const bool lo = i == 1, hi = !lo && i == n - 2;
        g[0] = pick(lo, T(0), pick(hi, W[1], S[0]));
        g[1] = pick(lo, W[0], pick(hi, W[2], S[1]));
        g[2] = pick(lo, W[1], pick(hi, T(0), S[2]));
    }
};
// Line system of any column from its rows: columns next to a wall, and every column of a non-uniform grid.
template <typename T, int NZ, bool D3>
__device__ __forceinline__ void line_matrix_general(const LvArgs<T> &L, int i, int j, const LineRows<T, D3> &R, const T (&cp)[6], T (&lo)[NZ],
                                                    T (&di)[NZ], T (&up)[NZ], T &e2) {
#pragma clang fp contract(off)
    T XG[3], YG[3];
    R.ghost_level(R.X1, R.XW, i, L.nxg, XG);
    if constexpr (D3) R.ghost_level(R.Y1, R.YW, j, L.nyg, YG);
    {
        const T *Sz = L.sz + 6;
        const T om = T(1) - L.zs[1];
        const T s2 = om * cp[3], s4 = om * cp[4], s5 = cp[0];
        const T hx = cp[1], hy = D3 ? cp[2] : T(0);
        const T cz = fma1(hy, s4, fma1(hx, s2, s5));
        T a1 = cz * Sz[1] + hx * R.X1[1];
        if constexpr (D3) a1 = a1 + hy * R.Y1[1];
        lo[0] = T(0); di[0] = cz * Sz[0]; up[0] = a1; e2 = cz * Sz[2];
    }
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) {
        const T *Z1 = L.sz + k * 6, *Z2 = Z1 + 3;
        const T om = T(1) - L.zs[k];
        const T s2 = om * cp[3], s4 = om * cp[4], s3 = om * cp[5], s5 = cp[0];
        const T czz = fma1(s5, s5, fma1(s2, s2, s4 * s4));
        T a[3];
#pragma unroll
        for (int m = 0; m < 3; m++) a[m] = fma1(s3, Z1[m], czz * Z2[m]);
        a[1] += R.X2[1];
#pragma unroll
        for (int m = 0; m < 3; m++) a[m] = a[m] + (T(2) * s2 * Z1[m]) * (k - 1 + m == 0 ? XG[1] : R.X1[1]);
        if constexpr (D3) {
            a[1] += R.Y2[1];
#pragma unroll
            for (int m = 0; m < 3; m++) a[m] = a[m] + (T(2) * s4 * Z1[m]) * (k - 1 + m == 0 ? YG[1] : R.Y1[1]);
        }
        lo[k] = a[0]; di[k] = a[1]; up[k] = a[2];
    }
}
template <typename T, int NZ, bool D3, int SXS>
__device__ __forceinline__ void line_rhs_general(const LvArgs<T> &L, int i, int j, const LineRows<T, D3> &R, T c3, T c4, const T (&bw)[4],
                                                 const T *c, int SYS, const T (&b)[NZ], T (&rh)[NZ]) {
#pragma clang fp contract(off)
    T XG[3], YG[3], xm[NZ], xp[NZ], ym[NZ], yp[NZ];
    R.ghost_level(R.X1, R.XW, i, L.nxg, XG);
    if constexpr (D3) R.ghost_level(R.Y1, R.YW, j, L.nyg, YG);
#pragma unroll
    for (int k = 0; k < NZ; k++) {
        xm[k] = c[k - SXS]; xp[k] = c[k + SXS];
        if constexpr (D3) { ym[k] = c[k - SYS]; yp[k] = c[k + SYS]; }
    }
    {
        T off = bw[0] * xm[1];
        off = off + bw[1] * xp[1];
        if constexpr (D3) {
            off = off + bw[2] * ym[1];
            off = off + bw[3] * yp[1];
        }
        rh[0] = b[0] - off;
    }
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) {
        const T *Z1 = L.sz + k * 6;
        const T om = T(1) - L.zs[k];
        const T s2 = om * c3, s4 = om * c4;
        T off = R.X2[0] * xm[k];
        off = off + R.X2[2] * xp[k];
#pragma unroll
        for (int m = 0; m < 3; m++) {
            const int kk = k - 1 + m;
            const T w = T(2) * s2 * Z1[m];
            off = off + (w * (kk == 0 ? XG[0] : R.X1[0])) * xm[kk];
            off = off + (w * (kk == 0 ? XG[2] : R.X1[2])) * xp[kk];
        }
        if constexpr (D3) {
            off = off + R.Y2[0] * ym[k];
            off = off + R.Y2[2] * yp[k];
#pragma unroll
            for (int m = 0; m < 3; m++) {
                const int kk = k - 1 + m;
                const T w = T(2) * s4 * Z1[m];
                off = off + (w * (kk == 0 ? YG[0] : R.Y1[0])) * ym[kk];
                off = off + (w * (kk == 0 ? YG[2] : R.Y1[2])) * yp[kk];
            }
        }
        rh[k] = b[k] - off;
    }
    rh[NZ - 1] = b[NZ - 1];
}

// line_rhs_general by two lanes per column, 32 apart: `hi` of them forms the upper half of the rows (half the time of
// the longest path of a small level's sweep; the rows of a wall column are about three times an interior
// column's).  The lower lanes receive all rows.
template <typename T, int NZ, bool D3, int SXS>
__device__ __forceinline__ void line_rhs_pair(const LvArgs<T> &L, int i, int j, bool hi, const LineRows<T, D3> &R, T c3, T c4, const T (&bw)[4],
                                              const T *c, int SYS, const T (&b)[NZ], T (&rh)[NZ]) {
#pragma clang fp contract(off)
    constexpr int HALF = (NZ - 1) / 2;   // of the NZ - 2 rows
    T XG[3], YG[3], xm[HALF + 2], xp[HALF + 2], ym[HALF + 2], yp[HALF + 2], r[HALF];
    R.ghost_level(R.X1, R.XW, i, L.nxg, XG);
    if constexpr (D3) R.ghost_level(R.Y1, R.YW, j, L.nyg, YG);
#pragma unroll
    for (int m = 0; m < 3; m++) {   // the upper half has no sigma ghost level among its rows
        XG[m] = pick(hi, R.X1[m], XG[m]);
        if constexpr (D3) YG[m] = pick(hi, R.Y1[m], YG[m]);
    }
#pragma unroll
    for (int q = 0; q < HALF + 2; q++) {
        const int k = hi ? cmin(HALF + q, NZ - 1) : q;
        xm[q] = c[k - SXS]; xp[q] = c[k + SXS];
        if constexpr (D3) { ym[q] = c[k - SYS]; yp[q] = c[k + SYS]; }
    }
    {   // bottom row (used by the lower lanes)
        T off = bw[0] * xm[1];
        off = off + bw[1] * xp[1];
        if constexpr (D3) {
            off = off + bw[2] * ym[1];
            off = off + bw[3] * yp[1];
        }
        rh[0] = b[0] - off;
    }
#pragma unroll
    for (int q = 0; q < HALF; q++) {
        constexpr int TOP = NZ - 2;
        const int kl = 1 + q, kh = cmin(1 + q + HALF, TOP);
        const T om = T(1) - pick(hi, L.zs[kh], L.zs[kl]);
        const T s2 = om * c3, s4 = om * c4;
        T Z1[3];
#pragma unroll
        for (int m = 0; m < 3; m++) Z1[m] = pick(hi, L.sz[kh * 6 + m], L.sz[kl * 6 + m]);
        T off = R.X2[0] * xm[q + 1];
        off = off + R.X2[2] * xp[q + 1];
#pragma unroll
        for (int m = 0; m < 3; m++) {
            const T w = T(2) * s2 * Z1[m];
            off = off + (w * (q + m == 0 ? XG[0] : R.X1[0])) * xm[q + m];
            off = off + (w * (q + m == 0 ? XG[2] : R.X1[2])) * xp[q + m];
        }
        if constexpr (D3) {
            off = off + R.Y2[0] * ym[q + 1];
            off = off + R.Y2[2] * yp[q + 1];
#pragma unroll
            for (int m = 0; m < 3; m++) {
                const T w = T(2) * s4 * Z1[m];
                off = off + (w * (q + m == 0 ? YG[0] : R.Y1[0])) * ym[q + m];
                off = off + (w * (q + m == 0 ? YG[2] : R.Y1[2])) * yp[q + m];
            }
        }
        r[q] = pick(hi, b[kh], b[kl]) - off;
    }
#pragma unroll
    for (int q = 0; q < HALF; q++) {
        const T up = __shfl_xor(r[q], 32);
        rh[1 + q] = r[q];
        if (1 + q + HALF <= NZ - 2) rh[1 + q + HALF] = up;
    }
    rh[NZ - 1] = b[NZ - 1];
}

// What the sweeps of a level need of a column that depends on the bottom and the grid only (LvArgs::fac), one record
// per column: the factors of its line matrix f[0 .. NZ-2], up[0 .. NZ-2], inv[0 .. NZ-2], then h_x / h, h_y / h and
// the bottom row's weights of the four neighbours.  A colour's records are contiguous, so that the lanes of a wave
// read neighbouring ones with 16-byte loads (as 3 NZ planes with coalesced 4-byte loads a 257^2 sweep took
// 15.2 us, and 4 us of a small level's sweep were address arithmetic and load issue).
template <typename T, int NZ>
struct LineRecord {
    static constexpr int W = 16 / sizeof(T), N = (3 * NZ - 3 + 6 + W - 1) / W * W;
    static constexpr int C3 = 3 * NZ - 3, C4 = C3 + 1, BW = C3 + 2;
    __host__ __device__ static size_t index(int nxg, int nyg, int i, int j) {   // of column (i, j), in records
        return ((size_t)((i + j) & 1) * nyg + j) * ((nxg + 1) / 2) + (i >> 1);
    }
    __host__ __device__ static size_t count(int nxg, int nyg) { return (size_t)2 * nyg * ((nxg + 1) / 2); }
};
template <typename T, int NZ, bool D3>
__global__ __launch_bounds__(256) void k_mg_factor(LvArgs<T> L, T *__restrict__ fac) {
#pragma clang fp contract(off)
    using Rec = LineRecord<T, NZ>;
    const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (p >= L.nxy) return;
    const int j = p / L.nxg, i = p - j * L.nxg;
    if (i < 1 || i > L.nxg - 2 || (D3 && (j < 1 || j > L.nyg - 2))) return;
    T cp[6], lo[NZ], di[NZ], up[NZ], f[NZ], inv[NZ], e2;
#pragma unroll
    for (int q = 0; q < 6; q++) cp[q] = L.col[(size_t)q * L.nxy + p];
    LineRows<T, D3> R;
    R.load(L, i, j);
    const bool edge = i < 2 || i > L.nxg - 3 || (D3 && (j < 2 || j > L.nyg - 3));
    if (edge || !L.uni) line_matrix_general<T, NZ, D3>(L, i, j, R, cp, lo, di, up, e2);
    else line_matrix_uniform<T, NZ, D3>(L, cp, R.X1, R.Y1, lo, di, up, e2);
    line_factor<T, NZ>(lo, di, up, e2, f, inv);
    const size_t r = Rec::index(L.nxg, L.nyg, i, j);
    auto put = [&](int q, T v) { fac[L.facq ? ((size_t)(q / Rec::W) * L.facq + r) * Rec::W + q % Rec::W : r * Rec::N + q] = v; };
#pragma unroll
    for (int k = 0; k < NZ - 1; k++) { put(k, f[k]); put(NZ - 1 + k, up[k]); put(2 * NZ - 2 + k, inv[k]); }
    put(Rec::C3, cp[3]); put(Rec::C4, cp[4]);
    put(Rec::BW, cp[1] * R.X1[0]); put(Rec::BW + 1, cp[1] * R.X1[2]);
    put(Rec::BW + 2, D3 ? cp[2] * R.Y1[0] : T(0)); put(Rec::BW + 3, D3 ? cp[2] * R.Y1[2] : T(0));
}

// Prolongation fused into the first post-smoothing sweep of a level with interpolation tables
// (k_mg_prolong_tab's tables and arithmetic; the coarse level is coarsened in x and y, not in sigma).
template <typename T>
struct ProArgs {
    const T *ec;              // coarse correction
    const T *pxw, *pyw;       // per fine column / row: left weight, right weight, 1 / sum
    int nxgc;                 // coarse row length
    int ghosts;               // 0: nothing reads the wall ghost points of the sweep's result before they are set anew
};

// First interior column (from 1) of tile t of nt over n columns: tiles of equal width but for one column.  The
// grids have 2^p m + 1 columns, so tiles of a fixed width of 2^q leave a last one with a single column; here every
// tile has two or more, as its wall ghost values need.
__host__ __device__ inline int tile_begin(int n, int t, int nt) { return 1 + (int)((long)n * t / nt); }

// Tile of the zebra sweep: at most TX x TY interior columns (TY = 1: x-z problems), one thread per column of a colour
// of the tile and its one-column ring, and one more wave for the columns next to a wall.
template <int NZ, int TX, int TY>
struct SweepTile {
    static constexpr bool D3 = TY > 1;
    static constexpr int H = 2, WX = TX + 2 * H, WY = D3 ? TY + 2 * H : 1, NZP = NZ | 1;
    static constexpr int RX = TX / 2 + 1, RY = D3 ? TY + 2 : 1;     // columns of a colour per row, rows (with the ring)
    static constexpr int NR = (RX * RY + 63) / 64 * 64, NT = NR + 64;
    static constexpr int BX = D3 ? TX / 2 + 1 : 0, BY = D3 ? TY / 2 + 1 : 1;   // wall columns of a colour per side
    static constexpr int GX = D3 ? TX + 2 : 0, GY = D3 ? TY + 2 : 1;           // wall ghost columns beside the ring per side
    static_assert(TX % 2 == 0 && (TY % 2 == 0 || TY == 1), "even tiles");
    static_assert(2 * (BX + BY) <= 64, "wall columns of a colour fit one wave");
    static_assert(2 * (GX + GY) <= NT, "one thread per wall ghost column");
    static_assert((WX / 2) * WY <= NT, "one thread per window column of a colour");
};

// One full zebra sweep (red columns, then black columns) in one launch, out of place (xin -> xout: a block's
// staged neighbours must not change while other blocks write their results).  A block owns a tile of
// at most TX x TY interior columns.  The red half-sweep covers the tile and its one-column ring (a red column reads only black
// neighbours, which do not change in the red half-sweep, so the ring gets exactly the values the owning blocks
// compute), the black half-sweep the tile.  The wall ghost pass before the sweep is done on the staged window
// and the one after it for the ghost points next to the tile, so one launch does (ghost pass, red, black, ghost
// pass) with x read once and written once.
//
// One thread per column: right-hand side, coefficients and the tridiagonal system live in its registers, and
// LDS holds only what columns read of each other.  A red column reads black ones and no column reads its own
// old value, so only black columns are staged (and, in tiles at a wall, red ones for the ghost pass).
// Columns next to a wall take a longer path; they have a wave of their own, so that no other wave runs both.
//
// MODE 1: the first sweep of a preconditioner application, from x = 0 with the right-hand side given as
// the FP64 residual r0: x is not read, b = (T) r0 is written to bout (unless NULL) for the points the tile owns (its
// columns and the ghost points the post-sweep ghost pass gives it), which together cover the level.
// MODE 2: the last sweep of an application: the owned points of the result go to uout as FP64 instead of to
// xout.  MODE 3: the coarse correction P is added to x first (prolongation); MODE 4: MODE 3 with the result to
// uout.  MODE 5: the first sweep of a coarse level: x = 0 (not read) and b is zero on the wall ghost columns, as
// the restrictions leave it, so that the ghost values are zero too and the red columns' rows are b alone.
// For levels whose columns' records are kept (L.fac): small levels, where a sweep is a chain of latencies, so every
// load is issued before the first wait and the red columns' loads before the black ones'.  What such a launch takes
// hardly depends on the level's size (FP32 / FP64, 33^2 to 129^2 columns of 10 values): from zero 5.8 / 6.8 us, with
// the correction 7.1-9.4 / 9.6-11.6 us, where a row of the line systems per thread, the systems passed through LDS and
// the Thomas solves on a few threads took 12.5 / 15-17 and 13.3-14.4 / 16-19 us.
template <typename T, int NZ, int TX, int TY, int MODE>
__global__ __launch_bounds__((SweepTile<NZ, TX, TY>::NT)) void k_mg_sweep(LvArgs<T> L, const T *__restrict__ xin, T *__restrict__ xout,
                                                                          const T *__restrict__ b, const double *__restrict__ r0,
                                                                          T *__restrict__ bout, double *__restrict__ uout, ProArgs<T> P) {
#pragma clang fp contract(off)
    constexpr bool ZX = MODE == 1, ZB = MODE == 5, ZO = MODE == 2 || MODE == 4, PRO = MODE == 3 || MODE == 4;
    using G = SweepTile<NZ, TX, TY>;
    constexpr bool D3 = G::D3, PAIR = 2 * (G::BX + G::BY) <= 32;   // PAIR: two lanes per wall column
    constexpr int H = G::H, WX = G::WX, WY = G::WY, NZP = G::NZP, SXS = NZP, SYS = WX * NZP;
    using Rec = LineRecord<T, NZ>;
    __shared__ T sX[WX * WY * NZP];
    const int nxg = L.nxg, nyg = L.nyg, th = (int)threadIdx.x;
    const int i0 = tile_begin(nxg - 2, (int)blockIdx.x, (int)gridDim.x), ie = tile_begin(nxg - 2, (int)blockIdx.x + 1, (int)gridDim.x);
    const int j0 = D3 ? tile_begin(nyg - 2, (int)blockIdx.y, (int)gridDim.y) : 0;
    const int je = D3 ? tile_begin(nyg - 2, (int)blockIdx.y + 1, (int)gridDim.y) : 1;
    const int lox = cmax(i0 - H, 0), loy = D3 ? cmax(j0 - H, 0) : 0;
    const int wcols = cmin(ie + H, nxg) - lox, wrows = D3 ? cmin(je + H, nyg) - loy : 1;
    const bool ww = i0 == 1, we = ie == nxg - 1, ws = D3 && j0 == 1, wn = D3 && je == nyg - 1;
    const bool wall = ww || we || ws || wn;
    const bool edge = th >= G::NR;   // the wave of the columns next to a wall
    const bool upper = PAIR && th >= G::NR + 32;
    using O = typename std::conditional<ZO, double, T>::type;
    O *const out = ZO ? (O *)uout : (O *)xout;
    auto lds = [&](int i, int j) -> T * { return sX + ((j - loy) * WX + (i - lox)) * NZP; };

    // a thread's column of a colour, and what its solve needs besides its neighbours
    struct Column {
        int i, j;
        bool on;
        T b[NZ], rec[Rec::N];
        LineRows<T, D3> R;
    };
    auto load = [&](Column &c, auto colour_tag) {
        constexpr int COL = decltype(colour_tag)::value;
        const int ilo = COL == 0 ? cmax(i0 - 1, 1) : i0, ihi = COL == 0 ? cmin(ie, nxg - 2) : ie - 1;
        const int jlo = !D3 ? 0 : (COL == 0 ? cmax(j0 - 1, 1) : j0), jhi = !D3 ? 0 : (COL == 0 ? cmin(je, nyg - 2) : je - 1);
        if (!edge) {   // away from the walls
            const int r = th / G::RX, t = th - r * G::RX;
            c.j = jlo + r;
            c.i = ilo + (((ilo + c.j) & 1) != COL ? 1 : 0) + 2 * t;
            c.on = c.i <= ihi && c.j <= jhi && c.i >= 2 && c.i <= nxg - 3 && (!D3 || (c.j >= 2 && c.j <= nyg - 3));
        } else {       // south row, north row, then west and east column
            const int l = PAIR ? (th - G::NR) & 31 : th - G::NR;
            if (D3 && l < 2 * G::BX) {
                const bool first = l < G::BX;
                const int t = first ? l : l - G::BX;
                c.j = first ? 1 : nyg - 2;
                c.i = ilo + (((ilo + c.j) & 1) != COL ? 1 : 0) + 2 * t;
                c.on = c.i <= ihi && c.j >= jlo && c.j <= jhi && (first || nyg > 3);
            } else {
                const int q = l - 2 * G::BX;
                const bool first = q < G::BY;
                const int t = first ? q : q - G::BY;
                c.i = first ? 1 : nxg - 2;
                c.j = jlo + (((c.i + jlo) & 1) != COL ? 1 : 0) + 2 * t;
                c.on = t < G::BY && c.i >= ilo && c.i <= ihi && c.j <= jhi && (first || nxg > 3) && !(D3 && (c.j == 1 || c.j == nyg - 2));
            }
        }
        const int i = c.on ? c.i : 1, j = c.on ? c.j : (D3 ? 1 : 0);   // (idle lanes load a valid column)
        const size_t p = (size_t)j * nxg + i;
        if constexpr (ZX) load_column<NZ>(r0 + p * NZ, c.b);
        else load_column<NZ>(b + p * NZ, c.b);
        load_record(L.fac + Rec::index(nxg, nyg, i, j) * Rec::N, c.rec);
        if (edge) c.R.load(L, i, j);
    };
    // a window column of one colour per thread: x, with the prolongated correction added
    struct Staged {
        int i, j;
        bool on;
        T x[NZ];
    };
    auto stage_load = [&](Staged &c, int col) {
        const int r = th / (WX / 2), t = th - r * (WX / 2);
        c.j = loy + r;
        c.i = lox + (((lox + c.j) & 1) != col ? 1 : 0) + 2 * t;
        c.on = r < wrows && c.i < lox + wcols;
        if (!c.on) return;
        if constexpr (ZX || ZB) {
#pragma unroll
            for (int k = 0; k < NZ; k++) c.x[k] = T(0);
        } else {
            load_column<NZ>(xin + ((size_t)c.j * nxg + c.i) * NZ, c.x);
        }
        if constexpr (PRO) {
            // interior columns, sigma levels 1 .. NZ - 2; column i lies on coarse column 1 + (i - 1) / 2 or between it
            // and the next
            if (c.i >= 1 && c.i <= nxg - 2 && c.j >= 1 && c.j <= nyg - 2) {
                const int2 xi = make_int2(1 + ((c.i - 1) >> 1), 1 + (c.i >> 1)), yi = make_int2(1 + ((c.j - 1) >> 1), 1 + (c.j >> 1));
                const T wxl = P.pxw[3 * c.i], wxr = P.pxw[3 * c.i + 1], sxw = P.pxw[3 * c.i + 2];
                const T wyl = P.pyw[3 * c.j], wyr = P.pyw[3 * c.j + 1], syw = P.pyw[3 * c.j + 2];
                T ea[NZ], eb[NZ], ec[NZ], ed[NZ];
                load_column<NZ>(P.ec + ((size_t)yi.x * P.nxgc + xi.x) * NZ, ea);
                load_column<NZ>(P.ec + ((size_t)yi.x * P.nxgc + xi.y) * NZ, eb);
                load_column<NZ>(P.ec + ((size_t)yi.y * P.nxgc + xi.x) * NZ, ec);
                load_column<NZ>(P.ec + ((size_t)yi.y * P.nxgc + xi.y) * NZ, ed);
#pragma unroll
                for (int k = 1; k < NZ - 1; k++) {
                    const T el = fma1(wxl, ea[k], wxr * eb[k]) * sxw, er = fma1(wxl, ec[k], wxr * ed[k]) * sxw;
                    c.x[k] = fma1(fma1(wyl, el, wyr * er), syw, c.x[k]);
                }
            }
        }
    };
    auto stage_store = [&](const Staged &c) {
        if (!c.on) return;
        T *d = lds(c.i, c.j);
#pragma unroll
        for (int k = 0; k < NZ; k++) d[k] = c.x[k];
    };
    // the thread's wall ghost column of the ring-extended tile (west, east, south, north; corners with west and east):
    // right-hand side and Neumann row (weight of the ghost, of the two columns beside it)
    int gi = -1, gj = 0;
    T gb[NZ], dg = T(1), wa = T(0), wb = T(0);
    if (wall) {
        if (th < 2 * G::GY) {
            const bool first = th < G::GY;
            const int r = (D3 ? j0 - 1 : 0) + (first ? th : th - G::GY);
            if ((first ? ww : we) && r <= (D3 ? je : 0)) { gi = first ? 0 : nxg - 1; gj = r; }
        } else if (th < 2 * (G::GX + G::GY)) {
            const int q = th - 2 * G::GY;
            const bool first = q < G::GX;
            const int c = i0 - 1 + (first ? q : q - G::GX);
            if ((first ? ws : wn) && c <= ie && !(ww && c == 0) && !(we && c == nxg - 1)) { gi = c; gj = first ? 0 : nyg - 1; }
        }
        if (gi >= 0) {
            const size_t p = (size_t)gj * nxg + gi;
            if constexpr (ZX) load_column<NZ>(r0 + p * NZ, gb);
            else load_column<NZ>(b + p * NZ, gb);
            const bool gx = gi == 0 || gi == nxg - 1, low = gx ? gi == 0 : gj == 0;
            const T *S = gx ? L.sx + (low ? 1 : nxg - 2) * 6 : L.sy + (low ? 1 : nyg - 2) * 6;
            const T w0 = S[0], w1 = S[1], w2 = S[2];
            dg = low ? w0 : w2; wa = low ? w1 : w0; wb = low ? w2 : w1;
        }
    }
    // its value from the staged interior values (GaussSeidelSpecialPoints.f90 rows: identity on the sigma ghost
    // level and at corners, the Neumann row relaxed pointwise elsewhere)
    auto ghost = [&](T (&v)[NZ]) {
        const bool gx = gi == 0 || gi == nxg - 1, gy = D3 && (gj == 0 || gj == nyg - 1);
        if (gx && gy) {
#pragma unroll
            for (int k = 0; k < NZ; k++) v[k] = gb[k];
            return;
        }
        const bool low = gx ? gi == 0 : gj == 0;
        const T *xa = gx ? lds(low ? 1 : nxg - 3, gj) : lds(gi, low ? 1 : nyg - 3);
        const T *xb = gx ? lds(low ? 2 : nxg - 2, gj) : lds(gi, low ? 2 : nyg - 2);
        v[0] = gb[0];
#pragma unroll
        for (int k = 1; k < NZ; k++) {
            const T sum = fma1(wb, xb[k], wa * xa[k]);
            v[k] = (gb[k] - sum) / dg;
        }
    };
    auto half = [&](const Column &c, auto x0) {
        constexpr bool X0 = decltype(x0)::value;   // all neighbours are zero
        if (c.on) {
            T *d = lds(c.i, c.j);
            T f[NZ], up[NZ], inv[NZ], rh[NZ], x[NZ], bw[4];
            const T c3 = c.rec[Rec::C3], c4 = c.rec[Rec::C4];
#pragma unroll
            for (int q = 0; q < 4; q++) bw[q] = c.rec[Rec::BW + q];
#pragma unroll
            for (int k = 0; k < NZ - 1; k++) { f[k] = c.rec[k]; up[k] = c.rec[NZ - 1 + k]; inv[k] = c.rec[2 * NZ - 2 + k]; }
            if constexpr (X0) {
#pragma unroll
                for (int k = 0; k < NZ; k++) rh[k] = c.b[k];
            } else if (!edge && L.uni) {
                line_rhs_uniform<T, NZ, D3, SXS>(L, c3, c4, bw, d, SYS, c.b, rh);
            } else if (PAIR && edge) {
                line_rhs_pair<T, NZ, D3, SXS>(L, c.i, c.j, upper, c.R, c3, c4, bw, d, SYS, c.b, rh);
            } else {
                LineRows<T, D3> R = c.R;
                if (!edge) R.load(L, c.i, c.j);
                line_rhs_general<T, NZ, D3, SXS>(L, c.i, c.j, R, c3, c4, bw, d, SYS, c.b, rh);
            }
            line_solve<T, NZ>(f, up, inv, rh, x);
            if (!upper) {
#pragma unroll
                for (int k = 0; k < NZ; k++) d[k] = x[k];
                if (c.i >= i0 && c.i < ie && c.j >= j0 && c.j < je) {
                    const size_t q = ((size_t)c.j * nxg + c.i) * NZ;
                    store_column<NZ>(out + q, x);
                    if constexpr (ZX) { if (bout) store_column<NZ>(bout + q, c.b); }
                }
            }
        }
    };
    Column red, black;
    load(red, std::integral_constant<int, 0>{});
    if constexpr (!ZB) {
        Staged s1, s0;
        if (!ZX || wall) {
            stage_load(s1, 1);
            if (wall) stage_load(s0, 0);
        }
        if (solve_done(L.skip)) return;
        if (!ZX || wall) {
            stage_store(s1);
            if (wall) stage_store(s0);
        }
        load(black, std::integral_constant<int, 1>{});
        if (!ZX || wall) lds_barrier();
        // the ghost pass before the sweep, on the ring-extended tile (the sweep reads no ghost point outside it)
        if (wall) {
            if (gi >= 0) {
                T v[NZ];
                ghost(v);
                T *d = lds(gi, gj);
#pragma unroll
                for (int k = 0; k < NZ; k++) d[k] = v[k];
            }
            lds_barrier();
        }
    } else {
        load(black, std::integral_constant<int, 1>{});
        if (solve_done(L.skip)) return;
        if (gi >= 0) {
            T *d = lds(gi, gj);
#pragma unroll
            for (int k = 0; k < NZ; k++) d[k] = T(0);
        }
    }
    // (MODE 1 away from the walls: nothing is staged, so the red columns must not read their neighbours)
    if (ZB || (ZX && !wall)) half(red, std::integral_constant<bool, ZX || ZB>{});
    else half(red, std::false_type{});
    lds_barrier();
    half(black, std::false_type{});
    // the ghost points this tile owns: wall columns beside its rows, wall rows beside its columns, and the corners of the
    // tiles at the corners of the domain
    const bool own = gi >= 0 && gi >= (ww ? 0 : i0) && gi < (we ? nxg : ie) && gj >= (ws ? 0 : j0) && gj < (wn ? nyg : je);
    const size_t gq = ((size_t)gj * nxg + gi) * NZ;
    if constexpr (ZX) {
        if (own && bout) store_column<NZ>(bout + gq, gb);
    }
    if (!wall || !P.ghosts) return;
    lds_barrier();
    if (own) {   // the ghost pass after the sweep
        T v[NZ];
        ghost(v);
        store_column<NZ>(out + gq, v);
    }
}


// rows x cols columns from LDS to HBM the same way.
template <int NZ, int ROWS, int COLS, int NT, int NZP, int RS, typename T, typename O>
__device__ __forceinline__ void store_rows(O *__restrict__ dst, size_t pitch, const T *lds, int rows, int cols) {
    constexpr int E = NZ % 2 == 0 ? 2 : 1, CH = COLS * NZ / E, PER = (CH + NT - 1) / NT;
#pragma unroll
    for (int p = 0; p < PER; p++) {
        const int e = ((int)threadIdx.x + p * NT) * E, c = e / NZ, k = e - c * NZ;
        if (e >= cols * NZ) continue;
        const T *s = lds + c * NZP + k;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            if (r >= rows) continue;
            if constexpr (E == 2) *reinterpret_cast<ColPair<O> *>(dst + (size_t)r * pitch + e) = ColPair<O>{(O)s[r * RS * NZP], (O)s[r * RS * NZP + 1]};
            else dst[(size_t)r * pitch + e] = (O)s[r * RS * NZP];
        }
    }
}

// k_mg_sweep for large 3D levels (same modes, same arithmetic): there the sweep is bound by the throughput of its
// HBM accesses and by its arithmetic, not by latency (513^2 x 10, first / last sweep of an application, FP32: 30.0 /
// 28.4 us, of which 12 are the loads, 12 the line solves and 2 the stores, 46-48 with the row-per-thread form; FP64
// 39.6 / 49.8 us, 71-73 before).  All fields move through LDS in whole rows (column by column,
// each lane's 40 bytes apart, the address units were busy 60% of a 513^2 sweep's 26 us), the line matrices are
// formed in registers (reading the records costs more bytes than the arithmetic costs time), the coarse window and
// then the right-hand sides share one LDS region, and the columns next to a wall are a second pass of the tiles
// that have some.
template <int NZ, int TX, int TY>
struct TiledSweep {
    static constexpr int H = 2, WX = TX + 2 * H, WY = TY + 2 * H, NZP = NZ | 1, BXC = TX + 2, BYC = TY + 2;
    static constexpr int RX = TX / 2 + 1, RY = TY + 2, NT = (RX * RY + 63) / 64 * 64;
    static constexpr int BX = TX / 2 + 1, BY = TY / 2 + 1;              // wall columns of a colour per side
    static constexpr int CWX = WX / 2 + 2, CWY = WY / 2 + 2;            // coarse window
    static constexpr int X = WX * WY * NZP, B = cmax(BXC * BYC, CWX * CWY) * NZP, TOTAL = X + B;
    static_assert(TX % 2 == 0 && TY % 2 == 0, "even tiles");
    static_assert(2 * (BX + BY) <= NT && 2 * (BXC + BYC) <= NT && (WX / 2) * WY <= 2 * NT, "threads cover the tile's lists");
};
template <typename T, int NZ, int TX, int TY, int MODE>
__global__ __launch_bounds__((TiledSweep<NZ, TX, TY>::NT)) void k_mg_sweep_tiled(
    LvArgs<T> L, const T *__restrict__ xin, T *__restrict__ xout, const T *__restrict__ b, const double *__restrict__ r0, T *__restrict__ bout,
    double *__restrict__ uout, ProArgs<T> P) {
#pragma clang fp contract(off)
    constexpr bool ZX = MODE == 1, ZB = MODE == 5, ZO = MODE == 2 || MODE == 4, PRO = MODE == 3 || MODE == 4;
    using G = TiledSweep<NZ, TX, TY>;
    constexpr int H = G::H, WX = G::WX, WY = G::WY, NZP = G::NZP, NT = G::NT, BXC = G::BXC, BYC = G::BYC, SXS = NZP, SYS = WX * NZP;
    if (solve_done(L.skip)) return;
    __shared__ T sX[G::X];
    __shared__ T sB[G::B];   // the coarse window, then the right-hand sides of the ring-extended tile
    const int nxg = L.nxg, nyg = L.nyg, nxy = L.nxy, th = (int)threadIdx.x;
    const int i0 = tile_begin(nxg - 2, (int)blockIdx.x, (int)gridDim.x), ie = tile_begin(nxg - 2, (int)blockIdx.x + 1, (int)gridDim.x);
    const int j0 = tile_begin(nyg - 2, (int)blockIdx.y, (int)gridDim.y), je = tile_begin(nyg - 2, (int)blockIdx.y + 1, (int)gridDim.y);
    const int lox = cmax(i0 - H, 0), loy = cmax(j0 - H, 0), wcols = cmin(ie + H, nxg) - lox, wrows = cmin(je + H, nyg) - loy;
    const int blox = i0 - 1, bloy = j0 - 1, bcols = ie + 1 - blox, brows = je + 1 - bloy;
    const bool ww = i0 == 1, we = ie == nxg - 1, ws = j0 == 1, wn = je == nyg - 1, wall = ww || we || ws || wn;
    using O = typename std::conditional<ZO, double, T>::type;
    O *const out = ZO ? (O *)uout : (O *)xout;
    auto lds = [&](int i, int j) -> T * { return sX + ((j - loy) * WX + (i - lox)) * NZP; };
    auto ldb = [&](int i, int j) -> T * { return sB + ((j - bloy) * BXC + (i - blox)) * NZP; };
    const size_t pitch = (size_t)nxg * NZ;
    // a thread's column of a colour away from the walls, its planes and first-derivative rows (loaded before the
    // window's wait; a column's solve would wait for them otherwise)
    struct Column {
        int i, j;
        bool on;
        T cp[6], s1x[3], s1y[3];
    };
    auto column = [&](Column &c, int col) {
        const int ilo = col == 0 ? cmax(i0 - 1, 1) : i0, ihi = col == 0 ? cmin(ie, nxg - 2) : ie - 1;
        const int jlo = col == 0 ? cmax(j0 - 1, 1) : j0, jhi = col == 0 ? cmin(je, nyg - 2) : je - 1;
        const int r = th / G::RX;
        c.j = jlo + r;
        c.i = ilo + (((ilo + c.j) & 1) != col ? 1 : 0) + 2 * (th - r * G::RX);
        c.on = c.i <= ihi && c.j <= jhi && c.i >= 2 && c.i <= nxg - 3 && c.j >= 2 && c.j <= nyg - 3;
        const int i = c.on ? c.i : 1, j = c.on ? c.j : 1;
#pragma unroll
        for (int q = 0; q < 6; q++) c.cp[q] = L.col[(size_t)q * nxy + (size_t)j * nxg + i];
#pragma unroll
        for (int m = 0; m < 3; m++) { c.s1x[m] = L.sx[i * 6 + m]; c.s1y[m] = L.sy[j * 6 + m]; }
    };
    Column red, black;
    {
        RowWindow<T, NZ, WY, WX, NT> xr;
        RowWindow<typename std::conditional<ZX, double, T>::type, NZ, BYC, BXC, NT> br;
        const int cxo = ((cmax(lox, 1) - 1) >> 1) + 1, cyo = ((cmax(loy, 1) - 1) >> 1) + 1;   // coarse window's first column, row
        if constexpr (PRO) {
            RowWindow<T, NZ, G::CWY, G::CWX, NT> pr;
            const int ccols = (cmin(lox + wcols - 1, nxg - 2) >> 1) + 2 - cxo, crows = (cmin(loy + wrows - 1, nyg - 2) >> 1) + 2 - cyo;
            pr.load(P.ec + ((size_t)cyo * P.nxgc + cxo) * NZ, (size_t)P.nxgc * NZ, crows, ccols);
            xr.load(xin + loy * pitch + (size_t)lox * NZ, pitch, wrows, wcols);
            br.load(b + bloy * pitch + (size_t)blox * NZ, pitch, brows, bcols);
            pr.template store<NZP, G::CWX>(sB, crows, ccols);
            xr.template store<NZP, WX>(sX, wrows, wcols);
            lds_barrier();
            // black columns take the correction (no column reads its own old value); in tiles at a wall red ones too,
            // for the ghost pass
            for (int q = th; q < (WX / 2) * WY * (wall ? 2 : 1); q += NT) {
                const int col = q < (WX / 2) * WY ? 1 : 0, e = col ? q : q - (WX / 2) * WY, r = e / (WX / 2);
                const int j = loy + r, i = lox + (((lox + j) & 1) != col ? 1 : 0) + 2 * (e - r * (WX / 2));
                if (r >= wrows || i >= lox + wcols || i < 1 || i > nxg - 2 || j < 1 || j > nyg - 2) continue;
                const T wxl = P.pxw[3 * i], wxr = P.pxw[3 * i + 1], sxw = P.pxw[3 * i + 2];
                const T wyl = P.pyw[3 * j], wyr = P.pyw[3 * j + 1], syw = P.pyw[3 * j + 2];
                const int xa = 1 + ((i - 1) >> 1) - cxo, xb = 1 + (i >> 1) - cxo, ya = 1 + ((j - 1) >> 1) - cyo, yb = 1 + (j >> 1) - cyo;
                const T *ea = sB + (ya * G::CWX + xa) * NZP, *eb = sB + (ya * G::CWX + xb) * NZP;
                const T *ec = sB + (yb * G::CWX + xa) * NZP, *ed = sB + (yb * G::CWX + xb) * NZP;
                T *x = lds(i, j);
#pragma unroll
                for (int k = 1; k < NZ - 1; k++) {
                    const T el = fma1(wxl, ea[k], wxr * eb[k]) * sxw, er = fma1(wxl, ec[k], wxr * ed[k]) * sxw;
                    x[k] = fma1(fma1(wyl, el, wyr * er), syw, x[k]);
                }
            }
            lds_barrier();
        } else {
            if constexpr (ZX) {
                br.load(r0 + bloy * pitch + (size_t)blox * NZ, pitch, brows, bcols);
            } else {
                if constexpr (!ZB) xr.load(xin + loy * pitch + (size_t)lox * NZ, pitch, wrows, wcols);
                br.load(b + bloy * pitch + (size_t)blox * NZ, pitch, brows, bcols);
            }
            if constexpr (ZX || ZB) {
                if (wall) for (int e = th; e < G::X; e += NT) sX[e] = T(0);
            } else {
                xr.template store<NZP, WX>(sX, wrows, wcols);
            }
        }
        column(red, 0);
        br.template store<NZP, BXC>(sB, brows, bcols);
        lds_barrier();
    }
    if (ZX && bout) store_rows<NZ, TY, TX, NT, NZP, BXC>(bout + j0 * pitch + (size_t)i0 * NZ, pitch, ldb(i0, j0), je - j0, ie - i0);
    // wall ghost column of thread th of the ring-extended tile (west, east, south, north; corners with west and east)
    int gi = -1, gj = 0;
    if (wall) {
        if (th < 2 * BYC) {
            const bool first = th < BYC;
            const int r = j0 - 1 + (first ? th : th - BYC);
            if ((first ? ww : we) && r <= je) { gi = first ? 0 : nxg - 1; gj = r; }
        } else if (th < 2 * (BXC + BYC)) {
            const int q = th - 2 * BYC;
            const bool first = q < BXC;
            const int c = i0 - 1 + (first ? q : q - BXC);
            if ((first ? ws : wn) && c <= ie && !(ww && c == 0) && !(we && c == nxg - 1)) { gi = c; gj = first ? 0 : nyg - 1; }
        }
    }
    auto ghost = [&](T (&v)[NZ]) {   // its value, as in k_mg_sweep
        const bool gx = gi == 0 || gi == nxg - 1, gy = gj == 0 || gj == nyg - 1;
        const T *gb = ldb(gi, gj);
        if (gx && gy) {
#pragma unroll
            for (int k = 0; k < NZ; k++) v[k] = gb[k];
            return;
        }
        const bool low = gx ? gi == 0 : gj == 0;
        const T *S = gx ? L.sx + (low ? 1 : nxg - 2) * 6 : L.sy + (low ? 1 : nyg - 2) * 6;
        const T w0 = S[0], w1 = S[1], w2 = S[2];
        const T dg = low ? w0 : w2, wa = low ? w1 : w0, wb = low ? w2 : w1;
        const T *xa = gx ? lds(low ? 1 : nxg - 3, gj) : lds(gi, low ? 1 : nyg - 3);
        const T *xb = gx ? lds(low ? 2 : nxg - 2, gj) : lds(gi, low ? 2 : nyg - 2);
        v[0] = gb[0];
#pragma unroll
        for (int k = 1; k < NZ; k++) {
            const T sum = fma1(wb, xb[k], wa * xa[k]);
            v[k] = (gb[k] - sum) / dg;
        }
    };
    if (wall && !ZB) {
        if (gi >= 0) {
            T v[NZ];
            ghost(v);
            T *d = lds(gi, gj);
#pragma unroll
            for (int k = 0; k < NZ; k++) d[k] = v[k];
        }
        lds_barrier();
    }
    // one column's line solve; x0: all neighbours are zero
    auto solve = [&](int i, int j, const T (&cp)[6], const T (&s1x)[3], const T (&s1y)[3], auto edge_tag, auto x0) {
        constexpr bool EDGE = decltype(edge_tag)::value, X0 = decltype(x0)::value;
        T bc[NZ], lo[NZ], di[NZ], up[NZ], f[NZ], inv[NZ], rh[NZ], x[NZ], e2;
        T *d = lds(i, j);
        const T *bl = ldb(i, j);
        LineRows<T, true> R;
        if (EDGE || !L.uni) {
            R.load(L, i, j);
            line_matrix_general<T, NZ, true>(L, i, j, R, cp, lo, di, up, e2);
        } else {
            line_matrix_uniform<T, NZ, true>(L, cp, s1x, s1y, lo, di, up, e2);
        }
        const T bw[4] = {cp[1] * s1x[0], cp[1] * s1x[2], cp[2] * s1y[0], cp[2] * s1y[2]};
        line_factor<T, NZ>(lo, di, up, e2, f, inv);   // before the right-hand side is formed: fewer live values
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < NZ; k++) bc[k] = bl[k];
        if constexpr (X0) {
#pragma unroll
            for (int k = 0; k < NZ; k++) rh[k] = bc[k];
        } else if (EDGE || !L.uni) {
            line_rhs_general<T, NZ, true, SXS>(L, i, j, R, cp[3], cp[4], bw, d, SYS, bc, rh);
        } else {
            line_rhs_uniform<T, NZ, true, SXS>(L, cp[3], cp[4], bw, d, SYS, bc, rh);
        }
        line_solve<T, NZ>(f, up, inv, rh, x);
#pragma unroll
        for (int k = 0; k < NZ; k++) d[k] = x[k];
    };
    auto half = [&](const Column &c, int col, auto x0) {
        if (c.on) solve(c.i, c.j, c.cp, c.s1x, c.s1y, std::false_type{}, x0);
        if (wall && th < 2 * (G::BX + G::BY)) {   // beside the walls: south row, north row, then west and east column
            const int ilo = col == 0 ? cmax(i0 - 1, 1) : i0, ihi = col == 0 ? cmin(ie, nxg - 2) : ie - 1;
            const int jlo = col == 0 ? cmax(j0 - 1, 1) : j0, jhi = col == 0 ? cmin(je, nyg - 2) : je - 1;
            int i, j;
            bool on;
            if (th < 2 * G::BX) {
                const bool first = th < G::BX;
                j = first ? 1 : nyg - 2;
                i = ilo + (((ilo + j) & 1) != col ? 1 : 0) + 2 * (first ? th : th - G::BX);
                on = i <= ihi && j >= jlo && j <= jhi && (first || nyg > 3);
            } else {
                const int q = th - 2 * G::BX;
                const bool first = q < G::BY;
                i = first ? 1 : nxg - 2;
                j = jlo + (((i + jlo) & 1) != col ? 1 : 0) + 2 * (first ? q : q - G::BY);
                on = i >= ilo && i <= ihi && j <= jhi && (first || nxg > 3) && j != 1 && j != nyg - 2;
            }
            if (on) {
                T cp[6], s1x[3], s1y[3];
#pragma unroll
                for (int q = 0; q < 6; q++) cp[q] = L.col[(size_t)q * nxy + (size_t)j * nxg + i];
#pragma unroll
                for (int m = 0; m < 3; m++) { s1x[m] = L.sx[i * 6 + m]; s1y[m] = L.sy[j * 6 + m]; }
                solve(i, j, cp, s1x, s1y, std::true_type{}, x0);
            }
        }
        lds_barrier();
    };
    column(black, 1);
    if (ZB || (ZX && !wall)) half(red, 0, std::integral_constant<bool, ZX || ZB>{});
    else half(red, 0, std::false_type{});
    half(black, 1, std::false_type{});
    store_rows<NZ, TY, TX, NT, NZP, WX>(out + j0 * pitch + (size_t)i0 * NZ, pitch, lds(i0, j0), je - j0, ie - i0);
    if (gi >= 0 && gi >= (ww ? 0 : i0) && gi < (we ? nxg : ie) && gj >= (ws ? 0 : j0) && gj < (wn ? nyg : je)) {
        const size_t q = gj * pitch + (size_t)gi * NZ;
        T v[NZ];
        if (ZX && bout) {
#pragma unroll
            for (int k = 0; k < NZ; k++) v[k] = ldb(gi, gj)[k];
            store_column<NZ>(bout + q, v);
        }
        if (P.ghosts) {
            ghost(v);
            store_column<NZ>(out + q, v);
        }
    }
}

template <typename T>
__global__ void k_mg_ghost_p(LvArgs<T> L, T *__restrict__ x, const T *__restrict__ b) {
    if (solve_done(L.skip)) return;
    ghost_point(L, (int)(blockIdx.x * blockDim.x + threadIdx.x), x, b);
}

// LDS-tiled residual r = b - L x (16 x TY columns per block, halo 2 on domain ends as the matvec; x-z
// problems: one row of 16 * TY columns), level coefficients staged in LDS with the tile.
template <typename T, int NZ, int TY>
__global__ __launch_bounds__(16 * TY) void k_mg_residual_t(LvArgs<T> L, const T *__restrict__ x, const T *__restrict__ b, T *__restrict__ r) {
    if (!L.spec && solve_done(L.skip)) return;
    constexpr int TX = 16, R = 2, WX = TX + 2 * R, WY = TY + 2 * R, NZP = NZ | 1, NT = TX * TY;
    constexpr int RS2 = TX * TY + 2 * R;       // x-z problems: the tile is one row of TX * TY columns
    constexpr int LX = WX * WY > RS2 ? WX * WY : RS2;
    __shared__ T sX[LX * NZP];
    __shared__ T sC[CoefLds<WX, WY, NZ>::TOTAL > CoefLds<RS2, 1, NZ>::TOTAL ? CoefLds<WX, WY, NZ>::TOTAL : CoefLds<RS2, 1, NZ>::TOTAL];
    const int nxg = L.nxg, nyg = L.nyg, d3 = L.dim3;
    const int i0 = d3 ? (int)blockIdx.x * TX : (int)blockIdx.x * (TX * TY), j0 = d3 ? (int)blockIdx.y * TY : 0;
    const int tw = d3 ? TX : TX * TY;        // columns per tile row
    const int lox = cmax(cmin(i0 - R, nxg - 4), 0);
    const int loy = d3 ? cmax(cmin(j0 - R, nyg - 4), 0) : 0;
    const int wcols = cmin(tw + 2 * R, nxg - lox), wrows = d3 ? cmin(WY, nyg - loy) : 1;
    const int rowstride = d3 ? WX : RS2;
    const int tx = d3 ? (int)threadIdx.x % TX : (int)threadIdx.x, ty = d3 ? (int)threadIdx.x / TX : 0;
    const int i = i0 + tx, j = j0 + ty;
    const bool active = i < nxg && j < nyg;
    // every HBM load of the block (coefficients, x window, the thread's column of b) is in flight before
    // the first wait
    T bc[NZ];
    const T *bp = b + ((size_t)i + (size_t)nxg * j) * NZ;
#pragma unroll
    for (int k = 0; k < NZ; k++) bc[k] = active ? bp[k] : T(0);
    CoefS<T> C;
    if (d3) {
        CoefRegs<T, NZ, WX, WY, NT> cr;
        WindowRegs<T, NZ, WY, WX, NT> xr;
        cr.load(L, lox, loy, wcols, wrows);
        xr.load(x + ((size_t)loy * nxg + lox) * NZ, (size_t)nxg * NZ, wrows, wcols);
        if (L.spec && solve_done(L.skip)) return;
        C = cr.store(sC);
        xr.template store<NZP, WX>(sX, wrows, wcols);
    } else {
        CoefRegs<T, NZ, RS2, 1, NT> cr;
        WindowRegs<T, NZ, 1, RS2, NT> xr;
        cr.load(L, lox, loy, wcols, wrows);
        xr.load(x + (size_t)lox * NZ, 0, 1, wcols);
        if (L.spec && solve_done(L.skip)) return;
        C = cr.store(sC);
        xr.template store<NZP, RS2>(sX, 1, wcols);
    }
    __syncthreads();
    auto X = [&](int k, int ii, int jj) -> T { return sX[((jj - loy) * rowstride + (ii - lox)) * NZP + k]; };
    T o[NZ];
    if (active) residual_column<T, NZ>(L, C, i, j, X, bc, o);
    __syncthreads();
    if (active) {
        T *dst = sX + ((j - loy) * rowstride + (i - lox)) * NZP;
#pragma unroll
        for (int k = 0; k < NZ; k++) dst[k] = o[k];
    }
    __syncthreads();
    const int ie = cmin(i0 + tw, nxg), je = d3 ? cmin(j0 + TY, nyg) : 1;
    for (int rr = 0; rr < je - j0; rr++)
        store_row<NZ, NZP, NT>(r + ((size_t)(j0 + rr) * nxg + i0) * NZ, sX + ((j0 + rr - loy) * rowstride + (i0 - lox)) * NZP, ie - i0);
}

// Restriction (MGRestriction3DExplicit.f90): separable full weighting x -> y -> z on interior
// points below the free surface, then injection; coarse ghost entries are zero.
struct RestrictGeo {
    int nxgf, nygf, nzgf, nxf, nyf, nzf, gx, gy;     // fine
    int nxgc, nygc, nzgc, nxc, nyc, nzc;             // coarse
    int xc, yc, zc;
    const double *xf, *yf, *zf;                      // fine coordinates
    const int *skip;                                 // solve_done flag (nullptr: always run)
    int spec;                                        // 1: loads are issued before skip is tested
};
// Restricted residual at coarse point (kc, ic, jc) (0 on ghost points), the residual read through R(k, i, j).
template <typename T, class RA>
__device__ __forceinline__ T restrict_at(const RestrictGeo &G, int kc, int ic, int jc, const RA &R) {
    const int icn = ic - G.gx, jcn = jc - G.gy;
    if (kc < 1 || icn < 0 || icn >= G.nxc || jcn < 0 || jcn >= G.nyc) return T(0);
    const int kf = 1 + (kc - 1) * (1 + G.zc), ifn = G.gx + icn * (1 + G.xc), jfn = G.gy + jcn * (1 + G.yc);
    // x pass value at (k,i,j)
    auto Xv = [&](int k, int i, int j) -> T {
        if (G.xc && k >= 1 && k <= G.nzf - 1 && j >= G.gy && j <= G.nyf + G.gy - 1 && ((i - G.gx) % 2 == 0) && i >= G.gx && i <= G.nxf + G.gx - 1) {
            const T dW = (T)(G.xf[i] - G.xf[i - 1]), dE = (T)(G.xf[i + 1] - G.xf[i]);
            const T dxc = T(1) / (dW + dE);
            return (T(0.5) * dxc) * ((dW * R(k, i - 1, j) + (dW + dE) * R(k, i, j)) + dE * R(k, i + 1, j));
        }
        return R(k, i, j);
    };
    auto Yv = [&](int k, int i, int j) -> T {
        if (G.yc && k >= 1 && k <= G.nzf - 1 && ((j - G.gy) % 2 == 0) && j >= G.gy && j <= G.nyf + G.gy - 1 &&
            i >= G.gx && i <= G.nxf + G.gx - 1 && (((i - G.gx) & G.xc) == 0)) {
            const T dS = (T)(G.yf[j] - G.yf[j - 1]), dN = (T)(G.yf[j + 1] - G.yf[j]);
            const T dyc = T(1) / (dS + dN);
            return (T(0.5) * dyc) * ((dS * Xv(k, i, j - 1) + (dN + dS) * Xv(k, i, j)) + dN * Xv(k, i, j + 1));
        }
        return Xv(k, i, j);
    };
    T v;
    if (G.zc && kf >= 1 && kf <= G.nzf - 1 && ((kf - 1) % 2 == 0)) {
        const T dU = (T)(G.zf[kf + 1] - G.zf[kf]), dD = (T)(G.zf[kf] - G.zf[kf - 1]);
        const T dzc = T(1) / (dD + dU);
        v = (T(0.5) * dzc) * (dD * Yv(kf - 1, ifn, jfn) + dU * Yv(kf + 1, ifn, jfn)) + T(0.5) * Yv(kf, ifn, jfn);
    } else v = Yv(kf, ifn, jfn);
    return v;
}
// Restricted residual at coarse point q < nxgc * nygc * nzgc.
template <typename T>
__device__ __forceinline__ T restrict_value(const RestrictGeo &G, size_t q, const T *__restrict__ rf) {
    const int kc = (int)(q % G.nzgc);
    const size_t col = q / G.nzgc;
    auto R = [&](int k, int i, int j) -> T { return rf[(size_t)(j * G.nxgf + i) * G.nzgf + k]; };
    return restrict_at<T>(G, kc, (int)(col % G.nxgc), (int)(col / G.nxgc), R);
}
template <typename T>
__global__ void k_mg_restrict(RestrictGeo G, const T *__restrict__ rf, T *__restrict__ rc, T *__restrict__ xz) {
    if (!G.spec && solve_done(G.skip)) return;
    const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (size_t)G.nxgc * G.nygc * G.nzgc) return;
    const T v = restrict_value(G, q, rf);
    if (G.spec && solve_done(G.skip)) return;
    if (xz) xz[q] = T(0);
    rc[q] = v;
}
// The same with one grid row of coarse columns per blockIdx.y and the coarse level count NZC known at
// compile time: the point decodes with no runtime division.
template <typename T, int NZC>
__global__ void k_mg_restrict_t(RestrictGeo G, const T *__restrict__ rf, T *__restrict__ rc, T *__restrict__ xz) {
    if (!G.spec && solve_done(G.skip)) return;
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= G.nxgc * NZC) return;
    const int ic = t / NZC, kc = t - ic * NZC, jc = (int)blockIdx.y;
    auto R = [&](int k, int i, int j) -> T { return rf[(size_t)(j * G.nxgf + i) * G.nzgf + k]; };
    const T v = restrict_at<T>(G, kc, ic, jc, R);
    if (G.spec && solve_done(G.skip)) return;
    const size_t q = (size_t)jc * G.nxgc * NZC + t;
    if (xz) xz[q] = T(0);
    rc[q] = v;
}

// Prolongation (MGProlongation3DExplicit.f90) of the coarse correction, added to x on interior
// columns below the free surface.
// Interpolated correction at fine point q < nxgf * nygf * nzgf; false where q takes none (ghost points,
// the sigma ghost level and the surface).  The coarse correction is read through E(kc, ic, jc).
// (The factors XF, YF, ZF are 1 or 2: x % F is x & (F - 1) and x / F is x >> (F - 1) on the
// non-negative offsets they are applied to.)
template <typename T, class EA>
__device__ __forceinline__ bool prolong_at(const RestrictGeo &G, int k, int i, int j, const EA &E, T &out) {
    if (k < 1 || k > G.nzf - 1 || i < G.gx || i > G.nxf + G.gx - 1 || j < G.gy || j > G.nyf + G.gy - 1) return false;
    const int XF = G.xc ? 2 : 1, YF = G.yc ? 2 : 1, ZF = G.zc ? 2 : 1;
    const int xs = G.xc ? 1 : 0, ys = G.yc ? 1 : 0, zs = G.zc ? 1 : 0;
    auto E0 = [&](int kk, int ii, int jj) -> T {
        if (kk < 1 || kk > G.nzf - 1 || ((kk - 1) & zs) != 0) return T(0);
        if (((ii - G.gx) & xs) != 0 || ((jj - G.gy) & ys) != 0) return T(0);
        const int kc = 1 + ((kk - 1) >> zs), ic = G.gx + ((ii - G.gx) >> xs), jc = G.gy + ((jj - G.gy) >> ys);
        if (kc > G.nzc - 1) return T(0);
        return E(kc, ic, jc);
    };
    auto EX = [&](int kk, int ii, int jj) -> T {
        if (XF == 2 && ((jj - G.gy) & ys) == 0 && ((ii - G.gx) % 2) == 1 && kk >= 1 && kk <= G.nzf - 1 && ((kk - 1) & zs) == 0) {
            const T dW = (T)(G.xf[ii] - G.xf[ii - 1]), dE = (T)(G.xf[ii + 1] - G.xf[ii]);
            const T dxf = T(1) / (dW + dE);
            return (dE * E0(kk, ii - 1, jj) + dW * E0(kk, ii + 1, jj)) * dxf;
        }
        return E0(kk, ii, jj);
    };
    auto EY = [&](int kk, int ii, int jj) -> T {
        if (kk > G.nzf - 1) return T(0);
        if (YF == 2 && ((jj - G.gy) % 2) == 1 && kk >= 1 && ((kk - 1) & zs) == 0) {
            const T dS = (T)(G.yf[jj] - G.yf[jj - 1]), dN = (T)(G.yf[jj + 1] - G.yf[jj]);
            const T dyf = T(1) / (dS + dN);
            return (dN * EX(kk, ii, jj - 1) + dS * EX(kk, ii, jj + 1)) * dyf;
        }
        return EX(kk, ii, jj);
    };
    T e;
    if (ZF == 2 && ((k - 1) % 2) == 1) {
        const T dD = (T)(G.zf[k] - G.zf[k - 1]), dU = (T)(G.zf[k + 1] - G.zf[k]);
        const T dzf = T(1) / (dD + dU);
        e = (dU * EY(k - 1, i, j) + dD * EY(k + 1, i, j)) * dzf;
    } else e = EY(k, i, j);
    out = e;
    return true;
}
template <typename T>
__device__ __forceinline__ bool prolong_value(const RestrictGeo &G, size_t q, const T *__restrict__ ec, T &out) {
    const int k = (int)(q % G.nzgf);
    const size_t col = q / G.nzgf;
    auto E = [&](int kc, int ic, int jc) -> T { return ec[(size_t)(jc * G.nxgc + ic) * G.nzgc + kc]; };
    return prolong_at<T>(G, k, (int)(col % G.nxgf), (int)(col / G.nxgf), E, out);
}
template <typename T>
__global__ void k_mg_prolong_add(RestrictGeo G, const T *__restrict__ ec, T *__restrict__ xf) {
    if (!G.spec && solve_done(G.skip)) return;
    const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (size_t)G.nxgf * G.nygf * G.nzgf) return;
    T e;
    if (!prolong_value(G, q, ec, e)) return;
    const T x0 = xf[q];
    if (G.spec && solve_done(G.skip)) return;
    xf[q] = x0 + e;
}
// The same with one grid row of fine columns per blockIdx.y and the fine level count NZF known at
// compile time.
template <typename T, int NZF>
__global__ void k_mg_prolong_add_t(RestrictGeo G, const T *__restrict__ ec, T *__restrict__ xf) {
    if (!G.spec && solve_done(G.skip)) return;
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= G.nxgf * NZF) return;
    const int i = t / NZF, k = t - i * NZF, j = (int)blockIdx.y;
    T e;
    auto E = [&](int kc, int ic, int jc) -> T { return ec[(size_t)(jc * G.nxgc + ic) * G.nzgc + kc]; };
    if (!prolong_at<T>(G, k, i, j, E, e)) return;
    const size_t q = (size_t)j * G.nxgf * NZF + t;
    const T x0 = xf[q];
    if (G.spec && solve_done(G.skip)) return;
    xf[q] = x0 + e;
}

// Residual of a column from its rows (residual_column's arithmetic, its roundings written out): c its level 0 in
// LDS, x- and y-neighbours at +- SXS and +- SYS; i, j the column (wall columns take the rows of the
// column beside them).
template <typename T, int NZ, bool D3, int SXS>
__device__ __forceinline__ void residual_rows(const LvArgs<T> &L, int i, int j, const LineRows<T, D3> &R, const T (&cp)[6], const T *c, int SYS,
                                              const T (&b)[NZ], T (&o)[NZ]) {
#pragma clang fp contract(off)
    auto dot3 = [](const T (&S)[3], T a, T m, T z) -> T {
#pragma clang fp contract(off)
        return fma1(S[2], z, fma1(S[0], a, S[1] * m));
    };
    const int nxg = L.nxg, nyg = L.nyg;
    const bool wx = i == 0 || i == nxg - 1, wy = D3 && (j == 0 || j == nyg - 1);
    if (wx || wy) {
        // identity at corners and on the sigma ghost level, else the Neumann row of the column beside the wall
        const int st = wx ? SXS : SYS, c0 = wx ? (i == 0 ? 0 : -2) : (j == 0 ? 0 : -2);
        T S[3];
#pragma unroll
        for (int m = 0; m < 3; m++) {
            if constexpr (D3) S[m] = pick(wx, R.X1[m], R.Y1[m]);
            else S[m] = R.X1[m];
        }
#pragma unroll
        for (int k = 0; k < NZ; k++) {
            const T *q = c + c0 * st + k;
            o[k] = (wx && wy) || k == 0 ? b[k] - c[k] : b[k] - dot3(S, q[0], q[st], q[2 * st]);
        }
        return;
    }
    T xc[NZ], dxl[NZ], dyl[NZ], xx[NZ];
#pragma unroll
    for (int k = 0; k < NZ; k++) {
        const T xm = c[k - SXS], xp = c[k + SXS];
        xc[k] = c[k];
        dxl[k] = dot3(R.X1, xm, xc[k], xp);
        dyl[k] = T(0);
        if (k > 0 && k < NZ - 1) xx[k] = dot3(R.X2, xm, xc[k], xp);
        if constexpr (D3) {
            const T ym = c[k - SYS], yp = c[k + SYS];
            dyl[k] = dot3(R.Y1, ym, xc[k], yp);
            if (k > 0 && k < NZ - 1) xx[k] = xx[k] + dot3(R.Y2, ym, xc[k], yp);
        }
    }
    // beside a wall the first derivative on the sigma ghost level takes the window shifted one column inwards
    if (i == 1 || i == nxg - 2) {
        const T *q = c + (i == 1 ? 0 : -2) * SXS;
        dxl[0] = dot3(R.XW, q[0], q[SXS], q[2 * SXS]);
    }
    if constexpr (D3) {
        if (j == 1 || j == nyg - 2) {
            const T *q = c + (j == 1 ? 0 : -2) * SYS;
            dyl[0] = dot3(R.YW, q[0], q[SYS], q[2 * SYS]);
        }
    }
    o[NZ - 1] = b[NZ - 1] - xc[NZ - 1];
#pragma unroll
    for (int k = 1; k < NZ - 1; k++) {
        const T *Z = L.sz + k * 6;
        const T Z1[3] = {Z[0], Z[1], Z[2]}, Z2[3] = {Z[3], Z[4], Z[5]};
        const T om = T(1) - L.zs[k];
        const T s2 = om * cp[3], s4 = om * cp[4], s3 = om * cp[5], s5 = cp[0];
        const T dz = dot3(Z1, xc[k - 1], xc[k], xc[k + 1]), dzz = dot3(Z2, xc[k - 1], xc[k], xc[k + 1]);
        const T dxz = dot3(Z1, dxl[k - 1], dxl[k], dxl[k + 1]), dyz = dot3(Z1, dyl[k - 1], dyl[k], dyl[k + 1]);
        const T mixed = fma1(s2, dxz, s4 * dyz), czz = fma1(s5, s5, fma1(s2, s2, s4 * s4));
        o[k] = b[k] - fma1(czz, dzz, fma1(T(2), mixed, fma1(s3, dz, xx[k])));
    }
    {
        const T *Z = L.sz + 6;
        const T Z1[3] = {Z[0], Z[1], Z[2]};
        const T om = T(1) - L.zs[1];
        const T s2 = om * cp[3], s4 = om * cp[4], s5 = cp[0], hx = cp[1], hy = D3 ? cp[2] : T(0);
        const T dz = dot3(Z1, xc[0], xc[1], xc[2]), cz = fma1(hy, s4, fma1(hx, s2, s5));
        // (read by the restriction onto a sigma-coarsened level only: there it must round as k_mg_residual_t does)
        o[0] = b[0] - fma1(hy, dyl[1], fma1(hx, dxl[1], cz * dz));
    }
}

// LDS elements of k_mg_residual_restrict: the x window, then the residual tile over it.
template <int NZ, int CX, int CY>
struct ResRestrictLds {
    static constexpr int FW = 2 * CX + 1, FH = 2 * CY + 1, WX = FW + 4, WY = FH + 4, NZP = NZ | 1;
    static constexpr int TOTAL = WX * WY * NZP;
};
// Residual of a level and its restriction onto a coarse level coarsened in x and y but not in sigma, in one
// launch (the arithmetic of k_mg_residual_t, then of restrict_at with the weights from tables).  A block owns CX x CY coarse
// columns (ghost columns included); it computes the fine residual on the (2 CX + 1) x (2 CY + 1) fine columns
// their restriction stencils reach, one thread per column (the fine column between two tiles is computed by
// both), keeps it in LDS over the staged x window and restricts from there, so the fine residual never goes
// to HBM.  Requires wall ghost layers in x and y (gx = gy = 1), as every level with restriction tables has.
// A thread's right-hand side, planes and stencil rows go straight to its registers: staging them in LDS by
// element took more instructions than the residual itself.  The barriers wait for LDS only, not for the loads in
// flight.  With 10 sigma levels, everything staged in LDS and then as here: FP32 at 513 x 513 columns 19.9 us
// before, 13.8 us after (bound by the instructions of the residual); at 257 x 257 10.2 and 7.4 us; on a level of
// one or two tiles 8.9 and 6.3 us (the chain load, residual, barrier, restriction, store).  FP64: 43.8 and
// 21.9 us, 17.9 and 10.0 us, 9.8 and 7.5 us.
template <typename T, int NZ, int CX, int CY, int NT>
__global__ __launch_bounds__(NT) void k_mg_residual_restrict(LvArgs<T> L, RestrictGeo G, const T *__restrict__ rxw, const T *__restrict__ ryw,
                                                             const T *__restrict__ x, const T *__restrict__ b, T *__restrict__ rc,
                                                             T *__restrict__ xz) {
#pragma clang fp contract(off)
    if (!L.spec && solve_done(L.skip)) return;
    using S = ResRestrictLds<NZ, CX, CY>;
    constexpr int FW = S::FW, FH = S::FH, WX = S::WX, WY = S::WY, NZP = S::NZP, R = 2, RES = (CY * CX * NZ + NT - 1) / NT;
    static_assert(FW * FH <= NT, "one thread per fine column of the tile");
    __shared__ T sX[S::TOTAL];
    const int nxg = L.nxg, nyg = L.nyg, t = (int)threadIdx.x;
    // XCD-aware tile order (xcd_tile over the row-major tile index): each XCD takes one contiguous band of
    // tile rows, so the halos neighbouring tiles share are re-read from that XCD's L2 (at 513^2: HBM fetch
    // 57 -> 29 MB, 22.2 -> 20.0 us)
    const int tb = xcd_tile((int)(blockIdx.y * gridDim.x + blockIdx.x), (int)(gridDim.x * gridDim.y));
    const int ic0 = (tb % (int)gridDim.x) * CX, jc0 = (tb / (int)gridDim.x) * CY;
    // fine column of coarse column ic is 2 ic - 1; the tile's stencils reach fine columns fi0 .. fi0 + FW - 1
    const int fi0 = 2 * ic0 - 2, fj0 = 2 * jc0 - 2;
    const int lox = cmax(cmin(fi0 - R, nxg - 4), 0), loy = cmax(cmin(fj0 - R, nyg - 4), 0);
    const int wcols = cmin(WX, nxg - lox), wrows = cmin(WY, nyg - loy);
    const int tx = t % FW, ty = t / FW;
    const int i = fi0 + tx, j = fj0 + ty;
    const bool active = t < FW * FH && i >= 0 && i < nxg && j >= 0 && j < nyg;
    // every HBM load of the block is in flight before the first wait
    RowWindow<T, NZ, WY, WX, NT, (WX * NZ / 2 <= NT / 2) ? 2 : 1> xr;
    xr.load(x + ((size_t)loy * nxg + lox) * NZ, (size_t)nxg * NZ, wrows, wcols);
    T bc[NZ], cp[6];
    LineRows<T, true> rows;
    {
        const int ii = active ? i : 0, jj = active ? j : 0;   // (idle threads load a valid column)
        const size_t p = (size_t)jj * nxg + ii;
        load_column<NZ>(b + p * NZ, bc);
#pragma unroll
        for (int q = 0; q < 6; q++) cp[q] = L.col[(size_t)q * L.nxy + p];
        rows.load(L, cclamp(ii, 1, nxg - 2), cclamp(jj, 1, nyg - 2));
    }
    // the thread's coarse points (CX * NZ contiguous values per coarse row) and their weights
    struct Point { int cc, rr, k; T x[4], y[4]; } pt[RES];
#pragma unroll
    for (int q = 0; q < RES; q++) {
        const int e = t + q * NT, c = e % (CX * NZ);
        pt[q].rr = e / (CX * NZ); pt[q].cc = c / NZ; pt[q].k = c - pt[q].cc * NZ;
        const int ic = cmin(ic0 + pt[q].cc, G.nxgc - 1), jc = cmin(jc0 + pt[q].rr, G.nygc - 1);
#pragma unroll
        for (int m = 0; m < 4; m++) { pt[q].x[m] = rxw[4 * ic + m]; pt[q].y[m] = ryw[4 * jc + m]; }
    }
    if (L.spec && solve_done(L.skip)) return;
    xr.template store<NZP, WX>(sX, wrows, wcols);
    lds_barrier();
    T o[NZ];
    if (active) residual_rows<T, NZ, true, NZP>(L, i, j, rows, cp, sX + ((j - loy) * WX + (i - lox)) * NZP, WX * NZP, bc, o);
    lds_barrier();
    if (active) {
        T *dst = sX + (ty * FW + tx) * NZP;
#pragma unroll
        for (int k = 0; k < NZ; k++) dst[k] = o[k];
    }
    lds_barrier();
    // restriction: smoothed along x on the coarse point's row and its two neighbour rows (injected on wall ghost rows),
    // then along y; injected on the top level; zero on coarse ghost points
#pragma unroll
    for (int q = 0; q < RES; q++) {
        const Point &p = pt[q];
        const int ic = ic0 + p.cc, jc = jc0 + p.rr;
        if (t + q * NT >= CY * CX * NZ || ic >= G.nxgc || jc >= G.nygc) continue;
        T v = T(0);
        if (p.k >= 1 && ic >= 1 && ic <= G.nxc && jc >= 1 && jc <= G.nyc) {
            const int ti = 2 * p.cc + 1, tj = 2 * p.rr + 1;   // tile position of fine column (2 ic - 1, 2 jc - 1)
            auto Rt = [&](int a, int bb) -> T { return sX[(bb * FW + a) * NZP + p.k]; };
            if (p.k <= G.nzf - 1) {
                const int jf = 2 * jc - 1;
                auto Xv = [&](int dj) -> T {
#pragma clang fp contract(off)
                    const int jj = jf + dj;
                    const T r1 = Rt(ti, tj + dj);
                    const T s = p.x[3] * fma1(p.x[2], Rt(ti + 1, tj + dj), fma1(p.x[0], Rt(ti - 1, tj + dj), p.x[1] * r1));
                    return jj < 1 || jj > G.nyf ? r1 : s;
                };
                v = p.y[3] * fma1(p.y[2], Xv(1), fma1(p.y[0], Xv(-1), p.y[1] * Xv(0)));
            } else {
                v = Rt(ti, tj);
            }
        }
        const size_t d = ((size_t)jc * G.nxgc + ic) * NZ + p.k;
        if (xz) xz[d] = T(0);
        rc[d] = v;
    }
}

// The same prolongation for a coarse level coarsened in x and y but not in sigma (kc = k), from per-column
// and per-row tables (left and right coarse index, weights left, right and 1 / sum, as prolong_at forms
// them): e = (wyl (wxl a + wxr b) sx + wyr (wxl c + wxr d) sx) sy over the (up to) four coarse neighbours,
// which is prolong_at's value with weights (1, 0, 1) on the coarse lines.  No branch on the point's parity.
template <typename T, int NZF>
__global__ void k_mg_prolong_tab(RestrictGeo G, const int2 *__restrict__ pxi, const T *__restrict__ pxw, const int2 *__restrict__ pyi,
                                 const T *__restrict__ pyw, const T *__restrict__ ec, T *__restrict__ xf) {
    if (!G.spec && solve_done(G.skip)) return;
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= G.nxgf * NZF) return;
    const int i = t / NZF, k = t - i * NZF, j = (int)blockIdx.y;
    const int2 yi = pyi[j], xi = pxi[i];
    if (yi.x < 0 || xi.x < 0 || k < 1 || k > G.nzf - 1) return;
    const T wxl = pxw[3 * i], wxr = pxw[3 * i + 1], sx = pxw[3 * i + 2];
    const T wyl = pyw[3 * j], wyr = pyw[3 * j + 1], sy = pyw[3 * j + 2];
    const size_t rl = (size_t)yi.x * G.nxgc, rr = (size_t)yi.y * G.nxgc;
    const T a = ec[(rl + xi.x) * NZF + k], b = ec[(rl + xi.y) * NZF + k];
    const T c = ec[(rr + xi.x) * NZF + k], d = ec[(rr + xi.y) * NZF + k];
    const T el = (wxl * a + wxr * b) * sx, er = (wxl * c + wxr * d) * sx;
    const T e = (wyl * el + wyr * er) * sy;
    const size_t q = (size_t)j * G.nxgf * NZF + t;
    const T x0 = xf[q];
    if (G.spec && solve_done(G.skip)) return;
    xf[q] = x0 + e;
}

// Row r's partial sums of x = Minv b for one wave: every lane's products of 16-byte chunks of the row and the matching
// values of b, in order (k_mg_coarse, and the dense solve of k_mg_bottom).
template <typename T, typename M>
__device__ __forceinline__ T coarse_chunk(const M *__restrict__ row, const T *b, int c0) {
    constexpr int V = 16 / (int)sizeof(M);
    const uint4 q = *reinterpret_cast<const uint4 *>(row + c0);
    M m[V];
    __builtin_memcpy(m, &q, 16);
    T bv[V];
    __builtin_memcpy(bv, __builtin_assume_aligned(b + c0, 16), V * sizeof(T));
    T p = T(0);
#pragma unroll
    for (int v = 0; v < V; v++) p += (T)m[v] * bv[v];
    return p;
}
// Coarsest level: x = Minv b with the dense inverse computed at set-up, stored as M (T, or FP16 with
// sums in T) in rows of `pitch` elements (a multiple of 8; zeros past n); b holds pitch elements (zeros
// past n).  One 64-lane wave per row: each lane reads 16 bytes of the row and the matching b values per
// step (vector loads), sums those products in order, and the lanes' sums are reduced in a fixed order.
template <typename T, typename M>
__global__ __launch_bounds__(256) void k_mg_coarse(int n, int pitch, const M *__restrict__ Minv, const T *__restrict__ b,
                                                   T *__restrict__ x, const int *skip) {
    if (solve_done(skip)) return;
    constexpr int V = 16 / (int)sizeof(M);
    const int lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= n) return;
    const M *row = Minv + (size_t)r * pitch;
    T s = T(0);
#pragma unroll 4
    for (int c0 = lane * V; c0 < n; c0 += 64 * V) s += coarse_chunk<T, M>(row, b, c0);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if (lane == 0) x[r] = s;
}

// The V cycle on the small levels in one workgroup: levels 0 .. top of the hierarchy (0 = coarsest, solved densely), whose
// finest member's right-hand side arrives in HBM and whose iterate starts from zero.  Same steps as the launches it
// replaces (per level: sweeps with their ghost passes, residual, restriction; dense solve; prolongation, sweeps).
// Each of those launches is a chain of latencies with a few hundred columns of work: its start, its loads, its stores
// and the drain before the next one take 5-10 us for 1-2 us of arithmetic.  Here the level vectors stay in LDS from the
// first restriction to the last prolongation and a step ends with an LDS barrier.  What bounds it is the instruction
// chain of a step on at most four waves per SIMD-quad, so columns keep everything in registers, stores come after all
// loads of a step, and the tables of a level (stencil rows, transfer weights) are copied to LDS once.
// One thread per column of a colour in a sweep, 256 threads: a wave per SIMD, so that a thread can hold the records
// of its red and its black column at once (up to 350 registers in FP64).  The records of these levels are stored by
// 16-byte chunk (LvArgs::facq): one compute unit serves a line per cycle and about one load instruction per 16, and
// the 64 lanes of a wave read 64 lines with a column's contiguous record per lane (4000-5500 cycles a step), 37
// instructions with a value per lane (4000-6500), 16 lines and a fourth or half of the instructions with a chunk.
constexpr int MG_BOTTOM_MAX = 10, MG_BOTTOM_NT = 256;
// A level handed to the kernel has at most one column of a colour per thread: columns away from the walls, and (in waves
// of their own, two lanes per column) those beside a wall.
__host__ __device__ inline int bottom_inner(int nxg, int nyg, bool d3) {   // columns of a colour, two or more from every wall
    return (nxg > 4 && (!d3 || nyg > 4)) ? (nxg - 3) / 2 * (d3 ? nyg - 4 : 1) : 0;
}
__host__ __device__ inline int bottom_edge(int nxg, int nyg, bool d3) { return d3 ? 2 * ((nxg - 1) / 2) + 2 * ((nyg - 1) / 2) : 2; }
__host__ __device__ inline int bottom_ghosts(int nxg, int nyg, bool d3) { return d3 ? 2 * nxg + 2 * (nyg - 2) : 2; }
inline bool bottom_fits(int nxg, int nyg, bool d3) {
    return (bottom_inner(nxg, nyg, d3) + 63) / 64 * 64 + (bottom_edge(nxg, nyg, d3) + 31) / 32 * 64 <= MG_BOTTOM_NT &&
           bottom_ghosts(nxg, nyg, d3) <= MG_BOTTOM_NT / 2 && nxg * nyg <= 2 * MG_BOTTOM_NT;
}
template <typename T>
struct BottomLevel {
    LvArgs<T> L;
    int xc, yc, zc, tab;                  // coarsening of the next coarser level; its transfers have weight tables (MgLevel::ptab)
    int nxgc, nygc, nzgc, pad;
    int x, b;                             // LDS offsets (elements) of iterate and right-hand side
    // offsets in the tables: stencil rows; restriction weights per coarse column and row (d_lo, d_lo + d_hi, d_hi,
    // 1 / (2 (d_lo + d_hi))) and level (d_lo, d_hi, 1 / (2 (d_lo + d_hi))); prolongation weights per fine column, row and
    // level (left, right, 1 / sum)
    int sx, sy, rx, ry, rz, px, py, pz;
};
template <typename T>
struct BottomArgs {
    int nlev, nu1, nu2, n0, pitch0, half0;   // pitch0: row pitch (elements) of minv; half0: it is FP16
    int r, tab, ntab, image;                 // LDS offsets of the residual and of the tables; elements of tables and of all x and b
    const void *minv;
    const T *tables;
    T *b, *x;                                // right-hand side of level nlev - 1; its result
    T *b0, *x0;                              // the same of level 0, and
    T *img;                                  // the LDS image, where the dense solve is a launch of its own
    BottomLevel<T> lev[MG_BOTTOM_MAX];
};
// Read-only device data behind a pointer that was itself loaded from memory: as constant address space, so that
// uniform reads are scalar loads and the others global (not flat) ones.
template <typename P>
__device__ __forceinline__ const P *ro(const P *p) {
    return (const P *)(const __attribute__((address_space(4))) P *)(unsigned long long)p;
}

template <typename T, int NZ, bool D3>
struct BottomStep {
    using Rec = LineRecord<T, NZ>;
    static constexpr int NZP = NZ | 1, NT = MG_BOTTOM_NT, NZH = (NZ - 2) / 2 + 2;   // NZH: depth of a sigma-coarsened level
    // The steps other than the sweeps' halves take two threads per column, NT / 2 apart: f(0) the levels below HALF, f(1)
    // the others (each thread's chain is half as long, and which half it is is known per wave).
    static constexpr int HALF = NZ / 2, NC = NT / 2;
    template <class F>
    __device__ __forceinline__ static void halves(const F &f) {
        if ((int)threadIdx.x < NC) f(std::integral_constant<int, 0>{});
        else f(std::integral_constant<int, 1>{});
    }
    struct Column {
        int i, j;
        bool on;
        T rec[Rec::N];
    };
    LvArgs<T> L;
    const T *tab;                // the tables in LDS
    T *X, *B;
    Column cur, nxt;             // the thread's red and black column
    T cp[6];                     // planes of the thread's next column in the residual
    bool edge, upper;
    int gi, gj;                  // the thread's wall ghost column (gi < 0: none)

    // Step l of the cycle: what does not depend on the step before is loaded here.
    __device__ __forceinline__ void load(const BottomLevel<T> &V, T *lds, const T *ltab, bool down) {
        L = V.L;
        L.sx = ltab + V.sx; L.sy = ltab + V.sy;
        L.sz = ro(L.sz); L.zs = ro(L.zs); L.col = ro(L.col); L.fac = ro(L.fac);
        tab = ltab;
        X = lds + V.x; B = lds + V.b;
        const int nxg = L.nxg, nyg = L.nyg, th = (int)threadIdx.x;
        const int nip = (bottom_inner(nxg, nyg, D3) + 63) / 64 * 64;
        edge = th >= nip;
        upper = edge && ((th - nip) & 32);
        column(cur, 0); column(nxt, 1);
        const int tc = th & (NC - 1);
        if (down) planes(cmin(tc, L.nxy - 1));
        gi = -1; gj = 0;
        if (tc < bottom_ghosts(nxg, nyg, D3)) {
            if (!D3) gi = tc == 0 ? 0 : nxg - 1;
            else if (tc < nxg) gi = tc;
            else if (tc < 2 * nxg) { gi = tc - nxg; gj = nyg - 1; }
            else if (tc < 2 * nxg + nyg - 2) { gi = 0; gj = 1 + tc - 2 * nxg; }
            else { gi = nxg - 1; gj = 1 + tc - 2 * nxg - (nyg - 2); }
        }
    }
    __device__ __forceinline__ void column(Column &C, int c) {   // of colour c
        const int nxg = L.nxg, nyg = L.nyg, th = (int)threadIdx.x;
        const int ni = bottom_inner(nxg, nyg, D3), nip = (ni + 63) / 64 * 64, hw = cmax((nxg - 3) / 2, 1);
        if (!edge) {
            const int r = D3 ? th / hw : 0, t = th - r * hw;
            C.j = D3 ? 2 + r : 0;
            C.i = 2 + ((C.j & 1) != c ? 1 : 0) + 2 * t;
            C.on = th < ni && C.i <= nxg - 3;
        } else {   // south row, north row, then west and east column
            const int l = ((th - nip) >> 6) * 32 + ((th - nip) & 31), bx = D3 ? (nxg - 1) / 2 : 0, by = D3 ? (nyg - 1) / 2 : 1;
            if (D3 && l < 2 * bx) {
                const bool first = l < bx;
                C.j = first ? 1 : nyg - 2;
                C.i = 1 + (((1 + C.j) & 1) != c ? 1 : 0) + 2 * (first ? l : l - bx);
                C.on = C.i <= nxg - 2 && (first || nyg > 3);
            } else {
                const int q = l - 2 * bx;
                const bool first = q < by;
                C.i = first ? 1 : nxg - 2;
                C.j = (D3 ? 1 : 0) + (((C.i + (D3 ? 1 : 0)) & 1) != c ? 1 : 0) + 2 * (first ? q : q - by);
                C.on = q < 2 * by && C.j <= (D3 ? nyg - 2 : 0) && (first || nxg > 3) && !(D3 && (C.j == 1 || C.j == nyg - 2));
            }
        }
        const int i = C.on ? C.i : 1, j = C.on ? C.j : (D3 ? 1 : 0);   // (idle lanes load a valid column)
        const int r = (int)Rec::index(nxg, nyg, i, j);
#pragma unroll
        for (int q = 0; q < Rec::N / Rec::W; q++) {
            T v[Rec::W];
            load_record(L.fac + (q * L.facq + r) * Rec::W, v);
#pragma unroll
            for (int m = 0; m < Rec::W; m++) C.rec[q * Rec::W + m] = v[m];
        }
    }
    __device__ __forceinline__ void planes(int c) {
#pragma unroll
        for (int q = 0; q < 6; q++) cp[q] = L.col[q * L.nxy + c];
    }
    __device__ __forceinline__ T *at(T *v, int i, int j) const { return v + (j * L.nxg + i) * NZP; }
    __device__ __forceinline__ void ghost_pass(bool zero) {   // k_mg_sweep's
        if (gi < 0) return;
        T *d = at(X, gi, gj);
        const T *gp = at(B, gi, gj);
        const int nxg = L.nxg, nyg = L.nyg;
        const bool gx = gi == 0 || gi == nxg - 1, gy = D3 && (gj == 0 || gj == nyg - 1);
        const bool low = gx ? gi == 0 : gj == 0;
        const T *S = gx ? L.sx + (low ? 1 : nxg - 2) * 6 : L.sy + (low ? 1 : nyg - 2) * 6;
        const T *xa = gx ? at(X, low ? 1 : nxg - 3, gj) : at(X, gi, low ? 1 : nyg - 3);
        const T *xb = gx ? at(X, low ? 2 : nxg - 2, gj) : at(X, gi, low ? 2 : nyg - 2);
        halves([&](auto h) {
#pragma clang fp contract(off)
            constexpr int K0 = h.value ? HALF : 0, K1 = h.value ? NZ : HALF;
            T v[NZ];
#pragma unroll
            for (int k = K0; k < K1; k++) v[k] = zero ? T(0) : gp[k];
            if (!zero && !(gx && gy)) {
                const T w0 = S[0], w1 = S[1], w2 = S[2];
                const T dg = low ? w0 : w2, wa = low ? w1 : w0, wb = low ? w2 : w1;
                T a[NZ], b[NZ];
#pragma unroll
                for (int k = cmax(K0, 1); k < K1; k++) { a[k] = xa[k]; b[k] = xb[k]; }
#pragma unroll
                for (int k = cmax(K0, 1); k < K1; k++) {
                    const T sum = fma1(wb, b[k], wa * a[k]);
                    v[k] = (v[k] - sum) / dg;
                }
            }
#pragma unroll
            for (int k = K0; k < K1; k++) d[k] = v[k];
        });
    }
    __device__ __forceinline__ void half(const Column &C, bool zero) {   // zero: all neighbours are
        if (!C.on) return;
        T *d = at(X, C.i, C.j);
        const T *bp = at(B, C.i, C.j);
        T f[NZ], up[NZ], inv[NZ], rh[NZ], x[NZ], bw[4], b[NZ];
        const T c3 = C.rec[Rec::C3], c4 = C.rec[Rec::C4];
#pragma unroll
        for (int k = 0; k < NZ; k++) b[k] = bp[k];
#pragma unroll
        for (int q = 0; q < 4; q++) bw[q] = C.rec[Rec::BW + q];
#pragma unroll
        for (int k = 0; k < NZ - 1; k++) { f[k] = C.rec[k]; up[k] = C.rec[NZ - 1 + k]; inv[k] = C.rec[2 * NZ - 2 + k]; }
        if (zero) {
#pragma unroll
            for (int k = 0; k < NZ; k++) rh[k] = b[k];
        } else if (!edge && L.uni) {
            line_rhs_uniform<T, NZ, D3, NZP>(L, c3, c4, bw, d, L.nxg * NZP, b, rh);
        } else {
            LineRows<T, D3> R;
            R.load(L, C.i, C.j);
            if (edge) line_rhs_pair<T, NZ, D3, NZP>(L, C.i, C.j, upper, R, c3, c4, bw, d, L.nxg * NZP, b, rh);
            else line_rhs_general<T, NZ, D3, NZP>(L, C.i, C.j, R, c3, c4, bw, d, L.nxg * NZP, b, rh);
        }
        line_solve<T, NZ>(f, up, inv, rh, x);
        if (!upper) {
#pragma unroll
            for (int k = 0; k < NZ; k++) d[k] = x[k];
        }
    }
    // nu sweeps, from zero before a descent; a ghost pass before each, and after the last one of a descent
    __device__ __forceinline__ void smooth(int nu, bool down) {
#pragma unroll 1
        for (int it = 0; it < nu + (down ? 1 : 0); it++) {
            const bool zero = down && it == 0;
            ghost_pass(zero);
            lds_barrier();
            if (it == nu) break;
            if (it > 0) { column(cur, 0); column(nxt, 1); }
#pragma unroll 1
            for (int c = 0; c < 2; c++) {   // (one copy of the code: see k_mg_bottom)
                half(cur, zero && c == 0);
                lds_barrier();
                cur = nxt;
            }
        }
    }
    // residual into r, restricted onto the coarse right-hand side (cb, column stride cs)
    __device__ __forceinline__ void descend(const BottomLevel<T> &V, T *r, T *cb, int cs) {
        const int nxg = L.nxg, nyg = L.nyg, th = (int)threadIdx.x;
        halves([&](auto h) {
            constexpr int K0 = h.value ? HALF : 0, K1 = h.value ? NZ : HALF;
#pragma unroll 1
            for (int c = th & (NC - 1); c < L.nxy; c += NC) {
                const int j = D3 ? c / nxg : 0, i = c - j * nxg;
                T b[NZ], o[NZ], cc[6];
#pragma unroll
                for (int q = 0; q < 6; q++) cc[q] = cp[q];
                planes(cmin(c + NC, L.nxy - 1));
                LineRows<T, D3> R;
                R.load(L, cclamp(i, 1, nxg - 2), D3 ? cclamp(j, 1, nyg - 2) : 0);
#pragma unroll
                for (int k = 0; k < NZ; k++) b[k] = B[c * NZP + k];
                residual_rows<T, NZ, D3, NZP>(L, i, j, R, cc, X + c * NZP, nxg * NZP, b, o);   // (the other half's rows are dead code)
#pragma unroll
                for (int k = K0; k < K1; k++) r[c * NZP + k] = o[k];
            }
        });
        lds_barrier();
        if ((D3 ? V.xc && V.yc : V.xc) && !V.zc) restrict_columns(V, r, cb, cs);
        else restrict_points(V, r, cb, cs);
        lds_barrier();
    }
    // Coarse column c of the restriction (restrict_at's arithmetic).  FULL: x and, in 3D, y are coarsened.
    template <bool FULL>
    struct Coarse {
        const T *q;          // its residual column
        T wx[4], wy[4];
        int row, py, ny;     // fine row, row pitch, rows
        bool in, xc, yc;     // in: no wall ghost column (those are zero)
        __device__ __forceinline__ void set(const BottomStep &S, const BottomLevel<T> &V, const T *r, int c) {
            const int jc = D3 ? c / V.nxgc : 0, ic = c - jc * V.nxgc;
            xc = FULL || V.xc; yc = D3 && (FULL || V.yc);
            in = ic >= 1 && ic <= V.nxgc - 2 && (!D3 || (jc >= 1 && jc <= V.nygc - 2));
            const int fi = in ? (xc ? 2 * ic - 1 : ic) : 1;
            row = in ? (yc ? 2 * jc - 1 : jc) : (D3 ? 1 : 0);   // (ghost columns read a valid one)
            py = S.L.nxg * NZP; ny = S.L.nyg;
            q = r + row * py + fi * NZP;
#pragma unroll
            for (int m = 0; m < 4; m++) { wx[m] = S.tab[V.rx + 4 * ic + m]; wy[m] = D3 ? S.tab[V.ry + 4 * jc + m] : T(0); }
        }
        __device__ __forceinline__ T line(const T *p, int dj) const {
#pragma clang fp contract(off)
            p += dj * py;
            const T r1 = p[0];
            if (!FULL && !xc) return r1;
            const T s = wx[3] * fma1(wx[2], p[NZP], fma1(wx[0], p[-NZP], wx[1] * r1));
            return D3 && (row + dj < 1 || row + dj > ny - 2) ? r1 : s;
        }
        __device__ __forceinline__ T plane(int k) const {   // smoothed in the plane of fine level k, 1 .. NZ - 2
#pragma clang fp contract(off)
            if (!D3 || (!FULL && !yc)) return line(q + k, 0);
            return wy[3] * fma1(wy[2], line(q + k, 1), fma1(wy[0], line(q + k, -1), wy[1] * line(q + k, 0)));
        }
    };
    // sigma not coarsened: two threads per coarse column
    __device__ __forceinline__ void restrict_columns(const BottomLevel<T> &V, const T *r, T *cb, int cs) {
        halves([&](auto h) {
            constexpr int K0 = h.value ? HALF : 0, K1 = h.value ? NZ : HALF;
#pragma unroll 1
            for (int c = (int)threadIdx.x & (NC - 1); c < V.nxgc * V.nygc; c += NC) {
                Coarse<true> P;
                P.set(*this, V, r, c);
                T y[NZ];
#pragma unroll
                for (int k = K0; k < K1; k++) y[k] = k == 0 ? T(0) : k == NZ - 1 ? P.q[k] : P.plane(k);
#pragma unroll
                for (int k = K0; k < K1; k++) cb[c * cs + k] = P.in ? y[k] : T(0);
            }
        });
    }
    // any coarsening: a thread per coarse point (the smallest levels)
    __device__ __forceinline__ void restrict_points(const BottomLevel<T> &V, const T *r, T *cb, int cs) {
#pragma clang fp contract(off)
        const int nzc = V.nzgc;
#pragma unroll 1
        for (int e = (int)threadIdx.x; e < V.nxgc * V.nygc * nzc; e += NT) {
            const int c = e / nzc, k = e - c * nzc;
            Coarse<false> P;
            P.set(*this, V, r, c);
            const int kf = V.zc ? 2 * k - 1 : k;
            T v = T(0);
            if (P.in && k > 0) {
                if (k == nzc - 1) v = P.q[NZ - 1];
                else {
                    v = P.plane(kf);
                    if (V.zc) {
                        const T *wz = tab + V.rz + 3 * k;
                        const T lo = kf == 1 ? P.q[0] : P.plane(kf - 1), hi = kf == NZ - 2 ? P.q[NZ - 1] : P.plane(kf + 1);
                        v = fma1(wz[2], fma1(wz[0], lo, wz[1] * hi), T(0.5) * v);
                    }
                }
            }
            cb[c * cs + k] = v;
        }
    }
    // Fine column c of the prolongation (prolong_at's and k_mg_prolong_tab's arithmetic), on the coarse correction ec.
    struct Fine {
        const T *ea, *eb, *el, *er;
        T wxl, wxr, sx, wyl, wyr, sy;
        bool in;
        __device__ __forceinline__ void set(const BottomStep &S, const BottomLevel<T> &V, const T *ec, int cs, int c) {
            const int nxg = S.L.nxg, j = D3 ? c / nxg : 0, i = c - j * nxg;
            in = i >= 1 && i <= nxg - 2 && (!D3 || (j >= 1 && j <= S.L.nyg - 2));
            const int xl = V.xc ? 1 + ((i - 1) >> 1) : i, xr = V.xc ? 1 + (i >> 1) : i;
            const int yl = !D3 ? 0 : V.yc ? 1 + ((j - 1) >> 1) : j, yr = !D3 ? 0 : V.yc ? 1 + (j >> 1) : j;
            wxl = S.tab[V.px + 3 * i]; wxr = S.tab[V.px + 3 * i + 1]; sx = S.tab[V.px + 3 * i + 2];
            if constexpr (D3) { wyl = S.tab[V.py + 3 * j]; wyr = S.tab[V.py + 3 * j + 1]; sy = S.tab[V.py + 3 * j + 2]; }
            ea = ec + (yl * V.nxgc + xl) * cs; eb = ec + (yl * V.nxgc + xr) * cs;
            el = ec + (yr * V.nxgc + xl) * cs; er = ec + (yr * V.nxgc + xr) * cs;
        }
        __device__ __forceinline__ T plane(int k) const {   // interpolated in the plane of coarse level k, without the last scale
#pragma clang fp contract(off)
            const T lo = fma1(wxl, ea[k], wxr * eb[k]);
            if constexpr (!D3) return lo;
            else {
                const T l1 = lo * sx, h1 = fma1(wxl, el[k], wxr * er[k]) * sx;
                return fma1(wyl, l1, wyr * h1);
            }
        }
        __device__ __forceinline__ T scale() const {
            if constexpr (D3) return sy;
            else return sx;
        }
    };
    // adds the prolongated coarse correction (ec, column stride cs)
    __device__ __forceinline__ void ascend(const BottomLevel<T> &V, const T *ec, int cs) {
        if (!V.zc) {   // two threads per column
            halves([&](auto h) {
#pragma clang fp contract(off)
                constexpr int K0 = h.value ? HALF : 1, K1 = h.value ? NZ - 1 : HALF;
#pragma unroll 1
                for (int c = (int)threadIdx.x & (NC - 1); c < L.nxy; c += NC) {
                    Fine P;
                    P.set(*this, V, ec, cs, c);
                    if (!P.in) continue;
                    T *d = X + c * NZP;
                    T x[NZ], m[NZ];
#pragma unroll
                    for (int k = K0; k < K1; k++) { x[k] = d[k]; m[k] = P.plane(k); }
#pragma unroll
                    for (int k = K0; k < K1; k++) d[k] = V.tab ? fma1(m[k], P.scale(), x[k]) : x[k] + m[k] * P.scale();
                }
            });
        } else {   // a thread per point (the smallest levels)
#pragma clang fp contract(off)
#pragma unroll 1
            for (int e = (int)threadIdx.x; e < L.nxy * (NZ - 2); e += NT) {
                const int c = e / (NZ - 2), k = 1 + e - c * (NZ - 2), kc = (k + 1) / 2;
                Fine P;
                P.set(*this, V, ec, cs, c);
                if (!P.in) continue;
                T *d = X + c * NZP + k;
                const T *wz = tab + V.pz + 3 * k;
                const bool odd = k % 2;   // on coarse level kc; else between kc and kc + 1 (none on the surface)
                const T lo = P.plane(kc) * P.scale();
                T hi = T(0);
                if (!odd && kc + 1 < NZH - 1) hi = P.plane(kc + 1) * P.scale();
                *d = *d + (odd ? lo : fma1(wz[0], lo, wz[1] * hi) * wz[2]);
            }
        }
        lds_barrier();
    }
};

// Runs `f` with the column depth nzg, one of NZ and its sigma coarsenings.
template <int NZ, class F>
__device__ __forceinline__ void bottom_depth(int nzg, const F &f) {
    if (nzg == NZ) f(std::integral_constant<int, NZ>{});
    else if constexpr (NZ % 2 == 0 && NZ >= 4) bottom_depth<(NZ - 2) / 2 + 2>(nzg, f);
}

// x = Minv b in one workgroup, k_mg_coarse's arithmetic: a wave takes RB rows at a time, and the reductions over its lanes
// pass half of the rows to the other half of the lanes at each of the first three steps (sums of the same pairs).
template <typename T, typename M>
__device__ __forceinline__ void bottom_dense(int n, int pitch, const M *__restrict__ minv, const T *b, T *x) {
    constexpr int V = 16 / (int)sizeof(M), RB = 8;
    const int lane = (int)threadIdx.x & 63;
    for (int r0 = ((int)threadIdx.x >> 6) * RB; r0 < n; r0 += MG_BOTTOM_NT / 64 * RB) {
        T s[RB];
#pragma unroll
        for (int q = 0; q < RB; q++) s[q] = T(0);
        for (int c0 = lane * V; c0 < n; c0 += 64 * V) {
#pragma unroll
            for (int q = 0; q < RB; q++) s[q] += coarse_chunk<T, M>(minv + cmin(r0 + q, n - 1) * pitch, b, c0);
        }
#pragma unroll
        for (int h = RB / 2, off = 32; h > 0; h >>= 1, off >>= 1) {
#pragma unroll
            for (int q = 0; q < h; q++) {
                const T keep = pick((lane & off) != 0, s[q + h], s[q]), give = pick((lane & off) != 0, s[q], s[q + h]);
                s[q] = keep + __shfl_xor(give, off, 64);
            }
        }
#pragma unroll
        for (int off = 4; off > 0; off >>= 1) s[0] += __shfl_xor(s[0], off, 64);
        const int r = r0 + ((lane & 32) ? 4 : 0) + ((lane & 16) ? 2 : 0) + ((lane & 8) ? 1 : 0);
        if ((lane & 7) == 0 && r < n) x[r] = s[0];
    }
}

// PART 0: the whole; 1: down to the right-hand side of level 0; 2: from its solution upwards.
// Size: at most 97 KB of code (FP64, 14 levels), less than the 128 KiB that a branch instruction reaches, in every
// instance; the loops over sweeps, colours and columns stay rolled for it.  A build with 235 KB (four unrolled copies of the
// residual), whose branches go through register-indirect jumps, gave wrong FP64 values with 10 sigma levels and right
// ones elsewhere.  Why is not known: the source was the same up to the unrolling, and the jumps are suspected only.
template <typename T, int NZ, bool D3>
__global__ __launch_bounds__(MG_BOTTOM_NT) void k_mg_bottom(const BottomArgs<T> *__restrict__ args, const int *skip, int part) {
    constexpr int NT = MG_BOTTOM_NT;
    extern __shared__ double bottom_lds[];
    T *lds = (T *)bottom_lds;
    const BottomArgs<T> *A = ro(args);
    const int top = A->nlev - 1, th = (int)threadIdx.x;
    const bool done = solve_done(skip);
    T *ltab = lds + A->tab;
    const T *tables = ro(A->tables);
    for (int e = th; e < A->ntab; e += NT) ltab[e] = tables[e];
    if (done) return;
    if (part == 2) {
        const T *img = ro((const T *)A->img), *x0 = ro((const T *)A->x0);
        for (int e = th; e < A->image; e += NT) lds[e] = img[e];
        lds_barrier();
        for (int e = th; e < A->n0; e += NT) lds[A->lev[0].x + e] = x0[e];
    } else {   // the right-hand side, and level 0's zeros up to the inverse's pitch
        const T *b = ro((const T *)A->b);
        T *B = lds + A->lev[top].b;
        for (int c = th; c < A->lev[top].L.nxy; c += NT) {
            T v[NZ];
            load_column<NZ>(b + c * NZ, v);
#pragma unroll
            for (int k = 0; k < NZ; k++) B[c * (NZ | 1) + k] = v[k];
        }
        for (int e = A->n0 + th; e < A->pitch0; e += NT) lds[A->lev[0].b + e] = T(0);
    }
    lds_barrier();
    // levels top .. 1 downwards, 0, and 1 .. top upwards
    const int last = part == 1 ? top - 1 : 2 * top;
    for (int st = part == 2 ? top + 1 : 0; st <= last; st++) {
        const bool down = st < top;
        const int l = down ? top - st : st - top;
        if (l == 0) {
            const T *b = lds + A->lev[0].b;
            T *x = lds + A->lev[0].x;
            if (sizeof(T) == 4 && A->half0) bottom_dense<T, __half>(A->n0, A->pitch0, ro((const __half *)A->minv), b, x);
            else bottom_dense<T, T>(A->n0, A->pitch0, ro((const T *)A->minv), b, x);
            lds_barrier();
            continue;
        }
        const BottomLevel<T> &V = A->lev[l], &C = A->lev[l - 1];
        const int cs = l == 1 ? C.L.nzg : (C.L.nzg | 1);   // level 0 is unpadded
        bottom_depth<NZ>(V.L.nzg, [&](auto depth) {
            BottomStep<T, decltype(depth)::value, D3> S;
            S.load(V, lds, ltab, down);
            if (!down) S.ascend(V, lds + C.x, cs);
            S.smooth(down ? A->nu1 : A->nu2, down);
            if (down) S.descend(V, lds + A->r, lds + C.b, cs);
        });
    }
    if (part == 1) {
        T *img = A->img, *b0 = A->b0;
        for (int e = th; e < A->image; e += NT) img[e] = lds[e];
        for (int e = th; e < A->n0; e += NT) b0[e] = lds[A->lev[0].b + e];
        return;
    }
    const T *X = lds + A->lev[top].x;
    T *out = A->x;
    for (int c = th; c < A->lev[top].L.nxy; c += NT) {
        T v[NZ];
#pragma unroll
        for (int k = 0; k < NZ; k++) v[k] = X[c * (NZ | 1) + k];
        store_column<NZ>(out + (size_t)c * NZ, v);
    }
}


}  // namespace ow3d
