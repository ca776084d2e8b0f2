// sem.hip -- SEM step kernels and the phc_sem_* C ABI.
//
// Reference hot path: SEMsolver::computeOneStep (src/sem/solver/SEMsolver.cpp:21-125)
//   K1 zero M, y                               SEMsolver.cpp:33-36
//   K2 source into pn(:,i2)                    SEMsolver.cpp:39-43
//   K3 per element: gather, computeB + gradPhiGradPhi, scatter M and y
//                                              SEMsolver.cpp:46-82, SEMQkGLIntegrals.hpp:206-565
//   K4 pn(:,i1) = 2 pn(:,i2) - pn(:,i1) - dt^2 y / M on interior nodes
//                                              SEMsolver.cpp:85-89
//
// Geometry and the lumped mass do not change between steps; they are built
// once in FP64 on the host (sem_setup.hpp) and the kernels read FP32 factors.
//
// Two step kernels:
//  * separable (default on the axis-aligned boxes SEMmesh builds): on such a
//    mesh the element Jacobians are diagonal, so the assembled stiffness is
//    Ax (x) Wz (x) Wy + Wx (x) Az (x) Wy + Wx (x) Wz (x) Ay with 1D assembled
//    operators A (banded, half width p) and lumped 1D masses W.  Dividing by
//    W = Wx Wy Wz turns the update into a radius-p star stencil whose
//    coefficients depend only on each index modulo p:
//        pnew = 2 p - pold - Q (Lx p + Ly p + Lz p),   Q = dt^2 W / M.
//    Each stencil row sums to zero, so it is evaluated on differences from
//    the centre node, which FP32 resolves far better than the plain sum.
//    It runs on the marching-tile scheme of the FD kernel: 16 B of HBM traffic
//    per node update (p, pold, Q read; pnew written).
//  * element: one thread per GLL point, the element's (p+1)^3 block and the
//    1D derivative matrix staged in LDS, sum-factorised gradient and
//    divergence contractions, atomic scatter of y into HBM, then a fused
//    leapfrog-update kernel that also clears y.  It takes per-point geometric
//    factors, so it serves general hexahedral geometry.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "fd_kernels.hpp"
#include "quad.hpp"
#include "march.hpp"
#include "xcd_sched.hpp"
#include "phc_common.hpp"
#include "readback.hpp"
#include "sem_setup.hpp"

namespace phc {

constexpr int SEM_MAX_P = 5;

struct SemSepArgs {
    const float *pn;   // level i2 (current)
    float *pnm1;       // level i1: read, overwritten by the new level
    const float *qf;   // dt^2 W / M per node (0 on boundary nodes)
    FdLayout L;        // i = iy, j = iz, k = ix; halo p (zeros)
    float cx[SEM_MAX_P][2 * SEM_MAX_P + 1];  // by ix mod p, offsets -p..p
    float cy[SEM_MAX_P][2 * SEM_MAX_P + 1];
    float cz[SEM_MAX_P][2 * SEM_MAX_P + 1];
    int64_t src_off;   // layout offset of the source node
    int inj;
    float inj_coef;    // dt^2 c^2 of the source element (SEMsolver.cpp:41-42)
    const float *rhs_next;  // in the run's sample window (device memory)
    float *trace;
    int tiles_k, tiles_j, chunk_i;
    // per-XCD schedule (null: one block per (tile, chunk of chunk_i planes)
    // in XCD block order): hardware block b marches tile column sched[b].x
    // over planes [sched[b].y, sched[b].z); an empty range does nothing
    const int4 *sched;
    // x-remainder slab: when the last 64-node x tile would hold at most 32
    // nodes, the tiles stop at x = krem and the blocks from nb_main on update
    // the interior nodes with x in [krem, nz - 1) one per thread
    int nb_main, krem;
    // receiver sampling of the level this launch reads as current (the
    // previous step's result) by rec_blocks extra blocks after the others,
    // one receiver per thread: rec_out[r * rec_stride + rec_step]; a receiver
    // on the source node takes rec_src[rec_step], recorded before injection
    const int64_t *rec_off;
    float *rec_out;
    const float *rec_src;
    int rec_n, rec_blocks, rec_stride, rec_step;
};

// out[r * stride + step] = level value of receiver r (the source node already
// holds the next sample's injection: its trace has the value before).
__device__ __forceinline__ void sem_sample_point(const float *p, const int64_t *offs, int r, float *out, int stride,
                                                 int step, int64_t src_off, const float *src_trace)
{
    const int64_t o = offs[r];
    out[(int64_t)r * stride + step] = (o == src_off) ? src_trace[step] : p[o];
}

// One node of the x-remainder slab per thread: the separable update with the
// same operations in the same order as the march (so a node gets the same
// bits from either path), its stencil values read from memory.
template <int P, typename IT>
__device__ __forceinline__ void sem_rem_points(const SemSepArgs &a, float rhs_next, int64_t t)
{
    constexpr int R = P, W = 2 * P + 1;
    constexpr IT S = sizeof(IT) == 4 ? 4 : 1;
    const FdLayout &L = a.L;
    const int nk = (L.nz - 1) - a.krem, nj = L.ny - 2;
    if (nk <= 0 || t >= (int64_t)nk * nj * (L.nx - 2)) return;
    const int k = a.krem + (int)(t % nk);
    const int64_t rest = t / nk;
    const int j = 1 + (int)(rest % nj);
    const int i = 1 + (int)(rest / nj);
    const IT si = (IT)L.pitch_j * S, sj = (IT)L.pitch_k * S;
    const IT o = (IT)fd_off(L, i, j, k) * S;
    const float pc = ldo(a.pn, o);
    const int my = i % P, mz = j % P, mx = k % P;
    float lap = 0.f;
#pragma unroll
    for (int d = 0; d < W; ++d) {
        if (d == R) continue;
        lap = fmaf(a.cy[my][d], ldo(a.pn, o + (d - R) * si) - pc, lap);
        lap = fmaf(a.cz[mz][d], ldo(a.pn, o + (d - R) * sj) - pc, lap);
        lap = fmaf(a.cx[mx][d], ldo(a.pn, o + (d - R) * S) - pc, lap);
    }
    float val = fmaf(-ldo(a.qf, o), lap, 2.f * pc - ldo(a.pnm1, o));
    if ((int64_t)(o / S) == a.src_off) {
        if (a.trace) *a.trace = val;
        if (a.inj) val = add_nc(val, mul_nc(a.inj_coef, rhs_next));
    }
    sto_nt(a.pnm1, o, val);
}

// Separable SEM step.  Same march as fd_step_kernel (register rings unrolled
// by 2P+2, halo FIFO, double-buffered LDS plane, LDS-only barrier); the
// stencil has per-position coefficients and a Dirichlet mask.
// Register budget: the one-row, 16-wave shapes of orders 1-4 fit in 64 VGPRs
// without spilling, i.e. 8 waves per SIMD instead of 6 (more loads in flight);
// the other shapes keep the budget their block size implies.
template <int P, int TY, int NJ, typename IT>
__global__ void __launch_bounds__(FD_TK *TY)
__attribute__((amdgpu_waves_per_eu((NJ == 1 && TY == 16 && P <= 4) ? 8 : (TY >= 4 ? TY / 4 : 1))))
sem_sep_kernel(SemSepArgs a)
{
    constexpr int R = P;
    constexpr int TJ = TY * NJ;
    constexpr int LW = FD_TK + 2 * R;
    constexpr int LH = TJ + 2 * R;
    constexpr int NH = (2 * R + TY - 1) / TY;
    constexpr int Q = 2 * R + 2;
    constexpr int F = R + 1;
    constexpr int W = 2 * R + 1;
    constexpr IT S = sizeof(IT) == 4 ? 4 : 1;
    __shared__ float tile[2][LH][LW];

    if ((int)blockIdx.x >= (int)gridDim.x - a.rec_blocks) {
        const int r = ((int)blockIdx.x - ((int)gridDim.x - a.rec_blocks)) * (FD_TK * TY) +
                      (int)(threadIdx.y * FD_TK + threadIdx.x);
        if (r < a.rec_n)
            sem_sample_point(a.pn, a.rec_off, r, a.rec_out, a.rec_stride, a.rec_step, a.src_off, a.rec_src);
        return;
    }
    const float rhs_next = uniform_value(a.rhs_next);
    if (a.nb_main && (int)blockIdx.x >= a.nb_main) {
        sem_rem_points<P, IT>(a, rhs_next, (int64_t)(blockIdx.x - a.nb_main) * (FD_TK * TY) +
                                     (int64_t)threadIdx.y * FD_TK + threadIdx.x);
        return;
    }
    const FdLayout &L = a.L;
    const int tx = threadIdx.x, ty = threadIdx.y;
    int w, i0, i1;
    if (a.sched) {
        const int4 e = a.sched[blockIdx.x];
        w = e.x;
        i0 = e.y;
        i1 = e.z;
        if (i0 >= i1) return;  // padding of a shorter XCD list (whole block)
    } else {
        const int b = xcd_block(blockIdx.x, a.nb_main ? a.nb_main : (int)gridDim.x - a.rec_blocks);
        const int ic = b / (a.tiles_k * a.tiles_j);
        w = b - ic * (a.tiles_k * a.tiles_j);
        i0 = ic * a.chunk_i;
        i1 = min(i0 + a.chunk_i, L.nx);
    }
    const int kt = w % a.tiles_k, jt = w / a.tiles_k;
    const int k0 = kt * FD_TK, j0 = 1 + jt * TJ;  // rows 0 and ny-1 are Dirichlet
    const int k = k0 + tx;
    const IT pitch = (IT)L.pitch_j * S;

    const bool kload = k < L.nz + R;
    const bool kin = k >= 1 && k < L.nz - 1;  // interior along x
    int jr[NJ];
    bool jcomp[NJ];
    IT colq[NJ];
    float czr[NJ][W];
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) {
        jr[jj] = j0 + ty * NJ + jj;
        const bool jl = kload && (jr[jj] < L.ny + R);
        jcomp[jj] = kin && jr[jj] >= 1 && jr[jj] < L.ny - 1;
        colq[jj] = (IT)fd_off(L, 0, jl ? jr[jj] : 0, jl ? k : 0) * S;
        const int mz = jr[jj] % P;
#pragma unroll
        for (int d = 0; d < W; ++d) czr[jj][d] = a.cz[mz][d];
    }
    float cxr[W];
    {
        const int mx = (k < L.nz ? k : 0) % P;
#pragma unroll
        for (int d = 0; d < W; ++d) cxr[d] = a.cx[mx][d];
    }
    const bool khalo = tx < 2 * R;
    const int kk = (tx < R) ? (k0 - R + tx) : (k0 + FD_TK + tx - R);
    const int kcol = kk - k0 + R;
    IT colk[NJ];
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) {
        const bool l = khalo && kk < L.nz + R && jr[jj] < L.ny + R;
        colk[jj] = (IT)fd_off(L, 0, l ? jr[jj] : 0, l ? kk : 0) * S;
    }
    int jhrow[NH];
    IT colh[NH];
#pragma unroll
    for (int m = 0; m < NH; ++m) {
        const int h = ty + TY * m;
        const int jh = (h < R) ? (j0 - R + h) : (j0 + TJ + h - R);
        jhrow[m] = jh - j0 + R;
        const bool l = (h < 2 * R) && (jh < L.ny + R) && kload;
        colh[m] = (IT)fd_off(L, 0, l ? jh : 0, l ? k : 0) * S;
    }

    float q[NJ][Q];
    float fk[NJ][F], fj[NH][F];
    float pm[2][NJ], qv[2][NJ];

    auto load_halo = [&](int slot, int p) {
        const IT po = (IT)p * pitch;
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) fk[jj][slot] = ldo(a.pn, colk[jj] + po);
#pragma unroll
        for (int m = 0; m < NH; ++m) fj[m][slot] = ldo(a.pn, colh[m] + po);
    };
    auto load_aux = [&](int set, int p) {
        const IT po = (IT)p * pitch;
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
            pm[set][jj] = ldo_nt(a.pnm1, colq[jj] + po);
            qv[set][jj] = ldo_nt(a.qf, colq[jj] + po);
        }
    };
    auto stage = [&](int buf, int qslot, int hslot) {
        float(*tl)[LW] = tile[buf];
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
            tl[ty * NJ + jj + R][tx + R] = q[jj][qslot];
            if (khalo) tl[ty * NJ + jj + R][kcol] = fk[jj][hslot];
        }
#pragma unroll
        for (int m = 0; m < NH; ++m)
            if (ty + TY * m < 2 * R) tl[jhrow[m]][tx + R] = fj[m][hslot];
    };

#pragma unroll
    for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
        for (int l = 0; l <= 2 * R; ++l) q[jj][l] = ldo(a.pn, colq[jj] + (IT)(i0 - R + l) * pitch);
#pragma unroll
    for (int d = 0; d <= R; ++d) load_halo(d, i0 + d);
    load_aux(0, i0);
    stage(0, R, 0);
    lds_barrier();

    // Unroll U planes per iteration.  U is a multiple of the ring length Q; at
    // order 4 it is lcm(Q, P) = 20 and chunks start at multiples of P, so the
    // coefficient row i % P of the march axis is a compile-time constant.
    constexpr int U = (P == 4) ? 20 : Q;
    for (int ib = i0; ib < i1; ib += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = ib + u;
            if (i >= i1) break;
            {
                const int pq = min(i + 1 + R, L.nx + R - 1);
                const IT po = (IT)pq * pitch;
#pragma unroll
                for (int jj = 0; jj < NJ; ++jj) q[jj][(u + 1 + 2 * R) % Q] = ldo(a.pn, colq[jj] + po);
                load_halo((u + 1 + R) % F, pq);
                load_aux((u + 1) & 1, min(i + 1, L.nx - 1));
            }
            const float(*tl)[LW] = tile[u & 1];
            const bool iin = i >= 1 && i < L.nx - 1;
            const int my = (P == 4) ? (u % P) : (i % P);
            const IT pi = (IT)i * pitch;
#pragma unroll
            for (int jj = 0; jj < NJ; ++jj) {
                if (!(jcomp[jj] && iin)) continue;
                const int r = ty * NJ + jj + R;
                const int c = tx + R;
                // rows sum to zero: sum over differences from the centre value
                // (the common part cancels exactly; FP32 keeps the differences)
                const float pc = q[jj][(u + R) % Q];
                float lap = 0.f;
#pragma unroll
                for (int d = 0; d < W; ++d) {
                    if (d == R) continue;
                    lap = fmaf(a.cy[my][d], q[jj][(u + d) % Q] - pc, lap);
                    lap = fmaf(czr[jj][d], tl[r - R + d][c] - pc, lap);
                    lap = fmaf(cxr[d], tl[r][c - R + d] - pc, lap);
                }
                float val = fmaf(-qv[u & 1][jj], lap, 2.f * pc - pm[u & 1][jj]);
                const IT o = colq[jj] + pi;
                if ((int64_t)(o / S) == a.src_off) {
                    if (a.trace) *a.trace = val;
                    if (a.inj) val = add_nc(val, mul_nc(a.inj_coef, rhs_next));
                }
                sto_nt(a.pnm1, o, val);
            }
            stage((u + 1) & 1, (u + 1 + R) % Q, (u + 1) % F);
            lds_barrier();
        }
    }
}

// The separable step with four nodes per lane, for the shapes with 4 rows per
// wavefront: the FD step's quad tile (fd_quad.hpp) with the separable
// operator's coefficients.  A lane holds 4 consecutive x nodes of one row; at
// orders 1, 2 and 4 a component's coefficient row along x is the same in
// every lane (its index mod p is the component's), at 3 and 5 it depends on
// the lane and is held in registers.  Every node takes the same operations in
// the same order as in sem_sep_kernel, so both give the same bits.
// Bound by the LDS reads and instructions of a node below the memory-side
// cache's size, by memory above it.  One node per lane (best shape) / four, us
// per step: 151^3 order 2 20.5 / 16.5, 151^3 order 3 22.5 / 16.7, 241^3 order
// 4 52.9 / 42.2, 186 x 111 x 146 order 5 21.8 / 19.0, 401^3 order 4 (774 MB,
// 16 B per node) 211 / 198.
template <int P>
struct SemQuadShape {
    static constexpr int HQ = (P + 3) / 4;               // halo quads per side of a row
    static constexpr int LQ = FD_TK / 4 + 2 * HQ;        // quads of an LDS row
    static constexpr int U = P == 4 ? 20 : 2 * P + 2;    // planes per turn (order 4: the march's row is u % 4)
};

template <int P, int TY, typename IT, bool NT>
__global__ void __launch_bounds__(FD_TK *TY) __attribute__((amdgpu_waves_per_eu(P == 5 ? 2 : 3)))
sem_quad_kernel(SemSepArgs a)
{
    constexpr int R = P, W = 2 * P + 1, TJ = 4 * TY, LH = TJ + 2 * R;
    constexpr int HQ = SemQuadShape<P>::HQ, LQ = SemQuadShape<P>::LQ;
    constexpr int T = FD_TK * TY;
    constexpr int NROW = 2 * R * (FD_TK / 4), NHQ = NROW + 2 * HQ * TJ;  // halo quads: rows, then row ends
    constexpr int NH = (NHQ + T - 1) / T;
    constexpr int Q = 2 * R + 2, F = R + 1, U = SemQuadShape<P>::U;
    constexpr IT S = sizeof(IT) == 4 ? 4 : 1;
    constexpr bool UNI = 4 % P == 0;  // a component's x row is the same in every lane
    __shared__ quad_f4 tile[2][LH][LQ];

    if ((int)blockIdx.x >= (int)gridDim.x - a.rec_blocks) {
        const int r = ((int)blockIdx.x - ((int)gridDim.x - a.rec_blocks)) * T +
                      (int)(threadIdx.y * FD_TK + threadIdx.x);
        if (r < a.rec_n)
            sem_sample_point(a.pn, a.rec_off, r, a.rec_out, a.rec_stride, a.rec_step, a.src_off, a.rec_src);
        return;
    }
    const float rhs_next = uniform_value(a.rhs_next);
    if (a.nb_main && (int)blockIdx.x >= a.nb_main) {
        sem_rem_points<P, IT>(a, rhs_next, (int64_t)(blockIdx.x - a.nb_main) * T +
                                               (int64_t)threadIdx.y * FD_TK + threadIdx.x);
        return;
    }
    const FdLayout &L = a.L;
    int w, i0, i1;
    if (a.sched) {
        const int4 e = a.sched[blockIdx.x];
        w = e.x;
        i0 = e.y;
        i1 = e.z;
        if (i0 >= i1) return;  // padding of a shorter XCD list (whole block)
    } else {
        const int b = xcd_block(blockIdx.x, a.nb_main ? a.nb_main : (int)gridDim.x - a.rec_blocks);
        const int ic = b / (a.tiles_k * a.tiles_j);
        w = b - ic * (a.tiles_k * a.tiles_j);
        i0 = ic * a.chunk_i;
        i1 = min(i0 + a.chunk_i, L.nx);
    }
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int k0 = (w % a.tiles_k) * FD_TK, j0 = 1 + (w / a.tiles_k) * TJ;  // rows 0 and ny-1 are Dirichlet
    const int qd = tx & 15, row = ty * 4 + (tx >> 4);
    const int k = k0 + 4 * qd, j = j0 + row;
    const IT pitch = (IT)L.pitch_j * S;

    const bool jk = j < L.ny - 1 && k < L.nz - 1;  // the lane updates at least one node of [1, nz-1)
    const bool ld = j < L.ny + R && k < L.nz + R;
    const IT colq = (IT)fd_off(L, 0, ld ? j : 0, ld ? k : 0) * S;
    int hrow[NH], hq[NH];
    IT colh[NH];
    bool hst[NH];
#pragma unroll
    for (int m = 0; m < NH; ++m) {
        const int h = ty * FD_TK + tx + T * m;
        int jh, kh;
        if (h < NROW) {
            const int hr = h >> 4;
            jh = hr < R ? j0 - R + hr : j0 + TJ + hr - R;
            kh = k0 + 4 * (h & 15);
            hrow[m] = hr < R ? hr : TJ + hr;
            hq[m] = (h & 15) + HQ;
        } else {
            const int e = h - NROW, s = e % (2 * HQ);
            jh = j0 + e / (2 * HQ);
            kh = s < HQ ? k0 + 4 * (s - HQ) : k0 + FD_TK + 4 * (s - HQ);
            hrow[m] = e / (2 * HQ) + R;
            hq[m] = s < HQ ? s : FD_TK / 4 + s;
        }
        hst[m] = h < NHQ;
        const bool l = hst[m] && jh < L.ny + R && kh < L.nz + R;
        colh[m] = (IT)fd_off(L, 0, l ? jh : 0, l ? kh : 0) * S;
    }
    float czr[W], cxv[UNI ? 1 : 4][W];
    {
        const int mz = j % P;
#pragma unroll
        for (int d = 0; d < W; ++d) czr[d] = a.cz[mz][d];
        if constexpr (!UNI) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int mx = (k + c) % P;
#pragma unroll
                for (int d = 0; d < W; ++d) cxv[c][d] = a.cx[mx][d];
            }
        }
    }
    int src_i = -1, src_c = 0;
    {
        const int64_t d = a.src_off - (int64_t)(colq / S);
        if (jk && d >= 0) {
            int64_t pi, c;
            if constexpr (sizeof(IT) == 4) {
                pi = (uint32_t)d / (uint32_t)L.pitch_j;
                c = (uint32_t)d % (uint32_t)L.pitch_j;
            } else {
                pi = d / L.pitch_j;
                c = d % L.pitch_j;
            }
            if (c < 4 && k + c >= 1 && k + c < L.nz - 1) {  // a boundary source is not injected by the step
                src_i = (int)pi;
                src_c = (int)c;
            }
        }
    }
    bool kin[4];  // interior along x
#pragma unroll
    for (int c = 0; c < 4; ++c) kin[c] = k + c >= 1 && k + c < L.nz - 1;

    quad_f4 q[Q], fh[NH][F], pm[2], qv[2];
    auto load_halo = [&](int slot, int p) {
        const IT po = (IT)p * pitch;
#pragma unroll
        for (int m = 0; m < NH; ++m) fh[m][slot] = ldq<false>(a.pn, colh[m] + po);
    };
    auto load_aux = [&](int set, int p) {
        const IT po = (IT)p * pitch;
        pm[set] = ldq<NT>(a.pnm1, colq + po);
        qv[set] = ldq<NT>(a.qf, colq + po);
    };
    auto stage = [&](int buf, int qslot, int hslot) {
        quad_f4(*tl)[LQ] = tile[buf];
        tl[row + R][qd + HQ] = q[qslot];
#pragma unroll
        for (int m = 0; m < NH; ++m)
            if (hst[m]) tl[hrow[m]][hq[m]] = fh[m][hslot];
    };
#pragma unroll
    for (int l = 0; l <= 2 * R; ++l) q[l] = ldq<false>(a.pn, colq + (IT)(i0 - R + l) * pitch);
#pragma unroll
    for (int d = 0; d <= R; ++d) load_halo(d, i0 + d);
    load_aux(0, i0);
    stage(0, R, 0);
    lds_barrier();

    auto plane = [&](auto uc, int i) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value;
        {
            const int pq = min(i + 1 + R, L.nx + R - 1);
            q[(u + 1 + 2 * R) % Q] = ldq<false>(a.pn, colq + (IT)pq * pitch);
            load_halo((u + F) % F, pq);
            load_aux((u + 1) & 1, min(i + 1, L.nx - 1));
        }
        if (jk && i >= 1 && i < L.nx - 1) {
            const quad_f4(*tl)[LQ] = tile[u & 1];
            const int my = (P == 4) ? (u % P) : (i % P);
            const int r = row + R;
            const quad_f4 pc = q[(u + R) % Q];
            quad_f4 zr[W];
            float x[4 * (2 * HQ + 1)];
#pragma unroll
            for (int d = 0; d < W; ++d)
                if (d != R) zr[d] = tl[r - R + d][qd + HQ];
#pragma unroll
            for (int s = 0; s < 2 * HQ + 1; ++s) {
                const quad_f4 v = s == HQ ? pc : tl[r][qd + s];
#pragma unroll
                for (int c = 0; c < 4; ++c) x[4 * s + c] = v[c];
            }
            float lap[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int d = 0; d < W; ++d) {
                if (d == R) continue;
#pragma unroll
                for (int c = 0; c < 4; ++c) lap[c] = fmaf(a.cy[my][d], q[(u + d) % Q][c] - pc[c], lap[c]);
#pragma unroll
                for (int c = 0; c < 4; ++c) lap[c] = fmaf(czr[d], zr[d][c] - pc[c], lap[c]);
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    lap[c] = fmaf(UNI ? a.cx[c % P][d] : cxv[UNI ? 0 : c][d], x[4 * HQ + c - R + d] - pc[c], lap[c]);
            }
            quad_f4 val;
#pragma unroll
            for (int c = 0; c < 4; ++c) val[c] = fmaf(-qv[u & 1][c], lap[c], 2.f * pc[c] - pm[u & 1][c]);
            if (src_i == i) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (src_c == c) {
                        if (a.trace) *a.trace = val[c];
                        if (a.inj) val[c] = add_nc(val[c], mul_nc(a.inj_coef, rhs_next));
                    }
            }
            // boundary nodes and what lies beyond the row keep their values
#pragma unroll
            for (int c = 0; c < 4; ++c) val[c] = kin[c] ? val[c] : pm[u & 1][c];
            stq<NT>(a.pnm1, colq + (IT)i * pitch, val);
        }
        stage((u + 1) & 1, (u + 1 + R) % Q, (u + 1) % F);
        lds_barrier();
    };
    for (int ib = i0; ib < i1; ib += U) march_turn(plane, ib, i1, std::make_integer_sequence<int, U>{});
}

// ------------------------------------------------------------ element path

struct SemElemArgs {
    const float *pn;     // level i2 in the node-order layout (no halo)
    float *y;            // assembled K p (atomic scatter target)
    const float *geo;    // per point: w_a w_b w_c * B (6 Voigt entries), for
                         // one element (stride 0) or every element
    int64_t geo_stride;  // floats between elements in geo
    float D[(SEM_MAX_P + 1) * (SEM_MAX_P + 1)];  // D[a][b] = l_a'(xi_b)
    float dgd[SEM_MAX_P + 1];  // MFMA kernel: gradient diagonal, -sum_{a != b} D[a][b]
    int ex, ey, ez, nx, ny, nz;
    int nelem;           // elements this launch covers
    // colour < 0: every element, atomic scatter.  colour c in 0..7: only the
    // elements with (ex_i, ez_i, ey_i) parities (c&1, c>>1&1, c>>2&1), which
    // share no node, scattered with plain read-add-write (deterministic)
    int colour;
    int ncx, ncz;        // elements of the colour along x and z
};

// Thread per GLL point; EPB elements per block.  The element's nodal block
// and the derivative matrix live in LDS; the gradient (3 q-term sums), the
// geometric factor product and the divergence (3 q-term sums) are done per
// point; y is scattered with float atomics.
template <int P, int EPB>
__global__ void __launch_bounds__(256)
sem_elem_kernel(SemElemArgs a)
{
    constexpr int q = P + 1, n3 = q * q * q;
    __shared__ float u[EPB][n3];
    __shared__ float g[EPB][3][n3];
    __shared__ float Ds[q * q];
    const int t = threadIdx.x;
    const int le = t / n3;          // element within the block
    const int pt = t - le * n3;     // GLL point (a fastest: x, then z (b), then y (c))
    const int k = blockIdx.x * EPB + le;  // element index within this launch
    const bool act = le < EPB && k < a.nelem;
    if (t < q * q) Ds[t] = a.D[t];
    const int pa = pt % q, pb = (pt / q) % q, pc = pt / (q * q);
    int node = 0, e = 0;
    if (act) {
        int exi, ezi, eyi;
        if (a.colour < 0) {
            exi = k % a.ex; ezi = (k / a.ex) % a.ez; eyi = k / (a.ex * a.ez);
        } else {
            exi = 2 * (k % a.ncx) + (a.colour & 1);
            ezi = 2 * ((k / a.ncx) % a.ncz) + ((a.colour >> 1) & 1);
            eyi = 2 * (k / (a.ncx * a.ncz)) + ((a.colour >> 2) & 1);
        }
        e = exi + ezi * a.ex + eyi * a.ex * a.ez;
        node = (exi * P + pa) + (ezi * P + pb) * a.nx + (eyi * P + pc) * a.nx * a.nz;
        u[le][pt] = a.pn[node];
    }
    __syncthreads();
    if (act) {
        // the derivative of a constant is zero (sum_m l_m' = 0): differences
        // from the point's own value keep FP32 precision on smooth fields
        const float uc = u[le][pt];
        float s1 = 0.f, s2 = 0.f, s3 = 0.f;
#pragma unroll
        for (int m = 0; m < q; ++m) {
            s1 = fmaf(Ds[m * q + pa], u[le][m + pb * q + pc * q * q] - uc, s1);
            s2 = fmaf(Ds[m * q + pb], u[le][pa + m * q + pc * q * q] - uc, s2);
            s3 = fmaf(Ds[m * q + pc], u[le][pa + pb * q + m * q * q] - uc, s3);
        }
        const float *G = a.geo + (int64_t)e * a.geo_stride + 6 * pt;
        // flux = (w w w B) grad u; B Voigt order 11, 22, 33, 12, 13, 23
        g[le][0][pt] = G[0] * s1 + G[3] * s2 + G[4] * s3;
        g[le][1][pt] = G[3] * s1 + G[1] * s2 + G[5] * s3;
        g[le][2][pt] = G[4] * s1 + G[5] * s2 + G[2] * s3;
    }
    __syncthreads();
    if (act) {
        float acc = 0.f;
#pragma unroll
        for (int m = 0; m < q; ++m) {
            acc = fmaf(Ds[pa * q + m], g[le][0][m + pb * q + pc * q * q], acc);
            acc = fmaf(Ds[pb * q + m], g[le][1][pa + m * q + pc * q * q], acc);
            acc = fmaf(Ds[pc * q + m], g[le][2][pa + pb * q + m * q * q], acc);
        }
        if (a.colour < 0) atomicAdd(&a.y[node], acc);
        else a.y[node] += acc;
    }
}

// The element operator with its contractions on the matrix cores (kernel
// PHC_SEM_ELEMENT_MFMA): one element per wavefront, four per block.  Each of
// the six contractions (three gradients, three divergence parts) is a product
// of the element's lines with the 1D derivative matrix,
//     out[line][j] = sum_m in[line][m] M[m][j],
// q^2 lines (rows) x q terms (K, padded to 8) x q outputs (N, padded to 16),
// taken as ceil(q^2/16) x 2 v_mfma_f32_16x16x4f32 products.  Operand layout
// of that instruction (one block): lane l supplies A[l%16][l/16] and
// B[l/16][l%16] of a 16x4 by 4x16 step and receives D[4 (l/16) + v][l%16],
// v = 0..3.  The gradient uses D with each column's diagonal entry dgd[b] =
// -sum_{a != b} D[a q + b] (so a constant has zero gradient, the exact
// property the vector kernel keeps with differences); the divergence uses D
// transposed.  Lines of direction x are (b, c) with the term index running
// over a, of z (a, c) over b, of y (a, b) over c; geometric factors are
// applied per point between the two products, and the three divergence parts
// are added per point before the colour scatter.
typedef float sem_f32x4 __attribute__((ext_vector_type(4)));

template <int P>
__device__ __forceinline__ int sem_line_point(int d, int line, int m)
{
    constexpr int q = P + 1;
    const int r0 = line % q, r1 = line / q;
    if (d == 0) return m + q * r0 + q * q * r1;   // x: line (b, c)
    if (d == 1) return r0 + q * m + q * q * r1;   // z: line (a, c)
    return r0 + q * r1 + q * q * m;               // y: line (a, b)
}

template <int P>
__global__ void __launch_bounds__(256) sem_elem_mfma_kernel(SemElemArgs a)
{
    constexpr int q = P + 1, n2 = q * q, n3 = q * n2;
    constexpr int RT = (n2 + 15) / 16;  // 16-line row tiles per direction
    static_assert(q <= 8 && n3 <= 256, "K padded to 8; points of an element within 4 lanes each");
    __shared__ float u[4][n3];
    __shared__ float gr[4][3][n3];  // gradients, then fluxes (per point)
    __shared__ float dv[4][3][n3];  // divergence parts (per point)
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int k = blockIdx.x * 4 + w;  // element of this launch
    if (k >= a.nelem) return;          // whole wavefront
    int exi, ezi, eyi;
    if (a.colour < 0) {
        exi = k % a.ex; ezi = (k / a.ex) % a.ez; eyi = k / (a.ex * a.ez);
    } else {
        exi = 2 * (k % a.ncx) + (a.colour & 1);
        ezi = 2 * ((k / a.ncx) % a.ncz) + ((a.colour >> 1) & 1);
        eyi = 2 * (k / (a.ncx * a.ncz)) + ((a.colour >> 2) & 1);
    }
    const int e = exi + ezi * a.ex + eyi * a.ex * a.ez;
    auto node_of = [&](int pt) {
        const int pa = pt % q, pb = (pt / q) % q, pc = pt / n2;
        return (exi * P + pa) + (ezi * P + pb) * a.nx + (eyi * P + pc) * a.nx * a.nz;
    };
    for (int pt = lane; pt < n3; pt += 64) u[w][pt] = a.pn[node_of(pt)];
    // B operands of the two K steps: gradient Dg[kk][j], divergence D[j][kk]
    const int j = lane & 15, kq = lane >> 4;
    float bg[2], bd[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        const int kk = 4 * st + kq;
        const bool in = kk < q && j < q;
        bg[st] = in ? (kk == j ? a.dgd[j] : a.D[kk * q + j]) : 0.f;
        bd[st] = in ? a.D[j * q + kk] : 0.f;
    }
    wave_lds_sync();
    // gradients
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            sem_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const int line = 16 * rt + j, kk = 4 * st + kq;
                const float av = (line < n2 && kk < q) ? u[w][sem_line_point<P>(d, line, kk)] : 0.f;
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bg[st], acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int line = 16 * rt + 4 * kq + v;
                if (line < n2 && j < q) gr[w][d][sem_line_point<P>(d, line, j)] = acc[v];
            }
        }
    wave_lds_sync();
    // fluxes, per point: (w w w B) grad u; B Voigt order 11, 22, 33, 12, 13, 23
    for (int pt = lane; pt < n3; pt += 64) {
        const float s1 = gr[w][0][pt], s2 = gr[w][1][pt], s3 = gr[w][2][pt];
        const float *G = a.geo + (int64_t)e * a.geo_stride + 6 * pt;
        gr[w][0][pt] = G[0] * s1 + G[3] * s2 + G[4] * s3;
        gr[w][1][pt] = G[3] * s1 + G[1] * s2 + G[5] * s3;
        gr[w][2][pt] = G[4] * s1 + G[5] * s2 + G[2] * s3;
    }
    wave_lds_sync();
    // divergence parts
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            sem_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const int line = 16 * rt + j, kk = 4 * st + kq;
                const float av = (line < n2 && kk < q) ? gr[w][d][sem_line_point<P>(d, line, kk)] : 0.f;
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bd[st], acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int line = 16 * rt + 4 * kq + v;
                if (line < n2 && j < q) dv[w][d][sem_line_point<P>(d, line, j)] = acc[v];
            }
        }
    wave_lds_sync();
    for (int pt = lane; pt < n3; pt += 64) {
        const float acc = (dv[w][0][pt] + dv[w][1][pt]) + dv[w][2][pt];
        const int node = node_of(pt);
        if (a.colour < 0) atomicAdd(&a.y[node], acc);
        else a.y[node] += acc;
    }
}

// ------------------------------------------------ element path, write-once
//
// The element operator assembled without a scatter to memory and with the
// leapfrog update fused (SEMsolver.cpp:46-89 in one pass).  A block owns the
// nodes of a tile of TE x TE elements in x and z (node x in [ex0 p, (ex0+TE) p),
// likewise z) over a range of element layers along y, and marches the layers
// one by one:
//  * the node patch of the layer's (TE+1)^2 elements (the tile plus one
//    element below it in x and z, whose faces carry owned nodes) is staged
//    in LDS, its p+1 node planes in a ring (a layer's top plane is the next
//    layer's bottom one and stays in place);
//  * each lane takes one node plane (local y index c) of one element: it
//    keeps the plane's (p+1)^2 values in registers, forms the x and z
//    derivatives there (the 1D derivative matrix entries are kernel-argument
//    constants), reads the y derivative's p+1 values from the patch, and
//    applies the geometric factors (SEMQkGLIntegrals.hpp:363-520: gradient,
//    flux, divergence); the y fluxes go through LDS for the y part of the
//    divergence, the x and z ones stay in registers;
//  * each element's K_e u_e is left in LDS and every owned node sums the
//    (at most 4) contributions of the layer's elements that hold it, in a
//    fixed order, plus the carried contribution of the layer below to its
//    bottom plane: no atomics, the same bits on every run;
//  * the node planes of the layer below its top face are then complete: the
//    owner applies the leapfrog update to its interior nodes and writes each
//    of them once; the top plane's sum is carried to the next layer in
//    registers (a thread keeps the same node columns all along).
// A range of layers [ey0, ey1) owns node planes [ey0 p, ey1 p) and first
// computes layer ey0 - 1 to complete its lowest plane.  Each node is written
// by exactly one block and only level i2 is read across blocks, so the new
// level can overwrite level i1 in place.
struct SemMarchArgs {
    const float *pn;     // level i2, node order
    float *pnm1;         // level i1: read, overwritten by the new level
    const float *dt2m;   // dt^2 / M per node
    const float *geo;    // per point w w w B (6 Voigt entries); element stride geo_stride
    int64_t geo_stride;
    float D[(SEM_MAX_P + 1) * (SEM_MAX_P + 1)];
    int ex, ey, ez, nx, ny, nz;
    int tiles_x, tiles_z, ychunk;
    int64_t src_node;
    int inj;
    float inj_coef;
    const float *rhs_next;  // in the run's sample window
    float *trace;
};

// Elements per tile side of the march kernel: (TE+1)^2 (p+1) element planes
// fit one 256-thread block.
constexpr int sem_march_te(int p)
{
    return p == 1 ? 10 : p == 2 ? 8 : p == 3 ? 7 : p == 4 ? 6 : 5;
}
constexpr int SEM_MARCH_NT = 256;

template <int P, int NT>
__global__ void __launch_bounds__(NT) sem_march_kernel(SemMarchArgs a)
{
    constexpr int TE = sem_march_te(P);
    constexpr int q = P + 1, n2 = q * q, n3 = q * n2;
    constexpr int NE = (TE + 1) * (TE + 1);            // elements of a layer's patch
    constexpr int PW = (TE + 1) * P + 1;               // patch nodes per axis (x, z)
    constexpr int OW = TE * P;                         // owned nodes per axis
    constexpr int NPF = (P * PW * PW + NT - 1) / NT;   // prefetched patch values per thread
    constexpr int NCOL = (OW * OW + NT - 1) / NT;      // owned node columns per thread
    static_assert(NE * q <= NT, "one lane per element plane");
    __shared__ float u[q][PW][PW];    // node patch, ring of planes [y][z][x]
    __shared__ float fv[NE][q][n2];   // y fluxes, then K_e u_e, per element [y][z][x]
    __shared__ float Gs[n3 * 6];      // geometric factors (one element: the box mesh)
    __shared__ float Ds[n2];
    const int tid = threadIdx.x;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int txi = b % a.tiles_x, rest = b / a.tiles_x;
    const int tzi = rest % a.tiles_z, yr = rest / a.tiles_z;
    const int ex0 = txi * TE, ez0 = tzi * TE;
    const int ey0 = yr * a.ychunk, ey1 = min(ey0 + a.ychunk, a.ey);
    const int X0 = ex0 * P - P, Z0 = ez0 * P - P;  // patch origin (node coordinates)
    const int64_t plane = (int64_t)a.nx * a.nz;
    const bool gshared = a.geo_stride == 0;
    for (int t = tid; t < n2; t += NT) Ds[t] = a.D[t];
    if (gshared)
        for (int t = tid; t < 6 * n3; t += NT) Gs[t] = a.geo[t];
    // the lane's element plane
    const int le = tid / q, pc = tid - le * q;
    const int lx = le % (TE + 1), lz = le / (TE + 1);
    const int exg = ex0 - 1 + lx, ezg = ez0 - 1 + lz;
    const bool act = le < NE && exg >= 0 && exg < a.ex && ezg >= 0 && ezg < a.ez;
    const int xb = lx * P, zb = lz * P;
    // patch value t of the planes above the bottom one of layer ey
    auto patch_load = [&](int ey, int t) {
        const int c = 1 + t / (PW * PW), r = t % (PW * PW), z = r / PW, x = r - z * PW;
        const int gx = X0 + x, gz = Z0 + z;
        float v = 0.f;
        if (t < P * PW * PW && gx >= 0 && gx < a.nx && gz >= 0 && gz < a.nz)
            v = a.pn[(int64_t)(ey * P + c) * plane + (int64_t)gz * a.nx + gx];
        return v;
    };
    float carry[NCOL];
#pragma unroll
    for (int c = 0; c < NCOL; ++c) carry[c] = 0.f;
    float pf[NPF];
    const int eyf = max(ey0 - 1, 0);
    int base = 0;  // ring slot of the layer's bottom plane
    for (int t = tid; t < PW * PW; t += NT) {
        const int z = t / PW, x = t - z * PW, gx = X0 + x, gz = Z0 + z;
        u[0][z][x] = (gx >= 0 && gx < a.nx && gz >= 0 && gz < a.nz)
                         ? a.pn[(int64_t)(eyf * P) * plane + (int64_t)gz * a.nx + gx] : 0.f;
    }
#pragma unroll
    for (int f = 0; f < NPF; ++f) pf[f] = patch_load(eyf, tid + f * NT);
    __syncthreads();  // Ds, Gs
    float dcol[q], drow[q];  // D[m][c], D[c][m] of the lane's plane c
#pragma unroll
    for (int m = 0; m < q; ++m) {
        dcol[m] = Ds[m * q + pc];
        drow[m] = Ds[pc * q + m];
    }
    for (int ey = eyf; ey < ey1; ++ey) {
        int slot[q];  // ring slot of the layer's plane c
#pragma unroll
        for (int c = 0; c < q; ++c) slot[c] = (base + c) % q;
        // planes 1..P of this layer from the registers
#pragma unroll
        for (int f = 0; f < NPF; ++f) {
            const int t = tid + f * NT;
            if (t < P * PW * PW) {
                const int c = 1 + t / (PW * PW);
                (&u[slot[c]][0][0])[t % (PW * PW)] = pf[f];
            }
        }
        __syncthreads();
        // the next layer's planes load while this layer is computed
        if (ey + 1 < ey1) {
#pragma unroll
            for (int f = 0; f < NPF; ++f) pf[f] = patch_load(ey + 1, tid + f * NT);
        }
        // gradient and flux of the lane's plane
        float U[q][q], F0[q][q], F1[q][q];
        if (act) {
            const float(*up)[PW] = u[slot[pc]];
#pragma unroll
            for (int pb = 0; pb < q; ++pb)
#pragma unroll
                for (int pa = 0; pa < q; ++pa) U[pb][pa] = up[zb + pb][xb + pa];
            const float *Gg = gshared ? Gs : a.geo + (exg + (int64_t)ezg * a.ex + (int64_t)ey * a.ex * a.ez) *
                                                         a.geo_stride;
#pragma unroll
            for (int pb = 0; pb < q; ++pb)
#pragma unroll
                for (int pa = 0; pa < q; ++pa) {
                    const float uc = U[pb][pa];
                    float s1 = 0.f, s2 = 0.f, s3 = 0.f;
#pragma unroll
                    for (int m = 0; m < q; ++m) {
                        s1 = fmaf(a.D[m * q + pa], U[pb][m] - uc, s1);
                        s2 = fmaf(a.D[m * q + pb], U[m][pa] - uc, s2);
                        s3 = fmaf(dcol[m], u[slot[m]][zb + pb][xb + pa] - uc, s3);
                    }
                    const float *G = Gg + 6 * (pa + q * pb + n2 * pc);
                    const float g0 = G[0], g1 = G[1], g2 = G[2], g3 = G[3], g4 = G[4], g5 = G[5];
                    F0[pb][pa] = g0 * s1 + g3 * s2 + g4 * s3;
                    F1[pb][pa] = g3 * s1 + g1 * s2 + g5 * s3;
                    fv[le][pc][pb * q + pa] = g4 * s1 + g5 * s2 + g2 * s3;
                }
        }
        __syncthreads();
        // divergence: x and z parts from registers, y part from the fluxes
        // of the element's other planes
        if (act) {
#pragma unroll
            for (int pb = 0; pb < q; ++pb)
#pragma unroll
                for (int pa = 0; pa < q; ++pa) {
                    float v = 0.f;
#pragma unroll
                    for (int m = 0; m < q; ++m) {
                        v = fmaf(a.D[pa * q + m], F0[pb][m], v);
                        v = fmaf(a.D[pb * q + m], F1[m][pa], v);
                        v = fmaf(drow[m], fv[le][m][pb * q + pa], v);
                    }
                    U[pb][pa] = v;
                }
        }
        __syncthreads();
        if (act) {
#pragma unroll
            for (int pb = 0; pb < q; ++pb)
#pragma unroll
                for (int pa = 0; pa < q; ++pa) fv[le][pc][pb * q + pa] = U[pb][pa];
        }
        __syncthreads();
        // assembly of the owned nodes (interior ones: every element holding
        // one is inside the mesh), leapfrog, one store per node
#pragma unroll
        for (int c = 0; c < NCOL; ++c) {
            const int col = tid + c * NT;
            if (col >= OW * OW) continue;
            const int oz = col / OW, ox = col - oz * OW;
            const int gx = ex0 * P + ox, gz = ez0 * P + oz;
            if (gx < 1 || gx >= a.nx - 1 || gz < 1 || gz >= a.nz - 1) continue;
            const int X = ox + P, Z = oz + P;
            const int lxa = X / P, pxa = X - lxa * P, lza = Z / P, pza = Z - lza * P;
            // contributing (element, local index) pairs along x and z: the
            // element below first when the node is on a face
            const int nxe = pxa == 0 ? 2 : 1, nze = pza == 0 ? 2 : 1;
            const int ex_[2] = {pxa == 0 ? lxa - 1 : lxa, lxa}, ax_[2] = {pxa == 0 ? P : pxa, 0};
            const int ez_[2] = {pza == 0 ? lza - 1 : lza, lza}, az_[2] = {pza == 0 ? P : pza, 0};
#pragma unroll
            for (int cc = 0; cc <= P; ++cc) {
                float g = cc == 0 ? carry[c] : 0.f;
                for (int iz = 0; iz < nze; ++iz)
                    for (int ix = 0; ix < nxe; ++ix)
                        g += fv[ez_[iz] * (TE + 1) + ex_[ix]][cc][az_[iz] * q + ax_[ix]];
                if (cc == P) {
                    carry[c] = g;
                } else if (ey >= ey0) {
                    const int gy = ey * P + cc;
                    if (gy >= 1 && gy < a.ny - 1) {
                        const int64_t n = (int64_t)gy * plane + (int64_t)gz * a.nx + gx;
                        float val = fmaf(-a.dt2m[n], g, 2.f * u[slot[cc]][Z][X] - a.pnm1[n]);
                        if (n == a.src_node) {
                            if (a.trace) *a.trace = val;
                            if (a.inj) val = add_nc(val, mul_nc(a.inj_coef, uniform_value(a.rhs_next)));
                        }
                        a.pnm1[n] = val;
                    }
                }
            }
        }
        __syncthreads();
        base = slot[P];  // the top plane is the next layer's bottom one
    }
}

// Leapfrog update of interior nodes (SEMsolver.cpp:85-89) with dt^2/M
// precomputed, fused with clearing y for the next step and with the source
// injection of the next time sample.
__global__ void sem_update_kernel(float *pold, const float *pcur, float *y, const float *dt2m,
                                  int nx, int ny, int nz, int src_node, int inj, float inj_coef,
                                  const float *rhs_next, float *trace)
{
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nn = (int64_t)nx * ny * nz;
    if (n >= nn) return;
    const int ix = (int)(n % nx), iz = (int)((n / nx) % nz), iy = (int)(n / ((int64_t)nx * nz));
    const float yv = y[n];
    y[n] = 0.f;
    if (ix < 1 || ix >= nx - 1 || iz < 1 || iz >= nz - 1 || iy < 1 || iy >= ny - 1) return;
    float val = fmaf(-dt2m[n], yv, 2.f * pcur[n] - pold[n]);
    if (n == src_node) {
        if (trace) *trace = val;
        if (inj) val = add_nc(val, mul_nc(inj_coef, uniform_value(rhs_next)));
    }
    pold[n] = val;
}

__global__ void sem_inject_kernel(float *p, int64_t off, float coef, const float *rhs, int it)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) p[off] = add_nc(p[off], mul_nc(coef, rhs[it]));
}

// One source term handed over by the caller: p[off] += coef * value.
__global__ void sem_add_value_kernel(float *p, int64_t off, float coef, float value)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) p[off] = add_nc(p[off], mul_nc(coef, value));
}

__global__ void sem_copy_point_kernel(const float *p, int64_t off, float *dst)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *dst = p[off];
}

__global__ void sem_sample_kernel(const float *p, const int64_t *offs, int nrec, float *out,
                                  int stride, int step, int64_t src_off, const float *src_trace)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nrec) sem_sample_point(p, offs, r, out, stride, step, src_off, src_trace);
}

// Start of a run: its source samples into the window, the first one into the
// current level (SEMsolver.cpp:39-43).
__global__ void sem_begin_run_kernel(float *p, int64_t off, float coef, const float *rhs, int it0, int n,
                                     float *window)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) window[t] = rhs[it0 + t];
    if (t == 0) p[off] = add_nc(p[off], mul_nc(coef, rhs[it0]));
}

using SemSepFn = void (*)(SemSepArgs);

template <int P, int TY, int NJ>
static SemSepFn sep_idx(bool idx32)
{
    return idx32 ? sem_sep_kernel<P, TY, NJ, uint32_t> : sem_sep_kernel<P, TY, NJ, int64_t>;
}

template <int P, int TY>
static SemSepFn quad_idx(bool idx32, bool nt)
{
    if (!idx32) return sem_quad_kernel<P, TY, int64_t, true>;
    return nt ? sem_quad_kernel<P, TY, uint32_t, true> : sem_quad_kernel<P, TY, uint32_t, false>;
}

template <int P>
static SemSepFn sep_shape(int ty, int nj, bool idx32, bool nt)
{
    if (ty == 8 && nj == 4) return quad_idx<P, 8>(idx32, nt);
    if (ty == 4 && nj == 4) return quad_idx<P, 4>(idx32, nt);
    if (ty == 16 && nj == 1) return sep_idx<P, 16, 1>(idx32);
    if (ty == 16 && nj == 2) return sep_idx<P, 16, 2>(idx32);
    if (ty == 8 && nj == 2) return sep_idx<P, 8, 2>(idx32);
    if (ty == 8 && nj == 1) return sep_idx<P, 8, 1>(idx32);
    if (ty == 4 && nj == 2) return sep_idx<P, 4, 2>(idx32);
    if (ty == 4 && nj == 1) return sep_idx<P, 4, 1>(idx32);
    return nullptr;
}

static SemSepFn sem_pick_sep(int p, int ty, int nj, bool idx32, bool nt)
{
    switch (p) {
    case 1: return sep_shape<1>(ty, nj, idx32, nt);
    case 2: return sep_shape<2>(ty, nj, idx32, nt);
    case 3: return sep_shape<3>(ty, nj, idx32, nt);
    case 4: return sep_shape<4>(ty, nj, idx32, nt);
    case 5: return sep_shape<5>(ty, nj, idx32, nt);
    default: return nullptr;
    }
}

using SemMarchFn = void (*)(SemMarchArgs);
static SemMarchFn sem_pick_march(int p)
{
    switch (p) {
    case 1: return sem_march_kernel<1, SEM_MARCH_NT>;
    case 2: return sem_march_kernel<2, SEM_MARCH_NT>;
    case 3: return sem_march_kernel<3, SEM_MARCH_NT>;
    case 4: return sem_march_kernel<4, SEM_MARCH_NT>;
    case 5: return sem_march_kernel<5, SEM_MARCH_NT>;
    default: return nullptr;
    }
}

using SemElemFn = void (*)(SemElemArgs);
static SemElemFn sem_pick_elem(int p, bool mfma, int *epb)
{
    if (mfma) {
        *epb = 4;  // one element per wavefront
        switch (p) {
        case 1: return sem_elem_mfma_kernel<1>;
        case 2: return sem_elem_mfma_kernel<2>;
        case 3: return sem_elem_mfma_kernel<3>;
        case 4: return sem_elem_mfma_kernel<4>;
        case 5: return sem_elem_mfma_kernel<5>;
        default: *epb = 0; return nullptr;
        }
    }
    switch (p) {
    case 1: *epb = 32; return sem_elem_kernel<1, 32>;
    case 2: *epb = 9; return sem_elem_kernel<2, 9>;
    case 3: *epb = 4; return sem_elem_kernel<3, 4>;
    case 4: *epb = 2; return sem_elem_kernel<4, 2>;
    case 5: *epb = 1; return sem_elem_kernel<5, 1>;
    default: *epb = 0; return nullptr;
    }
}

} // namespace phc

// ====================================================================== API
using namespace phc;

struct phc_sem {
    int ex, ey, ez, p, nx, ny, nz;
    int64_t nn;
    int kernel;
    float dt;
    int nsamples;
    std::vector<float> model;
    int src_element, src_node;
    bool src_interior = true;  // boundary nodes are never updated: no fused injection
    float inj_coef;
    hipStream_t stream = nullptr;
    // separable path
    FdLayout L;
    DevBuf lev[2], qf;
    // chunk_i < 0: the per-XCD schedule, rebuilt when it or the block shape changes
    DevBuf sched;
    int sched_nb = 0, sched_tj = -1;
    int cus = 256;
    float cx[SEM_MAX_P][2 * SEM_MAX_P + 1], cy[SEM_MAX_P][2 * SEM_MAX_P + 1],
        cz[SEM_MAX_P][2 * SEM_MAX_P + 1];
    int ty = 16, nj = 1, chunk_i = 0;
    int index64 = 0;  // 64-bit offsets even for arrays < 4 GiB
    int krem_mode = 0;  // phc_sem_params.k_remainder
    // element path
    DevBuf y, dt2m, geo, rhs;
    float Dm[(SEM_MAX_P + 1) * (SEM_MAX_P + 1)];
    std::vector<float> hmass;
    // traces, and the running chunk's source samples
    DevBuf trace, window, rec, recoff, readback;
    int nrec = 0, last_n = 0, last_nrec = 0;
    int timing = 0;
    double last_ms = 0.0;
    RunGraphs graph[2];  // of phc_sem_run, by i1
};

static int64_t sem_off(const phc_sem *h, int64_t node)
{
    const int ix = (int)(node % h->nx), iz = (int)((node / h->nx) % h->nz),
              iy = (int)(node / ((int64_t)h->nx * h->nz));
    if (h->kernel == PHC_SEM_SEPARABLE) return fd_off(h->L, iy, iz, ix);
    return node;
}

static void sem_drop_graph(phc_sem *h)
{
    for (RunGraphs &g : h->graph) g.drop();
}

// A node-order host field into a level (layout conversion for the
// separable path; halo stays zero).
static phc_status sem_put(phc_sem *h, DevBuf &dst, const float *host)
{
    if (h->kernel == PHC_SEM_SEPARABLE) {
        return write_field(h->stream, h->readback, dst.as<float>(), h->L, 0, 0, 0, host);
    } else {
        PHC_HIP(hipMemcpy(dst.ptr, host, sizeof(float) * h->nn, hipMemcpyHostToDevice));
    }
    return PHC_OK;
}

static phc_status sem_get(phc_sem *h, const DevBuf &src, float *host)
{
    if (h->kernel == PHC_SEM_SEPARABLE) {
        return read_field(h->stream, h->readback, src.as<float>(), h->L, 0, 0, 0, FieldDamping{}, nullptr, host);
    } else {
        PHC_HIP(hipStreamSynchronize(h->stream));
        PHC_HIP(hipMemcpy(host, src.ptr, sizeof(float) * h->nn, hipMemcpyDeviceToHost));
    }
    return PHC_OK;
}

// Per-XCD schedule of the separable kernel (chunk_i = -m, m = 1..4): slots
// = blocks resident per XCD, plane ranges between 4-plane groups.
static void sem_build_sched(int nx, int ncol, int slots, int m, std::vector<int4> &tab)
{
    build_xcd_schedule(nx, 0, ncol, std::max(slots, 1), m, 4, tab);
}

// x tiles of the separable kernel (over x in [0, nz - 1), interior from 1),
// and the first x of the remainder slab (0: none).
static int sem_tiles_k(const phc_sem *h, int *krem)
{
    const int span = std::max(h->L.nz - 1, 1), full = span / FD_TK, rem = span - full * FD_TK;
    // mode 0 with four nodes per lane: a tile (as nodes it cost 1-13% more at
    // 76^3 and 151^3 order 3, nothing elsewhere)
    const bool use = h->krem_mode >= (h->nj == 4 ? 1 : 0) && full > 0 && rem > 0 &&
                     (h->krem_mode == 1 || rem <= FD_TK / 2);
    if (krem) *krem = use ? FD_TK * full : 0;
    return use ? full : (span + FD_TK - 1) / FD_TK;
}

static SemSepFn sem_handle_kernel(const phc_sem *h)
{
    // non-temporal pnm1 and coefficients (quad kernels) from where the three
    // arrays no longer stay in the 256 MB memory-side cache, as in the FD step
    return sem_pick_sep(h->p, h->ty, h->nj, !h->index64 && h->L.total * 4 < ((int64_t)1 << 32),
                        12 * h->L.total > (int64_t)300e6);
}

// Blocks of the handle's shape resident per CU.
static int sem_resident(const phc_sem *h)
{
    int per_cu = 1;
    SemSepFn fn = sem_handle_kernel(h);
    if (!fn || hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(fn),
                                                            FD_TK * h->ty, 0) != hipSuccess || per_cu < 1)
        per_cu = 1;
    return per_cu;
}

// Block shape and per-XCD split where the caller gives none.
// Below 600,000 nodes 8 waves x 1 row, split 2: four nodes per lane leave too
// few wavefronts there (51^3 order 5: 9.6 against 10.9 us per step, 81^3 order
// 4: 9.7 / 10.3; 101^3, at once above the line: order 1 10.2 / 8.7, order 2
// 11.9 / 9.5, order 5 15.3 / 14.3).  Above, 4 waves x 16 rows, split 1, the
// best or within 5% of the best table entry from 101^3 to 321^3 (order 1
// alone prefers chunks of 12-24 planes by up to 14%).  For large arrays the
// shape and split with the least work on the busiest CU, as in the FD step: us
// per step of 8 x 1 / 4 x 16 split 1 / chosen: 331 x 346 x 331 order 3 127 / 112
// / 104, 353 x 361 x 345 order 4 148 / 141 / 122, 351 x 361 x 351 order 5 186 /
// 138 / 126, 481^3-sized orders 3, 4, 5 373, 346, 377 / - / 295, 281, 279.  The
// lines lie where 4 x 16 split 1 stops winning (it / the choice, MB of arrays):
//   order 1  331^3  511  99.9 / 102.2   341^3  542 110.2 / 115.6 | 356^3  640 136.5 / 132.5
//   order 2  327^3  505 101.6 / 109.3   333^3  523 102.2 / 102.0 | 341^3  548 115.8 / 108.2
//   order 3  292^3  375  75.6 /  76.2   313^3  430  83.5 /  91.9 | 325^3  505 105.7 /  95.0
//   order 4  313^3  435  83.8 /  94.2   321^3  499  87.9 /  92.6 | 325^3  511 109.6 /  98.9
//   order 5  291^3  383  82.1 /  79.9   311^3  435  98.9 /  94.2 | 321^3  505 102.9 /  95.4
// 321 nodes are 5 whole tiles along x; the sixth and the next row of tiles
// cost split 1 its balance.
// Flat meshes have few planes to cut: 8 ranges of whole groups leave XCDs idle
// below 32 planes and prime the ring over and over.  Up to 25 planes the XCDs
// take bands of columns over the whole axis (split 4), up to 63 halves of it
// (split 3).  Us per step of 4 x 16 split 1 (8 x 1 split 2 below 600,000 nodes) /
// 16 x 1 whole axis / this, orders 1 and 5: 801 x 5 x 801 47 / 15 / 14, 84 / 27 / 24;
// 401 x 21 x 401 19 / 18 / 14, 31 / 22 / 20; 17 x 21 x 3001 13 / 17 / 11, 27 / 22 / 18;
// 801 x 49 x 801 109 / 88 / 88, 141 / 106 / 100; 1767 x 51 x 341 98 / 90 / 83, 140 /
// 117 / 99; 361 x 61 x 541 39 / 46 / 41, 50 / 52 / 40.  At 65 planes split 1 is level
// or ahead at orders 1, 2 and 4.  Planes under 25,000 nodes keep 8 x 1 (145 x 33 x
// 145 order 4 10.0 against 10.7).
static void sem_default_shape(phc_sem *h)
{
    h->ty = 8;
    h->nj = 1;
    h->chunk_i = -2;
    const bool flat = h->ny < 64 && (int64_t)h->nx * h->nz >= 25000;
    if (h->nn < 600000 && !flat) return;
    h->ty = 4;
    h->nj = 4;
    h->chunk_i = !flat ? -1 : h->ny <= 25 ? -4 : -3;
    if (12 * h->L.total < (h->p <= 2 ? (int64_t)545e6 : (int64_t)500e6)) return;
    double best = -1.0;
    int ty = 4, m = 1;
    for (int t : {8, 4}) {
        h->ty = t;
        const int TJ = 4 * t, ncol = sem_tiles_k(h, nullptr) * ((std::max(h->L.ny - 2, 1) + TJ - 1) / TJ);
        const int cux = std::max(h->cus / 8, 1), slots = cux * sem_resident(h);
        std::vector<int4> tab;
        for (int s = 1; s <= 4; ++s) {
            sem_build_sched(h->L.nx, ncol, slots, s, tab);
            const double c = xcd_schedule_cost(tab, cux, TJ, 0.35 * 2 * h->p, 2 * h->p);
            if (best < 0.0 || c < best) {
                best = c;
                ty = t;
                m = s;
            }
        }
    }
    h->ty = ty;
    h->chunk_i = -m;
}

static phc_status sem_prepare_sched(phc_sem *h)
{
    const int TJ = h->ty * h->nj;
    const int key = ((TJ * 8 - h->chunk_i) * 4 + (h->krem_mode + 1)) * 32 + h->ty;
    if (h->kernel != PHC_SEM_SEPARABLE || h->chunk_i >= 0 || h->sched_tj == key) return PHC_OK;
    const int ncol = sem_tiles_k(h, nullptr) * ((std::max(h->L.ny - 2, 1) + TJ - 1) / TJ);
    // blocks of this shape resident per CU (the table deals one round of
    // them per XCD at a time)
    std::vector<int4> tab;
    sem_build_sched(h->L.nx, ncol, std::max(h->cus / 8, 1) * sem_resident(h), -h->chunk_i, tab);
    PHC_HIP(hipStreamSynchronize(h->stream));  // queued launches may still read the old table
    sem_drop_graph(h);
    PHC_TRY(h->sched.alloc(sizeof(int4) * tab.size()));
    PHC_HIP(hipMemcpy(h->sched.ptr, tab.data(), sizeof(int4) * tab.size(), hipMemcpyHostToDevice));
    h->sched_nb = (int)tab.size();
    h->sched_tj = key;
    return PHC_OK;
}

// One step: level i1 <- update(level i1, level i2); optional fused injection
// of the sample at rhs_next (device memory) and source trace.  rec_step >= 0:
// the separable launch also samples level i2's receivers into that step of a
// run of rec_stride steps.
static phc_status sem_launch(phc_sem *h, int i1, int i2, const float *rhs_next, float *trace, hipEvent_t e0,
                             hipEvent_t e1, int rec_step = -1, int rec_stride = 0)
{
    const int inj = rhs_next != nullptr;
    if (h->kernel == PHC_SEM_SEPARABLE) {
        SemSepArgs a;
        std::memset(&a, 0, sizeof(a));
        a.pn = h->lev[i2].as<float>();
        a.pnm1 = h->lev[i1].as<float>();
        a.qf = h->qf.as<float>();
        a.L = h->L;
        std::memcpy(a.cx, h->cx, sizeof(a.cx));
        std::memcpy(a.cy, h->cy, sizeof(a.cy));
        std::memcpy(a.cz, h->cz, sizeof(a.cz));
        a.src_off = sem_off(h, h->src_node);
        a.inj = inj;
        a.inj_coef = h->inj_coef;
        a.rhs_next = rhs_next;
        a.trace = trace;
        // tiles over the interior: k = 1..nz-2 (from k = 0), rows 1..ny-2
        const int TJ = h->ty * h->nj;
        a.tiles_k = sem_tiles_k(h, &a.krem);
        a.tiles_j = (std::max(h->L.ny - 2, 1) + TJ - 1) / TJ;
        int nb;
        if (h->chunk_i < 0) {
            // the table is built outside graph capture (phc_sem_run prepares it first)
            PHC_TRY(sem_prepare_sched(h));
            a.sched = h->sched.as<int4>();
            a.chunk_i = 0;
            nb = h->sched_nb;
        } else {
            if (h->chunk_i == 0) return fail(PHC_ERR_INVALID, "chunk_i is 0");
            a.chunk_i = h->chunk_i;
            // order 4: chunks start at multiples of 4 (the kernel's coefficient rows assume it)
            if (h->p == 4 && a.chunk_i < h->L.nx && a.chunk_i % 4) a.chunk_i += 4 - a.chunk_i % 4;
            nb = a.tiles_k * a.tiles_j * ((h->L.nx + a.chunk_i - 1) / a.chunk_i);
        }
        if (a.krem > 0) {
            const int64_t pts = (int64_t)(h->L.nz - 1 - a.krem) * (h->L.ny - 2) * (h->L.nx - 2);
            a.nb_main = nb;
            nb += (int)((pts + FD_TK * h->ty - 1) / (FD_TK * h->ty));
        }
        if (rec_step >= 0) {
            a.rec_off = h->recoff.as<int64_t>();
            a.rec_out = h->rec.as<float>();
            a.rec_src = h->trace.as<float>();
            a.rec_n = h->nrec;
            a.rec_stride = rec_stride;
            a.rec_step = rec_step;
            a.rec_blocks = (h->nrec + FD_TK * h->ty - 1) / (FD_TK * h->ty);
            nb += a.rec_blocks;
        }
        SemSepFn fn = sem_handle_kernel(h);
        if (!fn) return fail(PHC_ERR_INVALID, "no separable kernel for p=%d", h->p);
        if (e0) PHC_HIP(hipEventRecord(e0, h->stream));
        hipLaunchKernelGGL(fn, dim3(nb), dim3(FD_TK, h->ty), 0, h->stream, a);
        PHC_HIP(hipGetLastError());
        if (e1) PHC_HIP(hipEventRecord(e1, h->stream));
    } else if (h->kernel == PHC_SEM_ELEMENT_MARCH) {
        SemMarchArgs a;
        std::memset(&a, 0, sizeof(a));
        a.pn = h->lev[i2].as<float>();
        a.pnm1 = h->lev[i1].as<float>();
        a.dt2m = h->dt2m.as<float>();
        a.geo = h->geo.as<float>();
        a.geo_stride = 0;
        std::memcpy(a.D, h->Dm, sizeof(a.D));
        a.ex = h->ex; a.ey = h->ey; a.ez = h->ez;
        a.nx = h->nx; a.ny = h->ny; a.nz = h->nz;
        const int TE = sem_march_te(h->p);
        a.tiles_x = (h->ex + TE - 1) / TE;
        a.tiles_z = (h->ez + TE - 1) / TE;
        // layer ranges along y: the count that minimises the most layers any
        // CU marches (blocks per CU x (layers per range + the range's
        // priming layer))
        const int cols = a.tiles_x * a.tiles_z;
        int ranges = 1;
        long best = -1;
        for (int r = 1; r <= std::min(h->ey, 64); ++r) {
            const int chunk = (h->ey + r - 1) / r, nr = (h->ey + chunk - 1) / chunk;
            const long cost = (long)((cols * nr + h->cus - 1) / h->cus) * (chunk + (nr > 1 ? 1 : 0));
            if (best < 0 || cost < best) { best = cost; ranges = nr; }
        }
        a.ychunk = (h->ey + ranges - 1) / ranges;
        const int nb = cols * ((h->ey + a.ychunk - 1) / a.ychunk);
        a.src_node = h->src_node;
        a.inj = inj;
        a.inj_coef = h->inj_coef;
        a.rhs_next = rhs_next;
        a.trace = trace;
        SemMarchFn fn = sem_pick_march(h->p);
        if (!fn) return fail(PHC_ERR_INVALID, "no element march kernel for p=%d", h->p);
        if (e0) PHC_HIP(hipEventRecord(e0, h->stream));
        hipLaunchKernelGGL(fn, dim3(nb), dim3(SEM_MARCH_NT), 0, h->stream, a);
        PHC_HIP(hipGetLastError());
        if (e1) PHC_HIP(hipEventRecord(e1, h->stream));
    } else {
        SemElemArgs a;
        std::memset(&a, 0, sizeof(a));
        a.pn = h->lev[i2].as<float>();
        a.y = h->y.as<float>();
        a.geo = h->geo.as<float>();
        a.geo_stride = 0;
        std::memcpy(a.D, h->Dm, sizeof(a.D));
        a.ex = h->ex; a.ey = h->ey; a.ez = h->ez;
        a.nx = h->nx; a.ny = h->ny; a.nz = h->nz;
        int epb = 0;
        SemElemFn fn = sem_pick_elem(h->p, h->kernel == PHC_SEM_ELEMENT_MFMA, &epb);
        {
            const int q = h->p + 1;
            for (int c = 0; c < q; ++c) {
                double sum = 0.0;
                for (int m = 0; m < q; ++m)
                    if (m != c) sum += (double)h->Dm[m * q + c];
                a.dgd[c] = (float)(-sum);
            }
        }
        if (!fn) return fail(PHC_ERR_INVALID, "no element kernel for p=%d", h->p);
        if (e0) PHC_HIP(hipEventRecord(e0, h->stream));
        if (h->kernel == PHC_SEM_ELEMENT) {
            a.colour = -1;
            a.nelem = h->ex * h->ey * h->ez;
            hipLaunchKernelGGL(fn, dim3((a.nelem + epb - 1) / epb), dim3(256), 0, h->stream, a);
            PHC_HIP(hipGetLastError());
        } else {
            // 8 colours in a fixed order: each node receives its (at most 8)
            // element contributions in the same order on every run
            for (int c = 0; c < 8; ++c) {
                a.colour = c;
                a.ncx = (h->ex - (c & 1) + 1) / 2;
                a.ncz = (h->ez - ((c >> 1) & 1) + 1) / 2;
                const int ncy = (h->ey - ((c >> 2) & 1) + 1) / 2;
                a.nelem = a.ncx * a.ncz * ncy;
                if (a.nelem == 0) continue;
                hipLaunchKernelGGL(fn, dim3((a.nelem + epb - 1) / epb), dim3(256), 0, h->stream, a);
                PHC_HIP(hipGetLastError());
            }
        }
        hipLaunchKernelGGL(sem_update_kernel, dim3((unsigned)((h->nn + 255) / 256)), dim3(256), 0,
                           h->stream, h->lev[i1].as<float>(), h->lev[i2].as<float>(),
                           h->y.as<float>(), h->dt2m.as<float>(), h->nx, h->ny, h->nz,
                           h->src_node, inj, h->inj_coef, rhs_next, trace);
        PHC_HIP(hipGetLastError());
        if (e1) PHC_HIP(hipEventRecord(e1, h->stream));
    }
    return PHC_OK;
}

// First node of element e, globalNodesList(e, 0) (SEMmesh.cpp:214-223: elements
// numbered x fastest, then z, then y).
static int64_t sem_first_node(const phc_sem *h, int64_t e)
{
    const int64_t exi = e % h->ex, ezi = (e / h->ex) % h->ez, eyi = e / ((int64_t)h->ex * h->ez);
    return exi * h->p + (ezi * h->p) * h->nx + (eyi * h->p) * (int64_t)h->nx * h->nz;
}

// The source of the fused loop: element, samples, injection coefficient
// dt^2 c^2 of the element (SEMsolver.cpp:38-42, rounded left to right).
static phc_status sem_source(phc_sem *h, int src_element, int nsamples, const float *rhs)
{
    const int64_t nE = (int64_t)h->ex * h->ey * h->ez;
    if (src_element < 0 || src_element >= nE)
        return fail(PHC_ERR_INVALID, "source element %d outside 0..%lld", src_element, (long long)nE - 1);
    if (nsamples < 0 || (nsamples > 0 && !rhs)) return fail(PHC_ERR_INVALID, "bad rhs");
    h->src_element = src_element;
    h->src_node = (int)sem_first_node(h, src_element);
    const float c = h->model[src_element];
    h->inj_coef = ((h->dt * h->dt) * c) * c;
    const int64_t sn = h->src_node;
    const int sx = (int)(sn % h->nx), sz = (int)((sn / h->nx) % h->nz), sy = (int)(sn / ((int64_t)h->nx * h->nz));
    h->src_interior = sx >= 1 && sx < h->nx - 1 && sz >= 1 && sz < h->nz - 1 && sy >= 1 && sy < h->ny - 1;
    h->nsamples = nsamples;
    PHC_TRY(h->rhs.alloc(sizeof(float) * std::max(1, nsamples)));
    if (nsamples > 0) PHC_HIP(hipMemcpy(h->rhs.ptr, rhs, sizeof(float) * nsamples, hipMemcpyHostToDevice));
    return PHC_OK;
}

static phc_status sem_inject(phc_sem *h, int level, int it)
{
    hipLaunchKernelGGL(sem_inject_kernel, dim3(1), dim3(64), 0, h->stream, h->lev[level].as<float>(),
                       sem_off(h, h->src_node), h->inj_coef, h->rhs.as<float>(), it);
    PHC_HIP(hipGetLastError());
    return PHC_OK;
}

extern "C" {

int phc_sem_element_from_point(int ex, int ey, int ez, float lx, float ly, float lz, float x,
                               float y, float z)
{
    // SEMmesh.cpp:266-285 with the float element sizes of SEMmesh.cpp:20-22
    const float hx = (float)((double)lx / (1. * ex)), hy = (float)((double)ly / (1. * ey)),
                hz = (float)((double)lz / (1. * ez));
    int eX = 0, eY = 0, eZ = 0;
    for (int i = 0; i < ex; ++i)
        if (x >= i * hx && x < (i + 1) * hx) eX = i;
    for (int i = 0; i < ey; ++i)
        if (y >= i * hy && y < (i + 1) * hy) eY = i;
    for (int i = 0; i < ez; ++i)
        if (z >= i * hz && z < (i + 1) * hz) eZ = i;
    return eX + eZ * ex + eY * ex * ez;
}

phc_status phc_sem_schedule_table(int march_planes, int tile_columns, int cus, int split, int *entries,
                                  int *n_entries)
{
    if (!n_entries) return fail(PHC_ERR_INVALID, "n_entries is NULL");
    if (march_planes < 1 || tile_columns < 1 || cus < 1 || split < 1 || split > 4)
        return fail(PHC_ERR_INVALID, "planes %d, columns %d, CUs %d, split %d", march_planes, tile_columns, cus,
                    split);
    std::vector<int4> tab;
    sem_build_sched(march_planes, tile_columns, std::max(cus / 8, 1), split, tab);
    if (entries) {
        if (*n_entries < (int)tab.size())
            return fail(PHC_ERR_INVALID, "table has %d entries, room for %d", (int)tab.size(), *n_entries);
        for (size_t b = 0; b < tab.size(); ++b) {
            entries[3 * b] = tab[b].x;
            entries[3 * b + 1] = tab[b].y;
            entries[3 * b + 2] = tab[b].z;
        }
    }
    *n_entries = (int)tab.size();
    return PHC_OK;
}

phc_status phc_sem_create(const phc_sem_params *p, phc_sem **out)
{
    if (!out) return fail(PHC_ERR_INVALID, "out is NULL");
    *out = nullptr;
    if (!p) return fail(PHC_ERR_INVALID, "params is NULL");
    if (p->ex < 1 || p->ey < 1 || p->ez < 1)
        return fail(PHC_ERR_INVALID, "mesh %d x %d x %d has no elements", p->ex, p->ey, p->ez);
    if (p->order < 1 || p->order > SEM_MAX_P)
        return fail(PHC_ERR_INVALID, "order %d outside 1..%d", p->order, SEM_MAX_P);
    if (!(p->lx > 0) || !(p->ly > 0) || !(p->lz > 0)) return fail(PHC_ERR_INVALID, "bad domain size");
    if (!p->model) return fail(PHC_ERR_INVALID, "model is NULL");
    if (p->nsamples < 0 || (p->nsamples > 0 && !p->rhs)) return fail(PHC_ERR_INVALID, "bad rhs");
    if (p->kernel != PHC_SEM_SEPARABLE && p->kernel != PHC_SEM_ELEMENT && p->kernel != PHC_SEM_ELEMENT_COLOR &&
        p->kernel != PHC_SEM_ELEMENT_MARCH && p->kernel != PHC_SEM_ELEMENT_MFMA)
        return fail(PHC_ERR_INVALID, "unknown SEM kernel %d", p->kernel);
    const int64_t nE = (int64_t)p->ex * p->ey * p->ez;
    if (p->src_element < 0 || p->src_element >= nE)
        return fail(PHC_ERR_INVALID, "source element %d outside 0..%lld", p->src_element, (long long)nE - 1);
    for (int64_t e = 0; e < nE; ++e)
        if (!(p->model[e] > 0.f) || !std::isfinite(p->model[e]))
            return fail(PHC_ERR_INVALID, "wave speed of element %lld is not positive", (long long)e);
    // element sizes as the reference uses them for coordinates: the float
    // quotient lx/ex (SEMmesh.cpp:20) passed through an int parameter
    const int hxi = (int)(float)((double)p->lx / (1. * p->ex));
    const int hyi = (int)(float)((double)p->ly / (1. * p->ey));
    const int hzi = (int)(float)((double)p->lz / (1. * p->ez));
    if (hxi < 1 || hyi < 1 || hzi < 1)
        return fail(PHC_ERR_INVALID, "element size below 1 (the reference truncates it to an int)");

    phc_sem *h = new phc_sem();
    auto bail = [&](phc_status s) { phc_sem_destroy(h); return s; };
    h->ex = p->ex; h->ey = p->ey; h->ez = p->ez; h->p = p->order;
    h->nx = p->ex * p->order + 1;
    h->ny = p->ey * p->order + 1;
    h->nz = p->ez * p->order + 1;
    h->nn = (int64_t)h->nx * h->ny * h->nz;
    h->kernel = p->kernel;
    h->dt = p->dt;
    h->nsamples = p->nsamples;
    h->model.assign(p->model, p->model + nE);
    h->src_element = p->src_element;
    {
        const int e = p->src_element;
        const int exi = e % h->ex, ezi = (e / h->ex) % h->ez, eyi = e / (h->ex * h->ez);
        h->src_node = exi * h->p + (ezi * h->p) * h->nx + (eyi * h->p) * h->nx * h->nz;
        const float c = h->model[e];
        h->inj_coef = ((h->dt * h->dt) * c) * c;  // SEMsolver.cpp:41-42
        const int sx = exi * h->p, sz = ezi * h->p, sy = eyi * h->p;
        h->src_interior = sx >= 1 && sx < h->nx - 1 && sz >= 1 && sz < h->nz - 1 && sy >= 1 && sy < h->ny - 1;
    }
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(PHC_ERR_HIP, "hipStreamCreate failed"));

    // ---- FP64 setup
    const int P = h->p, qn = P + 1, W = 2 * P + 1;
    const GllBasis g = make_gll(P, p->weights_ref != 0);
    const SemAxis ax = make_axis(g, h->ex, hxi), ay = make_axis(g, h->ey, hyi),
                  az = make_axis(g, h->ez, hzi);
    // lumped mass: sum over elements of (w_a hx/2)(w_b hz/2)(w_c hy/2)/c^2
    std::vector<double> M((size_t)h->nn, 0.0);
    for (int64_t e = 0; e < nE; ++e) {
        const int exi = (int)(e % h->ex), ezi = (int)((e / h->ex) % h->ez), eyi = (int)(e / ((int64_t)h->ex * h->ez));
        const double ic2 = 1.0 / ((double)h->model[e] * h->model[e]);
        for (int c = 0; c < qn; ++c)
            for (int b = 0; b < qn; ++b)
                for (int a = 0; a < qn; ++a) {
                    const int64_t node = (exi * P + a) + (int64_t)(ezi * P + b) * h->nx +
                                         (int64_t)(eyi * P + c) * h->nx * h->nz;
                    M[node] += (g.w[a] * ax.half) * (g.w[b] * az.half) * (g.w[c] * ay.half) * ic2;
                }
    }
    h->hmass.resize(h->nn);
    for (int64_t n = 0; n < h->nn; ++n) h->hmass[n] = (float)M[n];
    const double dt2 = (double)h->dt * (double)h->dt;
    PHC_TRY(h->rhs.alloc(sizeof(float) * std::max(1, h->nsamples)));
    if (h->nsamples > 0 && hipMemcpy(h->rhs.ptr, p->rhs, sizeof(float) * h->nsamples, hipMemcpyHostToDevice))
        return bail(fail(PHC_ERR_HIP, "rhs upload failed"));

    phc_status st;
    if (h->kernel == PHC_SEM_SEPARABLE) {
        h->L = make_fd_layout(h->ny, h->nz, h->nx, P);  // i = iy, j = iz, k = ix
        const size_t bytes = sizeof(float) * (size_t)h->L.total;
        if ((st = h->lev[0].alloc(bytes)) || (st = h->lev[1].alloc(bytes)) || (st = h->qf.alloc(bytes)))
            return bail(st);
        for (DevBuf *b : {&h->lev[0], &h->lev[1], &h->qf})
            if ((st = fill_field(h->stream, b->as<float>(), h->L.total, 0.f))) return bail(st);
        // Q = dt^2 Wx Wz Wy / M on interior nodes, 0 elsewhere
        std::vector<float> Qn((size_t)h->nn, 0.f);
        for (int iy = 1; iy < h->ny - 1; ++iy)
            for (int iz = 1; iz < h->nz - 1; ++iz)
                for (int ix = 1; ix < h->nx - 1; ++ix) {
                    const int64_t n = ix + (int64_t)iz * h->nx + (int64_t)iy * h->nx * h->nz;
                    Qn[n] = (float)(dt2 * ax.Wg[ix] * az.Wg[iz] * ay.Wg[iy] / M[n]);
                }
        if ((st = sem_put(h, h->qf, Qn.data()))) return bail(st);
        h->readback.release();  // not held by a handle whose fields are never read
        // stencil rows by index mod p (identical on every row of an axis with
        // the same residue: the mesh is uniform along each axis)
        std::memset(h->cx, 0, sizeof(h->cx));
        std::memset(h->cy, 0, sizeof(h->cy));
        std::memset(h->cz, 0, sizeof(h->cz));
        auto rows = [&](const SemAxis &A, float (*c)[2 * SEM_MAX_P + 1]) {
            for (int m = 0; m < P; ++m) {
                // a representative interior row with residue m
                int i = m;
                if (i == 0) i = (A.n > P + 1) ? P : 0;
                if (i == 0 || i >= A.n - 1) continue;  // no interior node with this residue
                for (int d = 0; d < W; ++d) c[m][d] = (float)A.A[(size_t)i * W + d];
            }
        };
        rows(ax, h->cx);
        rows(ay, h->cy);
        rows(az, h->cz);
        h->ty = p->block_waves ? p->block_waves : 16;
        h->nj = p->tile_j ? p->tile_j / h->ty : 1;
        h->chunk_i = p->chunk_i ? p->chunk_i : h->ny;
        h->index64 = p->index64 ? 1 : 0;
        h->krem_mode = p->k_remainder;
        if (h->krem_mode < -1 || h->krem_mode > 1)
            return bail(fail(PHC_ERR_INVALID, "k_remainder must be -1, 0 or 1 (got %d)", h->krem_mode));
        if (h->chunk_i < -4)
            return bail(fail(PHC_ERR_INVALID, "chunk_i %d: planes per chunk, or -1..-4 for the per-XCD schedule",
                             h->chunk_i));
        if (!sem_pick_sep(P, h->ty, h->nj, true, true))
            return bail(fail(PHC_ERR_INVALID, "no separable kernel for p=%d with %d waves x %d rows",
                             P, h->ty, h->nj));
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess &&
            prop.multiProcessorCount > 0)
            h->cus = prop.multiProcessorCount;
        if (!p->block_waves && !p->tile_j && !p->chunk_i) sem_default_shape(h);
    } else {
        const size_t bytes = sizeof(float) * (size_t)h->nn;
        if ((st = h->lev[0].alloc(bytes)) || (st = h->lev[1].alloc(bytes)) || (st = h->y.alloc(bytes)) ||
            (st = h->dt2m.alloc(bytes)) || (st = h->geo.alloc(sizeof(float) * 6 * qn * qn * qn)))
            return bail(st);
        PHC_HIP(hipMemset(h->lev[0].ptr, 0, bytes));
        PHC_HIP(hipMemset(h->lev[1].ptr, 0, bytes));
        PHC_HIP(hipMemset(h->y.ptr, 0, bytes));
        std::vector<float> d2m((size_t)h->nn, 0.f);
        for (int64_t n = 0; n < h->nn; ++n) d2m[n] = (float)(dt2 / M[n]);
        if (hipMemcpy(h->dt2m.ptr, d2m.data(), bytes, hipMemcpyHostToDevice))
            return bail(fail(PHC_ERR_HIP, "mass upload failed"));
        // geometric factors of the (uniform) box element: w_a w_b w_c |J| J^-1 J^-T,
        // J = diag(hx/2, hz/2, hy/2) in the local (x, z, y) order
        std::vector<float> G((size_t)6 * qn * qn * qn, 0.f);
        const double ja = ax.half, jb = az.half, jc = ay.half, det = ja * jb * jc;
        for (int c = 0; c < qn; ++c)
            for (int b = 0; b < qn; ++b)
                for (int a = 0; a < qn; ++a) {
                    const int pt = a + b * qn + c * qn * qn;
                    const double wq = g.w[a] * g.w[b] * g.w[c] * det;
                    G[6 * pt + 0] = (float)(wq / (ja * ja));
                    G[6 * pt + 1] = (float)(wq / (jb * jb));
                    G[6 * pt + 2] = (float)(wq / (jc * jc));
                }
        if (hipMemcpy(h->geo.ptr, G.data(), sizeof(float) * G.size(), hipMemcpyHostToDevice))
            return bail(fail(PHC_ERR_HIP, "geometry upload failed"));
        for (int i = 0; i < qn * qn; ++i) h->Dm[i] = (float)g.D[i];
    }
    *out = h;
    return PHC_OK;
}

phc_status phc_sem_destroy(phc_sem *h)
{
    if (!h) return PHC_OK;
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    sem_drop_graph(h);
    for (DevBuf *b : {&h->lev[0], &h->lev[1], &h->qf, &h->y, &h->dt2m, &h->geo, &h->rhs, &h->window, &h->readback, &h->trace,
                      &h->rec, &h->recoff})
        b->release();
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
    return PHC_OK;
}

phc_status phc_sem_sizes(phc_sem *h, int *num_nodes, int *nx, int *ny, int *nz)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    if (num_nodes) *num_nodes = (int)h->nn;
    if (nx) *nx = h->nx;
    if (ny) *ny = h->ny;
    if (nz) *nz = h->nz;
    return PHC_OK;
}

phc_status phc_sem_compute_one_step(phc_sem *h, int time_sample, int i1, int i2)
{
    RoctxRange rr_("phc_sem_compute_one_step");
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    if (i1 < 0 || i1 > 1 || i2 < 0 || i2 > 1 || i1 == i2)
        return fail(PHC_ERR_INVALID, "levels i1=%d i2=%d must be 0 and 1", i1, i2);
    if (time_sample < 0 || time_sample >= h->nsamples)
        return fail(PHC_ERR_INVALID, "time sample %d outside 0..%d", time_sample, h->nsamples - 1);
    PHC_TRY(sem_inject(h, i2, time_sample));
    return sem_launch(h, i1, i2, nullptr, nullptr, nullptr, nullptr);
}

phc_status phc_sem_compute_one_step_rhs(phc_sem *h, int i1, int i2, int nrhs, const int *rhs_element,
                                        const float *rhs_value)
{
    RoctxRange rr_("phc_sem_compute_one_step_rhs");
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    if (i1 < 0 || i1 > 1 || i2 < 0 || i2 > 1 || i1 == i2)
        return fail(PHC_ERR_INVALID, "levels i1=%d i2=%d must be 0 and 1", i1, i2);
    if (nrhs < 0 || (nrhs > 0 && (!rhs_element || !rhs_value)))
        return fail(PHC_ERR_INVALID, "bad source list (%d sources)", nrhs);
    const int64_t nE = (int64_t)h->ex * h->ey * h->ez;
    for (int r = 0; r < nrhs; ++r) {
        if (rhs_element[r] < 0 || rhs_element[r] >= nE)
            return fail(PHC_ERR_INVALID, "source %d: element %d outside 0..%lld", r, rhs_element[r],
                        (long long)nE - 1);
        if (!std::isfinite(rhs_value[r])) return fail(PHC_ERR_INVALID, "source %d: value is not finite", r);
    }
    // SEMsolver.cpp:37-42: pnGlobal(node0(e), i2) += dt dt c c rhs, source by source
    for (int r = 0; r < nrhs; ++r) {
        const int e = rhs_element[r];
        const float c = h->model[e];
        hipLaunchKernelGGL(sem_add_value_kernel, dim3(1), dim3(64), 0, h->stream, h->lev[i2].as<float>(),
                           sem_off(h, sem_first_node(h, e)), ((h->dt * h->dt) * c) * c, rhs_value[r]);
        PHC_HIP(hipGetLastError());
    }
    return sem_launch(h, i1, i2, nullptr, nullptr, nullptr, nullptr);
}

phc_status phc_sem_set_source(phc_sem *h, int src_element, int nsamples, const float *rhs)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    PHC_HIP(hipStreamSynchronize(h->stream));
    sem_drop_graph(h);
    return sem_source(h, src_element, nsamples, rhs);
}

// A run's steps on h->stream (sem_begin_run_kernel has filled the window and
// injected its first sample).  Names no time sample, so that a captured run
// serves every chunk.  The separable step's launch samples the receivers of
// the step before; the element kernels' receivers, and the last step's, are
// sampled by launches of their own.
static phc_status sem_enqueue_run(phc_sem *h, int nsteps, int i1, int i2, std::vector<hipEvent_t> *ev)
{
    const int64_t src = sem_off(h, h->src_node);
    const float *win = h->window.as<float>();
    const bool fused = h->kernel == PHC_SEM_SEPARABLE && h->nrec > 0;
    for (int s = 0; s < nsteps; ++s) {
        const int rs = fused ? s - 1 : -1;
        hipEvent_t e0 = ev ? (*ev)[2 * s] : nullptr, e1 = ev ? (*ev)[2 * s + 1] : nullptr;
        if (h->src_interior) {
            PHC_TRY(sem_launch(h, i1, i2, s + 1 < nsteps ? win + s + 1 : nullptr, h->trace.as<float>() + s, e0, e1,
                               rs, nsteps));
        } else {
            // source on a (never updated) boundary node: inject in place each
            // step, as SEMsolver.cpp:39-43 does, and read the node back
            if (s > 0) {
                hipLaunchKernelGGL(sem_inject_kernel, dim3(1), dim3(64), 0, h->stream, h->lev[i2].as<float>(), src,
                                   h->inj_coef, win, s);
                PHC_HIP(hipGetLastError());
            }
            PHC_TRY(sem_launch(h, i1, i2, nullptr, nullptr, e0, e1, rs, nsteps));
            hipLaunchKernelGGL(sem_copy_point_kernel, dim3(1), dim3(64), 0, h->stream, h->lev[i1].as<float>(),
                               src, h->trace.as<float>() + s);
            PHC_HIP(hipGetLastError());
        }
        if (h->nrec > 0 && (!fused || s == nsteps - 1)) {
            hipLaunchKernelGGL(sem_sample_kernel, dim3((h->nrec + 255) / 256), dim3(256), 0, h->stream,
                               h->lev[i1].as<float>(), h->recoff.as<int64_t>(), h->nrec,
                               h->rec.as<float>(), nsteps, s, src, h->trace.as<float>());
            PHC_HIP(hipGetLastError());
        }
        std::swap(i1, i2);
    }
    return PHC_OK;
}

phc_status phc_sem_run(phc_sem *h, int it0, int nsteps, int *i1p, int *i2p)
{
    RoctxRange rr_("phc_sem_run");
    if (!h || !i1p || !i2p) return fail(PHC_ERR_INVALID, "NULL argument");
    const int i1 = *i1p, i2 = *i2p;
    if (i1 < 0 || i1 > 1 || i2 < 0 || i2 > 1 || i1 == i2)
        return fail(PHC_ERR_INVALID, "levels i1=%d i2=%d must be 0 and 1", i1, i2);
    if (nsteps < 0) return fail(PHC_ERR_INVALID, "negative step count");
    if (nsteps == 0) return PHC_OK;
    if (it0 < 0 || it0 + nsteps > h->nsamples)
        return fail(PHC_ERR_INVALID, "steps %d..%d outside the %d source samples", it0,
                    it0 + nsteps - 1, h->nsamples);
    PHC_TRY(sem_prepare_sched(h));  // before any capture
    if (h->trace.bytes < sizeof(float) * nsteps || h->window.bytes < sizeof(float) * nsteps) {
        PHC_HIP(hipStreamSynchronize(h->stream));
        sem_drop_graph(h);
        PHC_TRY(h->trace.alloc(sizeof(float) * nsteps));
        PHC_TRY(h->window.alloc(sizeof(float) * nsteps));
    }
    if (h->nrec > 0 && h->rec.bytes < sizeof(float) * (size_t)nsteps * h->nrec) {
        PHC_HIP(hipStreamSynchronize(h->stream));
        sem_drop_graph(h);
        PHC_TRY(h->rec.alloc(sizeof(float) * (size_t)nsteps * h->nrec));
    }
    // changes the current level: launched once nothing but launches can fail
    auto begin = [&]() -> phc_status {
        hipLaunchKernelGGL(sem_begin_run_kernel, dim3((nsteps + 255) / 256), dim3(256), 0, h->stream,
                           h->lev[i2].as<float>(), sem_off(h, h->src_node), h->inj_coef, h->rhs.as<float>(), it0, nsteps,
                           h->window.as<float>());
        PHC_HIP(hipGetLastError());
        return PHC_OK;
    };
    if (h->timing) {
        std::vector<hipEvent_t> ev(2 * (size_t)nsteps);
        for (auto &e : ev) PHC_HIP(hipEventCreate(&e));
        phc_status st = begin();
        if (st == PHC_OK) st = sem_enqueue_run(h, nsteps, i1, i2, &ev);
        if (st == PHC_OK) {
            PHC_HIP(hipStreamSynchronize(h->stream));
            double tot = 0.0;
            for (int s = 0; s < nsteps; ++s) {
                float ms = 0.f;
                PHC_HIP(hipEventElapsedTime(&ms, ev[2 * s], ev[2 * s + 1]));
                tot += ms;
            }
            h->last_ms = tot / nsteps;
        }
        for (auto &e : ev) (void)hipEventDestroy(e);
        PHC_TRY(st);
    } else {
        PHC_TRY(prepare_captured(h->stream, h->graph[i1], nsteps, 0, h->nrec,
                                 [&] { return sem_enqueue_run(h, nsteps, i1, i2, nullptr); }));
        PHC_TRY(begin());
        PHC_HIP(hipGraphLaunch(h->graph[i1].exec(), h->stream));
    }
    h->last_n = nsteps;
    h->last_nrec = h->nrec;
    if (nsteps % 2) std::swap(*i1p, *i2p);
    return PHC_OK;
}

phc_status phc_sem_set_receivers(phc_sem *h, int nrec, const int *nodes)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    if (nrec < 0 || (nrec > 0 && !nodes)) return fail(PHC_ERR_INVALID, "bad receiver list");
    std::vector<int64_t> offs(nrec);
    for (int r = 0; r < nrec; ++r) {
        if (nodes[r] < 0 || nodes[r] >= h->nn)
            return fail(PHC_ERR_INVALID, "receiver node %d outside 0..%lld", nodes[r], (long long)h->nn - 1);
        offs[r] = sem_off(h, nodes[r]);
    }
    PHC_HIP(hipStreamSynchronize(h->stream));
    sem_drop_graph(h);
    h->nrec = nrec;
    if (nrec > 0) {
        PHC_TRY(h->recoff.alloc(sizeof(int64_t) * nrec));
        PHC_HIP(hipMemcpy(h->recoff.ptr, offs.data(), sizeof(int64_t) * nrec, hipMemcpyHostToDevice));
    }
    return PHC_OK;
}

phc_status phc_sem_get_traces(phc_sem *h, float *src, float *rec)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    PHC_HIP(hipStreamSynchronize(h->stream));
    if (src && h->last_n > 0)
        PHC_HIP(hipMemcpy(src, h->trace.ptr, sizeof(float) * h->last_n, hipMemcpyDeviceToHost));
    if (rec && h->last_n > 0 && h->last_nrec > 0)
        PHC_HIP(hipMemcpy(rec, h->rec.ptr, sizeof(float) * (size_t)h->last_n * h->last_nrec,
                          hipMemcpyDeviceToHost));
    return PHC_OK;
}

phc_status phc_sem_get_field(phc_sem *h, int level, float *host)
{
    if (!h || !host) return fail(PHC_ERR_INVALID, "NULL argument");
    if (level < 0 || level > 1) return fail(PHC_ERR_INVALID, "level %d is not 0 or 1", level);
    return sem_get(h, h->lev[level], host);
}

phc_status phc_sem_set_field(phc_sem *h, int level, const float *host)
{
    if (!h || !host) return fail(PHC_ERR_INVALID, "NULL argument");
    if (level < 0 || level > 1) return fail(PHC_ERR_INVALID, "level %d is not 0 or 1", level);
    PHC_HIP(hipStreamSynchronize(h->stream));
    return sem_put(h, h->lev[level], host);
}

phc_status phc_sem_get_mass(phc_sem *h, float *host)
{
    if (!h || !host) return fail(PHC_ERR_INVALID, "NULL argument");
    std::memcpy(host, h->hmass.data(), sizeof(float) * h->nn);
    return PHC_OK;
}

phc_status phc_sem_apply_stiffness(phc_sem *h, const float *p, float *y)
{
    // y = M (pold - pnew) / dt^2 for pcur = p, pold = 0 would need the
    // update; instead run the kernel with pold = p and pcur = p: the new
    // value is 2p - p - (dt^2/M) y = p - (dt^2/M) y, so y = (p - new) M / dt^2.
    // Exact enough for tests of the operator (one FP32 rounding of p - new).
    if (!h || !p || !y) return fail(PHC_ERR_INVALID, "NULL argument");
    PHC_HIP(hipStreamSynchronize(h->stream));
    DevBuf s0, s1;
    const bool sep = h->kernel == PHC_SEM_SEPARABLE;
    const size_t bytes = sizeof(float) * (size_t)(sep ? h->L.total : h->nn);
    PHC_TRY(s0.alloc(bytes));
    PHC_TRY(s1.alloc(bytes));
    // swap the levels' buffers for the scratch ones for one launch
    std::swap(h->lev[0], s0);
    std::swap(h->lev[1], s1);
    phc_status st = PHC_OK;
    for (DevBuf *b : {&h->lev[0], &h->lev[1]}) {
        if (st == PHC_OK && sep) st = fill_field(h->stream, b->as<float>(), h->L.total, 0.f);  // the halo
        if (st == PHC_OK) st = sem_put(h, *b, p);
    }
    if (st == PHC_OK) st = sem_launch(h, 0, 1, nullptr, nullptr, nullptr, nullptr);
    std::vector<float> out((size_t)h->nn);
    if (st == PHC_OK) st = sem_get(h, h->lev[0], out.data());
    std::swap(h->lev[0], s0);
    std::swap(h->lev[1], s1);
    s0.release();
    s1.release();
    PHC_TRY(st);
    const double dt2 = (double)h->dt * h->dt;
    for (int64_t n = 0; n < h->nn; ++n) y[n] = (float)(((double)p[n] - out[n]) * h->hmass[n] / dt2);
    return PHC_OK;
}

phc_status phc_sem_check_finite(phc_sem *h, int level)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    std::vector<float> f((size_t)h->nn);
    PHC_TRY(phc_sem_get_field(h, level, f.data()));
    for (int64_t n = 0; n < h->nn; ++n)
        if (!std::isfinite(f[n])) return fail(PHC_ERR_NONFINITE, "level %d node %lld is not finite", level, (long long)n);
    return PHC_OK;
}

phc_status phc_sem_set_timing(phc_sem *h, int enable)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    h->timing = enable ? 1 : 0;
    return PHC_OK;
}

phc_status phc_sem_last_run_kernel_ms(phc_sem *h, double *ms)
{
    if (!h || !ms) return fail(PHC_ERR_INVALID, "NULL argument");
    *ms = h->last_ms;
    return PHC_OK;
}

phc_status phc_sem_synchronize(phc_sem *h)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    PHC_HIP(hipStreamSynchronize(h->stream));
    return PHC_OK;
}

} // extern "C"

// ================================================================ autotuner
// Separable kernel only: times block shapes and chunk lengths on scratch
// copies of the levels (state untouched), keeps the fastest; optional text
// cache "sem ex ey ez p waves tile_j chunk_i ms".
extern "C" phc_status phc_sem_autotune(phc_sem *h, int steps_per_trial, const char *cache_path,
                                       int *tile_j, int *block_waves, int *chunk_i)
{
    RoctxRange rr_("phc_sem_autotune");
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    if (steps_per_trial < 1) return fail(PHC_ERR_INVALID, "steps_per_trial must be >= 1");
    if (h->kernel != PHC_SEM_SEPARABLE) {
        if (tile_j) *tile_j = 0;
        if (block_waves) *block_waves = 0;
        if (chunk_i) *chunk_i = 0;
        return PHC_OK;
    }
    bool hit = false;
    if (cache_path) {
        FILE *f = std::fopen(cache_path, "r");
        if (f) {
            // one entry per line, "sem ex ey ez p kmode waves tile_j chunk_i ms";
            // lines with another tag (an FD entry in the same file) are skipped whole
            char line[256];
            while (std::fgets(line, sizeof(line), f)) {
                char tag[8];
                int ex, ey, ez, pp, km, a, b, c;
                double ms;
                if (std::sscanf(line, "%7s %d %d %d %d %d %d %d %d %lf", tag, &ex, &ey, &ez, &pp, &km, &a, &b, &c,
                                &ms) != 10)
                    continue;
                const bool chunk_ok = c > 0 || (c >= -4 && c <= -1);
                if (!std::strcmp(tag, "sem") && ex == h->ex && ey == h->ey && ez == h->ez && pp == h->p &&
                    km == h->krem_mode && a > 0 && b % a == 0 && chunk_ok && sem_pick_sep(h->p, a, b / a, true, true)) {
                    h->ty = a; h->nj = b / a; h->chunk_i = c;
                    hit = true;
                }
            }
            std::fclose(f);
        }
    }
    if (!hit) {
        const size_t bytes = sizeof(float) * (size_t)h->L.total;
        DevBuf s0, s1;
        PHC_TRY(s0.alloc(bytes));
        PHC_TRY(s1.alloc(bytes));
        PHC_HIP(hipMemcpyAsync(s0.ptr, h->lev[0].ptr, bytes, hipMemcpyDeviceToDevice, h->stream));
        PHC_HIP(hipMemcpyAsync(s1.ptr, h->lev[1].ptr, bytes, hipMemcpyDeviceToDevice, h->stream));
        std::swap(h->lev[0], s0);
        std::swap(h->lev[1], s1);
        hipEvent_t e0, e1;
        phc_status st = PHC_OK;
        if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
            st = fail(PHC_ERR_HIP, "event create failed");
        const int shapes[][2] = {{16, 16}, {16, 32}, {8, 32}, {8, 16}, {8, 8}, {4, 16}, {4, 8}, {4, 4}};
        // chunk lengths that split the march axis evenly (n chunks, multiples
        // of 4 planes): a short last chunk would be mostly ring priming
        std::vector<int> chunks;
        for (int n : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16}) {
            int c = (h->L.nx + n - 1) / n;
            c += (4 - c % 4) % 4;
            if (std::find(chunks.begin(), chunks.end(), c) == chunks.end()) chunks.push_back(c);
        }
        for (int m = 1; m <= 4; ++m) chunks.push_back(-m);  // the per-XCD schedules
        double best = 1e30;
        int bty = h->ty, bnj = h->nj, bci = h->chunk_i;
        for (auto &sh : shapes) {
            if (st != PHC_OK) break;
            if (!sem_pick_sep(h->p, sh[0], sh[1] / sh[0], true, true)) continue;
            for (int c : chunks) {
                h->ty = sh[0]; h->nj = sh[1] / sh[0]; h->chunk_i = c;
                float ms = 0.f;
                for (int rep = 0; rep < 2 && st == PHC_OK; ++rep) {
                    if (hipEventRecord(e0, h->stream) != hipSuccess) st = fail(PHC_ERR_HIP, "event record failed");
                    for (int s = 0; s < steps_per_trial && st == PHC_OK; ++s)
                        st = sem_launch(h, s & 1, 1 - (s & 1), nullptr, nullptr, nullptr, nullptr);
                    if (st == PHC_OK && (hipEventRecord(e1, h->stream) != hipSuccess ||
                                         hipEventSynchronize(e1) != hipSuccess ||
                                         hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
                        st = fail(PHC_ERR_HIP, "trial timing failed");
                }
                if (st != PHC_OK) break;
                if (ms < best) { best = ms; bty = h->ty; bnj = h->nj; bci = h->chunk_i; }
            }
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        (void)hipStreamSynchronize(h->stream);
        std::swap(h->lev[0], s0);
        std::swap(h->lev[1], s1);
        s0.release();
        s1.release();
        h->ty = bty; h->nj = bnj; h->chunk_i = bci;
        PHC_TRY(st);
        if (cache_path) {
            FILE *f = std::fopen(cache_path, "a");
            if (f) {
                std::fprintf(f, "sem %d %d %d %d %d %d %d %d %.5f\n", h->ex, h->ey, h->ez, h->p, h->krem_mode, bty,
                             bty * bnj,
                             bci, best / steps_per_trial);
                std::fclose(f);
            }
        }
    }
    sem_drop_graph(h);
    if (tile_j) *tile_j = h->ty * h->nj;
    if (block_waves) *block_waves = h->ty;
    if (chunk_i) *chunk_i = h->chunk_i;
    return PHC_OK;
}
