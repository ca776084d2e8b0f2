// fd_quad.hpp -- the marching tile body of the radius-4 FD step with four
// points per lane (inner3D + applySponge + fused source injection,
// src/fd/utilsFDTD/FDTDkernels.hpp:8-34, 108-128; pml3D, 36-73), for the
// shapes with 4 rows per wavefront.
#pragma once

#include "fd_tile.hpp"
#include "quad.hpp"

namespace phc {

// A block of TY wavefronts owns a 64(k) x 4 TY(j) column and marches along i
// as fd_tile does (register ring along i, halo ring, LDS plane, unconditional
// prefetch, unroll by the ring); here a lane holds 4 consecutive k points of
// one row (16 lanes per row, 4 rows per wavefront).
//   * Loads, stores and LDS accesses are 16 bytes.  The 8 neighbours along k
//     of a lane's 4 points are 2 LDS reads instead of 32, so a point costs 40
//     bytes of LDS reads instead of 64; one halo quad per thread covers the
//     whole halo of a plane.
//   * The sponge factors of a lane's points do not change between planes
//     inside the i range of the undamped box, so they are formed once; the
//     source test is one compare per plane.
// At sizes that live in the 256 MB cache or below, the one-point tile was
// bound by the sum of its VALU, LDS and address work per plane, not by memory
// (203 x 178 x 261: 38 us per step for 151 MB).
// Every point takes the same operations in the same order as in fd_tile, so
// both give the same bits.  NT: the streamed pnm1 and vp with non-temporal
// accesses (working sets past the cache), else cached ones.
template <int TY>
struct FdQuadShape {
    static constexpr int TJ = 4 * TY;
    static constexpr int LH = TJ + 8;
    static constexpr int LQ = FD_TK / 4 + 2;
};

template <int TY, int ARITH, typename IT, bool PML, bool NT, class G>
__device__ __forceinline__ void fd_quad(const FdStepArgs &a, const G &g, float rhs_next, int kt, int jt, int i0,
                                        int i1, quad_f4 (*tile)[FdQuadShape<TY>::LH][FdQuadShape<TY>::LQ])
{
    constexpr int R = 4;
    constexpr int TJ = 4 * TY;
    constexpr int LQ = FdQuadShape<TY>::LQ;
    constexpr int T = FD_TK * TY;
    constexpr int NHQ = 2 * R * (FD_TK / 4) + 2 * TJ;  // halo quads of a plane: 8 rows, then 2 per tile row
    constexpr int NH = (NHQ + T - 1) / T;
    constexpr int Q = 2 * R + 2;
    // halo ring: a plane's halo is requested when the neighbouring tile requests
    // the same rows as its interior (2 planes ahead instead of 5, with 4 waves
    // per SIMD instead of 3: 203 x 178 x 261 36 against 30 us, 512^3 398
    // against 357)
    constexpr int F = R + 1;
    constexpr IT S = sizeof(IT) == 4 ? 4 : 1;

    const FdLayout &L = g.L;
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int k0 = kt * FD_TK, j0 = jt * TJ;
    const int qd = tx & 15, row = ty * 4 + (tx >> 4);
    const int k = k0 + 4 * qd, j = j0 + row;
    const IT pitch = (IT)L.pitch_j * S;

    // Every load is unconditional, as in fd_tile: quads outside the stored
    // grid read the interior origin instead.
    const bool jk = j < L.ny && k < L.nz;  // the lane updates at least its first point
    const bool ld = j < L.ny + R && k < L.nz + R;
    const IT colq = (IT)fd_off(L, 0, ld ? j : 0, ld ? k : 0) * S;
    int hrow[NH], hq[NH];
    IT colh[NH];
    bool hst[NH];
#pragma unroll
    for (int m = 0; m < NH; ++m) {
        const int h = ty * FD_TK + tx + T * m;
        int jh, kh;
        if (h < 2 * R * (FD_TK / 4)) {
            const int hr = h >> 4;
            jh = hr < R ? j0 - R + hr : j0 + TJ + hr - R;
            kh = k0 + 4 * (h & 15);
            hrow[m] = hr < R ? hr : TJ + hr;
            hq[m] = (h & 15) + 1;
        } else {
            const int e = h - 2 * R * (FD_TK / 4);
            jh = j0 + (e >> 1);
            kh = (e & 1) ? k0 + FD_TK : k0 - 4;
            hrow[m] = (e >> 1) + R;
            hq[m] = (e & 1) ? LQ - 1 : 0;
        }
        hst[m] = h < NHQ;
        const bool l = hst[m] && jh < L.ny + R && kh < L.nz + R;
        colh[m] = (IT)fd_off(L, 0, l ? jh : 0, l ? kh : 0) * S;
    }

    // sponge factors of the lane's points on planes inside the undamped i
    // range (sin) and whether they take the plane's factor outside it (sfx)
    quad_f4 sin;
    bool sfx[4];
    const bool inJ = j >= a.sw && j < L.ny - a.sw;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const bool inK = k + c >= a.sw && k + c < L.nz - a.sw;
        sin[c] = 1.f;
        sfx[c] = inJ && inK;
        if (a.sw > 0 && jk) {
            if (inK && !inJ) sin[c] = g.fy[j];
            if (inJ && !inK && k + c < L.nz) sin[c] = g.fz[k + c];
        }
    }
    // PML: eta profiles of the lane's points, slab tests along j and k
    float ezv[6], eym = 0.f, ey0 = 0.f, eyp = 0.f;  // ezv[c..c+2]: eta_z at k+c-1, k+c, k+c+1
    bool kslab[4], jslab = false, qslab = false;
    if constexpr (PML) {
#pragma unroll
        for (int c = 0; c < 6; ++c) ezv[c] = (jk && k + c < L.nz + 2) ? a.pml_ez[k + c] : 0.f;
        if (jk) {
            eym = a.pml_ey[j];
            ey0 = a.pml_ey[j + 1];
            eyp = a.pml_ey[j + 2];
        }
        jslab = j < a.py3 || j >= a.py4;
        qslab = jslab;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            kslab[c] = k + c < a.pz3 || k + c >= a.pz4;
            qslab = qslab || kslab[c];
        }
    }
    // the plane and component of the source point, if the lane holds it
    int src_i = -1, src_c = 0;
    {
        const int64_t d = g.src_off - (int64_t)(colq / S);
        if (jk && d >= 0) {
            int64_t pi, c;
            if constexpr (sizeof(IT) == 4) {
                pi = (uint32_t)d / (uint32_t)L.pitch_j;
                c = (uint32_t)d % (uint32_t)L.pitch_j;
            } else {
                pi = d / L.pitch_j;
                c = d % L.pitch_j;
            }
            if (c < 4 && k + c < L.nz) {
                src_i = (int)pi;
                src_c = (int)c;
            }
        }
    }
    const int nval = min(4, L.nz - k);  // points of the quad inside the grid (<= 0: none)

    quad_f4 q[Q], fh[NH][F], pm[2], vv[2], ph[2];
    float ex[2][3];

    auto load_halo = [&](int slot, int p) {
        const IT po = (IT)p * pitch;
#pragma unroll
        for (int m = 0; m < NH; ++m) fh[m][slot] = ldq<false>(g.pn, colh[m] + po);
    };
    auto load_aux = [&](int set, int p) {
        const IT po = (IT)p * pitch;
        pm[set] = ldq<NT>(g.pnm1, colq + po);
        vv[set] = ldq<NT>(g.vp, colq + po);
        if constexpr (PML) {
            const bool sl = p < a.px3 || p >= a.px4;
            ph[set] = ldq<false>(a.pml_phi, (sl || qslab) ? colq + po : (IT)0);
            ex[set][0] = a.pml_ex[p];
            ex[set][1] = a.pml_ex[p + 1];
            ex[set][2] = a.pml_ex[p + 2];
        }
    };
    auto stage = [&](int buf, int qslot, int hslot) {
        quad_f4(*tl)[LQ] = tile[buf];
        tl[row + R][qd + 1] = q[qslot];
#pragma unroll
        for (int m = 0; m < NH; ++m)
            if (hst[m]) tl[hrow[m]][hq[m]] = fh[m][hslot];
    };

#pragma unroll
    for (int l = 0; l <= 2 * R; ++l) q[l] = ldq<false>(g.pn, colq + (IT)(i0 - R + l) * pitch);
#pragma unroll
    for (int d = 0; d < F; ++d) load_halo(d, i0 + d);
    load_aux(0, i0);
    stage(0, R, 0);
    lds_barrier();

    // one plane, u = its position in the ring's turn (a template argument: the
    // loop with its body is past the compiler's unroll limits)
    auto plane = [&](auto uc, int i) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value;
        {
            const int pq = min(i + 1 + R, L.nx + R - 1);
            q[(u + 1 + 2 * R) % Q] = ldq<false>(g.pn, colq + (IT)pq * pitch);
            load_halo((u + F) % F, pq);
            load_aux((u + 1) & 1, min(i + 1, L.nx - 1));
        }
        if (jk) {
            const quad_f4(*tl)[LQ] = tile[u & 1];
            const int r = row + R;
            const quad_f4 pc = q[(u + R) % Q];
            const quad_f4 pmr = pm[u & 1], vq = vv[u & 1];
            quad_f4 up[R + 1], dn[R + 1];
#pragma unroll
            for (int l = 1; l <= R; ++l) {
                up[l] = tl[r + l][qd + 1];
                dn[l] = tl[r - l][qd + 1];
            }
            const quad_f4 zl = tl[r][qd], zr = tl[r][qd + 2];
            float z[12];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                z[c] = zl[c];
                z[4 + c] = pc[c];
                z[8 + c] = zr[c];
            }
            float lapx[4], lapy[4], lapz[4], lap[4];
            if constexpr (ARITH == PHC_FD_ARITH_REF) {
#pragma clang fp contract(off)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    lapx[c] = lapy[c] = lapz[c] = lap[c] = 0.f;
#pragma unroll
                    for (int l = 1; l <= R; ++l)
                        lapx[c] += a.cx[l] * (q[(u + R + l) % Q][c] + q[(u + R - l) % Q][c]);
#pragma unroll
                    for (int l = 1; l <= R; ++l) lapy[c] += a.cy[l] * (up[l][c] + dn[l][c]);
#pragma unroll
                    for (int l = 1; l <= R; ++l) lapz[c] += a.cz[l] * (z[4 + c + l] + z[4 + c - l]);
                }
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    lapx[c] = lapy[c] = lapz[c] = 0.f;
                    lap[c] = a.c0f * pc[c];
                }
#pragma unroll
                for (int l = 1; l <= R; ++l) {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        lap[c] = fmaf(a.cx[l], q[(u + R + l) % Q][c] + q[(u + R - l) % Q][c], lap[c]);
#pragma unroll
                    for (int c = 0; c < 4; ++c) lap[c] = fmaf(a.cy[l], up[l][c] + dn[l][c], lap[c]);
#pragma unroll
                    for (int c = 0; c < 4; ++c) lap[c] = fmaf(a.cz[l], z[4 + c + l] + z[4 + c - l], lap[c]);
                }
            }
            quad_f4 val;
            {
                quad_f4 s = {1.f, 1.f, 1.f, 1.f};
                if (a.sw > 0) {
                    if (i >= a.sw && i < L.nx - a.sw) {
                        s = sin;
                    } else {
                        const float fxv = fd_face_damping(a, i, L.nx);
#pragma unroll
                        for (int c = 0; c < 4; ++c) s[c] = sfx[c] ? fxv : 1.f;
                    }
                }
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if constexpr (ARITH == PHC_FD_ARITH_REF) {
                        // deferred damping of the previous level (x1 is exact)
                        const float pmv = mul_nc(pmr[c], a.damp_prev ? s[c] : 1.f);
                        val[c] = fd_update_ref(pc[c], pmv, vq[c], a.coef0, lapx[c], lapy[c], lapz[c], s[c]);
                    } else {
                        const float pmv = pmr[c] * (a.damp_prev ? s[c] : 1.f);
                        val[c] = s[c] * fmaf(vq[c], lap[c], 2.f * pc[c] - pmv);
                    }
                }
            }
            const IT o = colq + (IT)i * pitch;
            if constexpr (PML) {
                const bool pslab_i = i < a.px3 || i >= a.px4;
                if (pslab_i || qslab) {
                    const float exm = ex[u & 1][0], ex0 = ex[u & 1][1], exp_ = ex[u & 1][2];
                    quad_f4 phn = ph[u & 1];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        float e, tg, v, pn;
                        fd_pml_terms<ARITH>(exm, ex0, exp_, eym, ey0, eyp, ezv[c], ezv[c + 1], ezv[c + 2],
                                            q[(u + R - 1) % Q][c], q[(u + R + 1) % Q][c], dn[1][c], up[1][c],
                                            z[3 + c], z[5 + c], a.pml_hd2, e, tg);
                        fd_pml_update<ARITH>(pc[c], pmr[c], vq[c], ph[u & 1][c], a.coef0, lapx[c], lapy[c],
                                             lapz[c], lap[c], e, tg, v, pn);
                        const bool sl = (pslab_i || jslab || kslab[c]) && c < nval;
                        val[c] = sl ? v : val[c];
                        phn[c] = sl ? pn : phn[c];
                    }
                    stq<true>(a.pml_phi, o, phn);
                }
            }
            if (src_i == i) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (src_c == c) {
                        if (g.trace) *g.trace = val[c];
                        if (g.inj) val[c] = add_nc(val[c], mul_nc(vq[c], rhs_next));
                    }
            }
            // a quad that ends beyond the grid keeps what the row's halo holds there
#pragma unroll
            for (int c = 1; c < 4; ++c) val[c] = c < nval ? val[c] : pmr[c];
            stq<NT>(g.pnm1, o, val);
        }
        stage((u + 1) & 1, (u + 1 + R) % Q, (u + 1) % F);
        lds_barrier();
    };
    for (int ib = i0; ib < i1; ib += Q) march_turn(plane, ib, i1, std::make_integer_sequence<int, Q>{});
}

} // namespace phc
