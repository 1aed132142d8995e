// adjoint.h -- the adjoint of one recorded anisotropic step with respect to the 16 mobility bins
// of UseMobilityModel 4 (a build extension with no reference counterpart).
//
// The differentiated map is one step from a held state: the fields, IDLocal, contours,
// junctions and boundary characteristics entering the step are constants, except that each
// recorded characteristic mobility is the mobility of its misorientation bin (what the step
// before recorded, and what ggx_set_mobility_bins refreshes).  The step's outputs are each
// grain's area and perimeter; redistancing does not move the zero level set they are measured
// on, so it is not on the path (the redistanced field is the held state of the next step).
// The discrete decisions of the step (sectors, nearest segments, argmax of the comparison,
// the set comparison's band, the contour's squares) are those of the recorded forward pass.
//
// The chain, reversed kernel by kernel:
//  * k_adj_contour: area = |sum (y_i + y_i+1)(x_i - x_i+1)| h^2 / 2 and perimeter = sum |p_i+1 - p_i| h
//    (ExplicitGrainBoundary::computeVolume / computePerimeter, grainBoundary.cpp:201-231) over
//    the contour points, each point the linear zero crossing of the set-compared field on one
//    square edge (MarchingSquaresAlgorithm, marchingSquares.cpp:204-265): x = l + v_l / (v_l - v_r).
//  * k_adj_route: the set comparison (box.cpp:847-855) s = (u - c) / 2 inside the band, u
//    outside, with c the comparison's maximum (box.cpp:923-934), so the adjoint of c goes to the
//    grain that won the pixel; the wall and uncovered pixels are constants, cleared pixels
//    (clearContourGrainArea) too.
//  * k_adj_weight: the corrector u = phi + (phi~ - phi) w where phi > -delta (box.cpp:472-510),
//    then w through ExplicitGrainBoundary::getWeight: constant sectors (the mean of their
//    junction weights), interpolating sectors (linear or quadratic in their end weights,
//    contourSector.cpp:211-271) and plain boundary points (e m of IDLocal's neighbour, floored at
//    0.01, box.cpp:544-554); junction weights through the drag 1 / (1 / (ds TPD) + 1 / mean m)
//    (junction.cpp:171-184).  Mobilities are bins[bin(misorientation)].
#pragma once
#include "aniso.h"

namespace ggx {

struct AdjContourArgs {
    int nslots;
    const int* flags_conv;      // flags as the step's corrector saw them
    const int* flags_out;       // flags after the step
    const Box* box;             // the step's input boxes
    const long long* off;       // and field offsets
    const double2* pts;         // the step's contours
    const long long* coff;
    const int* clen;
    const double* s;            // set-compared fields of the step (input layout)
    const int* win;             // per pixel: the comparison's winner (grain id), 0 wall, -1 none, -2 cleared
    const double* u;            // the corrected convolved fields
    const double* d_area;       // dJ/d area per grain id
    const double* d_perim;      // dJ/d perimeter per grain id
    const int* area_set;        // per grain: 1 where the step wrote a new area (a regular motion)
    double* lam_s;              // adjoint of s (zero at launch)
    double* lam_u;              // adjoint of u (zero at launch)
    double h, band;
};

__device__ __forceinline__ bool live_at_conv(int f) { return (f & kPresent) && (f & kExists); }

// One 64-lane workgroup per grain: the adjoint of the contour points, scattered onto the two
// pixels of each point's square edge.
__global__ void __launch_bounds__(64) k_adj_contour(AdjContourArgs A) {
#pragma clang fp contract(off)
    const int lane = (int)threadIdx.x;
    for (int g = 1 + (int)blockIdx.x; g < A.nslots; g += (int)gridDim.x) {
        if (!live_at_conv(A.flags_conv[g]) || !(A.flags_out[g] & kExists)) continue;
        const double da = A.area_set[g] ? A.d_area[g] : 0.0, dp = A.d_perim[g];
        if (da == 0.0 && dp == 0.0) continue;
        const int M = A.clen[g] - 1;  // distinct points; point M repeats point 0
        if (M < 2) continue;
        const double2* c = A.pts + A.coff[g];
        double v = 0.0;
        for (int i = lane; i < M; i += 64) v += (c[i].y + c[i + 1].y) * (c[i].x - c[i + 1].x);
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
        const double sa = (v >= 0 ? 1.0 : -1.0) * A.h * A.h * 0.5;
        const Box b = A.box[g];
        const long long o = A.off[g];
        auto value = [&](int row, int col, long long* k) -> bool {
            const int r = row - b.y0, q = col - b.x0;
            if ((unsigned)r >= (unsigned)b.n || (unsigned)q >= (unsigned)b.n) return false;
            *k = o + (long long)r * b.n + q;
            return true;
        };
        auto val = [&](long long k) { return A.win[k] == -2 ? -A.h : A.s[k]; };
        for (int i = lane; i < M; i += 64) {
            const double2 p = c[i], pp = c[(i - 1 + M) % M], pn = c[i + 1];
            double gx = da * sa * (pn.y - pp.y), gy = da * sa * (pp.x - pn.x);
            const double ax = p.x - pp.x, ay = p.y - pp.y, bx = pn.x - p.x, by = pn.y - p.y;
            const double la = sqrt(ax * ax + ay * ay), lb = sqrt(bx * bx + by * by);
            if (la > 0) { gx += dp * A.h * ax / la; gy += dp * A.h * ay / la; }
            if (lb > 0) { gx -= dp * A.h * bx / lb; gy -= dp * A.h * by / lb; }
            const double fx = floor(p.x), fy = floor(p.y);
            long long k0, k1;
            if (p.y != fy && p.x == fx) {  // on a column: y = t + v_t / (v_t - v_b)
                const int col = (int)fx, t = (int)fy;
                if (!value(t, col, &k0) || !value(t + 1, col, &k1)) continue;
                const double vt = val(k0), vb = val(k1), D = vt - vb;
                if (D == 0.0) continue;
                atomicAdd(&A.lam_s[k0], gy * (-vb / (D * D)));
                atomicAdd(&A.lam_s[k1], gy * (vt / (D * D)));
            } else if (p.x != fx && p.y == fy) {  // on a row: x = l + v_l / (v_l - v_r)
                const int row = (int)fy, l = (int)fx;
                if (!value(row, l, &k0) || !value(row, l + 1, &k1)) continue;
                const double vl = val(k0), vr = val(k1), D = vl - vr;
                if (D == 0.0) continue;
                atomicAdd(&A.lam_s[k0], gx * (-vr / (D * D)));
                atomicAdd(&A.lam_s[k1], gx * (vl / (D * D)));
            }
            // a point on a grid point (a zero of the field) or on the box edge: no derivative
        }
    }
}

// One workgroup per grain: the set comparison and the comparison's argmax, reversed.
__global__ void __launch_bounds__(256) k_adj_route(AdjContourArgs A) {
#pragma clang fp contract(off)
    for (int g = 1 + (int)blockIdx.x; g < A.nslots; g += (int)gridDim.x) {
        if (!live_at_conv(A.flags_conv[g])) continue;
        const Box b = A.box[g];
        const long long o = A.off[g];
        const long long nn = (long long)b.n * b.n;
        for (long long p = threadIdx.x; p < nn; p += blockDim.x) {
            const double ls = A.lam_s[o + p];
            if (ls == 0.0) continue;
            const int w = A.win[o + p];
            if (w == -2) continue;
            if (fabs(A.u[o + p]) < A.band) {
                atomicAdd(&A.lam_u[o + p], 0.5 * ls);
                if (w > 0 && w < A.nslots) {
                    const Box bw = A.box[w];
                    const int r = b.y0 + (int)(p / b.n) - bw.y0, q = b.x0 + (int)(p % b.n) - bw.x0;
                    if ((unsigned)r < (unsigned)bw.n && (unsigned)q < (unsigned)bw.n)
                        atomicAdd(&A.lam_u[A.off[w] + (long long)r * bw.n + q], -0.5 * ls);
                }
            } else {
                atomicAdd(&A.lam_u[o + p], ls);
            }
        }
    }
}

struct AdjWeightArgs {
    AnisoArgs<double> A;        // the corrector's inputs as the recorded step saw them
    const double* tilde0;       // the convolved fields before the corrector
    const double* lam_u;
    double* grad;               // 16 bins (accumulated)
    int loop;                   // loop index of the recorded step
};

// One workgroup per grain: the corrector and its weight field, reversed onto the bins.
__global__ void __launch_bounds__(256) k_adj_weight(AdjWeightArgs W) {
#pragma clang fp contract(off)
    const AnisoArgs<double>& A = W.A;
    __shared__ SectorSet S;
    __shared__ Junc s_j[kJuncCap];
    __shared__ double s_jw[kJuncCap];
    __shared__ JuncGrad s_jg[kJuncCap];
    __shared__ int s_nid[kNbCap], s_nbin[kNbCap];
    __shared__ double s_nw[kNbCap], s_ne[kNbCap];
    __shared__ double s_lcw[kJuncCap], s_lnw[kNbCap], s_grad[16];
    __shared__ int s_bad, s_any;
    if (W.loop == 0) return;  // no corrector at loop 0 (box.cpp:428-429)
    for (int g = 1 + (int)blockIdx.x; g < A.nslots; g += (int)gridDim.x) {
        __syncthreads();  // the previous grain's shared state is free
        const int f = A.flags[g];
        if (!live_at_conv(f) || !(f & kRegular)) continue;
        const Box b = A.box[g];
        const long long o = A.off[g];
        const int np = A.n_prev[g];
        const long long op = A.off_prev[g];
        const int2 org = A.S.idl_org[g];
        const int ix0 = max(org.x, b.x0), ix1 = min(org.x + np, b.x0 + b.n);
        const int iy0 = max(org.y, b.y0), iy1 = min(org.y + np, b.y0 + b.n);
        const int wx = ix1 - ix0, wy = iy1 - iy0;
        if (threadIdx.x == 0) { s_any = 0; s_bad = 0; }
        __syncthreads();
        if (wx <= 0 || wy <= 0) continue;
        bool any = false;
        for (int p = threadIdx.x; p < wx * wy && !any; p += blockDim.x) {
            const int i = iy0 + p / wx, j = ix0 + p % wx;
            any = W.lam_u[o + (long long)(i - b.y0) * b.n + (j - b.x0)] != 0.0;
        }
        if (any) s_any = 1;
        __syncthreads();
        if (!s_any) continue;
        const int L = A.clen[g];
        const int nj = min(A.S.jcnt[g], kJuncCap);
        const double2* c = A.pts + A.coff[g];
        const int nbc = A.nb_cnt[g];
        const double4 qme = A.S.quat[g];
        for (int k = threadIdx.x; k < nbc; k += blockDim.x) {
            const int id = A.nb_id[(size_t)g * kNbCap + k];
            s_nid[k] = id;
            const double e = A.S.nb_e[(size_t)g * kNbCap + k], m = A.S.nb_m[(size_t)g * kNbCap + k];
            s_nw[k] = (e * m > 0.01) ? e * m : 0.01;
            s_ne[k] = e;
            s_nbin[k] = (e > 0 && e * m > 0.01) ? mobility_bin(A.K, misorientation(qme, A.S.quat[id])) : -1;
            s_lnw[k] = 0.0;
        }
        for (int k = threadIdx.x; k < nj; k += blockDim.x) {
            s_j[k] = A.S.junc[(size_t)g * kJuncCap + k];
            double w = 1.0;
            if (!junction_weight(A, g, s_j[k], &w, &s_jg[k])) s_bad = 1;
            s_jw[k] = w;
            s_lcw[k] = 0.0;
        }
        if (threadIdx.x < 16) s_grad[threadIdx.x] = 0.0;
        __syncthreads();
        if (threadIdx.x < 64 && !s_bad) build_sectors(c, L, s_j, nj, s_jw, A.h, A.K.csr, A.K.isr, S);
        __syncthreads();
        if (threadIdx.x == 0 && !s_bad && S.err) s_bad = 1;
        __syncthreads();
        if (s_bad) continue;  // the forward step reported this grain (kErrAniso)
        const int ncons = S.ncons, ninterp = S.ninterp;
        for (int p = threadIdx.x; p < wx * wy; p += blockDim.x) {
            const int i = iy0 + p / wx, j = ix0 + p % wx;
            const long long q = o + (long long)(i - b.y0) * b.n + (j - b.x0);
            const double lu = W.lam_u[q];
            if (lu == 0.0) continue;
            const double val = A.phi[q];
            if (!(val > -A.delta)) continue;  // u = -delta: a constant
            const double lw = lu * (W.tilde0[q] - val);
            double lambda = 0;
            const int segment = project_to_contour(c, L, (double)j, (double)i, &lambda);
            if (segment < 0) continue;
            int found = -1;
            for (int s = 0; s < ncons && found < 0; ++s)
                if (sector_within(S.cr[s], S.cl[s], L, segment)) found = s;
            if (found >= 0) {
                atomicAdd(&s_lcw[found], lw);
                continue;
            }
            for (int s = 0; s < ninterp && found < 0; ++s)
                if (sector_within(S.ir[s], S.il[s], L, segment)) found = s;
            double wv;
            int slot;
            if (found < 0) {
                if (gb_weight_at(A, op, np, org.x, org.y, s_nid, s_nw, nbc, i, j, &wv, &slot) && slot >= 0)
                    atomicAdd(&s_lnw[slot], lw);
                continue;
            }
            const int s = found, rcs = L - 1;
            // the end weights and where they come from: a constant sector (>= 0) or a neighbour slot
            double left_w, right_w;
            int lslot = -1, rslot = -1;
            if (S.ils[s] >= 0) left_w = S.cw[S.ils[s]];
            else if (!gb_weight_at(A, op, np, org.x, org.y, s_nid, s_nw, nbc, (int)c[S.il[s]].y, (int)c[S.il[s]].x,
                                   &left_w, &lslot)) continue;
            if (S.irs[s] >= 0) right_w = S.cw[S.irs[s]];
            else if (!gb_weight_at(A, op, np, org.x, org.y, s_nid, s_nw, nbc, (int)c[S.ir[s]].y, (int)c[S.ir[s]].x,
                                   &right_w, &rslot)) continue;
            double t = 0;
            int k = S.ir[s];
            for (; k != segment; k = (k + 1 + rcs) % rcs) t += seg_len(c[k + 1], c[k]) * A.h;
            t += scaled_len(c[(k + 1 + rcs) % rcs], c[k], lambda);
            t /= S.ilen[s];
            if (t < 0) t = 0;
            if (t > 1) t = 1;
            double dl, dr;
            if (S.ils[s] >= 0 && S.irs[s] >= 0) {
                const double2 sample = c[(S.ir[s] + 1) % rcs];
                double bw;
                int bslot = -1;
                if (!gb_weight_at(A, op, np, org.x, org.y, s_nid, s_nw, nbc, (int)sample.y, (int)sample.x, &bw, &bslot))
                    continue;
                const double two_isr = 2 * A.K.isr;
                const double quot = (S.ilen[s] > two_isr ? two_isr : S.ilen[s]);
                const double kap = quot / two_isr;  // d amplitude / d bw
                const double d0 = t * t - 1.5 * t + 0.5, d1 = t * t - t, d2 = t * t - 0.5 * t;
                dr = 2 * d0 - 2 * (1 - kap) * d1;
                dl = 2 * d2 - 2 * (1 - kap) * d1;
                if (bslot >= 0) atomicAdd(&s_lnw[bslot], lw * (-4 * kap * d1));
            } else {
                dl = t;
                dr = 1 - t;
            }
            if (S.ils[s] >= 0) atomicAdd(&s_lcw[S.ils[s]], lw * dl);
            else if (lslot >= 0) atomicAdd(&s_lnw[lslot], lw * dl);
            if (S.irs[s] >= 0) atomicAdd(&s_lcw[S.irs[s]], lw * dr);
            else if (rslot >= 0) atomicAdd(&s_lnw[rslot], lw * dr);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            // constant sectors: the mean of their junctions' weights; junctions: three mobilities
            for (int k = 0; k < ncons; ++k) {
                if (s_lcw[k] == 0.0) continue;
                const double share = s_lcw[k] / S.cnj[k];
                for (int r = 0; r < S.cnj[k]; ++r) {
                    const JuncGrad& jg = s_jg[S.cj[k][r]];
                    for (int m = 0; m < 3; ++m)
                        if (jg.bin[m] >= 0) s_grad[jg.bin[m]] += share * jg.d[m];
                }
            }
            // neighbour weights e m
            for (int k = 0; k < nbc; ++k)
                if (s_nbin[k] >= 0 && s_lnw[k] != 0.0) s_grad[s_nbin[k]] += s_lnw[k] * s_ne[k];
        }
        __syncthreads();
        if (threadIdx.x < 16 && s_grad[threadIdx.x] != 0.0) atomicAdd(&W.grad[threadIdx.x], s_grad[threadIdx.x]);
    }
}

// After the bins change: every recorded characteristic mobility (energy > 0) becomes the mobility
// of its misorientation's bin again, as the neighbour wave of the level-set kernel computes it.
__global__ void __launch_bounds__(256) k_refresh_mobility(int nslots, const int* __restrict__ nb_cnt,
                                                         const int* __restrict__ nb_id, const double* __restrict__ nb_e,
                                                         double* __restrict__ nb_m, const double4* __restrict__ quat,
                                                         AnisoConst K) {
    const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (g < 1 || g >= nslots) return;
    const int c = min(nb_cnt[g], kNbCap);
    for (int k = 0; k < c; ++k) {
        const size_t e = (size_t)g * kNbCap + k;
        if (nb_e[e] > 0) nb_m[e] = gb_mobility(K, misorientation(quat[g], quat[nb_id[e]]));
    }
}

}  // namespace ggx
