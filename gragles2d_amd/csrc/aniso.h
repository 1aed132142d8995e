// aniso.h -- anisotropic grain boundaries (IsIsotropicNetwork = 0).
//
// Two halves:
//  * boundary properties that the level-set kernel records while it traces a grain: the
//    misorientation of two orientations (Quaternion::misorientationCubicQxQ,
//    Quaternion.cpp:309-367, floored at one degree by LSbox::computeMisorientation,
//    box.cpp:1766-1780), the Read-Shockley energy (LSbox::GBEnergyReadShockley,
//    box.cpp:1785-1823), the mobility models (LSbox::GBmobilityModel, box.cpp:1825-1865) and the
//    projection of a point onto a contour (ExplicitGrainBoundary::projectToGrainBondary,
//    grainBoundary.cpp:365-447);
//  * k_sectors and k_aniso, the velocity corrector of LSbox::executeConvolution (box.cpp:428-510),
//    run on the convolved fields of all grains before the comparison reads them: per grain the
//    contour sectors of the previous contour (ExplicitGrainBoundary::buildBoundarySectors,
//    setPointsOnBoundary, grainBoundary.cpp:233-330,524-559; ContourSector, contourSector.cpp)
//    with the junction weights (GrainJunction::getWeight, junction.cpp:23-192), laid out per
//    contour segment; then per pixel of IDLocal's window intersected with the box:
//    out = in + (out - in) * weight where in > -delta, else -delta.
// All of it is FP64 whatever the field type, with contraction off so that every decision
// (nearest vertex, sector bounds, floors) sees the rounding of a scalar CPU build.
#pragma once
#include "kernels.h"

namespace ggx {

constexpr int kJuncCap = 32;           // junctions recorded per grain (m_grainJunctions)
constexpr int kSecCap = 2 * kJuncCap;  // interpolating sectors per grain (two per constant sector)
constexpr int kAnisoContourLds = 320;  // contour points staged in LDS (longer contours are read in place)

struct AnisoConst {
    int on;              // 1: anisotropic network
    int research_mode;   // Settings::ResearchMode (0 or 1)
    int mobility_model;  // Settings::UseMobilityModel: 0, 1, 2, or 4 (16 misorientation bins)
    int pad;
    double tpd;          // Settings::TriplePointDrag
    double ds;           // grainhdl::ds (grainhdl.cpp:81-82)
    double csr, isr;     // sector radii in grid points times h (grainhdl.cpp:130-131)
    double bins[16];     // model 4: mobility of bin b = [b, b+1) x 62.8 deg / 16
};

// A junction of the marching squares (GrainJunction, junction.h:45-67) after its projection
// onto the contour: coordinates, contourSegment and lambda, the distinct grains in corner order.
struct Junc {
    double x, y, lambda;
    int seg, order;
    uint32_t gr[4];
};

// Device arrays of an anisotropic context.
struct AnisoState {
    const double4* quat;   // orientation per grain id (slot 0, the domain boundary: identity)
    double* nb_e;          // per direct neighbour: energy density (characteristics::energyDensity)
    double* nb_m;          // per direct neighbour: mobility
    Junc* junc;            // kJuncCap per grain
    int* jcnt;
    int2* idl_org;         // origin of the IDLocal window the last comparison wrote
};

constexpr double kPiD = 3.14159265358979323846;
constexpr double kDeg = 1 * kPiD / 180.0;

__device__ __forceinline__ double misorientation_cubic(double4 p, double4 q) {
#pragma clang fp contract(off)
    const double q0 = p.x, q1 = -p.y, q2 = -p.z, q3 = -p.w;
    const double a = +q0 * q.x - q1 * q.y - q2 * q.z - q3 * q.w;
    const double b = +q1 * q.x + q0 * q.y - q3 * q.z + q2 * q.w;
    const double c = +q2 * q.x + q3 * q.y + q0 * q.z - q1 * q.w;
    const double d = +q3 * q.x - q2 * q.y + q1 * q.z + q0 * q.w;
    const double fac = 1.0 / sqrt(2.0);
    double omega = 0.0;
    auto take = [&](double v) { if (fabs(v) > omega) omega = fabs(v); };
    take((a + b) * fac); take((a - b) * fac); take((c + d) * fac); take((c - d) * fac);
    take((a + c) * fac); take((a - c) * fac); take((b + d) * fac); take((b - d) * fac);
    take((a + d) * fac); take((a - d) * fac); take((b + c) * fac); take((b - c) * fac);
    take((a + b + c + d) * 0.5); take((a + b - c - d) * 0.5); take((a - b + c - d) * 0.5); take((a - b - c + d) * 0.5);
    take((a + b + c - d) * 0.5); take((a + b - c + d) * 0.5); take((a - b + c + d) * 0.5); take((a - b - c - d) * 0.5);
    take(a); take(b); take(c); take(d);
    if (omega > 1.0) omega = (double)(int)omega;
    return 2 * acos(omega);
}

__device__ __forceinline__ double misorientation(double4 p, double4 q) {
    const double r = misorientation_cubic(p, q);
    return r > kDeg ? r : kDeg;
}

// Read-Shockley with a 15 degree cutoff (ResearchMode 0); 1.0 for ResearchMode 1 outside the
// test-case generator.
__device__ __forceinline__ double gb_energy(const AnisoConst& K, double theta) {
#pragma clang fp contract(off)
    if (K.research_mode != 0) return 1.0;
    const double gamma_hagb = 1.0, theta_ref = 15.0 * kPiD / 180.0;
    double gamma;
    if (theta > theta_ref) {
        gamma = gamma_hagb;
    } else {
        if (theta < 1.0 * kPiD / 180.0) theta = 1.0 * kPiD / 180.0;
        gamma = gamma_hagb * (theta / theta_ref) * (1.0 - log(theta / theta_ref));
        if (gamma != gamma) gamma = 0.01;
    }
    return gamma;
}

// Mobility models 0-2 without twin identification; model 4 (no reference counterpart): the
// mobility of the misorientation's bin, 16 bins over [0, 62.8 deg).
__device__ __forceinline__ double gb_mobility(const AnisoConst& K, double theta) {
#pragma clang fp contract(off)
    const int model = K.mobility_model;
    if (model == 0 || K.research_mode != 0) return 1.0;
    if (model == 1) return 1 - (0.99 * exp(-5.0 * (pow(theta / (15.0 * kPiD / 180.0), 9.0))));
    if (model == 2) {
        if (theta < 25 * kPiD / 180 || theta > 33 * kPiD / 180) return 0.1;
        return (sin((theta - 25 * kPiD / 180) / (8 * kPiD / 180) * kPiD) * 0.9) + 0.1;
    }
    if (model == 4) {
        int b = (int)(theta / (62.8 * kPiD / 180.0 / 16.0));
        b = b < 0 ? 0 : (b > 15 ? 15 : b);
        return K.bins[b];
    }
    return 1.0;
}

// The bin of a misorientation under model 4 (the bin whose mobility gb_mobility returns), or -1
// where the mobility does not come from the bins.
__device__ __forceinline__ int mobility_bin(const AnisoConst& K, double theta) {
#pragma clang fp contract(off)
    if (K.mobility_model != 4 || K.research_mode != 0) return -1;
    int b = (int)(theta / (62.8 * kPiD / 180.0 / 16.0));
    return b < 0 ? 0 : (b > 15 ? 15 : b);
}

// a + (b - a) * t without contraction (SPoint arithmetic, spoint.h:47-66)
__device__ __forceinline__ double lerp_nc(double a, double b, double t) {
#pragma clang fp contract(off)
    return a + (b - a) * t;
}

// projectToGrainBondary over a contour of `size` points (the last repeats the first): the nearest
// vertex (the first of the nearest in contour order), then the better of the segments after and
// before it.  -1 for fewer than two points.
__device__ __forceinline__ int nearest_vertex(const double2* c, int size, double px, double py) {
#pragma clang fp contract(off)
    double minDist = 1000000.0;
    int nearest = -1;
    for (int k = 0; k < size - 1; k++) {
        const double2 v = c[k];
        const double dx = px - v.x, dy = py - v.y;
        const double dist = dx * dx + dy * dy;
        if (dist < minDist) { nearest = k; minDist = dist; }
    }
    return nearest;
}

// nearest_vertex for the 64 pixels of an 8 x 8 tile by one wave, the same vertex: the scan is cut to
// the vertices that can be a pixel's nearest.  With vmin the vertex nearest to the tile's centre c,
// a vertex v is nearer than vmin to some point of the tile only if
//   |v - c|^2 - |vmin - c|^2 <= 7 (|vx - vminx| + |vy - vminy|)
// (the half-plane nearer to v meets the square of half side 3.5), tested in float with a margin
// above its rounding; the others are scanned in contour order with the strict comparison of the
// full scan.  A contour point every 0.8 grid points leaves 20 to 25 of a contour's 110 vertices.
// (tx, ty): the tile's first pixel; px, py: the lane's pixel.  All lanes of the wave call this.
__device__ __forceinline__ int nearest_vertex_tile(const double2* c, int size, int tx, int ty, double px, double py) {
#pragma clang fp contract(off)
    const int lane = (int)(threadIdx.x & 63), nv = size - 1;
    if (nv < 1) return -1;
    const double cx = tx + 3.5, cy = ty + 3.5;
    float dm = 3.0e38f, mx = 0.0f, my = 0.0f;
    for (int k = lane; k < nv; k += 64) {
        const double2 v = c[k];
        const float dx = (float)(v.x - cx), dy = (float)(v.y - cy), d = dx * dx + dy * dy;
        if (d < dm) { dm = d; mx = dx; my = dy; }
    }
    float lo = dm;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) lo = fminf(lo, __shfl_xor(lo, d));
    const int at = (int)__builtin_ctzll(__ballot(dm == lo));
    mx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx), at));
    my = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my), at));
    double minDist = 1000000.0;
    int nearest = -1;
    for (int c0 = 0; c0 < nv; c0 += 64) {
        bool may = false;
        if (c0 + lane < nv) {
            const double2 v = c[c0 + lane];
            const float dx = (float)(v.x - cx), dy = (float)(v.y - cy), d = dx * dx + dy * dy;
            may = d - lo <= 7.0f * (fabsf(dx - mx) + fabsf(dy - my)) + (1e-5f * d + 0.01f);
        }
        unsigned long long todo = __ballot(may);
        while (todo) {
            const int k = c0 + (int)__builtin_ctzll(todo);
            todo &= todo - 1ull;
            const double2 v = c[k];
            const double dx = px - v.x, dy = py - v.y;
            const double dist = dx * dx + dy * dy;
            if (dist < minDist) { nearest = k; minDist = dist; }
        }
    }
    return nearest;
}

// The segment part of projectToGrainBondary: the better of the segments after and before the
// nearest vertex, lambda clamped to [0, 1].
__device__ __forceinline__ int segment_at(const double2* c, int size, int nearest, double px, double py,
                                          double* out_lambda) {
#pragma clang fp contract(off)
    if (nearest < 0) return -1;
    int minimal_segment = nearest;
    auto len_sqr = [](double x, double y) { return x * x + y * y; };
    double minDist = 1000000.0;
    double dist;
    {
        const double2 a = c[nearest], b = c[nearest + 1];
        const double ux = b.x - a.x, uy = b.y - a.y;
        double lambda = (px - a.x) * ux + (py - a.y) * uy;
        lambda /= ux * ux + uy * uy;
        if (lambda < 0) dist = len_sqr(px - a.x, py - a.y);
        else if (lambda > 1) dist = len_sqr(b.x - px, b.y - py);
        else dist = len_sqr(px - (a.x + ux * lambda), py - (a.y + uy * lambda));
        if (dist < minDist) { minimal_segment = nearest; minDist = dist; *out_lambda = lambda; }
    }
    if (nearest == 0) nearest = size - 1;
    {
        const int previous = nearest - 1;
        const double2 a = c[previous], b = c[nearest];
        const double ux = b.x - a.x, uy = b.y - a.y;
        double lambda = (px - a.x) * ux + (py - a.y) * uy;
        lambda /= ux * ux + uy * uy;
        if (lambda < 0) dist = len_sqr(px - a.x, py - a.y);
        else if (lambda > 1) dist = len_sqr(b.x - px, b.y - py);
        else dist = len_sqr(px - (a.x + ux * lambda), py - (a.y + uy * lambda));
        if (dist < minDist) { minimal_segment = previous; minDist = dist; *out_lambda = lambda; }
    }
    if (*out_lambda > 1) *out_lambda = 1;
    if (*out_lambda < 0) *out_lambda = 0;
    return minimal_segment;
}

__device__ __forceinline__ int project_to_contour(const double2* c, int size, double px, double py, double* out_lambda) {
    return segment_at(c, size, nearest_vertex(c, size, px, py), px, py, out_lambda);
}

// ------------------------------------------------------------------------------------------
// The velocity corrector.
// ------------------------------------------------------------------------------------------

// What k_sectors leaves per grain for the pixels: the weights of the constant sectors, and of the
// interpolating sectors the length and the weight's polynomial in the relative arc length
// (contourSector.cpp:211-271): quadratic between two constant sectors, else between two end weights.
struct SectorRecord {
    int ok;                       // 0: nothing to correct (or the grain reports an error)
    int pad;
    double cw[kJuncCap];
    int kind[kSecCap];            // kLinear, kQuadratic, or kNoWeight where IDLocal has no value at an end
    double len[kSecCap], a[kSecCap], b[kSecCap], c[kSecCap];
};
enum { kLinear = 0, kQuadratic = 1, kNoWeight = 2 };
// Sector codes of a segment: constant sector, kInterp + interpolating sector, or a plain boundary point.
enum { kInterp = kJuncCap, kPlain = 255 };
static_assert(kInterp + kSecCap < kPlain, "sector codes");

template <class T>
struct AnisoArgs {
    const int* list;
    const int* count;
    const Box* box;
    const long long* off;
    const T* phi;                 // the fields before convolution (in)
    T* tilde;                     // the convolved fields (out), corrected in place
    const uint32_t* idl;          // IDLocal written by the previous step
    const long long* off_prev;    // its layout: offset, side and origin per grain
    const int* n_prev;
    const int* flags;
    int* err;
    int nslots;
    const double2* pts;           // contours of the previous step
    const long long* coff;
    const int* clen;
    const int* nb_cnt;
    const int* nb_id;
    AnisoState S;
    AnisoConst K;
    const int* loop;
    double h, delta;
    unsigned char* seg_code;      // per contour point: the sector its segment lies in (k_sectors)
    double* seg_arc;              // and, in an interpolating sector, the arc length from its right end
    SectorRecord* sectors;        // per grain
};

// Sectors of one grain (ContourSector: left and right contour points, the
// constant sectors' junctions, the interpolating sectors' bounding constant sectors, lengths).
struct SectorSet {
    int ncons, ninterp, err;
    int cl[kJuncCap], cr[kJuncCap], cnj[kJuncCap];
    unsigned char cj[kJuncCap][kJuncCap];
    double cw[kJuncCap];
    int il[kSecCap], ir[kSecCap], ils[kSecCap], irs[kSecCap];
    double ilen[kSecCap];
};

// grainhdl::getGrainByID at convolution time: the grains deleted earlier in this step (kGone)
// are still there when the reference convolves.
__device__ __forceinline__ bool present_at_conv(const int* flags, int nslots, uint32_t id) {
    if (id == 0u) return true;
    return id < (uint32_t)nslots && (flags[id] & (kPresent | kGone));
}

__device__ __forceinline__ bool sector_within(int right, int left, int size, int segment) {
    const int totalP = size - 1;
    if (right == left && left == -1) return true;
    if (right > left) return (segment >= 0 && segment <= left) || (segment >= right && segment < totalP);
    return segment >= right && segment <= left;
}

__device__ __forceinline__ double seg_len(double2 a, double2 b) {
#pragma clang fp contract(off)
    const double x = a.x - b.x, y = a.y - b.y;
    return sqrt(x * x + y * y);
}

__device__ __forceinline__ double scaled_len(double2 b, double2 a, double f) {
#pragma clang fp contract(off)
    const double x = (b.x - a.x) * f, y = (b.y - a.y) * f;
    return sqrt(x * x + y * y);
}

// GrainJunction::getWeight (junction.cpp:23-192), read-from-file microstructures, research
// project 0 (an unset project is taken as 0: the precedence slip `!project == 1` is true and an
// incomplete junction weighs 1).  False where the reference would dereference a null grain.
// Partial derivatives of a junction weight with respect to the three boundary mobilities it
// averages, and the mobility bins those come from (-1: not from a bin).
struct JuncGrad {
    double d[3];
    int bin[3];
};

template <class T>
__device__ bool junction_weight(const AnisoArgs<T>& A, int me, const Junc& J, double* out, JuncGrad* jg = nullptr) {
#pragma clang fp contract(off)
    uint32_t nb[3] = {0xFFFFFFu, 0xFFFFFFu, 0xFFFFFFu};
    for (int i = 0, j = 0; i < J.order; i++) {
        if ((uint32_t)me != J.gr[i]) {
            if (j >= 3) return false;
            nb[j] = J.gr[i];
            j++;
        }
    }
    if (jg)
        for (int i = 0; i < 3; ++i) { jg->d[i] = 0.0; jg->bin[i] = -1; }
    if (nb[0] == 0xFFFFFFu || nb[1] == 0xFFFFFFu) { *out = 1; return true; }
    if (!present_at_conv(A.flags, A.nslots, nb[0]) || !present_at_conv(A.flags, A.nslots, nb[1])) return false;
    const AnisoConst& K = A.K;
    double averageMobility = 0;
    double gamma0, gamma1, gamma2;
    if (K.research_mode == 0) {
        const double4 qm = A.S.quat[me], q0 = A.S.quat[nb[0]], q1 = A.S.quat[nb[1]];
        double th = misorientation(qm, q0);
        averageMobility += gb_mobility(K, th);
        if (jg) jg->bin[0] = mobility_bin(K, th);
        gamma0 = gb_energy(K, th);
        th = misorientation(q0, q1);
        double m01 = 1.0;  // nb[0]'s characteristic of nb[1] (default mobility 1)
        const int c0 = nb[0] == 0u ? 0 : A.nb_cnt[nb[0]];
        for (int k = 0; k < c0; ++k)
            if ((uint32_t)A.nb_id[(size_t)nb[0] * kNbCap + k] == nb[1]) {
                const size_t e = (size_t)nb[0] * kNbCap + k;
                m01 = A.S.nb_m[e];
                // a recorded characteristic (energy > 0) holds the mobility of its bin; the manual
                // ones of a fresh network hold 0
                if (jg && A.S.nb_e[e] > 0) jg->bin[1] = mobility_bin(K, misorientation(q0, q1));
                break;
            }
        averageMobility += m01;
        gamma1 = gb_energy(K, th);
        th = misorientation(qm, q1);
        averageMobility += gb_mobility(K, th);
        if (jg) jg->bin[2] = mobility_bin(K, th);
        gamma2 = gb_energy(K, th);
    } else {
        gamma0 = gamma1 = gamma2 = 1.0;
    }
    double sigma = gamma0 - gamma1 + gamma2;
    double dsigma = 0.0;  // d sigma / d (each of the three mobilities)
    if (K.mobility_model > 0 && K.tpd > 0) {
        averageMobility /= 3;
        const double drag = 1 / ((1 / (K.ds * K.tpd)) + 1 / averageMobility);
        dsigma = sigma * (drag * drag) / (averageMobility * averageMobility) / 3;
        sigma *= drag;
    }
    if (sigma < 0.01) { sigma = 0.01; dsigma = 0.0; }
    if (jg)
        for (int i = 0; i < 3; ++i) jg->d[i] = jg->bin[i] >= 0 ? dsigma : 0.0;
    *out = sigma;
    return true;
}

// ExplicitGrainBoundary::buildBoundarySectors with setPointsOnBoundary and the interpolating
// sector generators, by one wave (S in LDS): the walks along the contour, a chain of square roots
// each, run one junction or constant sector per lane; only the merging of constant sectors, a few
// comparisons per junction, is serial.  jw: the junction weights.  Sets S.err on a contour too short
// to end the reference's length-bounded walks, or beyond the capacities.
__device__ void build_sectors(const double2* c, int size, const Junc* J, int nj, const double* jw, double h,
                              double csr, double isr, SectorSet& S) {
#pragma clang fp contract(off)
    const int lane = (int)(threadIdx.x & 63);
    if (lane == 0) { S.ncons = 0; S.ninterp = 0; S.err = 0; }
    wave_lds_sync();
    if (nj == 0) return;
    if (size < 2) {
        if (lane == 0) S.err = 1;
        wave_lds_sync();
        return;
    }
    const int P = size - 1;  // PERIODIC modulus (grainBoundary.cpp:27)
    auto per = [P](int x) { return (x + P) % P; };
    const int cap = 1 << 24;
    bool bad = false;
    if (lane < nj) {  // setPointsOnBoundary of junction `lane`; kept in il / ir until the merge is done
        double dist = 0;
        int l = J[lane].seg, it = 0;
        dist += scaled_len(c[per(l + 1)], c[l], 1 - J[lane].lambda) * h;
        l = per(l + 1);
        while (dist < csr && !bad) {
            dist += seg_len(c[per(l + 1)], c[l]) * h;
            l = per(l + 1);
            if (++it > cap) bad = true;
        }
        dist = 0;
        int r = J[lane].seg;
        dist += scaled_len(c[per(r + 1)], c[r], J[lane].lambda) * h;
        r = per(r);
        it = 0;
        while (dist < csr && !bad) {
            dist += seg_len(c[per(r - 1)], c[r]) * h;
            r = per(r - 1);
            if (++it > cap) bad = true;
        }
        S.ir[lane] = r;
        S.il[lane] = l;
    }
    if (__ballot(bad)) {
        if (lane == 0) S.err = 1;
        wave_lds_sync();
        return;
    }
    wave_lds_sync();
    if (lane == 0) {
        int ncons = 1, cur = 0, err = 0;
        S.cl[0] = S.il[0]; S.cr[0] = S.ir[0]; S.cnj[0] = 1; S.cj[0][0] = 0;
        for (int i = 1; i < nj && !err; i++) {
            const int rr = S.ir[i], ll = S.il[i];
            if (sector_within(S.cr[cur], S.cl[cur], size, rr)) {
                if (S.cnj[cur] >= kJuncCap) { err = 1; break; }
                S.cj[cur][S.cnj[cur]++] = (unsigned char)i;
                S.cl[cur] = ll;
                if (i == nj - 1 && sector_within(S.cr[0], S.cl[0], size, S.cl[cur])) {
                    if (cur == 0) {
                        S.cl[0] = -1;
                        S.cr[0] = -1;
                    } else {
                        const int m = S.cnj[cur];
                        for (int q = 0; q < m; ++q) {
                            if (S.cnj[0] >= kJuncCap) { err = 1; break; }
                            S.cj[0][S.cnj[0]++] = S.cj[cur][q];
                        }
                        S.cr[0] = S.cr[cur];
                    }
                }
            } else if (i == nj - 1 && sector_within(S.cr[0], S.cl[0], size, ll)) {
                if (S.cnj[0] >= kJuncCap) { err = 1; break; }
                S.cr[0] = rr;
                S.cj[0][S.cnj[0]++] = (unsigned char)i;
            } else {
                const int k = ncons++;
                S.cl[k] = ll; S.cr[k] = rr; S.cnj[k] = 1; S.cj[k][0] = (unsigned char)i;
                cur++;
            }
        }
        S.ncons = ncons;
        S.err = err;
    }
    wave_lds_sync();
    if (S.err) return;
    const int ncons = S.ncons;
    // ContourSector::getWeight of a constant sector: the mean of its junctions' weights
    if (lane < ncons) {
        double weight = 0;
        for (int q = 0; q < S.cnj[lane]; ++q) weight += jw[S.cj[lane][q]];
        S.cw[lane] = weight / S.cnj[lane];
    }
    wave_lds_sync();
    if (ncons < 2) return;
    // between constant sector `lane` and the next one: their interpolating contours, one sector each,
    // or one sector for both where the two contours meet
    const int sr = lane, sl = (lane + 1 + ncons) % ncons;
    int nr_left = 0, nr_right = 0, nl_left = 0, nl_right = 0;
    double nr_len = 0, nl_len = 0, both_len = 0;
    bool merged = false;
    if (lane < ncons) {
        // generateLeftInterpolatingContour of sector sr (contourSector.cpp:108-127)
        double dist = 0;
        int j, it = 0;
        for (j = S.cl[sr]; dist <= isr && !bad; j = (j + 1 + P) % P) {
            dist += seg_len(c[j], c[(j + 1 + P) % P]) * h;
            if (++it > cap) bad = true;
        }
        nr_left = (j + 1 + P) % P;
        nr_right = S.cl[sr];
        nr_len = dist;
        // generateRightInterpolatingContour of sector sl (contourSector.cpp:149-169)
        dist = 0;
        for (j = S.cr[sl]; dist <= isr && !bad; j = (j - 1 + P) % P) {
            dist += seg_len(c[j], c[(j - 1 + P) % P]) * h;
            if (++it > cap) bad = true;
        }
        nl_left = S.cr[sl];
        nl_right = (j - 1 + P) % P;
        nl_len = dist;
        for (int q = nr_right; q != per(nr_left + 1) && !bad; q = per(q + 1)) {
            if (q == nl_left || q == nl_right) merged = true;
            if (++it > cap) bad = true;
        }
        if (merged)  // generateInterpolatingSector: this = sector sl, other = sector sr
            for (int q = S.cl[sr]; q != S.cr[sl] && !bad; q = (q + 1 + P) % P) {
                both_len += seg_len(c[q], c[(q - 1 + P) % P]) * h;
                if (++it > cap) bad = true;
            }
    }
    // places in the order of the constant sectors: one entry where merged, two else
    const unsigned long long here = ncons < 64 ? (1ull << ncons) - 1ull : ~0ull, one = __ballot(merged) & here;
    const unsigned long long below = (1ull << lane) - 1ull;
    const int k = 2 * __popcll(here & below) - __popcll(one & below);
    const int count = 2 * __popcll(here) - __popcll(one);
    if (__ballot(bad) || count > kSecCap) {
        if (lane == 0) S.err = 1;
        wave_lds_sync();
        return;
    }
    wave_lds_sync();  // il / ir served the merge until here
    if (lane < ncons) {
        if (merged) {
            S.il[k] = S.cr[sl]; S.ils[k] = sl; S.ir[k] = S.cl[sr]; S.irs[k] = sr; S.ilen[k] = both_len;
        } else {
            S.il[k] = nr_left; S.ir[k] = nr_right; S.ils[k] = -1; S.irs[k] = sr; S.ilen[k] = nr_len;
            S.il[k + 1] = nl_left; S.ir[k + 1] = nl_right; S.ils[k + 1] = sl; S.irs[k + 1] = -1; S.ilen[k + 1] = nl_len;
        }
    }
    if (lane == 0) S.ninterp = count;
    wave_lds_sync();
}

// LSbox::getGBEnergyTimesGBMobility(i, j) (box.cpp:544-554): IDLocal's neighbour at (i, j), its
// energy x mobility in this grain's direct neighbourhood (0.01 floor; 1 when absent).  False
// where IDLocal::getValueAt would throw.
// slot (optional): the neighbour entry the weight came from, -1 for the default.
template <class T>
__device__ __forceinline__ bool gb_weight_at(const AnisoArgs<T>& A, long long op, int np, int ix0, int iy0,
                                             const int* s_nid, const double* s_nw, int nbc, int i, int j, double* w,
                                             int* slot = nullptr) {
    uint32_t k = (uint32_t)i - (uint32_t)iy0;
    k *= (uint32_t)np;
    k += (uint32_t)j - (uint32_t)ix0;
    if ((unsigned long long)k >= (unsigned long long)np * (unsigned long long)np) return false;
    const uint32_t id = A.idl[op + k];
    double v = 1.0;
    int sl = -1;
    if (present_at_conv(A.flags, A.nslots, id)) {
        for (int q = 0; q < nbc; ++q)
            if ((uint32_t)s_nid[q] == id) { v = s_nw[q]; sl = q; break; }
    }
    *w = v;
    if (slot) *slot = sl;
    return true;
}

// k_sectors: one wave per grain.  The sectors of the previous contour and, laid out for k_aniso,
// the sector of every contour segment, the arc length before it and every sector's weight.  Bound
// by the latency of the walks (square roots in a chain): a kernel of its own, so that the pixels'
// waves do not hold their registers and LDS through it.  10000 grains: 0.13 ms.
template <class T>
__global__ void __launch_bounds__(64) k_sectors(AnisoArgs<T> A) {
#pragma clang fp contract(off)
    __shared__ SectorSet S;
    __shared__ Junc s_j[kJuncCap];
    __shared__ double s_jw[kJuncCap];
    __shared__ int s_nid[kNbCap];
    __shared__ double s_nw[kNbCap];
    __shared__ double2 s_c[kAnisoContourLds];
    __shared__ unsigned char s_code[kAnisoContourLds];
    const int total = *A.count;
    const int loop = *A.loop;
    const int lane = (int)threadIdx.x;
    for (int item = blockIdx.x; item < total; item += gridDim.x) {
        wave_lds_sync();  // the previous grain's shared state is free
        const int g = A.list[item];
        SectorRecord& R = A.sectors[g];
        if (loop == 0 || !(A.flags[g] & kRegular)) {  // box.cpp:428-429
            if (lane == 0) R.ok = 0;
            continue;
        }
        const int L = A.clen[g];
        const int nj = min(A.S.jcnt[g], kJuncCap);
        const long long co = A.coff[g];
        const double2* cg = A.pts + co;
        const int nbc = A.nb_cnt[g];
        const long long op = A.off_prev[g];
        const int np = A.n_prev[g];
        const int2 org = A.S.idl_org[g];
        const bool staged = L <= kAnisoContourLds;
        if (staged)
            for (int k = lane; k < L; k += 64) s_c[k] = cg[k];
        for (int k = lane; k < nbc; k += 64) {
            s_nid[k] = A.nb_id[(size_t)g * kNbCap + k];
            const double e = A.S.nb_e[(size_t)g * kNbCap + k], m = A.S.nb_m[(size_t)g * kNbCap + k];
            s_nw[k] = (e * m > 0.01) ? e * m : 0.01;
        }
        bool bad = false;
        if (lane < nj) {
            s_j[lane] = A.S.junc[(size_t)g * kJuncCap + lane];
            double w = 1.0;
            if (!junction_weight(A, g, s_j[lane], &w)) bad = true;
            s_jw[lane] = w;
        }
        wave_lds_sync();
        // the contour in LDS when it fits; separate code, so that the walks read LDS and not through
        // a generic pointer in the usual case
        auto build = [&](const double2* c) -> bool {
            build_sectors(c, L, s_j, nj, s_jw, A.h, A.K.csr, A.K.isr, S);
            if (S.err) return false;
            const int ncons = S.ncons, ninterp = S.ninterp, P = L - 1;
            if (lane < ncons) R.cw[lane] = S.cw[lane];
            if (lane < ninterp) {
                // end weights: a constant sector's, or the boundary's at the end point
                const int s = lane;
                double left_w = 0, right_w = 0, bw = 0;
                bool ok = true;
                if (S.ils[s] >= 0) left_w = S.cw[S.ils[s]];
                else ok = gb_weight_at(A, op, np, org.x, org.y, s_nid, s_nw, nbc, (int)c[S.il[s]].y, (int)c[S.il[s]].x, &left_w);
                if (S.irs[s] >= 0) right_w = S.cw[S.irs[s]];
                else ok = ok && gb_weight_at(A, op, np, org.x, org.y, s_nid, s_nw, nbc, (int)c[S.ir[s]].y, (int)c[S.ir[s]].x, &right_w);
                const bool both = S.ils[s] >= 0 && S.irs[s] >= 0;
                R.len[s] = S.ilen[s];
                if (both) {
                    const double2 sample = c[(S.ir[s] + 1) % P];
                    ok = ok && gb_weight_at(A, op, np, org.x, org.y, s_nid, s_nw, nbc, (int)sample.y, (int)sample.x, &bw);
                    const double two_isr = 2 * A.K.isr;
                    const double quot = (S.ilen[s] > two_isr ? two_isr : S.ilen[s]);
                    const double amplitude = (bw - (left_w + right_w) / 2) / (two_isr) * quot + (left_w + right_w) / 2;
                    const double a0 = 2 * right_w, a1 = -4 * amplitude, a2 = 2 * left_w;
                    R.a[s] = a0 + a1 + a2;
                    R.b[s] = -(a0 * 1.5 + a1 + a2 * 0.5);
                    R.c[s] = a0 * 0.5;
                } else {
                    R.a[s] = left_w;
                    R.b[s] = right_w;
                }
                R.kind[s] = ok ? (both ? kQuadratic : kLinear) : kNoWeight;
            }
            for (int k = lane; k < P; k += 64) {
                int code = kPlain;
                for (int s = 0; s < ncons && code == kPlain; ++s)
                    if (sector_within(S.cr[s], S.cl[s], L, k)) code = s;
                for (int s = 0; s < ninterp && code == kPlain; ++s)
                    if (sector_within(S.ir[s], S.il[s], L, k)) code = kInterp + s;
                A.seg_code[co + k] = (unsigned char)code;
                if (staged) s_code[k] = (unsigned char)code;
            }
            wave_lds_sync();
            // arc length from an interpolating sector's right end to each of its segments, a sector per
            // lane; a segment in two sectors keeps the first one's (the one its code names)
            auto arcs = [&](int s, auto mine) {
                double arc = 0;
                int k = S.ir[s];
                for (int it = 0; it < P; ++it) {
                    if (mine(k)) A.seg_arc[co + k] = arc;
                    if (k == S.il[s]) break;
                    arc += seg_len(c[k + 1], c[k]) * A.h;
                    k = (k + 1 + P) % P;
                }
            };
            if (staged) {
                if (lane < ninterp) arcs(lane, [&](int k) { return (int)s_code[k] == kInterp + lane; });
            } else if (lane == 0) {
                for (int s = ninterp - 1; s >= 0; --s) arcs(s, [](int) { return true; });
            }
            return true;
        };
        const bool ok = !__ballot(bad) && (staged ? build(s_c) : build(cg));
        if (lane == 0) {
            R.ok = ok ? 1 : 0;
            if (!ok) A.err[g] = kErrAniso;
        }
    }
}

// k_aniso: the corrected field.  One workgroup per grain, a wave per 8 x 8 tile of pixels (the tile
// keeps the pixels' candidate vertices few); contour, segment codes and arc lengths in LDS.  Bound
// by the vertex scan and the two projections (FP64 VALU).  10000 grains: 0.38 ms, with k_sectors
// 0.51 ms, where one kernel with a lane-0 sector build, chunk boxes per pixel and a walk to each
// pixel's segment took 2.5 to 3.0 ms.
template <class T>
__global__ void __launch_bounds__(256) k_aniso(AnisoArgs<T> A) {
#pragma clang fp contract(off)
    __shared__ double2 s_c[kAnisoContourLds];
    __shared__ double s_arc[kAnisoContourLds];
    __shared__ unsigned char s_code[kAnisoContourLds];
    __shared__ int s_nid[kNbCap];
    __shared__ double s_nw[kNbCap];
    const int total = *A.count;
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6), nw = (int)(blockDim.x >> 6);
    for (int item = blockIdx.x; item < total; item += gridDim.x) {
        __syncthreads();  // the previous grain's shared state is free
        const int g = A.list[item];
        const SectorRecord& R = A.sectors[g];
        if (!R.ok) continue;
        const int L = A.clen[g];
        const long long co = A.coff[g];
        const bool staged = L <= kAnisoContourLds;
        if (staged)
            for (int k = threadIdx.x; k < L; k += blockDim.x) {
                s_c[k] = A.pts[co + k];
                s_arc[k] = A.seg_arc[co + k];
                s_code[k] = A.seg_code[co + k];
            }
        const int nbc = A.nb_cnt[g];
        for (int k = threadIdx.x; k < nbc; k += blockDim.x) {
            s_nid[k] = A.nb_id[(size_t)g * kNbCap + k];
            const double e = A.S.nb_e[(size_t)g * kNbCap + k], m = A.S.nb_m[(size_t)g * kNbCap + k];
            s_nw[k] = (e * m > 0.01) ? e * m : 0.01;
        }
        // pixels: IDLocal's window (previous step) intersected with the box (box.cpp:452-470)
        const Box b = A.box[g];
        const long long o = A.off[g];
        const int np = A.n_prev[g];
        const long long op = A.off_prev[g];
        const int2 org = A.S.idl_org[g];
        const int ix0 = max(org.x, b.x0), ix1 = min(org.x + np, b.x0 + b.n);
        const int iy0 = max(org.y, b.y0), iy1 = min(org.y + np, b.y0 + b.n);
        __syncthreads();
        if (ix0 >= ix1 || iy0 >= iy1) continue;
        const int tw = (ix1 - ix0 + 7) >> 3, th = (iy1 - iy0 + 7) >> 3;
        auto process = [&](const double2* c, const unsigned char* code_of, const double* arc_of) {
            for (int tile = wave; tile < tw * th; tile += nw) {
                const int ty = iy0 + (tile / tw) * 8, tx = ix0 + (tile % tw) * 8;
                const int i = ty + (lane >> 3), j = tx + (lane & 7);
                const bool on = i < iy1 && j < ix1;
                const long long q = o + (long long)(i - b.y0) * b.n + (j - b.x0);
                const double val = on ? (double)A.phi[q] : -A.delta;
                const bool act = on && val > -A.delta;
                if (on && !act) A.tilde[q] = (T)(-A.delta);
                if (!__ballot(act)) continue;
                // ExplicitGrainBoundary::getWeight (grainBoundary.cpp:344-363)
                const int nearest = nearest_vertex_tile(c, L, tx, ty, (double)j, (double)i);
                if (!act) continue;
                double lambda = 0, weight = 0;
                const int segment = segment_at(c, L, nearest, (double)j, (double)i, &lambda);
                bool ok = segment >= 0;
                if (ok) {
                    const int code = code_of[segment];
                    if (code < kInterp) {
                        weight = R.cw[code];
                    } else if (code == kPlain) {
                        ok = gb_weight_at(A, op, np, org.x, org.y, s_nid, s_nw, nbc, i, j, &weight);
                    } else {
                        // ContourSector::getWeight of an interpolating sector (contourSector.cpp:211-271)
                        const int s = code - kInterp, rcs = L - 1, kind = R.kind[s];
                        double t = arc_of[segment];
                        t += scaled_len(c[(segment + 1 + rcs) % rcs], c[segment], lambda);
                        t /= R.len[s];
                        if (t < 0) t = 0;
                        if (t > 1) t = 1;
                        if (kind == kQuadratic) weight = R.a[s] * t * t + R.b[s] * t + R.c[s];
                        else if (kind == kLinear) weight = t * R.a[s] + (1 - t) * R.b[s];
                        else ok = false;
                    }
                }
                if (!ok) {
                    A.err[g] = kErrAniso;
                    continue;
                }
                const double radiuscorrection = 1.0;  // box.cpp:501
                const double t = (double)A.tilde[q];
                A.tilde[q] = (T)(val + (t - val) * weight * radiuscorrection);
            }
        };
        if (staged) process(s_c, s_code, s_arc);
        else process(A.pts + co, A.seg_code + co, A.seg_arc + co);
    }
}

}  // namespace ggx
