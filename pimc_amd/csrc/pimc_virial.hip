// pimc_virial.hip -- the virial and centroid-virial pair terms of a closed path
// (LocalAction::rDOTgradUterm1/2, deltadotgradUterm1/2, gradVSquared,
// src/action.cpp:1188-1223, :1446-1762) and the link sums of
// VirialEnergyEstimator::accumulate (src/estimator.cpp:1125-1146).
//
// For every bead i of slice m, over every partner j of the slice (no cutoff, as the
// reference; slices of up to 1024 beads as unordered pairs, k_virial_sym, larger
// ones one lane per bead):
//   F_i = sum_j gradV(r_i - r_j),   gradV(r) = (lookupdVdr[k] / |r|) r
//   T_i = sum_j [ r r^T d2V / |r|^2 - r r^T dV / |r|^3 + I dV / |r| ]
// with d2V = lookupd2Vdr2[k] and dV = |gradV(r)| (a magnitude, as the
// reference takes it), then writes seven per-bead terms
//   F.r_i, (T F).r_i, F.delta_i, (T F).delta_i, |F|^2, -vel1.vel2, -vel2.vel2
// where delta_i is the bead's offset from the centroid of its worldline window
// (virialWindow links each way) and vel1 / vel2 the window and one-link
// displacements along the next links.  Each workgroup reduces its beads in a
// fixed order, so the per-slice sums the host forms are deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "pimc_kernels.hpp"

namespace pimc {

namespace {

// Position of bead (m, i) and the minimum-image separation of two beads
// (Path::getSeparation, include/path.h:179-184).
struct PathView {
    const double* pos;
    int64_t plane;
    int nalloc;
    __device__ __forceinline__ void at(int m, int i, double r[3]) const {
        const double* p = pos + (int64_t)m * nalloc + i;
        r[0] = p[0];
        r[1] = p[plane];
        r[2] = p[2 * plane];
    }
};

__device__ __forceinline__ void sep_of(const double a[3], const double b[3], const BoxDev& box, double s[3]) {
    for (int q = 0; q < 3; ++q) s[q] = min_image_exact(a[q] - b[q], box.L, box.invL);
}

__device__ __forceinline__ double dot3(const double a[3], const double b[3]) {
#pragma clang fp contract(off)
    double s = a[0] * b[0];
    s = s + a[1] * b[1];
    s = s + a[2] * b[2];
    return s;
}

__device__ __forceinline__ void step_link(const int* links, int M, int nalloc, int& m, int& i, int dir) {
    if (links) {
        const int64_t t = (int64_t)m * nalloc + i;
        const int nm = links[2 * t], ni = links[2 * t + 1];
        m = nm;
        i = ni;
    } else {
        m = dir > 0 ? (m + 1 == M ? 0 : m + 1) : (m == 0 ? M - 1 : m - 1);
    }
}

// One pair's terms from the (not yet minimum-imaged) separation d = r_i - r_j:
// g = gradV(s) and, when need_t, the symmetric t (xx, xy, xz, yy, yz, zz); s gets
// the minimum image.  False outside (0, tableLength), where both are 0.
template <int MODE>
__device__ __forceinline__ bool virial_pair(double dx, double dy, double dz, const BoxDev& box, const AzizDev& a,
                                            double inv_dr, bool need_t, double s[3], double g[3], double t[6]) {
    double rn, ir;
    int k;
    if (MODE == 0) {
        s[0] = min_image_fast(dx, box.L, box.invL);
        s[1] = min_image_fast(dy, box.L, box.invL);
        s[2] = min_image_fast(dz, box.L, box.invL);
        k = bin_rsq(norm2_exact(s[0], s[1], s[2]), inv_dr, &rn, &ir);
    } else {
        s[0] = min_image_exact(dx, box.L, box.invL);
        s[1] = min_image_exact(dy, box.L, box.invL);
        s[2] = min_image_exact(dz, box.L, box.invL);
        k = bin_exact(norm2_exact(s[0], s[1], s[2]), a.dr, &rn);
        // one division per pair: the reference's quotients by |r|, |r|^2 and
        // |r|^3 become products with 1/|r| (a rounding apart)
        ir = 1.0 / rn;
    }
    if ((unsigned)(k - a.k_eps) >= (unsigned)(a.table_length - a.k_eps)) return false;
    const double d = (MODE == 2) ? a.dtable[k] : (MODE == 1 ? aziz_dvdr64(k, a) : aziz_dvdr_mix(k, a));
    const double f = d * ir;
#pragma unroll
    for (int q = 0; q < 3; ++q) g[q] = f * s[q];
    if (need_t) {
        const double d2 = (MODE == 2) ? a.d2table[k] : (MODE == 1 ? aziz_d2vdr2_64(k, a) : aziz_d2vdr2_mix(k, a));
        // |gradV| = |dV/dr|; r r^T (d2V/r^2 - |gradV|/r^3) + I |gradV|/r
        const double diag = __builtin_fabs(d) * ir;
        const double c = (d2 - diag) * (ir * ir);
        const double c0 = c * s[0], c1 = c * s[1], c2 = c * s[2];
        t[0] = fma(c0, s[0], diag);
        t[1] = c0 * s[1];
        t[2] = c0 * s[2];
        t[3] = fma(c1, s[1], diag);
        t[4] = c1 * s[2];
        t[5] = fma(c2, s[2], diag);
    }
    return true;
}

// The minimum image s of d, seen from the partner, is -s; at half a box it may be s
// (floor folds L/2 and -L/2 alike): -1 for such a component, else 1.
template <int MODE>
__device__ __forceinline__ double fold_sign(double back, double s, const BoxDev& box) {
    const double r = MODE == 0 ? min_image_fast(back, box.L, box.invL) : min_image_exact(back, box.L, box.invL);
    return r * s > 0.0 ? -1.0 : 1.0;
}

// The sum over partners [j0, j1) of one bead: F (3) and, when need_t, T.
template <int MODE, typename P>
__device__ __forceinline__ void bead_pairs(P px, P py, P pz, int j0, int j1, int i, const BoxDev& box,
                                           const AzizDev& a, bool need_t, double F[3], double T[6]) {
    const double xi = px[i], yi = py[i], zi = pz[i];
    const double inv_dr = 1.0 / a.dr;
    for (int j = j0; j < j1; ++j) {
        if (j == i) continue;
        double s[3], g[3], t[6];
        if (!virial_pair<MODE>(xi - px[j], yi - py[j], zi - pz[j], box, a, inv_dr, need_t, s, g, t)) continue;
#pragma unroll
        for (int q = 0; q < 3; ++q) F[q] += g[q];
        if (need_t) {
#pragma unroll
            for (int q = 0; q < 6; ++q) T[q] += t[q];
        }
    }
}

// The per-bead terms from the bead's F and T: (T F).r, the window centroid
// offset delta and the link displacements, into o[kVirialTerms].
template <bool LINKS>
__device__ __forceinline__ void bead_finish(const VirialArgs& A, int m, int i, const double F[3], const double T[6],
                                            double* o) {
#pragma clang fp contract(off)
    // T F (apply_matrix_vector_product, include/common.h:187-199)
    double TF[3];
    TF[0] = ((0.0 + T[0] * F[0]) + T[1] * F[1]) + T[2] * F[2];
    TF[1] = ((0.0 + T[1] * F[0]) + T[3] * F[1]) + T[4] * F[2];
    TF[2] = ((0.0 + T[2] * F[0]) + T[4] * F[1]) + T[5] * F[2];
    const PathView P{A.pos, A.plane, A.nalloc};
    double r1[3];
    P.at(m, i, r1);
    // One walk along the next links (window of them) and one along the prev
    // links (window - 1): the window centroid (src/action.cpp:1621-1645: running
    // separations from the bead, the bead itself counted for gamma = 0) and the
    // link displacements (src/estimator.cpp:1125-1146).  Without link arrays the
    // addresses need no load, so a few steps' loads are in flight at once.
    double more[3] = {0.0, 0.0, 0.0}, less[3] = {0.0, 0.0, 0.0}, com[3] = {0.0, 0.0, 0.0};
    double vel2[3] = {0.0, 0.0, 0.0};
    int nm = m, ni = i, pm = m, pi = i;
    double nold[3] = {r1[0], r1[1], r1[2]}, pold[3] = {r1[0], r1[1], r1[2]};
    for (int q = 0; q < 3; ++q) com[q] += r1[q] + r1[q];
#pragma unroll 4
    for (int gamma = 1; gamma < A.window; ++gamma) {
        step_link(LINKS ? A.next : nullptr, A.num_slices, A.nalloc, nm, ni, 1);
        step_link(LINKS ? A.prev : nullptr, A.num_slices, A.nalloc, pm, pi, -1);
        double rn[3], rp[3], sn[3], sp[3];
        P.at(nm, ni, rn);
        P.at(pm, pi, rp);
        sep_of(rn, nold, A.box, sn);
        sep_of(rp, pold, A.box, sp);
        for (int q = 0; q < 3; ++q) {
            more[q] += sn[q];
            less[q] += sp[q];
            com[q] += (r1[q] + more[q]) + (r1[q] + less[q]);
            nold[q] = rn[q];
            pold[q] = rp[q];
            if (gamma == 1) vel2[q] = sn[q];
        }
    }
    double delta[3];
    for (int q = 0; q < 3; ++q) {
        com[q] /= (2.0 * A.window);
        delta[q] = min_image_exact(r1[q] - com[q], A.box.L, A.box.invL);
    }
    step_link(LINKS ? A.next : nullptr, A.num_slices, A.nalloc, nm, ni, 1);
    double rk[3], sk[3], vel1[3];
    P.at(nm, ni, rk);
    sep_of(rk, nold, A.box, sk);
    for (int q = 0; q < 3; ++q) {
        vel1[q] = more[q] + sk[q];
        if (A.window == 1) vel2[q] = sk[q];
    }
    o[0] = dot3(F, r1);
    o[1] = dot3(TF, r1);
    o[2] = dot3(F, delta);
    o[3] = dot3(TF, delta);
    o[4] = dot3(F, F);
    o[5] = -dot3(vel1, vel2);
    o[6] = -dot3(vel2, vel2);
}

template <int MODE>
__global__ __launch_bounds__(256) void k_virial(VirialArgs A, AzizDev az) {
    extern __shared__ double lds[];
    __shared__ double red[4][kVirialTerms];
    const int m = blockIdx.y, b = blockIdx.x;
    const int n = A.nbs[m];
    const double* px = A.pos + (int64_t)m * A.nalloc;
    const double* py = px + A.plane;
    const double* pz = py + A.plane;
    const bool in_lds = n <= A.lds_beads;
    double* lx = lds;
    double* ly = lds + A.lds_beads;
    double* lz = lds + 2 * A.lds_beads;
    if (in_lds)
        for (int t = threadIdx.x; t < n; t += 256) {
            lx[t] = px[t];
            ly[t] = py[t];
            lz[t] = pz[t];
        }
    __syncthreads();
    const int i = b * 256 + threadIdx.x;
    double o[kVirialTerms];
#pragma unroll
    for (int q = 0; q < kVirialTerms; ++q) o[q] = 0.0;
    if (i < n) {
        const bool need_t = (m & 1) ? A.t_odd : A.t_even;
        double F[3] = {0.0, 0.0, 0.0}, T[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if (in_lds)
            bead_pairs<MODE>(lx, ly, lz, 0, n, i, A.box, az, need_t, F, T);
        else
            bead_pairs<MODE>(px, py, pz, 0, n, i, A.box, az, need_t, F, T);
        A.next ? bead_finish<true>(A, m, i, F, T, o) : bead_finish<false>(A, m, i, F, T, o);
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < kVirialTerms; ++q) {
        const double v = wave_sum(o[q]);
        if (lane == 0) red[wave][q] = v;
    }
    __syncthreads();
    if (threadIdx.x < kVirialTerms) {
        const int q = threadIdx.x;
        A.part[((int64_t)m * gridDim.x + b) * kVirialTerms + q] = ((red[0][q] + red[1][q]) + red[2][q]) + red[3][q];
        if (A.part_on_host) __threadfence_system();
    }
}

// Partner chunks when the slices alone leave CUs idle: block (b C + c, m)
// writes the partial F and T of rows 256 b ... against partners [c Nc, (c+1) Nc).
template <int MODE>
__global__ __launch_bounds__(256) void k_virial_chunk(VirialArgs A, AzizDev az) {
    extern __shared__ double lds[];
    const int C = A.chunks;
    const int m = blockIdx.y, b = blockIdx.x / C, c = blockIdx.x - b * C;
    const int n = A.nbs[m];
    const double* px = A.pos + (int64_t)m * A.nalloc;
    const double* py = px + A.plane;
    const double* pz = py + A.plane;
    const bool in_lds = n <= A.lds_beads;
    double* lx = lds;
    double* ly = lds + A.lds_beads;
    double* lz = lds + 2 * A.lds_beads;
    if (in_lds)
        for (int t = threadIdx.x; t < n; t += 256) {
            lx[t] = px[t];
            ly[t] = py[t];
            lz[t] = pz[t];
        }
    __syncthreads();
    const int i = b * 256 + threadIdx.x;
    if (i >= n) return;
    const int nc = (n + C - 1) / C;
    const int j0 = c * nc, j1 = min(n, j0 + nc);
    const bool need_t = (m & 1) ? A.t_odd : A.t_even;
    double F[3] = {0.0, 0.0, 0.0}, T[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (in_lds)
        bead_pairs<MODE>(lx, ly, lz, j0, j1, i, A.box, az, need_t, F, T);
    else
        bead_pairs<MODE>(px, py, pz, j0, j1, i, A.box, az, need_t, F, T);
    double* o = A.fpart + (((int64_t)m * C + c) * A.nalloc + i) * 9;
    for (int q = 0; q < 3; ++q) o[q] = F[q];
    if (need_t)
        for (int q = 0; q < 6; ++q) o[3 + q] = T[q];
}

// How k_virial_sym shares the slices' offsets among its workgroups: a slice has
// `steps` of them, each of weight w (8 where T is needed, 5 elsewhere: about their
// issue slots), and workgroup g takes the steps that end in its equal share of the
// total weight: one that straddles two shares goes to the later workgroup.  Every
// workgroup's share is at least one step.  The whole numbers stay far below 2^52 and so their FP64 quotients floor exactly
// (a 64-bit integer division is a hundred scalar instructions).
struct SymShare {
    double steps, we, wo, total, wgs;
    __device__ __host__ SymShare(int tiles, int M, int t_even, int t_odd, int wgs_)
        : steps(32.0 * tiles), we(t_even ? 8.0 : 5.0), wo(t_odd ? 8.0 : 5.0), wgs(wgs_) {
        total = start(M);
    }
    __device__ __host__ static double quot(double a, double b) { return floor(a / b); }
    __device__ __host__ double weight(int m) const { return (m & 1) ? wo : we; }
    __device__ __host__ double start(int m) const { return steps * (((m + 1) >> 1) * we + (m >> 1) * wo); }
    // the first step of workgroup g as (slice, step); workgroup wgs: (M, 0)
    __device__ __host__ void first(int g, int* m, int* s) const {
        const double b = quot(g * total, wgs), two = steps * (we + wo), p = quot(b, two);
        *m = 2 * (int)p + (b - p * two >= steps * we ? 1 : 0);
        *s = (int)quot(b - start(*m), weight(*m));
    }
    // the workgroup that takes step s of slice m
    __device__ __host__ int owner(int m, double s) const {
        return (int)quot((start(m) + (s + 1.0) * weight(m)) * wgs - 1.0, total);
    }
};

// Slices of at most kVirialSymBeads beads: each unordered pair once, F_j -= g and
// T_j += t beside F_i += g and T_i += t.  FP64 bound (about 165 issue slots for a
// pair with T, 100 without; as ordered pairs twice that).
// The slice's beads form `tiles` tiles of 64.  A wave owns tile w of one of waves
// / tiles groups and meets tile w + r in round r; within a round the waves of a group
// write different tiles of the group's LDS sums, and the rounds are separated by
// barriers, so every sum has one fixed order.  In the last round of an even number
// of tiles both waves of a tile pair take half of the offsets.  The groups share out
// the offsets; waves beyond the last whole group only help to stage the slice (5 of 8
// waves work at five tiles, 6 of 8 at three and six, 9 of 16 at nine).  16 waves per CU
// (126 VGPRs), each workgroup with an equal share of all slices' offsets: with half a slice with T or a whole one without it
// as the unit, N = 256 and M = 166 took 72 us (two uneven rounds of the CUs).
// A sum entry is nine doubles (18 banks: the 32 lanes of a half-wave hit 32 different
// pairs of banks).
// N = 256, M = 166, T on odd slices: 41 us (61 % of it issuing VALU instructions),
// against 55 us as ordered pairs with chunks of partners.
template <int MODE>
__global__ __launch_bounds__(1024) void k_virial_sym(VirialArgs A, AzizDev az) {
    extern __shared__ double lds[];
    const int tiles = A.tiles, W = tiles << 6, threads = 64 * A.waves, groups = A.waves / tiles;
    double* lx = lds;
    double* ly = lx + W;
    double* lz = ly + W;
    double* sums = lz + W;   // [groups][W][9]
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int grp = wave / tiles, tile = wave - grp * tiles;
    const bool works = grp < groups;
    const int i = (tile << 6) + lane;
    double* gs = sums + (works ? grp : 0) * 9 * W;
    const double inv_dr = 1.0 / az.dr;
    // a component this near L/2 may fold the same way from either end
    const double tie = 0.5 * (1.0 - 1e-12) * A.box.L;
    const SymShare share(tiles, A.num_slices, A.t_even, A.t_odd, A.wgs);
    int m0, s0, m1, s1;
    share.first(blockIdx.x, &m0, &s0);
    share.first(blockIdx.x + 1, &m1, &s1);
    for (int m = m0; m < A.num_slices && (m < m1 || (m == m1 && s1 > 0)); ++m) {
        const int from = m == m0 ? s0 : 0, to = m == m1 ? s1 : (int)share.steps;
        const int n = A.nbs[m];
        const bool need_t = (m & 1) ? A.t_odd : A.t_even;
        for (int t = threadIdx.x; t < n; t += threads) {
            const double* p = A.pos + (int64_t)m * A.nalloc + t;
            lx[t] = p[0];
            ly[t] = p[A.plane];
            lz[t] = p[2 * A.plane];
        }
        for (int t = threadIdx.x; t < groups * 9 * W; t += threads) sums[t] = 0.0;
        __syncthreads();
        double F[3] = {0.0, 0.0, 0.0}, T[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        double xi = 0.0, yi = 0.0, zi = 0.0;
        if (works && i < n) {
            xi = lx[i];
            yi = ly[i];
            zi = lz[i];
        }
        int base = 0;   // the round's first step
        for (int rd = 0; 2 * rd <= tiles; ++rd) {
            int tj = tile + rd;
            if (tj >= tiles) tj -= tiles;
            const bool half = rd == 0 || 2 * rd == tiles;
            const int len = half ? 32 : 64;
            const int shift = (rd == 0 || (half && tile > tj)) ? 1 : 0;   // offsets 1 .. 32, not 0 .. 31
            const int lo = max(from - base, 0), hi = min(to - base, len);
            base += len;
            for (int u = lo + grp; works && u < hi; u += groups) {
                // one step's sums are in LDS before the next step reads them (the
                // wave runs in step; this keeps the compiler from reordering)
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const int off = u + shift;
                const int j = (tj << 6) + ((lane + off) & 63);
                if (i >= n || j >= n || (rd == 0 && off == 32 && lane >= 32)) continue;
                double s[3], g[3], t[6];
                if (!virial_pair<MODE>(xi - lx[j], yi - ly[j], zi - lz[j], A.box, az, inv_dr, need_t, s, g, t)) continue;
#pragma unroll
                for (int q = 0; q < 3; ++q) F[q] += g[q];
                if (need_t) {
#pragma unroll
                    for (int q = 0; q < 6; ++q) T[q] += t[q];
                }
                const double far = fmax(fmax(__builtin_fabs(s[0]), __builtin_fabs(s[1])), __builtin_fabs(s[2]));
                if (__builtin_expect(far >= tie, 0)) {
                    const double a0 = fold_sign<MODE>(lx[j] - xi, s[0], A.box);
                    const double a1 = fold_sign<MODE>(ly[j] - yi, s[1], A.box);
                    const double a2 = fold_sign<MODE>(lz[j] - zi, s[2], A.box);
                    g[0] *= a0;
                    g[1] *= a1;
                    g[2] *= a2;
                    if (need_t) {
                        t[1] *= a0 * a1;
                        t[2] *= a0 * a2;
                        t[4] *= a1 * a2;
                    }
                }
                double* e = gs + 9 * j;
#pragma unroll
                for (int q = 0; q < 3; ++q) e[q] -= g[q];
                if (need_t) {
#pragma unroll
                    for (int q = 0; q < 6; ++q) e[3 + q] += t[q];
                }
            }
            __syncthreads();
        }
        if (works && i < n) {
            double* e = gs + 9 * i;
#pragma unroll
            for (int q = 0; q < 3; ++q) e[q] += F[q];
            if (need_t) {
#pragma unroll
                for (int q = 0; q < 6; ++q) e[3 + q] += T[q];
            }
        }
        __syncthreads();
        // (without T its entries are zeros, which nothing reads)
        double* o = A.fpart + ((int64_t)m * A.chunks + ((int)blockIdx.x - share.owner(m, 0))) * 9 * A.nalloc;
        for (int t = threadIdx.x; t < 9 * n; t += threads) {
            double v = sums[t];
            for (int h = 1; h < groups; ++h) v += sums[h * 9 * W + t];
            o[t] = v;
        }
        __syncthreads();
    }
}

// The chunks of each row summed in chunk order, then the per-bead terms.
__global__ __launch_bounds__(256) void k_virial_sum(VirialArgs A) {
    __shared__ double red[4][kVirialTerms];
    const int m = blockIdx.y, b = blockIdx.x;
    const bool need_t = (m & 1) ? A.t_odd : A.t_even;
    int C = A.chunks;
    if (A.tiles) {
        const SymShare share(A.tiles, A.num_slices, A.t_even, A.t_odd, A.wgs);
        C = share.owner(m, share.steps - 1) - share.owner(m, 0) + 1;
    }
    const int n = A.nbs[m];
    const int i = b * 256 + threadIdx.x;
    double o[kVirialTerms];
#pragma unroll
    for (int q = 0; q < kVirialTerms; ++q) o[q] = 0.0;
    if (i < n) {
        double F[3] = {0.0, 0.0, 0.0}, T[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int c = 0; c < C; ++c) {
            const double* p = A.fpart + (((int64_t)m * A.chunks + c) * A.nalloc + i) * 9;
            for (int q = 0; q < 3; ++q) F[q] += p[q];
            if (need_t)
                for (int q = 0; q < 6; ++q) T[q] += p[3 + q];
        }
        A.next ? bead_finish<true>(A, m, i, F, T, o) : bead_finish<false>(A, m, i, F, T, o);
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < kVirialTerms; ++q) {
        const double v = wave_sum(o[q]);
        if (lane == 0) red[wave][q] = v;
    }
    __syncthreads();
    if (threadIdx.x < kVirialTerms) {
        const int q = threadIdx.x;
        A.part[((int64_t)m * ((A.nalloc + 255) >> 8) + b) * kVirialTerms + q] = ((red[0][q] + red[1][q]) + red[2][q]) + red[3][q];
        if (A.part_on_host) __threadfence_system();
    }
}

}  // namespace

void virial_chunks(VirialArgs* A, int num_cus) {
    if (A->nalloc > kVirialSymBeads) {
        A->tiles = A->wgs = 0;
        A->chunks = gradv2_chunks(A->nalloc, A->num_slices, num_cus);
        return;
    }
    A->tiles = std::max(1, (A->nalloc + 63) / 64);
    A->waves = A->tiles <= 8 ? 8 : 16;   // (4 for one to four tiles: no faster, twice the partials)
    // 16 waves per CU, those that work with at least one step each
    const int64_t steps = (int64_t)A->num_slices * 32 * A->tiles;
    A->wgs = (int)std::max<int64_t>(
        1, std::min<int64_t>(num_cus * (16 / A->waves), steps / (2 * (A->waves / A->tiles))));
    const SymShare share(A->tiles, A->num_slices, A->t_even, A->t_odd, A->wgs);
    A->chunks = 1;
    for (int m = 0; m < A->num_slices; ++m)
        A->chunks = std::max(A->chunks, share.owner(m, share.steps - 1) - share.owner(m, 0) + 1);
}

hipError_t launch_virial(int mode, hipStream_t st, const VirialArgs& A, const AzizDev& az, int* blocks_per_slice) {
    (void)hipGetLastError();
    const int B = (A.nalloc + 255) / 256;
    *blocks_per_slice = B;
    dim3 g(B, A.num_slices), b(256);
    if (A.tiles) {
        auto go = [&](auto kern, std::atomic<bool>& attr_set) -> hipError_t {
            // at most 3 * 1024 positions and 16 * 9 * 64 sums (fewer tiles: no more sums)
            constexpr size_t most = sizeof(double) * (3 * kVirialSymBeads + 16 * 9 * 64);
            if (!attr_set.load(std::memory_order_acquire)) {
                const hipError_t e =
                    hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
                if (e != hipSuccess) return e;
                attr_set.store(true, std::memory_order_release);
            }
            const size_t lds = sizeof(double) * (size_t)(3 * 64 * A.tiles + A.waves * 9 * 64);
            hipLaunchKernelGGL(kern, dim3(A.wgs), dim3(64 * A.waves), lds, st, A, az);
            return hipGetLastError();
        };
        static std::atomic<bool> set[3];
        const hipError_t e = mode == 2   ? go(k_virial_sym<2>, set[2])
                             : mode == 1 ? go(k_virial_sym<1>, set[1])
                                         : go(k_virial_sym<0>, set[0]);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_virial_sum, g, b, 0, st, A);
        return hipGetLastError();
    }
    const size_t lds = sizeof(double) * 3 * (size_t)A.lds_beads;
    if (A.chunks > 1) {
        dim3 gc(B * A.chunks, A.num_slices);
        if (mode == 2)
            hipLaunchKernelGGL(k_virial_chunk<2>, gc, b, lds, st, A, az);
        else if (mode == 1)
            hipLaunchKernelGGL(k_virial_chunk<1>, gc, b, lds, st, A, az);
        else
            hipLaunchKernelGGL(k_virial_chunk<0>, gc, b, lds, st, A, az);
        hipLaunchKernelGGL(k_virial_sum, g, b, 0, st, A);
        return hipGetLastError();
    }
    if (mode == 2)
        hipLaunchKernelGGL(k_virial<2>, g, b, lds, st, A, az);
    else if (mode == 1)
        hipLaunchKernelGGL(k_virial<1>, g, b, lds, st, A, az);
    else
        hipLaunchKernelGGL(k_virial<0>, g, b, lds, st, A, az);
    return hipGetLastError();
}

}  // namespace pimc
