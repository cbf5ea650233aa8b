// pimc_sq.hip -- density modes, S(q) and F(q,tau) for gfx950.
//
// The reference's estimators are direct pair sums:
//   S:  sf(q)      = sum_m [N_m + 2 sum_{i<j} cos(q . r_ij)]          (src/estimator.cpp:3705-3737)
//   F:  isf(q,tau) = sum_m sum_{i in m} sum_{j in m+tau} cos(q.r_i - q.r_j)  (:3923-3961)
// Both equal sums over the density mode rho_q(m) = sum_i exp(i q . r_i(m)):
//   sf(q) = sum_m |rho_q(m)|^2,   isf(q,tau) = sum_m Re rho_q(m) conj(rho_q(m+tau)),
// exactly for F and, for S, whenever q is a reciprocal-lattice vector of the
// periodic box (then the minimum image drops out of the phase).  The kernels
// build rho_q(m) once (O(n_q M N)) and then correlate in imaginary time
// (O(n_q M^2)) instead of O(n_q M^2 N^2) trigonometric pair terms.
//
// Lattice q = (2 pi / L) n: exp(i q.r) = prod_d exp(2 pi i n_d s_d), s_d = x_d / L.
// Each workgroup stages per-bead axis phasors exp(2 pi i n s_d) in LDS (phase in
// quarter turns reduced in FP64, sine and cosine of the rest as FP32 series, for n < 4
// and multiples of four; the others one product of those) and sums X Y Z over the beads
// with FP32 products and FP64 sums every 32 beads: as real matrix products on the matrix cores for a
// list of q (k_rho_matrix), or one lane per q (k_rho_lattice).  q and -q have
// conjugate modes and equal S and F, so a list's modes are formed once per pair.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "pimc_kernels.hpp"

namespace pimc {

constexpr int kRhoThreads = 256;
constexpr int kRhoBeadChunk = 32;  // beads per LDS phasor stage
constexpr int kMaxNmax = 40;       // largest |n_d| of a lattice q

// Per-bead axis phasors E(n) = exp(2 pi i n s), s = x_d / L, of one stage of
// kRhoBeadChunk beads (beads past the slice's last are zero), bead-major in LDS:
// x and z for 0 <= n <= H, y for -H <= n <= H, up to the list's own nmax[d] <= H.
// H is fixed at compile time, so a bead's rows are an immediate offset apart, and
// even, so the row lengths are odd and the beads start on distinct LDS banks.
// n < 4 and the multiples of four are evaluated (seeds(): the phase in quarter
// turns reduced in FP64, sine and cosine of the remainder in FP32), the others are
// one complex product E(4 a) E(b) of those (products(), after a barrier): no entry
// is more than one product away from an evaluated one.  Each pass walks (entry,
// bead), bead fastest, over the whole workgroup, the entries through descriptors
// made once.  Both kernels below read tables made here.
template <int H>
struct Phasors {
    static constexpr int WX = H + 1, WY = 2 * H + 1, WZ = H + 1;
    static constexpr int X = 0, Y = kRhoBeadChunk * WX, Z = Y + kRhoBeadChunk * WY;
    // and 16 more: the matrix form reads columns up to 15 past a row's end (unused)
    static constexpr int kEntries = Z + kRhoBeadChunk * WZ + 16;
    static constexpr int kSeeds = 3 * (4 + H / 4), kProducts = 3 * (H - 3 - H / 4);
    struct Entries {
        int4 seed[kSeeds];       // place, row length | (place of -n, + 1) << 8, 4 n, 32 axis
        int4 product[kProducts]; // place, row length | (place of -n, + 1) << 8, places of the factors
        int n_seeds, n_products;
    };
    static __device__ __forceinline__ int count_seeds(int h) { return h < 4 ? h + 1 : 4 + h / 4; }
    // by every lane, before a barrier
    static __device__ __forceinline__ void make_entries(Entries& E, const int nmax[3]) {
        const int base[3] = {X, Y + H, Z}, width[3] = {WX, WY, WZ};
        int s0 = 0, p0 = 0;
#pragma unroll
        for (int axis = 0; axis < 3; ++axis) {
            const int h = nmax[axis], ns = count_seeds(h), np = h + 1 - ns;
            for (int e = threadIdx.x; e < ns; e += (int)blockDim.x) {
                const int n = e < 4 ? e : 4 * (e - 3);
                const int back = axis == 1 && n ? base[1] - n + 1 : 0;
                E.seed[s0 + e] = make_int4(base[axis] + n, width[axis] | back << 8, 4 * n, kRhoBeadChunk * axis);
            }
            for (int e = threadIdx.x; e < np; e += (int)blockDim.x) {
                const int n4 = 4 * (1 + e / 3), n1 = 1 + e % 3, n = n4 + n1;
                const int back = axis == 1 ? base[1] - n + 1 : 0;
                E.product[p0 + e] = make_int4(base[axis] + n, width[axis] | back << 8, base[axis] + n4, base[axis] + n1);
            }
            s0 += ns;
            p0 += np;
        }
        if (threadIdx.x == 0) {
            E.n_seeds = s0;
            E.n_products = p0;
        }
    }
    // at: the beads' positions in box units, |at| <= 1/2, [3][kRhoBeadChunk] in LDS
    static __device__ __forceinline__ void seeds(float2* t, const Entries& E, const double* at, int nb) {
        const int bb = threadIdx.x & (kRhoBeadChunk - 1);
        for (int e = threadIdx.x / kRhoBeadChunk; e < E.n_seeds; e += (int)blockDim.x / kRhoBeadChunk) {
            const int4 d = E.seed[e];
            // quarter turns: the nearest whole number k and the rest, |r| <= 1/2,
            // whose FP32 rounding is under 2.4e-8 of a radian
            const double v = (double)d.z * at[d.w + bb];
            const double k = rint(v);
            const float r = (float)(v - k) * 1.57079632679489662f;
            const int quad = (int)k;
            // sine and cosine by their series, |r| <= pi/4 (last terms r^9/9!, r^10/10!)
            const float r2 = r * r;
            float sn = fmaf(r2, 2.7557319e-6f, -1.9841270e-4f);
            sn = fmaf(r2, sn, 8.3333333e-3f);
            sn = fmaf(r2, sn, -1.6666667e-1f);
            sn = fmaf(r2 * r, sn, r);
            float cs = fmaf(r2, -2.7557319e-7f, 2.4801587e-5f);
            cs = fmaf(r2, cs, -1.3888889e-3f);
            cs = fmaf(r2, cs, 4.1666667e-2f);
            cs = fmaf(r2, cs, -0.5f);
            cs = fmaf(r2, cs, 1.0f);
            const bool odd = quad & 1;
            float c = odd ? sn : cs, s = odd ? cs : sn;
            // E rotates by i every quarter turn: (c, s) -> (-s, c)
            c = ((quad + 1) & 2) ? -c : c;
            s = (quad & 2) ? -s : s;
            if (bb >= nb) c = s = 0.f;
            const int w = d.y & 255, back = d.y >> 8;
            t[d.x + bb * w] = make_float2(c, s);
            if (back) t[back - 1 + bb * w] = make_float2(c, -s);
        }
    }
    static __device__ __forceinline__ void products(float2* t, const Entries& E) {
        const int bb = threadIdx.x & (kRhoBeadChunk - 1);
        for (int e = threadIdx.x / kRhoBeadChunk; e < E.n_products; e += (int)blockDim.x / kRhoBeadChunk) {
            const int4 d = E.product[e];
            const int w = d.y & 255, back = d.y >> 8;
            const float2 p = t[d.z + bb * w], q = t[d.w + bb * w];
            const float c = fmaf(p.x, q.x, -p.y * q.y);
            const float s = fmaf(p.x, q.y, p.y * q.x);
            t[d.x + bb * w] = make_float2(c, s);
            if (back) t[back - 1 + bb * w] = make_float2(c, -s);
        }
    }
};
static_assert(kMaxNmax <= 40 && 2 * 40 + 1 < 256, "row lengths take 8 bits");

// A coordinate in box units, less its whole boxes (they drop out of lattice phases).
__device__ __forceinline__ double box_fraction(double x, double invL) {
    const double s = x * invL;
    return s - rint(s);
}

// rho at +n_z (sg = +1) or -n_z (sg = -1) of a row (n_x, n_y) from its four real
// sums over the beads, with X Y = xr + i xi and Z(|n_z|) = c + i s:
//   rc = sum xr c, rs = sum xr s, ic = sum xi c, is = sum xi s.
__device__ __forceinline__ double2 rho_of_sums(double rc, double rs, double ic, double is, double sg) {
    return make_double2(rc - sg * is, ic + sg * rs);
}

// rho_q(m) for lattice q, one lane per q (lane t of a workgroup takes q = base +
// t + 256 k, k < QPT): the form for q lists too sparse for the matrix form below and,
// a lane for every q of the list, of the callers that make no plan (pimc_ssf_noalloc and
// the server; 4913 q, N = 256 x 167: 164 us a call).  q and -q are conjugates, so a q is first turned into
// the half space n_x > 0, or n_x = 0 and n_y > 0, ...: the sums, their order
// (32 beads in FP32, then FP64) and so the bits are those of the matrix form.
template <int QPT, int H>
__global__ __launch_bounds__(kRhoThreads) void k_rho_lattice(RhoArgs A) {
    using T = Phasors<H>;
    __shared__ float2 ph[T::kEntries];
    __shared__ typename T::Entries E;
    __shared__ double at[3 * kRhoBeadChunk];
    const int m = blockIdx.y;
    const int n_beads = A.nbs[m];
    const double* px = A.pos + (int64_t)m * A.nalloc;
    const int qbase = blockIdx.x * kRhoThreads * QPT + threadIdx.x;
    int ix[QPT], iy[QPT], iz[QPT];
    double sg[QPT], cj[QPT];
#pragma unroll
    for (int k = 0; k < QPT; ++k) {
        const int qi = qbase + k * kRhoThreads;
        int nx = 0, ny = 0, nz = 0;
        if (qi < A.nq) {
            nx = A.qn[3 * qi];
            ny = A.qn[3 * qi + 1];
            nz = A.qn[3 * qi + 2];
        }
        const bool flip = nx < 0 || (nx == 0 && (ny < 0 || (ny == 0 && nz < 0)));
        cj[k] = flip ? -1.0 : 1.0;
        ix[k] = flip ? -nx : nx;
        iy[k] = H + (flip ? -ny : ny);
        iz[k] = nz < 0 ? -nz : nz;
        sg[k] = (flip ? -nz : nz) < 0 ? -1.0 : 1.0;
    }
    double rc[QPT], rs[QPT], ic[QPT], is[QPT];
#pragma unroll
    for (int k = 0; k < QPT; ++k) rc[k] = rs[k] = ic[k] = is[k] = 0.0;
    T::make_entries(E, A.nmax);
    for (int b0 = 0; b0 < n_beads; b0 += kRhoBeadChunk) {
        const int nb = min(kRhoBeadChunk, n_beads - b0);
        __syncthreads();
        if (threadIdx.x < 3 * kRhoBeadChunk) {
            const int axis = threadIdx.x / kRhoBeadChunk, bb = threadIdx.x % kRhoBeadChunk;
            at[threadIdx.x] = bb < nb ? box_fraction(px[axis * A.plane + b0 + bb], A.invL) : 0.0;
        }
        __syncthreads();
        T::seeds(ph, E, at, nb);
        __syncthreads();
        T::products(ph, E);
        __syncthreads();
        float frc[QPT], frs[QPT], fic[QPT], fis[QPT];
#pragma unroll
        for (int k = 0; k < QPT; ++k) frc[k] = frs[k] = fic[k] = fis[k] = 0.f;
        // byte offsets walked bead by bead, the compiler not told how far apart they are:
        // it would read two beads at once (ds_read2_b64), which keeps the LDS busy four
        // cycles a value where ds_read_b64 takes some two, and the kernel is bound by that
        // (9261 q, N = 2048 x 100: 957 -> 769 us)
        unsigned ox[QPT], oy[QPT], oz[QPT];
#pragma unroll
        for (int k = 0; k < QPT; ++k) {
            ox[k] = sizeof(float2) * (T::X + ix[k]);
            oy[k] = sizeof(float2) * (T::Y + iy[k]);
            oz[k] = sizeof(float2) * (T::Z + iz[k]);
        }
        auto entry = [&](unsigned& o, unsigned step) {
            const float2 v = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(ph) + o);
            o += sizeof(float2) * step;
            asm("" : "+v"(o));
            return v;
        };
        auto bead = [&]() {
#pragma unroll
            for (int k = 0; k < QPT; ++k) {
                const float2 ex = entry(ox[k], T::WX);
                const float2 ey = entry(oy[k], T::WY);
                const float2 ez = entry(oz[k], T::WZ);
                const float xr = fmaf(ex.x, ey.x, -ex.y * ey.y);
                const float xi = fmaf(ex.x, ey.y, ex.y * ey.x);
                frc[k] = fmaf(xr, ez.x, frc[k]);
                frs[k] = fmaf(xr, ez.y, frs[k]);
                fic[k] = fmaf(xi, ez.x, fic[k]);
                fis[k] = fmaf(xi, ez.y, fis[k]);
            }
        };
        int left = nb;
        for (; left >= 4; left -= 4) {
            bead();
            bead();
            bead();
            bead();
        }
        for (; left > 0; --left) bead();
#pragma unroll
        for (int k = 0; k < QPT; ++k) {
            rc[k] += (double)frc[k];
            rs[k] += (double)frs[k];
            ic[k] += (double)fic[k];
            is[k] += (double)fis[k];
        }
    }
#pragma unroll
    for (int k = 0; k < QPT; ++k) {
        const int qi = qbase + k * kRhoThreads;
        if (qi < A.nq) {
            const double2 v = rho_of_sums(rc[k], rs[k], ic[k], is[k], sg[k]);
            reinterpret_cast<double2*>(A.rho)[(int64_t)m * A.nq + qi] = make_double2(v.x, cj[k] * v.y);
        }
    }
}

// rho_q(m) of a whole list of lattice q as real matrix products.  For a slice the
// rows (n_x, n_y) of the list's half space and the columns |n_z| make
//   rho(n_x, n_y, +-n_z) = sum_b X Y(row, b) Z(n_z, b)^(+-1),
// four real products (Re or Im of X Y against cos or sin of Z) whose sums give
// both signs of n_z (rho_of_sums).  A wave takes a job of 16 rows by 16 columns:
// four accumulators of v_mfma_f32_16x16x4_f32 (lane l: row and column l % 16,
// bead l / 16 of the four of a step; the unit adds the four products in bead
// order with one rounding each, as the chain of FP32 FMA it replaces).  The X Y
// operand is formed in registers from the phasor tables, four FMA per step, so
// nothing but the tables is staged; up to 16 waves of a workgroup share them.
// Every 32 beads the FP32 sums go into FP64 ones, as in k_rho_lattice.  Three
// table buffers: while stage c is summed, stage c + 1 gets its products and
// stage c + 2 its seeds, one barrier per stage.
// Bound: the FP32 matrix rate (126 TFLOP/s measured here), 128 SIMD cycles per job
// and four beads; the unit shares the vector unit's multipliers, so the tables, the
// X Y operands and the FP64 sums (about a third of the time) add to it.  At N = 2048
// x 250 the 50 201 modes of 100 401 q take 2.0 ms (one lane per mode 8.1 ms), at N = 256
// x 167 the 2689 modes of 5377 q 33 us (57 us).  Waves that only make tables beside
// waves that only sum were
// slower (2.8 ms), as were 8 waves to a workgroup (2.9 ms).
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kRhoWaves = 16;

template <int H>
__global__ __launch_bounds__(64 * kRhoWaves) void k_rho_matrix(RhoMatrixArgs A) {
    using T = Phasors<H>;
    extern __shared__ float2 ph[];                 // [3][T::kEntries]
    __shared__ typename T::Entries E;
    __shared__ double at[2][3 * kRhoBeadChunk];   // positions in box units, two stages
    const int m = blockIdx.y;
    const int n_beads = A.nbs[m];
    const int stages = (n_beads + kRhoBeadChunk - 1) / kRhoBeadChunk;
    const double* px = A.pos + (int64_t)m * A.nalloc;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int j = A.job0 + blockIdx.x * ((int)blockDim.x >> 6) + wave;
    const bool work = j < A.job_end;
    const RhoJob job = work ? A.jobs[j] : RhoJob{0, 0};
    const int l16 = lane & 15, l4 = lane >> 4;
    const int2 row = work ? A.rows[16 * job.tile + l16] : make_int2(0, 0);
    const int ix = T::X + l4 * T::WX + row.x;
    const int iy = T::Y + l4 * T::WY + H + row.y;
    const int iz = T::Z + l4 * T::WZ + job.col0 + l16;
    double sum[4][4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[k][r] = 0.0;
    auto make_seeds = [&](int c) {
        if (c < stages)
            T::seeds(ph + (c % 3) * T::kEntries, E, at[c & 1], min(kRhoBeadChunk, n_beads - c * kRhoBeadChunk));
    };
    auto make_products = [&](int c) {
        if (c < stages) T::products(ph + (c % 3) * T::kEntries, E);
    };
    // a stage's positions: lanes 0 .. 95 load them one stage before they are put
    // into LDS, so no pass waits for memory
    const int p_axis = threadIdx.x / kRhoBeadChunk, p_bead = threadIdx.x % kRhoBeadChunk;
    auto load_pos = [&](int c) {
        const int b = c * kRhoBeadChunk + p_bead;
        return p_axis < 3 && b < n_beads ? box_fraction(px[p_axis * A.plane + b], A.invL) : 0.0;
    };
    auto put_pos = [&](int c, double v) {
        if (p_axis < 3) at[c & 1][threadIdx.x] = v;
    };
    auto sum_stage = [&](int c) {
        if (!work) return;
        const float2* t = ph + (c % 3) * T::kEntries;
        const float2 *bx = t + ix, *by = t + iy, *bz = t + iz;
        const int steps = (min(kRhoBeadChunk, n_beads - c * kRhoBeadChunk) + 3) >> 2;
        f32x4 acc[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto step = [&](int k) {
            const float2 ex = bx[4 * k * T::WX], ey = by[4 * k * T::WY], ez = bz[4 * k * T::WZ];
            const float xr = fmaf(ex.x, ey.x, -ex.y * ey.y);
            const float xi = fmaf(ex.x, ey.y, ex.y * ey.x);
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xr, ez.x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xr, ez.y, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(xi, ez.x, acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(xi, ez.y, acc[3], 0, 0, 0);
        };
        if (steps == kRhoBeadChunk / 4) {
#pragma unroll
            for (int k = 0; k < kRhoBeadChunk / 4; ++k) step(k);
        } else {
            for (int k = 0; k < steps; ++k) step(k);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[k][r] += (double)acc[k][r];
    };
    T::make_entries(E, A.nmax);
    put_pos(0, load_pos(0));
    put_pos(1, load_pos(1));
    __syncthreads();
    double ahead = load_pos(2);
    make_seeds(0);
    make_seeds(1);
    __syncthreads();
    make_products(0);
    put_pos(2, ahead);
    __syncthreads();
    for (int c = 0; c < stages; ++c) {
        ahead = load_pos(c + 3);
        make_products(c + 1);
        make_seeds(c + 2);
        sum_stage(c);
        put_pos(c + 3, ahead);   // the other of the two: seeds of stage c + 1 are done
        __syncthreads();
    }
    if (!work) return;
    // lane l, register r: row 4 (l / 16) + r, column l % 16
    double2* out = reinterpret_cast<double2*>(A.rho) + (int64_t)m * A.nu;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int* slot = A.slot + (int64_t)(16 * job.tile + 4 * l4 + r) * 2 * A.width + job.col0 + l16;
        const int up = slot[0], un = slot[A.width];
        if (up >= 0) out[up] = rho_of_sums(sum[0][r], sum[1][r], sum[2][r], sum[3][r], 1.0);
        if (un >= 0) out[un] = rho_of_sums(sum[0][r], sum[1][r], sum[2][r], sum[3][r], -1.0);
    }
}

// General q: rho_q(m) = sum_i exp(i q . r_i) with the phase reduced in FP64.
__global__ __launch_bounds__(kRhoThreads) void k_rho_general(RhoArgs A) {
    const int m = blockIdx.y;
    const int qi = blockIdx.x * kRhoThreads + threadIdx.x;
    if (qi >= A.nq) return;
    const double qx = A.q[3 * qi], qy = A.q[3 * qi + 1], qz = A.q[3 * qi + 2];
    const double* px = A.pos + (int64_t)m * A.nalloc;
    const double* py = px + A.plane;
    const double* pz = py + A.plane;
    const int n = A.nbs[m];
    double re = 0.0, im = 0.0;
    constexpr double kInv2Pi = 0.15915494309189533577;
    for (int b0 = 0; b0 < n; b0 += 64) {
        float sre = 0.f, sim = 0.f;
        const int e = min(n, b0 + 64);
        for (int b = b0; b < e; ++b) {
            const double phase = qx * px[b] + qy * py[b] + qz * pz[b];
            const double rev = phase * kInv2Pi;
            const double red = rev - rint(rev);
            float s, c;
            sincospif((float)(2.0 * red), &s, &c);
            sre += c;
            sim += s;
        }
        re += (double)sre;
        im += (double)sim;
    }
    A.rho[((int64_t)m * A.nq + qi) * 2 + 0] = re;
    A.rho[((int64_t)m * A.nq + qi) * 2 + 1] = im;
}

// F(q,tau) = sum_m Re rho(m) conj(rho(m+tau)).  A workgroup of 4 waves takes
// kIsfQ = 4 modes, one per wave; rho(m) is staged twice over (m and m + M) so lag
// tau reads row[m + tau] with no wrap test: rho(m) is an LDS broadcast,
// rho(m + tau) consecutive words, each lag at a fixed offset.  Rows are 2M + 64
// long: lanes past the last lag read the zero padding.  The sum over the closed
// path makes F(M - tau) = F(tau), so only the lags up to M / 2 are formed.  With
// dst, mode u's lags go to the rows dst[2 u] and dst[2 u + 1] (those of q and -q;
// -1: none), else to row u.
constexpr int kIsfQ = 4;
constexpr int kIsfLagsPerLane = 5;   // M / 2 + 1 <= 257
__global__ __launch_bounds__(256) void k_isf_from_rho(const double* __restrict__ rho, int nu, int u0, int u_end, int M,
                                                     double inv_n, const int* __restrict__ dst,
                                                     double* __restrict__ fqt) {
    extern __shared__ double2 sr[];  // [kIsfQ][2M + 64]
    const int R = 2 * M + 64;
    const int qb = u0 + blockIdx.x * kIsfQ;
    const int nql = min(kIsfQ, u_end - qb);
    for (int t = threadIdx.x; t < M * kIsfQ; t += 256) {
        const int m = t / kIsfQ, k = t % kIsfQ;
        double2 v = make_double2(0.0, 0.0);
        if (k < nql) v = reinterpret_cast<const double2*>(rho)[(int64_t)m * nu + qb + k];
        sr[(int64_t)k * R + m] = v;
        sr[(int64_t)k * R + m + M] = v;
    }
    for (int t = threadIdx.x; t < 64 * kIsfQ; t += 256) sr[(int64_t)(t / 64) * R + 2 * M + (t % 64)] = make_double2(0.0, 0.0);
    __syncthreads();
    const int k = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (k >= nql) return;
    const double2* row = sr + (int64_t)k * R;
    double acc[kIsfLagsPerLane];
#pragma unroll
    for (int u = 0; u < kIsfLagsPerLane; ++u) acc[u] = 0.0;
    const int half = M / 2 + 1;   // lags 0 .. M/2
    const int nl = (half + 63) / 64;
    const double2* b = row + lane;
    for (int m = 0; m < M; ++m, ++b) {
        const double2 a = row[m];
#pragma unroll
        for (int u = 0; u < kIsfLagsPerLane; ++u) {
            if (u < nl) {
                const double2 c = b[64 * u];
                acc[u] = fma(a.x, c.x, acc[u]);
                acc[u] = fma(a.y, c.y, acc[u]);
            }
        }
    }
    const int r0 = dst ? dst[2 * (qb + k)] : qb + k, r1 = dst ? dst[2 * (qb + k) + 1] : -1;
#pragma unroll
    for (int u = 0; u < kIsfLagsPerLane; ++u) {
        const int tau = lane + 64 * u;
        if (u < nl && tau < half) {
            const double v = acc[u] * inv_n;
            const int back = tau ? M - tau : 0;
            if (r0 >= 0) {
                fqt[(int64_t)r0 * M + tau] = v;
                fqt[(int64_t)r0 * M + back] = v;
            }
            if (r1 >= 0) {
                fqt[(int64_t)r1 * M + tau] = v;
                fqt[(int64_t)r1 * M + back] = v;
            }
        }
    }
}

// Rows of q that a list names again: one workgroup each.
__global__ __launch_bounds__(128) void k_isf_repeat(const int2* __restrict__ rep, int M, double* __restrict__ fqt) {
    const int2 r = rep[blockIdx.x];
    const double* from = fqt + (int64_t)r.y * M;
    double* to = fqt + (int64_t)r.x * M;
    for (int t = threadIdx.x; t < M; t += 128) to[t] = from[t];
}

// S(q) contribution = sum_m |rho_q(m)|^2 / N.  A workgroup takes 32 q (32
// consecutive entries of rho, coalesced) with 8 lanes each: lane g adds the
// slices [g seg, (g + 1) seg), seg = ceil(M / 8), in order, eight loads in flight,
// and the eight parts are added in order, so a value depends on M and rho alone.
// With a few hundred q the kernel is a chain of loads, which the 8 lanes cut to
// an eighth; with many it is bound by reading rho
// (50 201 modes x 250: 38 us, 5.3 TB/s).
// done (or null): the last workgroup to finish publishes seq there (ticket: the
// arrival counter, zero between calls); sq is then mapped host memory.
constexpr int kSsfQ = 32, kSsfParts = 8;
__global__ __launch_bounds__(kSsfQ* kSsfParts) void k_ssf_from_rho(const double* __restrict__ rho, int nq, int M,
                                                                  double inv_n, double* __restrict__ sq,
                                                                  unsigned* ticket, unsigned long long* done,
                                                                  unsigned long long seq) {
    __shared__ double part[kSsfParts][kSsfQ];
    const int g = threadIdx.x / kSsfQ, k = threadIdx.x % kSsfQ;
    const int qi = blockIdx.x * kSsfQ + k;
    const int seg = (M + kSsfParts - 1) / kSsfParts;
    double acc = 0.0;
    if (qi < nq) {
        const double2* r = reinterpret_cast<const double2*>(rho) + qi;   // rho_q(m) at r[m nq]
        constexpr int U = 8;
        int m = g * seg;
        const int m_end = min(M, m + seg);
        for (; m + U <= m_end; m += U) {
            double2 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = r[(int64_t)(m + u) * nq];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                acc = fma(v[u].x, v[u].x, acc);
                acc = fma(v[u].y, v[u].y, acc);
            }
        }
        for (; m < m_end; ++m) {
            const double2 v = r[(int64_t)m * nq];
            acc = fma(v.x, v.x, acc);
            acc = fma(v.y, v.y, acc);
        }
    }
    part[g][k] = acc;
    __syncthreads();
    if (g == 0 && qi < nq) {
        double s = part[0][k];
#pragma unroll
        for (int u = 1; u < kSsfParts; ++u) s += part[u][k];
        sq[qi] = s * inv_n;
        if (done) __threadfence_system();
    }
    if (!done) return;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (t + 1 == gridDim.x) {
            __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            publish_done(done, seq);
        }
    }
}

// Direct minimum-image S(q) pair sum for general q: one block per (q, slice).
__global__ __launch_bounds__(256) void k_ssf_pairs(const double* __restrict__ pos, int64_t plane, int nalloc,
                                                  const int* __restrict__ nbs, const double* __restrict__ q,
                                                  BoxDev box, double* __restrict__ partial) {
    __shared__ double red[4];
    const int qi = blockIdx.x, m = blockIdx.y;
    const double qx = q[3 * qi], qy = q[3 * qi + 1], qz = q[3 * qi + 2];
    const double* px = pos + (int64_t)m * nalloc;
    const double* py = px + plane;
    const double* pz = py + plane;
    const int n = nbs[m];
    constexpr double kInv2Pi = 0.15915494309189533577;
    double acc = 0.0;
    const int64_t total = (int64_t)n * n;
    for (int64_t t = threadIdx.x; t < total; t += 256) {
        const int i = (int)(t / n), j = (int)(t % n);
        if (j <= i) continue;
        const double dx = min_image_exact(px[i] - px[j], box.L, box.invL);
        const double dy = min_image_exact(py[i] - py[j], box.L, box.invL);
        const double dz = min_image_exact(pz[i] - pz[j], box.L, box.invL);
        const double rev = (dx * qx + dy * qy + dz * qz) * kInv2Pi;
        const double red2 = rev - rint(rev);
        acc += 2.0 * (double)cospif((float)(2.0 * red2));
    }
    const double s = block_sum<256>(acc, red);
    if (threadIdx.x == 0) partial[(int64_t)qi * gridDim.y + m] = s + (double)n;
}

// sq[q] = sum_m partial[q][m] / N in slice order
__global__ void k_ssf_finish(const double* __restrict__ partial, int nq, int M, double inv_n,
                             double* __restrict__ sq) {
    const int qi = blockIdx.x * blockDim.x + threadIdx.x;
    if (qi >= nq) return;
    double s = 0.0;
    for (int m = 0; m < M; ++m) s += partial[(int64_t)qi * M + m];
    sq[qi] = s * inv_n;
}

// The smallest table size that holds nmax: f(std::integral_constant<int, H>).  FINE: also
// sizes for |n| <= 20 and 24, with which six and five workgroups of k_rho_lattice fit a CU,
// four at 32 (3000 q with |n| <= 20, N = 2048 x 100: 479 -> 381 us).
template <bool FINE, typename F>
static hipError_t for_table_size(const int nmax[3], F f) {
    const int h = std::max(nmax[0], std::max(nmax[1], nmax[2]));
    if (h <= 4) return f(std::integral_constant<int, 4>{});
    if (h <= 8) return f(std::integral_constant<int, 8>{});
    if (h <= 16) return f(std::integral_constant<int, 16>{});
    if constexpr (FINE) {
        if (h <= 20) return f(std::integral_constant<int, 20>{});
        if (h <= 24) return f(std::integral_constant<int, 24>{});
    }
    if (h <= 32) return f(std::integral_constant<int, 32>{});
    return f(std::integral_constant<int, 40>{});
}

hipError_t launch_rho(bool lattice, hipStream_t st, const RhoArgs& A) {
    (void)hipGetLastError();  // drop any stale error of an earlier call
    if (A.nq <= 0) return hipSuccess;
    if (lattice) {
        // the most q per lane that still leaves >= 2048 workgroups
        auto blocks = [&](int qpt) { return (int64_t)((A.nq + kRhoThreads * qpt - 1) / (kRhoThreads * qpt)) * A.num_slices; };
        int qpt = 4;
        while (qpt > 1 && blocks(qpt) < 2048) qpt >>= 1;
        dim3 g((A.nq + kRhoThreads * qpt - 1) / (kRhoThreads * qpt), A.num_slices), b(kRhoThreads);
        (void)for_table_size<true>(A.nmax, [&](auto h) {
            constexpr int H = decltype(h)::value;
            if (qpt == 4) hipLaunchKernelGGL((k_rho_lattice<4, H>), g, b, 0, st, A);
            else if (qpt == 2) hipLaunchKernelGGL((k_rho_lattice<2, H>), g, b, 0, st, A);
            else hipLaunchKernelGGL((k_rho_lattice<1, H>), g, b, 0, st, A);
            return hipSuccess;
        });
    } else {
        dim3 g((A.nq + kRhoThreads - 1) / kRhoThreads, A.num_slices), b(kRhoThreads);
        hipLaunchKernelGGL(k_rho_general, g, b, 0, st, A);
    }
    return hipGetLastError();
}

hipError_t launch_rho_matrix(hipStream_t st, const RhoMatrixArgs& A) {
    (void)hipGetLastError();
    const int jobs = A.job_end - A.job0;
    if (jobs <= 0) return hipSuccess;
    // the jobs spread evenly over the fewest workgroups of up to 16 waves; at least
    // four waves, which share the table passes however few jobs there are
    const int groups = (jobs + kRhoWaves - 1) / kRhoWaves;
    const int waves = std::max(4, (jobs + groups - 1) / groups);
    const hipError_t e = for_table_size<false>(A.nmax, [&](auto h) {
        constexpr int H = decltype(h)::value;
        const size_t lds = 3 * sizeof(float2) * Phasors<H>::kEntries;   // at most 126 KB
        static std::atomic<bool> attr_set{false};
        if (!attr_set.load(std::memory_order_acquire)) {
            const hipError_t e1 = hipFuncSetAttribute((const void*)k_rho_matrix<H>,
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e1 != hipSuccess) return e1;
            attr_set.store(true, std::memory_order_release);
        }
        hipLaunchKernelGGL(k_rho_matrix<H>, dim3(groups, A.num_slices), dim3(64 * waves), lds, st, A);
        return hipSuccess;
    });
    return e != hipSuccess ? e : hipGetLastError();
}

hipError_t launch_isf(hipStream_t st, const double* rho, int nu, int u0, int u_end, int M, double inv_n,
                      const int* dst, double* fqt) {
    (void)hipGetLastError();  // drop any stale error of an earlier call
    if (u_end <= u0) return hipSuccess;
    dim3 g((u_end - u0 + kIsfQ - 1) / kIsfQ), b(256);
    const size_t lds = sizeof(double2) * kIsfQ * (2 * (size_t)M + 64);
    static std::atomic<bool> attr_set{false};
    if (!attr_set.load(std::memory_order_acquire)) {
        // rows of M <= 512 slices need up to 68 KB of the 160 KB LDS
        hipError_t e = hipFuncSetAttribute((const void*)k_isf_from_rho, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           160 * 1024);
        if (e != hipSuccess) return e;
        attr_set.store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL(k_isf_from_rho, g, b, lds, st, rho, nu, u0, u_end, M, inv_n, dst, fqt);
    return hipGetLastError();
}

hipError_t launch_isf_repeat(hipStream_t st, const int2* rep, int n, int M, double* fqt) {
    (void)hipGetLastError();
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_isf_repeat, dim3(n), dim3(128), 0, st, rep, M, fqt);
    return hipGetLastError();
}

hipError_t launch_ssf(hipStream_t st, const double* rho, int nq, int M, double inv_n, double* sq, unsigned* ticket,
                      unsigned long long* done, unsigned long long seq) {
    (void)hipGetLastError();
    if (nq <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ssf_from_rho, dim3((nq + kSsfQ - 1) / kSsfQ), dim3(kSsfQ * kSsfParts), 0, st, rho, nq, M,
                       inv_n, sq, ticket, done, seq);
    return hipGetLastError();
}

hipError_t launch_ssf_pairs(hipStream_t st, const double* pos, int64_t plane, int nalloc, int M, const int* nbs,
                            const double* q, int nq, const BoxDev& box, double* partial, double inv_n, double* sq) {
    (void)hipGetLastError();  // drop any stale error of an earlier call
    if (nq <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ssf_pairs, dim3(nq, M), dim3(256), 0, st, pos, plane, nalloc, nbs, q, box, partial);
    hipLaunchKernelGGL(k_ssf_finish, dim3((nq + 255) / 256), dim3(256), 0, st, partial, nq, M, inv_n, sq);
    return hipGetLastError();
}

int rho_max_nmax() { return kMaxNmax; }

}  // namespace pimc
