// pimc_capi_sq.hip -- host side of the structure-factor entry points and of the
// batched PotentialBase (Aziz) entry points of include/pimc_gpu.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <string>
#include <memory>
#include <utility>
#include <vector>

#include "pimc_host.hpp"

using namespace pimc;

namespace {

int sfail(pimc_ctx* c, int code, const std::string& m) {
    if (c) {
        c->err = m;
        ++c->fail_count;
    }
    return code;
}

#define SHIP(c, expr)                                                                          \
    do {                                                                                       \
        hipError_t _e = (expr);                                                                \
        if (_e != hipSuccess) return sfail((c), PIMC_E_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)

template <typename T>
int grow(pimc_ctx* c, T** p, size_t* cap, size_t need) {
    if (need <= *cap && *p) return PIMC_OK;
    if (*p) {
        (void)hipFree(*p);
        c->dev_allocs.erase(std::remove(c->dev_allocs.begin(), c->dev_allocs.end(), (void*)*p), c->dev_allocs.end());
        *p = nullptr;
    }
    size_t n = std::max<size_t>(need, 1);
    hipError_t e = hipMalloc((void**)p, sizeof(T) * n);
    if (e != hipSuccess) return sfail(c, PIMC_E_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    c->dev_allocs.push_back((void*)*p);
    *cap = n;
    return PIMC_OK;
}

int true_num_particles(pimc_ctx* c) {
    long on = 0;
    for (auto v : c->h_on) on += v;
    return (int)(on / c->desc.num_slices);
}

// Room for nq q-vectors in the device list of the general (non-lattice) forms.
int ensure_q(pimc_ctx* c, int nq) {
    size_t cap = (size_t)c->cap_q;
    const int r = grow(c, &c->d_q, &cap, (size_t)nq * 3);
    if (!r) c->cap_q = (int)cap;
    return r;
}

// The plan of a lattice q list on the device, one copy from pinned memory.
struct DevPlan {
    const int* dst = nullptr;    // [nu][2] list rows of each mode, for F
    const int2* repeat = nullptr;   // {row, row it repeats}, where the device copies them
    int n_repeat = 0;
    RhoMatrixArgs mat{};         // matrix form
    RhoArgs lane{};              // one lane per mode
};

// The rows of a list's repeated q are copied on the device before the result leaves it,
// but a few, whose copies on the host take no longer than a launch.  F of 20 000 q of
// which 11 800 repeat others, N = 16 x 125 (20 MB): 1.20 ms with the host's copies, 0.60 ms
// with the device's.
constexpr size_t kHostRepeatBytes = 64u << 10;

bool device_repeats(const RhoPlan& P, int M) { return P.repeat.size() * (size_t)M * sizeof(double) > kHostRepeatBytes; }

int upload_plan(pimc_ctx* c, const RhoPlan& P, const std::vector<int>& n3, bool want_dst, DevPlan* D) {
    const size_t n_rows = 2 * P.rows.size(), n_jobs = 2 * P.jobs.size(), n_slot = P.slot.size();
    const size_t n_dst = want_dst ? 2 * (size_t)P.nu : 0, n_list = P.matrix ? 0 : 3 * (size_t)P.nu;
    const size_t n_rep = want_dst && device_repeats(P, c->desc.num_slices) ? 2 * P.repeat.size() : 0;
    const size_t need = n_rows + n_jobs + n_rep + n_slot + n_dst + n_list;
    int r;
    if ((r = grow(c, &c->d_plan, &c->cap_plan, std::max<size_t>(need, 16384)))) return r;
    // packed in the context's pinned staging block where it fits (the block holds
    // the path, 24 M N bytes; nothing else uses it during the call)
    std::vector<int> unpinned;
    int* h = reinterpret_cast<int*>(c->h_stage);
    if (sizeof(int) * need > sizeof(double) * c->cap_stage) {
        unpinned.resize(need);
        h = unpinned.data();
    }
    int* d = c->d_plan;
    // the jobs, rows and repeats first: 8-byte records at an aligned start
    size_t o = 0;
    const size_t o_jobs = o;
    if (n_jobs) std::memcpy(h + o, P.jobs.data(), sizeof(int) * n_jobs);
    o += n_jobs;
    const size_t o_rows = o;
    if (n_rows) std::memcpy(h + o, P.rows.data(), sizeof(int) * n_rows);
    o += n_rows;
    const size_t o_rep = o;
    for (size_t t = 0; t < n_rep / 2; ++t) {
        h[o + 2 * t] = P.repeat[t];
        h[o + 2 * t + 1] = P.first[P.mode[P.repeat[t]]];
    }
    o += n_rep;
    const size_t o_slot = o;
    if (n_slot) std::memcpy(h + o, P.slot.data(), sizeof(int) * n_slot);
    o += n_slot;
    const size_t o_dst = o;
    for (int u = 0; u < (int)(n_dst / 2); ++u) {
        h[o + 2 * (size_t)u] = P.first[u];
        h[o + 2 * (size_t)u + 1] = P.second[u];
    }
    o += n_dst;
    const size_t o_list = o;
    for (int u = 0; u < (int)(n_list / 3); ++u)
        for (int k = 0; k < 3; ++k) h[o + 3 * (size_t)u + k] = n3[3 * (size_t)P.first[u] + k];
    SHIP(c, hipMemcpyAsync(d, h, sizeof(int) * need, hipMemcpyHostToDevice, c->stream));
    if (!unpinned.empty()) SHIP(c, hipStreamSynchronize(c->stream));
    D->dst = want_dst ? d + o_dst : nullptr;
    D->repeat = reinterpret_cast<const int2*>(d + o_rep);
    D->n_repeat = (int)(n_rep / 2);
    if (P.matrix) {
        RhoMatrixArgs& A = D->mat;
        A.pos = c->d_pos;
        A.plane = c->plane;
        A.nalloc = c->desc.num_alloc;
        A.num_slices = c->desc.num_slices;
        A.nbs = c->d_nbs;
        A.invL = 1.0 / c->desc.side;
        for (int k = 0; k < 3; ++k) A.nmax[k] = P.nmax[k];
        A.rows = reinterpret_cast<const int2*>(d + o_rows);
        A.jobs = reinterpret_cast<const RhoJob*>(d + o_jobs);
        A.job0 = 0;
        A.job_end = (int)P.jobs.size();
        A.slot = d + o_slot;
        A.width = P.width;
        A.nu = P.nu;
        A.rho = c->d_rho;
    } else {
        RhoArgs& A = D->lane;
        A.pos = c->d_pos;
        A.plane = c->plane;
        A.nalloc = c->desc.num_alloc;
        A.num_slices = c->desc.num_slices;
        A.nbs = c->d_nbs;
        A.invL = 1.0 / c->desc.side;
        A.nq = P.nu;
        A.qn = d + o_list;
        for (int k = 0; k < 3; ++k) A.nmax[k] = P.nmax[k];
        A.rho = c->d_rho;
    }
    return PIMC_OK;
}

// rho_u(m) of the plan's modes into c->d_rho [M][nu][2]
int lattice_rho(pimc_ctx* c, const RhoPlan& P, const std::vector<int>& n3, bool want_dst, DevPlan* D) {
    int r;
    if ((r = grow(c, &c->d_rho, &c->cap_rho, (size_t)c->desc.num_slices * P.nu * 2))) return r;
    if ((r = upload_plan(c, P, n3, want_dst, D))) return r;
    c->timed_begin(2);
    SHIP(c, P.matrix ? launch_rho_matrix(c->stream, D->mat) : launch_rho(true, c->stream, D->lane));
    c->timed_end();
    return PIMC_OK;
}

// rho_q(m) of general q into c->d_rho [M][nq][2]
int general_rho(pimc_ctx* c, const std::vector<double>& qv, int nq) {
    const int M = c->desc.num_slices;
    int r;
    if ((r = ensure_q(c, nq))) return r;
    if ((r = grow(c, &c->d_rho, &c->cap_rho, (size_t)M * nq * 2))) return r;
    RhoArgs A{};
    A.pos = c->d_pos;
    A.plane = c->plane;
    A.nalloc = c->desc.num_alloc;
    A.num_slices = M;
    A.nbs = c->d_nbs;
    A.invL = 1.0 / c->desc.side;
    A.nq = nq;
    A.q = c->d_q;
    A.rho = c->d_rho;
    SHIP(c, hipMemcpyAsync(c->d_q, qv.data(), sizeof(double) * 3 * nq, hipMemcpyHostToDevice, c->stream));
    c->timed_begin(2);
    SHIP(c, launch_rho(false, c->stream, A));
    c->timed_end();
    return PIMC_OK;
}

// F(q, tau) of a long lattice q list written straight into page-locked memory:
// the modes run in pieces of row tiles (a list of up to 16 jobs in one), each
// piece's modes and lags on the context's stream, and the list rows it completes
// are copied out while the next piece computes.  A mode's sums do not depend on what
// shares its launch, so the values are those of the one-launch path bit for bit.
// 100 401 q x 250 lags are 200 MB, 3.5 ms at the 57 GB/s the link gives, beside
// 2.8 ms of kernels; S(q) and F of that list took 39.6 ms together and now take
// 7.6 ms, F of 5377 q x 167 (one piece) 392 us and now 256 us.
constexpr int kIsfPieceMinQ = 2048;                // shorter lists: one copy
constexpr size_t kIsfPieceMinBytes = 4u << 20;     // smaller results: one copy
constexpr int kIsfPiecesMax = 16;

bool isf_pieces_pay(pimc_ctx* c, int n, int M, const double* fqt) {
    if (n < kIsfPieceMinQ || (size_t)n * M * sizeof(double) < kIsfPieceMinBytes) return false;
    // a timed call keeps one launch per kernel, so its durations stay per call
    if (c->timing && (c->timing_kinds & ((1u << 2) | (1u << 4)))) return false;
    // a pageable destination is copied through staging with the host waiting
    hipPointerAttribute_t at{};
    const hipError_t e = hipPointerGetAttributes(&at, fqt);
    (void)hipGetLastError();   // a pageable pointer may report an error here
    return e == hipSuccess && at.type == hipMemoryTypeHost;
}

// The list rows of modes [u0, u_end) as at most two runs {first row, rows}: their
// first q and their second q (those of -q), each a run when the rows named are
// consecutive (in either direction), which a list in the reference's order
// gives.  False when they are not.
bool isf_runs(const RhoPlan& P, int u0, int u_end, std::pair<int, int> run[2]) {
    const std::vector<int>* by[2] = {&P.first, &P.second};
    for (int s = 0; s < 2; ++s) {
        int lo = INT_MAX, hi = -1, cnt = 0;
        for (int u = u0; u < u_end; ++u) {
            const int k = (*by[s])[u];
            if (k < 0) continue;
            lo = std::min(lo, k);
            hi = std::max(hi, k);
            ++cnt;
        }
        if (cnt && hi - lo + 1 != cnt) return false;   // the rows of distinct modes are distinct
        run[s] = {cnt ? lo : 0, cnt};
    }
    return true;
}

int isf_lattice_pieces(pimc_ctx* c, const RhoPlan& P, const std::vector<int>& n3, int n, int M, double inv_n,
                        double* fqt) {
    int r;
    if ((r = grow(c, &c->d_rho, &c->cap_rho, (size_t)M * P.nu * 2))) return r;
    if ((r = grow(c, &c->d_fqt, &c->cap_fqt, (size_t)n * M))) return r;
    DevPlan D;
    if ((r = upload_plan(c, P, n3, true, &D))) return r;
    const int pieces = (int)P.piece_modes.size();
    while ((int)c->chunk_ev.size() < pieces) {
        hipEvent_t ev = nullptr;
        SHIP(c, hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        c->chunk_ev.push_back(ev);
    }
    hipError_t e = hipSuccess;
    int u0 = 0;
    std::vector<std::pair<int, int>> runs;   // two per piece
    bool late = false;                       // rows left for one copy at the end
    for (int k = 0; k < pieces && e == hipSuccess; ++k) {
        RhoMatrixArgs A = D.mat;
        A.job0 = P.piece_job[k];
        A.job_end = P.piece_job[k + 1];
        e = launch_rho_matrix(c->stream, A);
        const int u1 = P.piece_modes[k];
        if (e == hipSuccess) e = launch_isf(c->stream, c->d_rho, P.nu, u0, u1, M, inv_n, D.dst, c->d_fqt);
        if (e == hipSuccess) e = hipEventRecord(c->chunk_ev[k], c->stream);
        std::pair<int, int> run[2];
        late = late || !isf_runs(P, u0, u1, run);
        runs.insert(runs.end(), run, run + 2);
        u0 = u1;
    }
    if (e == hipSuccess && D.n_repeat) {
        e = launch_isf_repeat(c->stream, D.repeat, D.n_repeat, M, c->d_fqt);
        late = true;
    }
    // the copies go to the DMA engines, which leave the compute units to the next
    // piece (copy kernels on a second stream slowed the pieces 1.7 times at 100 401
    // q); the host, which would only wait, starts each piece's once the piece's
    // event has passed
    const bool dma = e == hipSuccess && !late && dma_open(&c->dma, c->d_fqt, fqt);
    bool moved = dma;
    if (dma) {
        for (int k = 0; k < pieces && moved && e == hipSuccess; ++k) {
            while ((e = hipEventQuery(c->chunk_ev[k])) == hipErrorNotReady) __builtin_ia32_pause();
            for (int s = 0; s < 2 && moved && e == hipSuccess; ++s) {
                const std::pair<int, int>& r2 = runs[2 * k + s];
                if (r2.second)
                    moved = dma_start(&c->dma, fqt + (size_t)r2.first * M, c->d_fqt + (size_t)r2.first * M,
                                      sizeof(double) * (size_t)r2.second * M);
            }
        }
        (void)hipGetLastError();   // hipErrorNotReady is no error
        moved = dma_wait(&c->dma) && moved;
    }
    if (e == hipSuccess && !moved)
        e = hipMemcpyAsync(fqt, c->d_fqt, sizeof(double) * (size_t)n * M, hipMemcpyDeviceToHost, c->stream);
    // the stream ends quiet, after an error too (no copy may land later)
    const hipError_t e1 = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) e = e1;
    if (e != hipSuccess) return sfail(c, PIMC_E_HIP, std::string("F(q,tau) in pieces: ") + hipGetErrorString(e));
    c->isf_chunks += pieces;
    if (moved) c->isf_dma += pieces;
    return PIMC_OK;
}

// The rows of a list's repeated q, from the rows of the modes' first q, where the
// device has not copied them.
void isf_repeats(const RhoPlan& P, int M, double* rows) {
    if (device_repeats(P, M)) return;
    for (int k : P.repeat)
        std::memcpy(rows + (size_t)k * M, rows + (size_t)P.first[P.mode[k]] * M, sizeof(double) * M);
}

// A list with nl lattice q among its nq, split: an all-lattice list keeps its
// order (idx_l empty, n3 as it is); otherwise the lattice q's components move to
// the front of n3 and idx_l / idx_g list both kinds' places.
void split_list(const double* q, int nq, int nl, const std::vector<uint8_t>& lat, std::vector<int>& n3,
                std::vector<int>& idx_l, std::vector<int>& idx_g, std::vector<double>& qg) {
    if (nl == nq) return;
    for (int k = 0; k < nq; ++k) {
        if (lat[k]) {
            for (int d = 0; d < 3; ++d) n3[3 * idx_l.size() + d] = n3[3 * (size_t)k + d];
            idx_l.push_back(k);
        } else {
            idx_g.push_back(k);
            qg.insert(qg.end(), q + 3 * (size_t)k, q + 3 * (size_t)k + 3);
        }
    }
}

}  // namespace

namespace pimc {

bool lattice_q(const double* q, double L, int* n3) {
    const double f = L / (2.0 * M_PI);
    for (int d = 0; d < 3; ++d) {
        const double x = q[d] * f;
        const double r = std::nearbyint(x);
        if (!(std::fabs(r) <= rho_max_nmax())) return false;
        const double back = r * 2.0 * M_PI / L;
        if (std::fabs(back - q[d]) > 1e-9 * std::max(1.0, std::fabs(q[d]))) return false;
        n3[d] = (int)r;
    }
    return true;
}

int lattice_qs(const double* q, int nq, double L, std::vector<int>& n3, std::vector<uint8_t>& lat) {
    // blocks whose components all lie well inside lattice_q's tolerance (straight
    // arithmetic the compiler vectorises: round to nearest by adding and taking
    // away 1.5 2^52, no division) need no second look
    constexpr int kBlock = 64;
    n3.resize(3 * (size_t)nq);
    lat.resize(nq);
    std::memset(lat.data(), 1, (size_t)nq);
    const double f = L / (2.0 * M_PI), g = 2.0 * M_PI / L, top = rho_max_nmax();
    constexpr double kRound = 6755399441055744.0;
    int count = 0;
    for (int k0 = 0; k0 < nq; k0 += kBlock) {
        const int n = 3 * std::min(kBlock, nq - k0);
        const double* s = q + 3 * (size_t)k0;
        int* o = n3.data() + 3 * (size_t)k0;
        double rr[3 * kBlock];
        int sure = 1;
        for (int t = 0; t < n; ++t) {
            const double r = (s[t] * f + kRound) - kRound;
            rr[t] = r;
            // NaN fails both
            sure &= (int)(std::fabs(r) <= top) & (int)(std::fabs(r * g - s[t]) <= 0.5e-9);
        }
        if (sure) {
            for (int t = 0; t < n; ++t) o[t] = (int)rr[t];
            count += n / 3;
            continue;
        }
        for (int k = 0; k < n / 3; ++k) {
            const bool ok = lattice_q(s + 3 * k, L, o + 3 * k);
            lat[k0 + k] = ok;
            count += ok;
        }
    }
    return count;
}

// A 16 x 16 block of the matrix form takes the same time whatever it holds (up to
// 512 modes, both signs of n_z), a mode of the lane form always its own.  Random
// parts of the 100 401 q at N = 2048 x 250: at 133 modes a block the matrix form
// takes 2.01 ms against 3.40 ms, at 72 1.98 against 2.02, at 42 1.72 against 1.18;
// of the 5377 q at N = 256 x 167: at 80 30.5 us against 30.9, at 47 30.0 against 27.3,
// at 29 29.0 against 26.4.  With a few blocks both are a chain of stages (105 modes in
// five blocks 24.6 us against 24.7).
constexpr int kModesPerBlock = 72, kFewBlocks = 4;

// Jobs of a piece: those of one workgroup of k_rho_matrix per slice, which at M = 250 is
// one round of the 256 CUs.  With fewer slices a piece leaves CUs idle, which its copy
// hides where the list is long: 42 499 q at N = 2048 take 1.42 ms at M = 40, 1.56 at 96
// and 1.96 at 167, of which the link takes 0.24, 0.57 and 1.00.
constexpr int kPieceJobs = 16;

void make_rho_plan(const int* n3, int nq, int max_pieces, RhoPlan* P) {
    int h[3] = {0, 0, 0};
    for (int k = 0; k < nq; ++k)
        for (int d = 0; d < 3; ++d) h[d] = std::max(h[d], std::abs(n3[3 * (size_t)k + d]));
    for (int d = 0; d < 3; ++d) P->nmax[d] = h[d];
    const int wy = 2 * h[1] + 1, wz = 2 * h[2] + 1;
    const int width = 16 * (h[2] / 16 + 1), blocks = width / 16;
    P->width = width;
    // modes by (n_x, n_y, n_z) of the half space, rows by (n_x, n_y): a table of the
    // box, or, of a large box that the list leaves mostly empty, {place, mode} in an open
    // hash table of at least two places a q (ten q at |n| <= 40, N = 16 x
    // 125: S(q) 33.6 -> 25.3 us, F 60.5 -> 51.4)
    const size_t box = (size_t)(h[0] + 1) * wy * wz;
    size_t places = 0;   // of the hash table, a power of two; 0: a table of the box
    if (box > 16384 && box / 8 > (size_t)nq)
        for (places = 64; places < 2 * (size_t)nq;) places *= 2;
    P->mode_at.assign(places ? 2 * places : box, -1);
    auto mode_of = [&](size_t at) -> int& {
        if (!places) return P->mode_at[at];
        size_t t = (uint32_t)at * 2654435761u & (places - 1);
        while (P->mode_at[2 * t] >= 0 && P->mode_at[2 * t] != (int)at) t = (t + 1) & (places - 1);
        P->mode_at[2 * t] = (int)at;
        return P->mode_at[2 * t + 1];
    };
    P->row_at.assign((size_t)(h[0] + 1) * wy, -1);
    P->mode.resize(nq);
    P->first.resize(nq);
    P->second.resize(nq);
    P->mode_row.resize(nq);
    P->mode_nz.resize(nq);
    P->repeat.clear();
    P->list_rows.clear();
    P->row_mode.clear();   // a row's first mode
    P->row_cols.clear();   // the 16-column blocks a row uses
    int nu = 0;
    for (int k = 0; k < nq; ++k) {
        int nx = n3[3 * (size_t)k], ny = n3[3 * (size_t)k + 1], nz = n3[3 * (size_t)k + 2];
        if (nx < 0 || (nx == 0 && (ny < 0 || (ny == 0 && nz < 0)))) {
            nx = -nx;
            ny = -ny;
            nz = -nz;
        }
        const size_t rk = (size_t)nx * wy + (ny + h[1]);
        int& u = mode_of(rk * wz + (nz + h[2]));
        if (u < 0) {
            u = nu++;
            P->first[u] = k;
            P->second[u] = -1;
            int& r = P->row_at[rk];
            if (r < 0) {
                r = (int)P->list_rows.size();
                P->list_rows.push_back(make_int2(nx, ny));
                P->row_mode.push_back(u);
                P->row_cols.push_back(0);
            }
            P->row_cols[r] |= 1 << (std::abs(nz) >> 4);
            P->mode_row[u] = r;
            P->mode_nz[u] = nz;
        } else if (P->second[u] < 0) {
            P->second[u] = k;
        } else {
            P->repeat.push_back(k);
        }
        P->mode[k] = u;
    }
    P->nu = nu;
    // the pieces' rows, sorted by their blocks (stable: then in the list's order),
    // 16 to a tile; a tile's jobs are the blocks its rows use
    const int n_rows = (int)P->list_rows.size();
    std::vector<int>& order = P->order;   // tile places -> rows (-1: unused)
    int pieces = 1;
    for (int pass = 0; pass < 2; ++pass) {
        order.clear();
        P->jobs.clear();
        P->piece_job.assign(1, 0);
        P->piece_modes.clear();
        for (int k = 0; k < pieces; ++k) {
            const int r0 = (int)((int64_t)n_rows * k / pieces), r1 = (int)((int64_t)n_rows * (k + 1) / pieces);
            const size_t o0 = order.size();
            for (int mask = (1 << blocks) - 1; mask > 0; --mask)
                for (int r = r0; r < r1; ++r)
                    if (P->row_cols[r] == mask) order.push_back(r);
            while (order.size() % 16) order.push_back(-1);
            for (size_t t = o0; t < order.size(); t += 16) {
                int mask = 0;
                for (int i = 0; i < 16; ++i)
                    if (order[t + i] >= 0) mask |= P->row_cols[order[t + i]];
                for (int c = 0; c < blocks; ++c)
                    if (mask & (1 << c)) P->jobs.push_back({(int)(t / 16), 16 * c});
            }
            P->piece_job.push_back((int)P->jobs.size());
            // the modes of the rows still to run start at the smallest first mode among them
            int least = nu;
            for (int r = r1; r < n_rows; ++r) least = std::min(least, P->row_mode[r]);
            P->piece_modes.push_back(least);
        }
        const int want = std::min(max_pieces, ((int)P->jobs.size() + kPieceJobs - 1) / kPieceJobs);
        if (pass || want <= 1) break;
        pieces = want;
    }
    P->matrix = (int)P->jobs.size() <= kFewBlocks || (int64_t)nu >= (int64_t)kModesPerBlock * (int64_t)P->jobs.size();
    if (!P->matrix) {
        P->jobs.clear();
        P->rows.clear();
        P->slot.clear();
        return;
    }
    P->rows.assign(order.size(), make_int2(0, 0));
    P->at.resize(n_rows);
    for (size_t t = 0; t < order.size(); ++t)
        if (order[t] >= 0) {
            P->rows[t] = P->list_rows[order[t]];
            P->at[order[t]] = (int)t;
        }
    P->slot.assign(order.size() * 2 * width, -1);
    for (int u = 0; u < nu; ++u) {
        const int nz = P->mode_nz[u];
        P->slot[((size_t)P->at[P->mode_row[u]] * 2 + (nz < 0 ? 1 : 0)) * width + std::abs(nz)] = u;
    }
}

}  // namespace pimc

extern "C" {

int pimc_ssf(pimc_ctx* c, const double* q, int nq, double* sq) {
    if (!c || (nq > 0 && (!q || !sq))) return sfail(c, PIMC_E_ARG, "null argument");
    if (!c->have_path) return sfail(c, PIMC_E_STATE, "no path uploaded");
    if (nq <= 0) return PIMC_OK;
    const int M = c->desc.num_slices;
    if (M > 512) return sfail(c, PIMC_E_UNSUPPORTED, "S(q) supports M <= 512 slices");
    const int Np = true_num_particles(c);
    if (Np <= 0) return sfail(c, PIMC_E_STATE, "no active particles");
    const double inv_n = 1.0 / Np;
    std::vector<int>& n3 = c->q_n3;
    std::vector<uint8_t>& lat = c->q_lat;
    std::vector<int> idx_l, idx_g;
    std::vector<double> qg;
    const int nl = lattice_qs(q, nq, c->desc.side, n3, lat);
    split_list(q, nq, nl, lat, n3, idx_l, idx_g, qg);
    int r;
    if (nl) {
        RhoPlan& P = c->plan;
        make_rho_plan(n3.data(), nl, 1, &P);
        DevPlan D;
        if ((r = lattice_rho(c, P, n3, false, &D))) return r;
        // a few thousand values go straight into mapped memory and the host spins
        // on the kernel's completion word; more are copied
        const bool mapped = P.nu <= pimc_ctx::kMappedSq;
        if (!mapped && (r = grow(c, &c->d_fqt, &c->cap_fqt, (size_t)P.nu))) return r;
        const unsigned long long seq = ++c->seq;
        c->timed_begin(3);
        SHIP(c, launch_ssf(c->stream, c->d_rho, P.nu, M, inv_n, mapped ? c->d_map + pimc_ctx::kSqSlot : c->d_fqt, c->d_ticket,
                           mapped ? c->d_done() : nullptr, seq));
        c->timed_end();
        const double* got = c->h_map + pimc_ctx::kSqSlot;
        std::vector<double> host;
        if (mapped) {
            if (c->wait_done(seq) != 0) {
                // the arrival counter may have been left part-way
                (void)hipMemsetAsync(c->d_ticket, 0, sizeof(unsigned), c->stream);
                return sfail(c, PIMC_E_HIP, "S(q): completion not published");
            }
        } else {
            double* to = c->h_stage;
            if ((size_t)P.nu > c->cap_stage) {
                host.resize(P.nu);
                to = host.data();
            }
            SHIP(c, hipMemcpyAsync(to, c->d_fqt, sizeof(double) * P.nu, hipMemcpyDeviceToHost, c->stream));
            SHIP(c, hipStreamSynchronize(c->stream));
            got = to;
        }
        if (idx_l.empty())
            for (int k = 0; k < nl; ++k) sq[k] = got[P.mode[k]];
        else
            for (int k = 0; k < nl; ++k) sq[idx_l[k]] = got[P.mode[k]];
    }
    if (!idx_g.empty()) {
        const int ng = (int)idx_g.size();
        if ((r = ensure_q(c, ng))) return r;
        if ((r = grow(c, &c->d_rho, &c->cap_rho, (size_t)ng * M))) return r;
        if ((r = grow(c, &c->d_fqt, &c->cap_fqt, (size_t)ng))) return r;
        SHIP(c, hipMemcpyAsync(c->d_q, qg.data(), sizeof(double) * 3 * ng, hipMemcpyHostToDevice, c->stream));
        c->timed_begin(3);
        SHIP(c, launch_ssf_pairs(c->stream, c->d_pos, c->plane, c->desc.num_alloc, M, c->d_nbs, c->d_q, ng, c->box,
                                 c->d_rho, inv_n, c->d_fqt));
        c->timed_end();
        std::vector<double> host(ng);
        SHIP(c, hipMemcpyAsync(host.data(), c->d_fqt, sizeof(double) * ng, hipMemcpyDeviceToHost, c->stream));
        SHIP(c, hipStreamSynchronize(c->stream));
        for (int k = 0; k < ng; ++k) sq[idx_g[k]] = host[k];
    }
    return PIMC_OK;
}

int pimc_isf(pimc_ctx* c, const double* q, int nq, double* fqt) {
    if (!c || (nq > 0 && (!q || !fqt))) return sfail(c, PIMC_E_ARG, "null argument");
    if (!c->have_path) return sfail(c, PIMC_E_STATE, "no path uploaded");
    if (nq <= 0) return PIMC_OK;
    const int M = c->desc.num_slices;
    if (M > 512) return sfail(c, PIMC_E_UNSUPPORTED, "F(q,tau) supports M <= 512 slices");
    const int Np = true_num_particles(c);
    if (Np <= 0) return sfail(c, PIMC_E_STATE, "no active particles");
    const double inv_n = 1.0 / Np;
    std::vector<int>& n3 = c->q_n3;
    std::vector<uint8_t>& lat = c->q_lat;
    std::vector<int> idx_l, idx_g;
    std::vector<double> qg;
    const int nl = lattice_qs(q, nq, c->desc.side, n3, lat);
    split_list(q, nq, nl, lat, n3, idx_l, idx_g, qg);
    for (int pass = 0; pass < 2; ++pass) {
        const int n = pass == 0 ? nl : nq - nl;
        if (n == 0) continue;
        int r;
        RhoPlan& P = c->plan;
        DevPlan D;
        if (pass == 0) {
            const bool pieces = n == nq && isf_pieces_pay(c, n, M, fqt);
            make_rho_plan(n3.data(), nl, pieces ? kIsfPiecesMax : 1, &P);
            if (pieces && P.matrix) {
                if ((r = isf_lattice_pieces(c, P, n3, n, M, inv_n, fqt))) return r;
                isf_repeats(P, M, fqt);
                continue;
            }
            if ((r = lattice_rho(c, P, n3, true, &D))) return r;
        } else if ((r = general_rho(c, qg, n))) {
            return r;
        }
        const int nu = pass == 0 ? P.nu : n;
        if (pass == 1) P.repeat.clear();
        if ((r = grow(c, &c->d_fqt, &c->cap_fqt, (size_t)n * M))) return r;
        c->timed_begin(4);
        SHIP(c, launch_isf(c->stream, c->d_rho, nu, 0, nu, M, inv_n, D.dst, c->d_fqt));
        c->timed_end();
        if (D.n_repeat) SHIP(c, launch_isf_repeat(c->stream, D.repeat, D.n_repeat, M, c->d_fqt));
        if (n == nq) {
            // every q in this pass, in order: straight into the caller's array
            SHIP(c, hipMemcpyAsync(fqt, c->d_fqt, sizeof(double) * n * M, hipMemcpyDeviceToHost, c->stream));
            SHIP(c, hipStreamSynchronize(c->stream));
            isf_repeats(P, M, fqt);
            continue;
        }
        std::unique_ptr<double[]> host(new double[(size_t)n * M]);
        SHIP(c, hipMemcpyAsync(host.get(), c->d_fqt, sizeof(double) * n * M, hipMemcpyDeviceToHost, c->stream));
        SHIP(c, hipStreamSynchronize(c->stream));
        isf_repeats(P, M, host.get());
        const std::vector<int>& idx = pass == 0 ? idx_l : idx_g;
        for (int k = 0; k < n; ++k) std::memcpy(fqt + (size_t)idx[k] * M, host.get() + (size_t)k * M, sizeof(double) * M);
    }
    return PIMC_OK;
}

}  // extern "C"

// ===========================================================================
// Batched PotentialBase for the Aziz pair potential
// ===========================================================================
struct pimc_aziz {
    AzizParams p{};
    AzizDev az{};
    int v_mode = PIMC_V_FP32;
    int year = 1979;
    double tailV = 0;
    hipStream_t stream = nullptr;
    double* d_in = nullptr;
    double* d_out = nullptr;
    size_t cap = 0;
    std::string err;
};

namespace {

int afail(pimc_aziz* a, int code, const std::string& m) {
    if (a) a->err = m;
    return code;
}

int aziz_run(pimc_aziz* a, const double* sep, double* out, int n, int what) {
    if (!a || (n > 0 && (!sep || !out))) return afail(a, PIMC_E_ARG, "null argument");
    if (n < 0) return afail(a, PIMC_E_ARG, "negative count");
    if (n == 0) return PIMC_OK;
    const size_t need = 3 * (size_t)n;
    if (need > a->cap) {
        if (a->d_in) (void)hipFree(a->d_in);
        if (a->d_out) (void)hipFree(a->d_out);
        a->d_in = a->d_out = nullptr;
        if (hipMalloc(&a->d_in, sizeof(double) * need) != hipSuccess ||
            hipMalloc(&a->d_out, sizeof(double) * need) != hipSuccess) {
            a->cap = 0;
            return afail(a, PIMC_E_NOMEM, "hipMalloc failed");
        }
        a->cap = need;
    }
    std::string err;
    AzizDev az = a->az;
    const double* d1 = nullptr;
    const double* d2 = nullptr;
    if (what == 0 && a->v_mode == PIMC_V_TABLE) {
        az.table = cached_table(a->year, 0, az.table_length, &err);
        if (!az.table) return afail(a, PIMC_E_NOMEM, err);
    }
    if (what == 1) {
        d1 = cached_table(a->year, 1, az.table_length, &err);
        if (!d1) return afail(a, PIMC_E_NOMEM, err);
    }
    if (what == 2) {
        d2 = cached_table(a->year, 2, az.table_length, &err);
        if (!d2) return afail(a, PIMC_E_NOMEM, err);
    }
    hipError_t e = hipMemcpyAsync(a->d_in, sep, sizeof(double) * need, hipMemcpyHostToDevice, a->stream);
    if (e == hipSuccess) e = launch_aziz_batch(a->v_mode, a->stream, a->d_in, n, az, d1, d2, what, a->d_out);
    const size_t outn = (what == 1) ? need : (size_t)n;
    if (e == hipSuccess) e = hipMemcpyAsync(out, a->d_out, sizeof(double) * outn, hipMemcpyDeviceToHost, a->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(a->stream);
    if (e != hipSuccess) return afail(a, PIMC_E_HIP, hipGetErrorString(e));
    return PIMC_OK;
}

}  // namespace

extern "C" {

int pimc_aziz_create(int year, double max_sep, double rc, int v_mode, pimc_aziz** out) {
    if (!out) return PIMC_E_ARG;
    *out = nullptr;
    pimc_aziz* a = new pimc_aziz();
    if (!aziz_params(year, &a->p) || !(max_sep > 0) || !(rc > 0) || v_mode < 0 || v_mode > 2) {
        delete a;
        return PIMC_E_ARG;
    }
    a->year = year;
    a->v_mode = v_mode;
    a->az = make_aziz_dev(a->p, max_sep);
    a->tailV = aziz_tail(a->p, rc);
    if (hipStreamCreateWithFlags(&a->stream, hipStreamNonBlocking) != hipSuccess) {
        delete a;
        return PIMC_E_HIP;
    }
    *out = a;
    return PIMC_OK;
}

void pimc_aziz_destroy(pimc_aziz* a) {
    if (!a) return;
    if (a->stream) (void)hipStreamSynchronize(a->stream);
    if (a->d_in) (void)hipFree(a->d_in);
    if (a->d_out) (void)hipFree(a->d_out);
    if (a->stream) (void)hipStreamDestroy(a->stream);
    delete a;
}

int pimc_aziz_V(pimc_aziz* a, const double* sep3, double* out, int n) { return aziz_run(a, sep3, out, n, 0); }
int pimc_aziz_gradV(pimc_aziz* a, const double* sep3, double* out3, int n) { return aziz_run(a, sep3, out3, n, 1); }
int pimc_aziz_grad2V(pimc_aziz* a, const double* sep3, double* out, int n) { return aziz_run(a, sep3, out, n, 2); }
double pimc_aziz_tailV(const pimc_aziz* a) { return a ? a->tailV : 0.0; }
int pimc_aziz_table_length(const pimc_aziz* a) { return a ? a->az.table_length : 0; }

}  // extern "C"
