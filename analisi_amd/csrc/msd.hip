// Mean square displacement (msd.cpp:40-146) on the device.
//
// vdata[t][type] = mean over (t0 = 0, skip, .. < n ; atoms of the type) of
// |x(t0) - x(t0+t) [- (cm(t0) - cm(t0+t))]|^2 and, with cm_msd, the second
// half vdata[t][nt + type] = mean over t0 of |cm(t0) - cm(t0+t)|^2.
//
// The atom part is a sum of non-negative terms: each thread accumulates one
// atom over all t0 for a tile of lags (FP64), the workgroup sums its atoms per
// type in slot order, and a second kernel adds the chunk partials in a fixed
// order and divides by the term count -- deterministic, and within a few ulps
// of the reference's running mean (no cancellation).  The centre-of-mass
// channel replays the reference's running mean exactly.  Several blocks
// (primo_b, n_b) run in one launch.
//
// msd_window_kernel: a wavefront holds R frames of its 64 atoms in registers,
// one per lag of its tile, and moving to the next t0 replaces one of them.
// The launch shape (R, wavefronts per workgroup) is tunable; tile 0 runs
// msd_atoms_kernel (eight lags per thread, every frame loaded), which a
// calculation with few lags per residue also takes by itself.
// A small calculation splits its t0 range into segments (msd_segments), summed
// in order by msd_finish_kernel; the split depends on the calculation alone,
// so every launch shape gives the same bits.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "anl_internal.h"

#pragma clang fp contract(off)

namespace anl {

constexpr int MSD_WG = 256;

// f(std::integral_constant<int, 0>) .. f(std::integral_constant<int, N-1>),
// unrolled at compile time.
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}
constexpr int MSD_TL = 8;  // lags per thread of msd_atoms_kernel

struct MsdBlock {
    uint64_t primo;
    uint32_t n;
    uint32_t nseg;  // segments of the t0 range
};

// Block table and term counts of a launch: in device memory, or, for one block
// and few types, in the kernel arguments (nothing to upload).
constexpr uint32_t MSD_INL = 8;
struct MsdTables {
    const MsdBlock *blocks;  // null: one
    const uint64_t *count;   // [nblocks][nt], null: cnt
    MsdBlock one;
    uint64_t cnt[MSD_INL];
    __device__ __forceinline__ MsdBlock block(uint32_t b) const { return blocks ? blocks[b] : one; }
    __device__ __forceinline__ uint64_t terms(uint32_t b, uint32_t tt, uint32_t nt) const {
        return count ? count[(uint64_t)b * nt + tt] : cnt[tt];
    }
};

// Segment seg of a block's t0 values k = 0 .. ceil(n / skip) - 1: first and count.
__device__ __forceinline__ void msd_segment(const MsdBlock &b, uint32_t skip, uint32_t seg, uint32_t &k0, uint32_t &nk) {
    const uint32_t K = (b.n + skip - 1) / skip, len = (K + b.nseg - 1) / b.nseg;
    k0 = min(K, seg * len);
    nk = min(len, K - k0);
}

// A thread holds eight lags of one atom and loads every frame.  The same
// operations in the same order as msd_window_kernel over one segment, and the
// same partial sums: per 64 slots, or per 256 (group 4).
template <bool CMSELF>
__global__ __launch_bounds__(MSD_WG) void msd_atoms_kernel(const double4 *__restrict__ pos, const double *__restrict__ cm,
                                                          const int32_t *__restrict__ type_slot, uint64_t N, uint32_t nt,
                                                          const MsdTables tb_, uint32_t skip, uint32_t leff,
                                                          uint32_t nchunks, uint32_t group, double *__restrict__ partial) {
    __shared__ double acc_lds[MSD_TL][MSD_WG];
    __shared__ int type_lds[MSD_WG];
    const MsdBlock blk = tb_.block(blockIdx.z);
    const uint64_t primo = blk.primo;
    const uint32_t n = blk.n;
    const uint64_t slot = (uint64_t)blockIdx.x * MSD_WG + threadIdx.x;
    const uint32_t tb = blockIdx.y * MSD_TL;
    double acc[MSD_TL];
#pragma unroll
    for (int l = 0; l < MSD_TL; l++) acc[l] = 0.0;
    int ti = -1;
    if (slot < N) {
        ti = type_slot[slot];
        auto frame = [&](uint64_t f) {
            const double4 x = pos[f * N + slot];
            if (!CMSELF) return make_double3(x.x, x.y, x.z);
            const double *c = cm + (f * nt + ti) * 3;
            return make_double3(x.x - c[0], x.y - c[1], x.z - c[2]);
        };
        for (uint32_t t0 = 0; t0 < n; t0 += skip) {
            const double3 y = frame(primo + t0);
#pragma unroll
            for (int l = 0; l < MSD_TL; l++) {
                const uint32_t t = tb + l;
                if (t < leff) {
                    const double3 z = frame(primo + t0 + t);
                    const double e0 = y.x - z.x, e1 = y.y - z.y, e2 = y.z - z.z;
                    acc[l] = fma(e0, e0, acc[l]);
                    acc[l] = fma(e1, e1, acc[l]);
                    acc[l] = fma(e2, e2, acc[l]);
                }
            }
        }
    }
#pragma unroll
    for (int l = 0; l < MSD_TL; l++) acc_lds[l][threadIdx.x] = acc[l];
    type_lds[threadIdx.x] = ti;
    __syncthreads();
    // thread (chunk, lag, type) sums 64 slots in order, or (lag, type) four such sums
    const uint32_t parts = 4 / group;
    for (uint32_t w = threadIdx.x; w < parts * MSD_TL * nt; w += MSD_WG) {
        const uint32_t p = w / (MSD_TL * nt), r = w % (MSD_TL * nt), l = r / nt, tt = r % nt;
        const uint32_t t = tb + l, chunk = blockIdx.x * parts + p;
        if (t >= leff || chunk >= nchunks) continue;
        double s = 0.0;
        for (uint32_t g = 0; g < group; g++) {
            double sum = 0.0;
            for (uint32_t k = 64 * (p + g); k < 64 * (p + g) + 64; k++)
                if (type_lds[k] == (int)tt) sum += acc_lds[l][k];
            s = g == 0 ? sum : s + sum;
        }
        partial[(((uint64_t)blockIdx.z * leff + t) * nchunks + chunk) * nt + tt] = s;  // one segment
    }
}

// Every t0 stride.  With t0 = skip k and lag = skip m + r, a residue r is a
// stride 1 problem on two thinned series, y_k = x(skip k) and z_j = x(skip j +
// r): lag m adds |y_k - z_{k+m}|^2.  Workgroup = 64 atom slots (the lanes) x WV
// wavefronts, each a tile of R consecutive m of one residue.  A wavefront's
// R frames z rotate through registers (the t0 loop is unrolled R times): per t0
// it loads y_k and one new z for R updates of 6 FP64 operations.  The FP64
// unit needs 3 or more wavefronts per SIMD to approach its rate (one issues an
// operation every 6 to 7 clocks, four together every 4.3), so the window of a
// wavefront stays in its own registers: an LDS ring shared by the workgroup's
// wavefronts left room for one per SIMD and was 10% slower.  The frames'
// addresses are uniform: scalar pointers that step by skip frames and stop at
// the last one.
// The 1-D grid is decoded so that the tiles and residues of one atom chunk are
// consecutive logical ids on one XCD (hardware id h runs on XCD h % 8), where
// they share its frames in L2.  With drift removal y and z lose the centre of
// mass of the atom's type as each frame is loaded.
// Measured: 8,192 atoms x 499 t0 x 499 lags 0.49 ms without drift removal
// (63% of the FP64 issue rate) and 0.60 ms with it (0.57 and 0.79 ms when
// every address was a vector computation and the tile 16); 4,001 atoms x 101
// t0 of stride 10 x 499 lags 0.097 ms (0.375 ms in msd_atoms_kernel).
template <int R, int WV, bool CMSELF>
__global__ __launch_bounds__(64 * WV, CMSELF ? (R <= 12 ? 4 : R <= 16 ? 3 : 2) : 1) void msd_window_kernel(const double4 *__restrict__ pos,
                                                           const double *__restrict__ cm,
                                                           const int32_t *__restrict__ type_slot, uint64_t N,
                                                           uint32_t nt, const MsdTables tables, uint32_t maxseg,
                                                           uint32_t skip, uint32_t leff, uint32_t nchunks,
                                                           uint32_t group, uint32_t ntiles, uint32_t nres,
                                                           uint32_t per_xcd, uint32_t total,
                                                           double *__restrict__ partial) {
    __shared__ double red[WV][R][64];
    __shared__ int type_lds[64];
    const uint32_t h = blockIdx.x;
    const uint32_t L = (h & 7u) * per_xcd + (h >> 3);
    if (L >= total) return;  // whole workgroup: uniform
    const uint32_t tile = L % ntiles;
    uint32_t rest = L / ntiles;
    const uint32_t res = rest % nres;
    rest /= nres;
    const uint32_t seg = rest % maxseg;
    rest /= maxseg;
    const uint32_t chunk = rest % nchunks, blk = rest / nchunks;
    const MsdBlock b = tables.block(blk);
    const uint32_t M = (leff - res + skip - 1) / skip;  // lags of this residue (res < nres <= leff)
    if (seg >= b.nseg || tile * (uint32_t)(R * WV) >= M) return;
    uint32_t k0, nk;
    msd_segment(b, skip, seg, k0, nk);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t mb = (tile * (uint32_t)WV + wave) * (uint32_t)R;  // first m of this wavefront
    // the last frame a counted (t0, lag) reads
    const uint64_t flast = b.primo + (uint64_t)b.n - 1u + (uint64_t)leff - 1u;
    // a uniform walk over frames f0, f0 + skip, .. that stays on the last one
    // within flast (the sums of the lags that would read on are not used)
    struct Walk {
        const double4 *p;
        const double *c;
        uint32_t left;
    };
    const uint64_t pstep = (uint64_t)skip * N, cstep = (uint64_t)skip * nt * 3;
    auto walk = [&](uint64_t f0) -> Walk {
        const uint64_t f = f0 < flast ? f0 : flast;
        return Walk{pos + f * N, cm + f * nt * 3, (uint32_t)((flast - f) / skip)};
    };
    // `group` chunks of 64 slots, one after the other, share a partial sum
    for (uint32_t g = 0; g < group; g++) {
        const uint64_t base = ((uint64_t)chunk * group + g) * 64u;
        if (base >= N) break;  // uniform
        const uint64_t slot = base + lane;
        const uint32_t sl = (uint32_t)(slot < N ? slot : N - 1);  // lanes past N load a real atom and are not summed
        const int ti = type_slot[sl];
        const uint32_t co = (uint32_t)ti * 3u;
        struct Raw {  // a frame as loaded
            double3 x, c;
        };
        auto take = [&](Walk &w) -> Raw {
            const double4 x = w.p[sl];
            Raw r{make_double3(x.x, x.y, x.z), make_double3(0.0, 0.0, 0.0)};
            if (CMSELF) r.c = make_double3(w.c[co], w.c[co + 1], w.c[co + 2]);
            const bool on = w.left > 0;
            w.p += on ? pstep : 0;
            if (CMSELF) w.c += on ? cstep : 0;
            w.left -= on ? 1u : 0u;
            return r;
        };
        auto frame = [&](const Raw &r) -> double3 {
            return CMSELF ? make_double3(r.x.x - r.c.x, r.x.y - r.c.y, r.x.z - r.c.z) : r.x;
        };
        double acc[R];
#pragma unroll
        for (int k = 0; k < R; k++) acc[k] = 0.0;
        if (mb < M) {  // uniform per wavefront
            Walk yw = walk(b.primo + (uint64_t)skip * k0);
            Walk zw = walk(b.primo + (uint64_t)skip * ((uint64_t)k0 + mb) + res);
            double3 W[R];
#pragma unroll
            for (int k = 0; k < R; k++) W[k] = frame(take(zw));
            // step s of a pass starting at k: W[(s + i) % R] holds z_{k+s+mb+i};
            // afterwards W[s] is refilled with the next one.  Every index is a
            // compile-time constant once the pass is unrolled, so the window
            // stays in registers.  y is loaded a step ahead; with drift removal
            // y and z wait as loaded until the step that uses them (a
            // subtraction right after the load would wait for it).
            Raw yr = take(yw);
            auto step = [&](auto sc) {
                constexpr int s = decltype(sc)::value;
                const double3 ya = frame(yr);
                yr = take(yw);
                Raw zr;
                if (CMSELF) zr = take(zw);
#pragma unroll
                for (int k = 0; k < R; k++) {
                    const double3 wv = W[(s + k) % R];
                    const double e0 = ya.x - wv.x, e1 = ya.y - wv.y, e2 = ya.z - wv.z;
                    acc[k] = fma(e0, e0, acc[k]);
                    acc[k] = fma(e1, e1, acc[k]);
                    acc[k] = fma(e2, e2, acc[k]);
                }
                if (CMSELF) {
                    __builtin_amdgcn_sched_barrier(0);
                    W[s] = frame(zr);
                } else {
                    W[s] = take(zw).x;
                }
            };
            uint32_t k = 0;
            for (; k + R <= nk; k += R)
                static_for<R>([&](auto sc) { step(sc); });
            // last partial pass (uniform condition per step)
            static_for<R>([&](auto sc) {
                if (k + (uint32_t)decltype(sc)::value < nk) step(sc);
            });
        }
        __syncthreads();  // the previous chunk's sums have been read
#pragma unroll
        for (int k = 0; k < R; k++) red[wave][k][lane] = acc[k];
        if (threadIdx.x < 64) type_lds[lane] = slot < N ? ti : -1;
        __syncthreads();
        // thread (wave, lag, type) sums the 64 slots in order
        for (uint32_t w = threadIdx.x; w < (uint32_t)WV * R * nt; w += 64u * WV) {
            const uint32_t wv = w / ((uint32_t)R * nt), r = w % ((uint32_t)R * nt);
            const uint32_t k = r / nt, tt = r % nt;
            const uint32_t m = (tile * (uint32_t)WV + wv) * (uint32_t)R + k;
            if (m >= M) continue;
            double sum = 0.0;
            for (int j = 0; j < 64; j++)
                if (type_lds[j] == (int)tt) sum += red[wv][k][j];
            const uint64_t t = (uint64_t)skip * m + res;
            double *o = &partial[((((uint64_t)blk * leff + t) * maxseg + seg) * nchunks + chunk) * nt + tt];
            *o = g == 0 ? sum : *o + sum;
        }
    }
}

// Sums the partials of one (block, lag, type) per wavefront: lane l adds the
// (segment, chunk) sums l, l + 64, .. in order, then the lanes add up in a
// fixed order.  The workgroups from nfin on run the centre-of-mass channel
// (msd.cpp:113-123: |cm(t0) - cm(t0+t)|^2 running mean over t0, per type), 64
// lags of a type each: three wavefronts form the squares of a stage of t0 while
// one runs the mean over the stage before, and 1/cont in two parts replaces the division by
// cont (exact, see div_by in gk.hip; a stage whose differences leave its range
// takes true divisions).
constexpr uint32_t MSD_CMS = 33;  // t0 of a centre-of-mass stage, 11 per producer
__global__ __launch_bounds__(256) void msd_finish_kernel(const double *__restrict__ partial, uint32_t nchunks,
                                                         uint32_t maxseg, uint32_t nt, uint32_t leff, uint32_t nblocks,
                                                         const MsdTables tables, uint32_t fcm,
                                                         const double *__restrict__ cm, uint32_t skip, uint32_t nfin,
                                                         double *__restrict__ out) {
    __shared__ double ds[2][MSD_CMS][64];
    __shared__ __align__(16) double2 ys[2][MSD_CMS];
    const uint32_t lane = threadIdx.x & 63u;
    if (blockIdx.x < nfin) {
        const uint32_t w = blockIdx.x * 4 + (threadIdx.x >> 6);
        if (w >= nblocks * leff * nt) return;
        const uint32_t b = w / (leff * nt), r = w % (leff * nt);
        const uint32_t t = r / nt, tt = r % nt;
        const double *p = partial + (((uint64_t)b * leff + t) * maxseg * nchunks) * nt + tt;
        const uint32_t np = tables.block(b).nseg * nchunks;
        double s = 0.0;
        for (uint32_t c = lane; c < np; c += 64) s += p[(uint64_t)c * nt];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
        const uint64_t cn = tables.terms(b, tt, nt);
        if (lane == 0) out[(uint64_t)b * leff * nt * fcm + (uint64_t)t * nt * fcm + tt] = cn ? s / (double)cn : 0.0;
        return;
    }
    uint32_t w = blockIdx.x - nfin;
    const uint32_t nl = (leff + 63) / 64, lt = w % nl;
    w /= nl;
    const uint32_t tt = w % nt, b = w / nt, t = lt * 64 + lane;
    const MsdBlock blk = tables.block(b);
    const uint32_t K = (blk.n + skip - 1) / skip;
    const uint64_t f0 = blk.primo, flast = blk.primo + (uint64_t)blk.n - 1u + (uint64_t)leff - 1u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t nst = (K + MSD_CMS - 1) / MSD_CMS;
    constexpr uint32_t PK = MSD_CMS / 3;
    double m = 0.0, e[PK][6];
    auto load = [&](uint32_t st) {
#pragma unroll
        for (uint32_t j = 0; j < PK; j++) {
            const uint32_t k = min(st * MSD_CMS + (wave - 1) * PK + j, K - 1);
            const uint64_t fa = f0 + (uint64_t)k * skip, fc = min(fa + t, flast);
            const double *a = cm + (fa * nt + tt) * 3, *c = cm + (fc * nt + tt) * 3;
#pragma unroll
            for (int x = 0; x < 3; x++) {
                e[j][x] = a[x];
                e[j][3 + x] = c[x];
            }
        }
    };
    if (wave > 0 && nst) load(0);
    for (uint32_t st = 0; st <= nst; st++) {  // stage st is formed, stage st - 1 averaged
        const uint32_t buf = st & 1u;
        if (wave > 0 && st < nst) {
#pragma unroll
            for (uint32_t j = 0; j < PK; j++) {
                const double e0 = e[j][0] - e[j][3], e1 = e[j][1] - e[j][4], e2 = e[j][2] - e[j][5];
                ds[buf][(wave - 1) * PK + j][lane] = (e0 * e0 + e1 * e1) + e2 * e2;
            }
            if (wave == 1 && lane < MSD_CMS) {
                const double c = (double)(st * MSD_CMS + lane + 1), y = 1.0 / c;
                ys[buf][lane] = make_double2(y, fma(-c, y, 1.0) / c);
            }
            if (st + 1 < nst) load(st + 1);
        } else if (wave == 0 && st > 0) {
            const uint32_t k0 = (st - 1) * MSD_CMS, ns = min(MSD_CMS, K - k0);
            const double m0 = m;
            double dmin = 1.0;
#pragma unroll 11
            for (uint32_t k = 0; k < ns; k++) {
                const double d = ds[buf ^ 1][k][lane] - m;
                dmin = fmin(dmin, d == 0.0 ? 1.0 : fabs(d));  // a zero (lag 0) divides exactly
                m = m + fma(d, ys[buf ^ 1][k].x, d * ys[buf ^ 1][k].y);
            }
            if (__ballot(!(dmin > 0x1p-900) || !(fabs(m) < 0x1p1000))) {
                m = m0;
                for (uint32_t k = 0; k < ns; k++) {
                    const double d = ds[buf ^ 1][k][lane] - m;
                    m = m + d / (double)(k0 + k + 1);
                }
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 64 && t < leff) out[(uint64_t)b * leff * nt * 2 + (uint64_t)t * nt * 2 + nt + tt] = m;
}

// Launch shapes of msd_window_kernel: (lag tile R, wavefronts per workgroup).
// A workgroup covers R * waves consecutive lags of 64 atoms and streams the
// atoms' frames once for all of them, so wider workgroups read each frame
// fewer times; the register window (R frames) and the workgroup size must
// fit the VGPRs (R 24 needs 256: at most 8 wavefronts; R 16 at most 12).
struct MsdShape {
    uint32_t tile, waves;
};
constexpr MsdShape MSD_SHAPES[] = {{8, 4}, {12, 4}, {16, 4}, {24, 4}, {16, 8}, {24, 8}, {12, 12}, {16, 12}, {8, 16}};
bool msd_shape_ok(uint32_t tile, uint32_t waves) {
    if (tile == 0) return true;  // the eight-lags-per-thread kernel (waves ignored)
    for (const MsdShape &m : MSD_SHAPES)
        if (m.tile == tile && m.waves == waves) return true;
    return false;
}

struct MsdPrepared {
    anl_traj *tr = nullptr;
    uint32_t skip = 1, leff = 0, nblocks = 0, nt = 0, fcm = 1, nchunks = 0, maxseg = 1;
    uint32_t group = 1;  // chunks of 64 slots per partial sum
    uint32_t tile = 0;   // lag tile R of msd_window_kernel; 0: msd_atoms_kernel
    uint32_t waves = 4;  // wavefronts per workgroup of msd_window_kernel
    bool cm_msd = false, cm_self = false;
    bool owns = true;    // the device buffers were allocated for this launch
    MsdTables tables{};
    void *d_tables = nullptr;  // block table and term counts, when not in the arguments
    double *d_partial = nullptr;
    ~MsdPrepared() {
        if (!owns) return;
        (void)hipFree(d_tables);
        (void)hipFree(d_partial);
    }
};

// Segments of the t0 range of a calculation: enough that a small one has 512
// workgroups of 64 atoms and 64 lags (two per CU), 64 t0 each at least (a
// workgroup first fills windows of 64 frames).  A function of the calculation
// alone: it sets the order of the sums.
static uint32_t msd_segments(uint64_t N, uint32_t nt, uint32_t n, uint32_t skip, uint32_t leff) {
    const uint64_t nres = std::min(skip, leff), M = (leff + skip - 1) / skip, K = (n + skip - 1) / skip;
    const uint64_t chunks = (N + 63) / 64, wgs = chunks * nres * ((M + 63) / 64);
    const uint64_t segs = std::max<uint64_t>(1, std::min<uint64_t>((512 + wgs - 1) / std::max<uint64_t>(wgs, 1), K / 64));
    return (uint64_t)leff * chunks * nt * segs * sizeof(double) <= (4ull << 20) ? (uint32_t)segs : 1;
}

// Lag tile of a calculation whose shape was not chosen (4 wavefronts per
// workgroup; all tiles give the same bits): the smallest estimate, lags in
// whole tiles times the measured time per lag on 8,192 atoms x 499 t0 x 499
// lags (us, without and with drift removal: tile 24 0.77 and 0.96, 16 1.18 and
// 1.63, 12 1.4 and 1.9, 8 1.6 and 2.5), among the tiles that give two
// wavefronts per SIMD.  Without one it is 16 (2,000 atoms: 141 us against 174
// with 24; 4,001 atoms, 50 lags per residue: 97 against 120).
// units: 64-atom chunks x residues x segments.
static uint32_t msd_auto_tile(uint64_t units, uint32_t M, bool cm_self) {
    static const struct {
        uint32_t R;
        double w[2];
    } T[] = {{24, {0.77, 0.96}}, {16, {1.18, 1.63}}, {12, {1.4, 1.9}}, {8, {1.6, 2.5}}};
    uint32_t best = 16;
    double cost = HUGE_VAL;
    for (const auto &t : T) {
        const uint32_t tiles = (M + t.R - 1) / t.R;
        const double c = (double)(tiles * t.R) * t.w[cm_self ? 1 : 0];
        if (units * tiles >= 2048 && c < cost) {
            cost = c;
            best = t.R;
        }
    }
    return best;
}

// Whether the shape chosen with anl_msd_set_tuning runs this calculation: at t0
// strides above 1 only where the lags of a residue fill its workgroups.  Else
// wavefronts, or most of their windows, would work for no lag: 8,000 atoms,
// stride 300, one lag per residue, shape (24, 8) 1,120 us, the calculation's
// own 49.
static bool msd_chosen_shape(const anl_traj *tr, uint32_t skip, uint32_t leff) {
    if (tr->msd_auto) return false;
    return skip == 1 || tr->msd_tile == 0 || (leff + skip - 1) / skip >= tr->msd_tile * tr->msd_waves;
}

// Whether msd_atoms_kernel is the faster one: few lags per residue (M) and few
// t0 (K), in a launch that fills the chip.  A wavefront of the window kernel
// then fills a window of 8 frames and uses M of them, msd_atoms_kernel forms 8
// lags of any residues in a thread.  20,000 atoms, stride 100 (us, window and
// atoms, without drift removal): M 1, K 2 143 and 55, K 20 389 and 249; M 2, K 8
// 217 and 198, K 20 401 and 453; M 3, K 4 182 and 152, K 6 203 and 209; with
// it M 2, K 20 635 and 451, M 3, K 20 639 and 672, M 4, K 6 322 and 272, K 12
// 466 and 540.  The line is where 10.7 M K + 33 meets 13.7 (K + 8), with drift
// removal 25 (K + 5).  Launches of 3,000 to 4,700 workgroups break even.
static bool msd_few_lags(uint64_t N, uint32_t nblocks, uint32_t n, uint32_t skip, uint32_t leff, bool cm_self) {
    const double M = (leff + skip - 1) / skip, K = (n + skip - 1) / skip;
    return skip > 1 && (N + 63) / 64 * std::min(skip, leff) * nblocks >= 8192 && (M - (cm_self ? 2.34 : 1.28)) * K < 8;
}

// msd.cpp:52-61 checks (leff is common to all blocks: min(n_b, tmax) must
// agree); fills P's sizes and the host tables of the block list and the
// term counts.  Touches no device memory.
static void msd_plan(anl_traj *tr, const uint64_t *primo, const uint32_t *n, uint32_t nblocks, uint32_t skip,
                     uint32_t tmax, int cm_msd, int cm_self, MsdPrepared *P, std::vector<MsdBlock> *hb,
                     std::vector<uint64_t> *hc) {
    if (nblocks == 0) fail(ANL_ERR_ARG, "no blocks");
    if (skip == 0) skip = 1;
    const uint32_t leff = (n[0] < tmax || tmax == 0) ? n[0] : tmax;  // msd.cpp:42
    for (uint32_t b = 0; b < nblocks; b++) {
        const uint32_t lb = (n[b] < tmax || tmax == 0) ? n[b] : tmax;
        if (lb != leff) fail(ANL_ERR_ARG, "blocks with different numbers of lags cannot be averaged together");
        if ((uint64_t)leff + n[b] + primo[b] > tr->F)
            fail(ANL_ERR_TOO_SHORT,
                 "trajectory is too short for this kind of calculation. Select a different starting timestep or "
                 "lower the size of the average or the lenght of the time lag");
        if ((uint64_t)leff + n[b] > tr->F)
            fail(ANL_ERR_NOT_LOADED, "there are not enough loaded timesteps inside the trajectory object. I need at "
                                     "least " + std::to_string((uint64_t)leff + n[b]) +
                                         " timesteps to do the requested calculation");
    }
    if ((cm_msd || cm_self) && !tr->cm) fail(ANL_ERR_ARG, "centre-of-mass series not provided");
    P->tr = tr;
    P->skip = skip;
    P->leff = leff;
    P->nblocks = nblocks;
    P->nt = tr->nt;
    P->fcm = cm_msd ? 2 : 1;
    P->cm_msd = cm_msd;
    P->cm_self = cm_self;
    const bool own = !msd_chosen_shape(tr, skip, leff);
    P->tile = tr->msd_tile;
    P->waves = tr->msd_waves;
    // a partial sum per 64 atoms; per 256 at the strides and in the kernel that
    // once had them all, where 64 would take more than 8 MiB (what fits a
    // caller's scratch stays what it was)
    const uint64_t c64 = (tr->N + 63) / 64;
    P->group = (P->tile == 0 || skip > 1) && (uint64_t)leff * c64 * tr->nt * sizeof(double) > (8ull << 20) ? 4 : 1;
    P->nchunks = (uint32_t)((c64 + P->group - 1) / P->group);
    P->maxseg = 1;
    hb->assign(nblocks, MsdBlock{});
    hc->assign((size_t)nblocks * tr->nt, 0);
    uint64_t segs = 0;
    uint32_t nmax = 0;
    for (uint32_t b = 0; b < nblocks; b++) {
        const uint32_t nseg = P->tile && leff ? msd_segments(tr->N, tr->nt, n[b], skip, leff) : 1;
        P->maxseg = std::max(P->maxseg, nseg);
        segs += nseg;
        nmax = std::max(nmax, n[b]);
        (*hb)[b] = MsdBlock{primo[b], n[b], nseg};
        const uint64_t n0 = (n[b] + skip - 1) / skip;
        for (uint32_t k = 0; k < tr->nt; k++) (*hc)[(size_t)b * tr->nt + k] = n0 * tr->type_count[k];
    }
    if (P->tile && own && leff) {
        const uint32_t M = (leff + skip - 1) / skip;
        P->tile = msd_auto_tile((uint64_t)P->nchunks * std::min(skip, leff) * segs, M, cm_self);
        P->waves = 4;
        if (P->maxseg == 1 && msd_few_lags(tr->N, nblocks, nmax, skip, leff, cm_self)) P->tile = 0;
    }
    if (nblocks == 1 && tr->nt <= MSD_INL) {
        P->tables.one = (*hb)[0];
        std::copy(hc->begin(), hc->end(), P->tables.cnt);
    }
}

// whether the tables of a planned launch travel in the kernel arguments
static bool msd_inline_tables(const MsdPrepared &P) { return P.nblocks == 1 && P.nt <= MSD_INL; }

// partial sums of a planned launch: [nblocks][leff][maxseg][nchunks][nt] doubles
static size_t msd_partial_len(const MsdPrepared &P) {
    return std::max<size_t>(1, (size_t)P.nblocks * P.leff * P.maxseg * P.nchunks * P.nt);
}

void *msd_prepare_blocks(anl_traj *tr, const uint64_t *primo, const uint32_t *n, uint32_t nblocks, uint32_t skip,
                         uint32_t tmax, int cm_msd, int cm_self, uint32_t *leff_out) {
    auto *P = new MsdPrepared();
    try {
        std::vector<MsdBlock> hb;
        std::vector<uint64_t> hc;
        msd_plan(tr, primo, n, nblocks, skip, tmax, cm_msd, cm_self, P, &hb, &hc);
        ensure_device();
        if (!msd_inline_tables(*P)) {
            const size_t nb = nblocks * sizeof(MsdBlock), nc = hc.size() * sizeof(uint64_t);
            ANL_HIP(hipMalloc(&P->d_tables, nb + nc));
            ANL_HIP(hipMemcpy(P->d_tables, hb.data(), nb, hipMemcpyHostToDevice));
            ANL_HIP(hipMemcpy((char *)P->d_tables + nb, hc.data(), nc, hipMemcpyHostToDevice));
            P->tables.blocks = (const MsdBlock *)P->d_tables;
            P->tables.count = (const uint64_t *)((const char *)P->d_tables + nb);
        }
        ANL_HIP(hipMalloc(&P->d_partial, msd_partial_len(*P) * sizeof(double)));
    } catch (...) {
        delete P;
        throw;
    }
    if (leff_out) *leff_out = P->leff;
    return P;
}

// out: [nblocks][leff][fcm][nt].  A launch holds less than 2^32 threads: more
// blocks than that go one range after the other.
void msd_enqueue_prepared(void *prep, double *out, hipStream_t s) {
    const MsdPrepared &P = *(const MsdPrepared *)prep;
    if (P.leff == 0) return;
    const anl_traj *tr = P.tr;
    const uint32_t span = P.waves * P.tile;  // lags per workgroup of the window kernel
    const uint32_t nres = std::min(P.skip, P.leff), M = (P.leff + P.skip - 1) / P.skip;
    const uint32_t ntiles = P.tile ? (M + span - 1) / span : 0, nlb = (P.leff + MSD_TL - 1) / MSD_TL;
    const uint32_t ncm = P.cm_msd ? P.nt * ((P.leff + 63) / 64) : 0;
    // threads of a block
    const uint64_t wgs = P.tile ? (uint64_t)ntiles * nres * P.maxseg * P.nchunks : 0;
    const uint64_t threads = std::max(wgs * 64 * P.waves, ((uint64_t)P.leff * P.nt / 4 + 1 + ncm) * 256);
    constexpr uint64_t LIMIT = (1ull << 32) - (1u << 14);  // grids are rounded up to 8 workgroups
    if (threads > LIMIT) fail(ANL_ERR_ARG, "MSD launch too large (reduce the number of lags)");
    const uint32_t range = (uint32_t)std::min<uint64_t>(P.tile ? P.nblocks : std::min(P.nblocks, 65535u), LIMIT / threads);
    for (uint32_t b0 = 0; b0 < P.nblocks; b0 += range) {
        const uint32_t nb = std::min(range, P.nblocks - b0);
        MsdTables tables = P.tables;
        if (tables.blocks) tables.blocks += b0;
        if (tables.count) tables.count += (uint64_t)b0 * P.nt;
        double *partial = P.d_partial + (uint64_t)b0 * P.leff * P.maxseg * P.nchunks * P.nt;
        if (P.tile) {
            const uint64_t total = wgs * nb, per = (total + 7) / 8;
            const dim3 grid((uint32_t)(8 * per));
#define ANL_MSD_WIN(R, W, C)                                                                             \
    hipLaunchKernelGGL((msd_window_kernel<R, W, C>), grid, dim3(64 * W), 0, s, tr->pos, tr->cm, tr->type_slot, \
                       tr->N, P.nt, tables, P.maxseg, P.skip, P.leff, P.nchunks, P.group, ntiles, nres,           \
                       (uint32_t)per, (uint32_t)total, partial)
#define ANL_MSD_CASE(R, W)                          \
    case (R) * 64 + (W) * 2: ANL_MSD_WIN(R, W, false); break; \
    case (R) * 64 + (W) * 2 + 1: ANL_MSD_WIN(R, W, true); break;
            switch (P.tile * 64 + P.waves * 2 + (P.cm_self ? 1 : 0)) {
                ANL_MSD_CASE(8, 4)
                ANL_MSD_CASE(12, 4)
                ANL_MSD_CASE(16, 4)
                ANL_MSD_CASE(24, 4)
                ANL_MSD_CASE(16, 8)
                ANL_MSD_CASE(24, 8)
                ANL_MSD_CASE(12, 12)
                ANL_MSD_CASE(16, 12)
                ANL_MSD_CASE(8, 16)
                default: fail(ANL_ERR_ARG, "unsupported MSD launch shape");
            }
#undef ANL_MSD_CASE
#undef ANL_MSD_WIN
        } else {
            auto kernel = P.cm_self ? msd_atoms_kernel<true> : msd_atoms_kernel<false>;
            hipLaunchKernelGGL(kernel, dim3((uint32_t)((tr->N + MSD_WG - 1) / MSD_WG), nlb, nb), dim3(MSD_WG), 0, s,
                               tr->pos, tr->cm, tr->type_slot, tr->N, P.nt, tables, P.skip, P.leff, P.nchunks, P.group,
                               partial);
        }
        ANL_HIP(hipGetLastError());
        const uint32_t nfin = (uint32_t)(((uint64_t)nb * P.leff * P.nt + 3) / 4);
        hipLaunchKernelGGL(msd_finish_kernel, dim3(nfin + nb * ncm), dim3(256), 0, s, partial, P.nchunks, P.maxseg, P.nt,
                           P.leff, nb, tables, P.fcm, tr->cm, P.skip, nfin,
                           out + (uint64_t)b0 * P.leff * P.nt * P.fcm);
        ANL_HIP(hipGetLastError());
    }
}

void msd_free_prepared(void *prep) { delete (MsdPrepared *)prep; }

// One MSD calculation whose block table, term counts and partial sums live
// in caller-provided device memory (scratch, scratch_bytes, 256-byte
// aligned); allocates nothing.  The tables are copied in on stream s, which
// is synchronised before returning (the host tables are locals).
void msd_calculate_in_scratch(anl_traj *tr, uint32_t skip, uint32_t tmax, int cm_msd, int cm_self, uint32_t n,
                              uint64_t primo, double *out, unsigned char *scratch, size_t scratch_bytes,
                              hipStream_t s) {
    MsdPrepared P;
    P.owns = false;
    std::vector<MsdBlock> hb;
    std::vector<uint64_t> hc;
    msd_plan(tr, &primo, &n, 1, skip, tmax, cm_msd, cm_self, &P, &hb, &hc);
    auto al = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t b_blocks = al(sizeof(MsdBlock)), b_count = al(hc.size() * sizeof(uint64_t));
    const size_t b_partial = al(msd_partial_len(P) * sizeof(double));
    if (b_blocks + b_count + b_partial > scratch_bytes)
        fail(ANL_ERR_ARG, "MSD of " + std::to_string(tr->N) + " atoms and " + std::to_string(P.leff) + " lags needs " +
                              std::to_string(b_blocks + b_count + b_partial) + " bytes of scratch, more than the " +
                              std::to_string(scratch_bytes) + " of the allocation-free entry point");
    P.d_partial = reinterpret_cast<double *>(scratch + b_blocks + b_count);
    if (!msd_inline_tables(P)) {
        P.tables.blocks = reinterpret_cast<MsdBlock *>(scratch);
        P.tables.count = reinterpret_cast<uint64_t *>(scratch + b_blocks);
        ANL_HIP(hipMemcpyAsync(scratch, hb.data(), sizeof(MsdBlock), hipMemcpyHostToDevice, s));
        ANL_HIP(hipMemcpyAsync(scratch + b_blocks, hc.data(), hc.size() * sizeof(uint64_t), hipMemcpyHostToDevice, s));
    }
    msd_enqueue_prepared(&P, out, s);
    ANL_HIP(hipStreamSynchronize(s));
}

// One calculation on stream s, finished on return, with a workspace of the
// trajectory's pool (an allocation and its free cost more than a small
// calculation).  The result goes to out_dev or, without it, through pinned
// memory to out_host.
static void msd_run(anl_traj *tr, uint32_t skip, uint32_t tmax, int cm_msd, int cm_self, uint32_t n, uint64_t primo,
                    double *out_dev, double *out_host, hipStream_t s) {
    MsdPrepared P;
    P.owns = false;
    std::vector<MsdBlock> hb;
    std::vector<uint64_t> hc;
    msd_plan(tr, &primo, &n, 1, skip, tmax, cm_msd, cm_self, &P, &hb, &hc);
    ensure_device();
    const size_t len = (size_t)P.leff * P.nt * P.fcm * sizeof(double);
    auto al = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t b_partial = al(msd_partial_len(P) * sizeof(double));
    const size_t b_tables = msd_inline_tables(P) ? 0 : al(sizeof(MsdBlock)) + al(hc.size() * sizeof(uint64_t));
    // a small result is written to pinned memory by the kernel itself
    const bool direct = out_host && len <= (64u << 10);
    const size_t b_out = out_host && !direct ? al(len) : 0;
    ScratchLease w(tr->scratch, b_partial + b_tables + b_out, out_host ? std::max<size_t>(len, 256) : 0);
    char *d = (char *)w.s.dev;
    P.d_partial = (double *)d;
    if (b_tables) {
        char *t = d + b_partial;
        P.tables.blocks = (const MsdBlock *)t;
        P.tables.count = (const uint64_t *)(t + al(sizeof(MsdBlock)));
        ANL_HIP(hipMemcpyAsync(t, hb.data(), sizeof(MsdBlock), hipMemcpyHostToDevice, s));
        ANL_HIP(hipMemcpyAsync(t + al(sizeof(MsdBlock)), hc.data(), hc.size() * sizeof(uint64_t),
                               hipMemcpyHostToDevice, s));
    }
    double *out = out_dev ? out_dev : direct ? (double *)w.s.pin : (double *)(d + b_partial + b_tables);
    // the workspace goes back to the pool after the stream is done with it,
    // on an error too
    try {
        msd_enqueue_prepared(&P, out, s);
        if (b_out) ANL_HIP(hipMemcpyAsync(w.s.pin, out, len, hipMemcpyDeviceToHost, s));
    } catch (...) {
        (void)hipStreamSynchronize(s);
        throw;
    }
    ANL_HIP(hipStreamSynchronize(s));
    if (out_host) std::memcpy(out_host, w.s.pin, len);
}

}  // namespace anl

using namespace anl;

extern "C" {

int anl_msd_calculate_async(anl_traj *tr, uint32_t skip, uint32_t tmax, int cm_msd, int cm_self, uint32_t n,
                            uint64_t primo, double *out_dev, void *stream) {
    return guard([&] {
        if (!tr || !out_dev) fail(ANL_ERR_ARG, "null pointer passed to anl_msd_calculate_async");
        msd_run(tr, skip, tmax, cm_msd, cm_self, n, primo, out_dev, nullptr, (hipStream_t)stream);
    });
}

int anl_msd_calculate(anl_traj *tr, uint32_t skip, uint32_t tmax, int cm_msd, int cm_self, uint32_t n, uint64_t primo,
                      double *out_host) {
    return guard([&] {
        if (!tr || !out_host) fail(ANL_ERR_ARG, "null pointer passed to anl_msd_calculate");
        msd_run(tr, skip, tmax, cm_msd, cm_self, n, primo, nullptr, out_host, nullptr);
    });
}

static const char *MSD_SHAPE_MSG =
    "MSD launch shape must be lag tile 0, or (lag tile, wavefronts) one of (8,4) (12,4) (16,4) (24,4) (16,8) "
    "(24,8) (12,12) (16,12) (8,16)";

int anl_msd_set_tuning(anl_traj *tr, uint32_t lag_tile, uint32_t waves) {
    return guard([&] {
        if (!tr) fail(ANL_ERR_ARG, "null trajectory");
        if (!msd_shape_ok(lag_tile, waves)) fail(ANL_ERR_ARG, MSD_SHAPE_MSG);
        tr->msd_tile = lag_tile;
        tr->msd_waves = lag_tile ? waves : 4;
        tr->msd_auto = false;
    });
}

int anl_msd_get_tuning(anl_traj *tr, uint32_t *lag_tile, uint32_t *waves) {
    return guard([&] {
        if (!tr || !lag_tile) fail(ANL_ERR_ARG, "null pointer passed to anl_msd_get_tuning");
        *lag_tile = tr->msd_tile;
        if (waves) *waves = tr->msd_waves;
    });
}

// Times the MSD calculation (reset(n) at primo) with each candidate lag tile:
// one untimed and one timed call each (HIP events on the null stream); keeps
// the fastest in the trajectory.
int anl_msd_autotune(anl_traj *tr, uint32_t skip, uint32_t tmax, int cm_msd, int cm_self, uint32_t n, uint64_t primo,
                     const uint32_t *cand, uint32_t ncand, float *ms_out, uint32_t *best_out) {
    return guard([&] {
        if (!tr) fail(ANL_ERR_ARG, "null trajectory");
        // (lag tile, wavefronts) pairs
        static const uint32_t defaults[] = {8, 4, 12, 4, 16, 4, 24, 4, 16, 8, 24, 8, 12, 12, 16, 12, 8, 16, 0, 4};
        if (!cand) {
            cand = defaults;
            ncand = sizeof(defaults) / sizeof(defaults[0]) / 2;
        }
        if (ncand == 0) fail(ANL_ERR_ARG, "no candidates");
        for (uint32_t c = 0; c < ncand; c++)
            if (!msd_shape_ok(cand[2 * c], cand[2 * c + 1]))
                fail(ANL_ERR_ARG, "candidate " + std::to_string(c) + ": " + MSD_SHAPE_MSG);
        ensure_device();
        const uint32_t saved = tr->msd_tile, saved_w = tr->msd_waves;
        const bool saved_auto = tr->msd_auto;
        tr->msd_auto = false;
        const uint32_t leff = (n < tmax || tmax == 0) ? n : tmax;
        double *d = nullptr;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        void *P = nullptr;
        float best = -1.0f;
        uint32_t besti = 0;
        try {
            ANL_HIP(hipMalloc(&d, std::max<size_t>(1, (size_t)leff * tr->nt * 2) * sizeof(double)));
            ANL_HIP(hipEventCreate(&e0));
            ANL_HIP(hipEventCreate(&e1));
            for (uint32_t c = 0; c < ncand; c++) {
                tr->msd_tile = cand[2 * c];
                tr->msd_waves = cand[2 * c] ? cand[2 * c + 1] : 4;
                P = msd_prepare_blocks(tr, &primo, &n, 1, skip, tmax, cm_msd, cm_self, nullptr);
                msd_enqueue_prepared(P, d, 0);
                ANL_HIP(hipEventRecord(e0, 0));
                msd_enqueue_prepared(P, d, 0);
                ANL_HIP(hipEventRecord(e1, 0));
                ANL_HIP(hipEventSynchronize(e1));
                msd_free_prepared(P);
                P = nullptr;
                float ms = 0.0f;
                ANL_HIP(hipEventElapsedTime(&ms, e0, e1));
                if (ms_out) ms_out[c] = ms;
                if (best < 0.0f || ms < best) {
                    best = ms;
                    besti = c;
                }
            }
        } catch (...) {
            tr->msd_tile = saved;
            tr->msd_waves = saved_w;
            tr->msd_auto = saved_auto;
            if (P) {
                (void)hipDeviceSynchronize();
                msd_free_prepared(P);
            }
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
            (void)hipFree(d);
            throw;
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        (void)hipFree(d);
        tr->msd_tile = cand[2 * besti];
        tr->msd_waves = cand[2 * besti] ? cand[2 * besti + 1] : 4;
        if (best_out) *best_out = besti;
    });
}

}  // extern "C"
