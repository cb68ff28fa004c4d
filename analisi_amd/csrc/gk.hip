// Green-Kubo N-component lag correlations (greenkuboNcomponentionicfluid.cpp:
// 156-356) on the device, in the reference's FP64 operation order so that the
// correlation functions, their integrals and the transport coefficients match
// the reference's values:
//  * gk_chain_kernel: a lane per (lag l, current pair ab, segment, block)
//    holds the running mean
//      JJ[ab] += ((Ja(t0).Jb(t0+l))/3 - JJ[ab]) / cont      (:200-228)
//    over t0 = align, align+skip, .. < seg*(iseg+1) of its segment;
//    gk_segments_kernel takes the running mean of the segment means
//    (:230-237).
//  * gk_mean_kernel / gk_integral_kernel / gk_schur_kernel: the serial
//    epilogue (:259-356) as column-parallel prefix scans and a lag-parallel
//    Schur complement of the symmetrised integral matrix.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <optional>
#include <thread>
#include <type_traits>

#include "anl_internal.h"

#pragma clang fp contract(off)

namespace anl {

constexpr int GK_MAXC = 4;  // up to 4 vector currents (16 correlation pairs)

constexpr uint32_t GK_MAXB = 64;  // blocks per launch

// Per-block t0 ranges of one launch: block b starts at row primo[b] and
// averages over n[b] t0 values; its output is out + b * out_stride.
struct GkBlocks {
    uint64_t primo[GK_MAXB];
    uint32_t n[GK_MAXB];
};

struct GkArgs {
    const double *data;
    const double2 *rec;  // [nrows] {RN(1/c), the rest of 1/c}, c = 1 ..
    uint64_t nrows;
    uint32_t ncols;
    uint32_t ncur;
    uint32_t idx[GK_MAXC];
    uint32_t n_seg, skip, leff, narr;
    uint32_t seg0;        // first segment of this launch
    uint64_t out_stride;
    double *out;   // [block][leff][narr]
    double *segm;  // segment means [block][segment][pair][lag], or null: fold into out
    GkBlocks bl;
};

// a / c for an integer c < 2^32 from y = {yh, yl}, yh = RN(1/c) and yl =
// 1/c - yh to about 2^-50 of itself: the correctly rounded quotient, in two
// operations.  yh + yl is 1/c to 2^-102 of it, and a yl rounds once, so the
// last rounding sees a/c to better than 2^-100 of it.  With the quotient
// scaled so that its rounding midpoints are odd integers M < 2^54, a/c is
// never a midpoint (c M has 54 significant bits or more, a has 53), so
// |a/c - M| >= 1/c > 2^-32, which is far more than 2^54 2^-100: both sides
// round to the same number.  Needs |a| in (GK_TINY, inf): below it a yl may
// lose bits to underflow, and inf * 0 is not a number.
constexpr double GK_TINY = 0x1p-900;
__device__ __forceinline__ double div_by(double a, double2 y) { return fma(a, y.x, a * y.y); }

__global__ __launch_bounds__(256) void gk_reciprocal_kernel(double2 *__restrict__ rec, uint64_t n) {
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double c = (double)(k + 1), y = 1.0 / c;
    rec[k] = make_double2(y, fma(-c, y, 1.0) / c);
}

// Lane J of each row of 16 lanes, in every lane of the row: what all lanes
// need of 16 t0 sits in one register and costs a move each, where an LDS
// broadcast moves 512 bytes through a port of 128 per clock.
template <int J>
__device__ __forceinline__ double row_lane(double v) {
#ifdef __HIP_DEVICE_COMPILE__
    const long long x = __builtin_bit_cast(long long, v);
    const long long r = __builtin_amdgcn_update_dpp(0ll, x, 0x150 + J, 0xf, 0xf, true);  // row_newbcast:J
    return __builtin_bit_cast(double, r);
#else
    return v;
#endif
}

// Smallest |d| so far, by the high words read as FP32: their order is that of
// the doubles (what reads as a NaN is 2^1017 or more, and either passes or
// sends the steps to true divisions); one operation for two values.
constexpr float GK_TINY_HI = 0x1.6p-112f;  // 0x07b00000, the high word of GK_TINY
__device__ __forceinline__ void track_min(float &m, double d0, double d1) {
    const int h0 = __double2hiint(d0), h1 = __double2hiint(d1);
    asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(h0), "v"(h1));
}

template <int N, int I = 0, class F>
__device__ __forceinline__ void gk_for(F &&f) {  // f(integral_constant 0) .. f(integral_constant N-1)
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        gk_for<N, I + 1>(f);
    }
}

// One workgroup = 64 lags of one current pair, one segment and one block, a
// running mean per lane:
//     JJ += ((Ja(t0).Jb(t0+l))/3 - JJ) / cont            (:200-228)
// The chain over t0 is serial (its roundings are the reference's): four
// dependent FP64 operations per t0, 5.4 clocks each, and a wavefront issues
// an instruction of any kind about every 4.3 clocks.  So wavefront 0 runs the
// chain and nothing else, and wavefronts 1 to 3 form the terms Ja.Jb/3 of the
// next round of T = 48 t0, 16 each, and hand them over in LDS (two buffers,
// one barrier per round).  They also stage the rows: global loads two rounds
// ahead into registers, then LDS.
// LDS: Jb as one plane per component; with t0 stride 1 a lane's rows of two
// consecutive t0 are adjacent and each row is stored with its successor, so
// that one 16-byte read serves both (ds_read2_b64 of the two measured twice
// the time).  LDS traffic is 20 clocks per t0.
// Divisions by 3 and by cont are two operations each (div_by); steps outside
// its range (a difference or product of zero included) take true divisions.
// Rows of a round: contiguous where skip <= 64 (row rr of the round is
// series row base + rr), else 64 rows per t0.
// Measured, 2 currents: 5,000 lags x 95,001 t0 2.85 ms (47 to 50 clocks per
// t0; one thread per lag with true divisions took 44.2 ms), 2,000 lags x 4
// segments of 4,500 t0 0.16 ms (8.37 ms).
constexpr uint32_t gk_rows(uint32_t T, uint32_t maxskip) { return 64 + (T - 1) * maxskip; }
// doubles of a plane of at least n: planes start 12 banks apart, so that the
// lanes of a store, which walk all planes, spread over the banks (with planes
// a multiple of 64 banks apart the stores conflicted six ways and took half of
// the LDS time)
constexpr uint32_t gk_plane(uint32_t n) { return (n + 25) / 32 * 32 + 6; }

template <uint32_t T, uint32_t MAXSKIP>
__global__ __launch_bounds__(256, 1) void gk_chain_kernel(const GkArgs a) {
    constexpr bool ONE = MAXSKIP == 1;
    constexpr uint32_t ROWS = gk_rows(T, MAXSKIP), NC = ONE ? 2 : 1, PL = gk_plane(NC * ROWS), G = T / 16;
    constexpr uint32_t NPT = 192, PF = (3 * ROWS + NPT - 1) / NPT;
    static_assert(3 * T <= NPT && T % 16 == 0 && G <= 3, "16 t0 and one Ja value per producer");
    __shared__ __align__(16) double Bs[2][3][PL];  // t0 stride 1: rows r and r + 1 at 2r
    __shared__ double As[2][3][T];
    __shared__ double Ys[4][2][T];
    __shared__ __align__(16) double2 Xs[2][T / 2][64];  // terms of t0 2i, 2i + 1
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u, l16 = lane & 15u;
    const uint32_t np = a.ncur * a.ncur, ntile = (a.leff + 63) / 64;
    const uint32_t pair = blockIdx.x / ntile, tile = blockIdx.x - pair * ntile;
    const uint32_t iseg = a.seg0 + blockIdx.y, blk = blockIdx.z;
    const uint64_t primo = a.bl.primo[blk];
    const uint32_t seg = a.bl.n[blk] / a.n_seg;
    const uint32_t first = seg * iseg + (seg * iseg) % a.skip, end = seg * (iseg + 1);  // :208
    const uint32_t n0 = first < end ? (end - first - 1) / a.skip + 1 : 0;
    const uint32_t nst = (n0 + T - 1) / T;
    double JJ = 0.0;
    if (wave == 0) {
        struct Sub {
            double2 x[8];
            double y0, y1;
        };
        float dmin = 1.0f;
        auto read = [&](Sub &r, uint32_t k, uint32_t g) {
#pragma unroll
            for (uint32_t j = 0; j < 8; j++) r.x[j] = Xs[k & 1u][8 * g + j][lane];
            r.y0 = Ys[k & 3u][0][16 * g + l16];
            r.y1 = Ys[k & 3u][1][16 * g + l16];
        };
        // the chain over the 16 steps in r, the operands of group g of round k
        // read into n between its operations: each of them waits for the one
        // before and leaves an issue slot (the barriers keep the order)
        auto steps = [&](const Sub &r, Sub &n, uint32_t k, uint32_t g) {
            const double2 *X = &Xs[k & 1u][8 * g][lane];
            double dlast = 0.0;
            gk_for<16>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                const double d = (j & 1 ? r.x[j / 2].y : r.x[j / 2].x) - JJ;
                const double yl = row_lane<j>(r.y1);
                __builtin_amdgcn_sched_barrier(0);
                const double m = d * yl;
                const double yh = row_lane<j>(r.y0);
                __builtin_amdgcn_sched_barrier(0);
                const double q = fma(d, yh, m);
                if constexpr (j & 1) n.x[j / 2] = X[j / 2 * 64];
                else if constexpr (j == 0) n.y0 = Ys[k & 3u][0][16 * g + l16];
                else if constexpr (j == 2) n.y1 = Ys[k & 3u][1][16 * g + l16];
                __builtin_amdgcn_sched_barrier(0);
                JJ = JJ + q;
                if constexpr (j & 1) track_min(dmin, dlast, d);
                dlast = d;
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        auto slow = [&](uint32_t k, uint32_t s0, uint32_t s1) {  // steps s0 .. s1 - 1 of round k with true divisions
            for (uint32_t s = s0; s < s1; s++) {
                const double2 x = Xs[k & 1u][s / 2][lane];
                const double d = (s & 1 ? x.y : x.x) - JJ;
                JJ = JJ + d / (double)(k * T + s + 1);
            }
        };
        __syncthreads();
        __syncthreads();
        for (uint32_t k = 0; k < nst; k++) {
            const uint32_t cnt = min(T, n0 - k * T), full = cnt / 16;
            const double J0 = JJ;
            dmin = 1.0f;
            Sub r0, r1;
            if (full) read(r0, k, 0);
            for (uint32_t g = 0; g < full; g += 2) {
                steps(r0, r1, k, min(g + 1, G - 1));
                if (g + 1 < full) steps(r1, r0, k, min(g + 2, G - 1));
            }
            if (__ballot(!(dmin > GK_TINY_HI) || !(fabs(JJ) < 0x1p1000))) {
                JJ = J0;
                slow(k, 0, 16 * full);
            }
            slow(k, 16 * full, cnt);  // the last round's remainder
            __syncthreads();
        }
    } else {
        const uint32_t p = threadIdx.x - 64u;  // producer thread
        const uint32_t ca = a.idx[pair / a.ncur], cb = a.idx[pair % a.ncur];
        const uint64_t ra = primo + first, rb = ra + (uint64_t)tile * 64u, last = a.nrows - 1;
        const uint32_t skip = a.skip, rs = min(skip, 64u);
        // this thread's loads of a round: PF values of Jb rows, one of Ja, one
        // part of 1/cont.  Rows past the series' end are clamped to the last
        // one (their lags are not used).
        struct Regs {
            double b[PF], a, y;
        };
        const double *pb[PF], *lb[PF];
#pragma unroll
        for (uint32_t j = 0; j < PF; j++) {
            const uint32_t e = p + NPT * j, rr = e / 3, x = e - 3 * rr;
            const uint64_t off = skip <= 64 ? rr : (uint64_t)(rr / 64) * skip + rr % 64;
            pb[j] = a.data + (rb + off) * a.ncols + cb + x;
            lb[j] = a.data + last * a.ncols + cb + x;
        }
        const uint32_t pa3 = min(p, 3 * T - 1), py = min(p, 2 * T - 1);
        const double *pa = a.data + (ra + (uint64_t)(pa3 / 3) * skip) * a.ncols + ca + pa3 % 3;
        const double *la = a.data + last * a.ncols + ca + pa3 % 3;
        const double *pyr = reinterpret_cast<const double *>(a.rec) + py;
        const double *ly = reinterpret_cast<const double *>(a.rec) + 2 * last + (py & 1u);
        const uint64_t step = (uint64_t)T * skip * a.ncols;
        auto fetch = [&](Regs &r) {  // the next round's
#pragma unroll
            for (uint32_t j = 0; j < PF; j++) {
                r.b[j] = *(pb[j] < lb[j] ? pb[j] : lb[j]);
                pb[j] += step;
            }
            r.a = *(pa < la ? pa : la);
            pa += step;
            r.y = *(pyr < ly ? pyr : ly);
            pyr += 2 * T;
        };
        auto stash = [&](const Regs &r, uint32_t k) {
#pragma unroll
            for (uint32_t j = 0; j < PF; j++) {
                const uint32_t e = p + NPT * j, rr = e / 3, x = e - 3 * rr;
                if (rr < ROWS) {
                    Bs[k & 1u][x][NC * rr] = r.b[j];
                    if (ONE && rr) Bs[k & 1u][x][2 * rr - 1] = r.b[j];
                }
            }
            if (p < 3 * T) As[k & 1u][p % 3][p / 3] = r.a;
            if (p < 2 * T) Ys[k & 3u][p & 1u][p / 2] = r.y;
        };
        const double2 third = make_double2(1.0 / 3.0, 0x1.5555555555555p-56);  // 1/3 - RN(1/3) = RN(1/3) 2^-54
        const uint32_t w = wave - 1;
        auto produce = [&](uint32_t k) {  // terms of t0 16w .. 16w + 15 of round k
            if (w >= G) return;
            const uint32_t buf = k & 1u;
            const double A0 = As[buf][0][16 * w + l16], A1 = As[buf][1][16 * w + l16], A2 = As[buf][2][16 * w + l16];
            double b[2][3][4];
            auto read = [&](double (&r)[3][4], uint32_t s) {  // steps s .. s + 3
#pragma unroll
                for (uint32_t c = 0; c < 3; c++) {
                    if (ONE) {
                        const double2 *q = reinterpret_cast<const double2 *>(&Bs[buf][c][2 * (lane + s)]);
                        const double2 u = q[0], v = q[2];
                        r[c][0] = u.x, r[c][1] = u.y, r[c][2] = v.x, r[c][3] = v.y;
                    } else {
#pragma unroll
                        for (uint32_t j = 0; j < 4; j++) r[c][j] = Bs[buf][c][(s + j) * rs + lane];
                    }
                }
            };
            read(b[0], 16 * w);
            gk_for<4>([&](auto mc) {
                constexpr int m = decltype(mc)::value;
                if constexpr (m < 3) read(b[(m + 1) & 1], 16 * w + 4 * m + 4);
                double pr[4], x[4];
                gk_for<4>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    double q = row_lane<4 * m + j>(A0) * b[m & 1][0][j];
                    q = q + row_lane<4 * m + j>(A1) * b[m & 1][1][j];
                    pr[j] = q + row_lane<4 * m + j>(A2) * b[m & 1][2][j];
                });
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) x[j] = div_by(pr[j], third);
                float least = 1.0f;
                track_min(least, pr[0], pr[1]);
                track_min(least, pr[2], pr[3]);
                if (__ballot(!(least > GK_TINY_HI))) {
#pragma unroll
                    for (uint32_t j = 0; j < 4; j++) x[j] = pr[j] / 3.0;
                }
                Xs[buf][8 * w + 2 * m][lane] = make_double2(x[0], x[1]);
                Xs[buf][8 * w + 2 * m + 1][lane] = make_double2(x[2], x[3]);
            });
        };
        Regs r0{}, r1{};
        fetch(r0);
        if (nst > 1) fetch(r1);
        stash(r0, 0);
        if (nst > 2) fetch(r0);
        __syncthreads();
        // while round k - 1 is summed: form round k, stage round k + 1, load round k + 3
        auto round = [&](Regs &r, uint32_t k) {
            if (k < nst) produce(k);
            if (k + 1 < nst) stash(r, k + 1);
            if (k + 3 < nst) fetch(r);
            __syncthreads();
        };
        for (uint32_t k = 0; k <= nst; k += 2) {
            round(r1, k);
            if (k + 1 <= nst) round(r0, k + 1);
        }
        return;
    }
    const uint32_t it = tile * 64 + lane;
    if (it >= a.leff) return;
    if (a.segm) {
        a.segm[(((uint64_t)blk * a.n_seg + iseg) * np + pair) * a.leff + it] = JJ;
        return;
    }
    double *o = a.out + blk * a.out_stride + (uint64_t)it * a.narr;
    const double v = iseg ? o[pair] : 0.0;
    o[pair] = v + (JJ - v) / (double)(iseg + 1);  // :230-237
    if (it == 0 && pair == 0)  // the integrals start from zero
        for (uint32_t k = np; k < a.narr; k++) o[k] = 0.0;
}

__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The same chains for launches that fill the chip, t0 stride 1: one wavefront
// = 64 lags of CH pairs (ja, jb0 ..) or, with one current, CH x 64 lags, CH
// running means per lane that share Ja and 1/cont.  What bounds it is the
// FP64 issue: 12 operations per mean and t0 and 5 / CH broadcast moves; the
// LDS port is next (3 rows of 8 bytes per mean and t0: 12 of 16 clocks).  A
// stage of 16 t0 goes through one LDS buffer: a wavefront's LDS operations
// stay in order, so the next stage's values, loaded to registers while this
// one is summed, are stored after its last read.  VALU busy 83% on 20,000
// lags x 60,000 t0 x 8 blocks, 2 currents; 32 such blocks 90 ms per call
// with its 72 MB copied to the host (186 ms with one thread per lag).
template <int NCUR, int CH>
__global__ __launch_bounds__(64, 3) void gk_dense_kernel(const GkArgs a) {
    constexpr bool LAGS = NCUR == 1;                     // the CH means are lags 64 apart
    constexpr uint32_t T = 16, CB = LAGS ? 1 : CH;       // columns of Jb
    constexpr uint32_t ROWS = 64 * (LAGS ? CH : 1) + T - 1, PL = gk_plane(2 * ROWS), NB = 3 * CB;
    constexpr uint32_t PF = (NB * ROWS + 63) / 64;
    constexpr uint32_t NJB = LAGS ? 1 : (NCUR + CH - 1) / CH;  // groups of CH columns
    __shared__ __align__(16) double Bs[NB][PL];
    const uint32_t lane = threadIdx.x, l16 = lane & 15u;
    constexpr uint32_t W = 64 * (LAGS ? CH : 1);
    const uint32_t ntile = (a.leff + W - 1) / W;
    uint32_t z = blockIdx.x;
    const uint32_t tile = z % ntile;
    z /= ntile;
    const uint32_t jb0 = z % NJB * CH, ja = z / NJB;
    const uint32_t iseg = a.seg0 + blockIdx.y, blk = blockIdx.z;
    const uint32_t seg = a.bl.n[blk] / a.n_seg, n0 = seg;  // stride 1: every t0 of the segment
    const uint64_t ra = a.bl.primo[blk] + (uint64_t)seg * iseg, rb = ra + (uint64_t)tile * W, last = a.nrows - 1;
    // columns past the last current repeat it (their means are not stored)
    uint32_t cb[CB];
#pragma unroll
    for (uint32_t c = 0; c < CB; c++) cb[c] = a.idx[min(jb0 + c, (uint32_t)NCUR - 1)];
    const double *pb[PF], *lb[PF];
#pragma unroll
    for (uint32_t j = 0; j < PF; j++) {
        const uint32_t e = lane + 64 * j, rr = e / NB, x = e - NB * rr;
        uint32_t col = cb[0] + x;
#pragma unroll
        for (uint32_t c = 1; c < CB; c++) col = x >= 3 * c ? cb[c] + x - 3 * c : col;
        pb[j] = a.data + (rb + rr) * a.ncols + col;
        lb[j] = a.data + last * a.ncols + col;
    }
    const double *pa = a.data + (ra + l16) * a.ncols + a.idx[ja], *la = a.data + last * a.ncols + a.idx[ja];
    const double2 *py = a.rec + l16, *ly = a.rec + last;
    const uint64_t step = (uint64_t)T * a.ncols;
    struct Lane {
        double a[3];
        double2 y;
    };
    double FB[PF];
    auto fetch = [&](Lane &f) {
#pragma unroll
        for (uint32_t j = 0; j < PF; j++) {
            FB[j] = *(pb[j] < lb[j] ? pb[j] : lb[j]);
            pb[j] += step;
        }
        const double *q = pa < la ? pa : la;
        f.a[0] = q[0], f.a[1] = q[1], f.a[2] = q[2];
        pa += step;
        f.y = *(py < ly ? py : ly);
        py += T;
    };
    auto stash = [&]() {
#pragma unroll
        for (uint32_t j = 0; j < PF; j++) {
            const uint32_t e = lane + 64 * j, rr = e / NB, x = e - NB * rr;
            if (rr < ROWS) {
                Bs[x][2 * rr] = FB[j];
                if (rr) Bs[x][2 * rr - 1] = FB[j];
            }
        }
    };
    const double2 third = make_double2(1.0 / 3.0, 0x1.5555555555555p-56);
    double JJ[CH];
#pragma unroll
    for (int c = 0; c < CH; c++) JJ[c] = 0.0;
    const uint32_t nst = (n0 + T - 1) / T;
    auto rows = [&](int c, int x, uint32_t s) {  // of steps s, s + 1 (s even) of mean c, component x
        return *reinterpret_cast<const double2 *>(&Bs[LAGS ? x : 3 * c + x][2 * (lane + (LAGS ? 64 * c : 0) + s)]);
    };
    auto stage = [&](uint32_t k, const Lane &f) {
        const uint32_t c0 = k * T, cnt = min(T, n0 - c0);
        double J0[CH];
        float dmin = 1.0f;
        bool bad = cnt < T;
#pragma unroll
        for (int c = 0; c < CH; c++) J0[c] = JJ[c];
        if (!bad) {
            gk_for<8>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                double2 b[CH][3];
#pragma unroll
                for (int c = 0; c < CH; c++)
#pragma unroll
                    for (int x = 0; x < 3; x++) b[c][x] = rows(c, x, 2 * i);
                double dl[CH];
                gk_for<2>([&](auto hc) {
                    constexpr int h = decltype(hc)::value, j = 2 * i + h;
                    const double a0 = row_lane<j>(f.a[0]), a1 = row_lane<j>(f.a[1]), a2 = row_lane<j>(f.a[2]);
                    const double2 y = make_double2(row_lane<j>(f.y.x), row_lane<j>(f.y.y));
#pragma unroll
                    for (int c = 0; c < CH; c++) {
                        double q = a0 * (h ? b[c][0].y : b[c][0].x);
                        q = q + a1 * (h ? b[c][1].y : b[c][1].x);
                        q = q + a2 * (h ? b[c][2].y : b[c][2].x);
                        const double d = div_by(q, third) - JJ[c];
                        if constexpr (h == 1) track_min(dmin, dl[c], d);
                        dl[c] = d;
                        JJ[c] = JJ[c] + div_by(d, y);
                    }
                });
            });
            bad = !(dmin > GK_TINY_HI);
#pragma unroll
            for (int c = 0; c < CH; c++) bad = bad || !(fabs(JJ[c]) < 0x1p1000);
        }
        if (__ballot(bad)) {
#pragma unroll
            for (int c = 0; c < CH; c++) JJ[c] = J0[c];
            for (uint32_t s = 0; s < cnt; s++) {
                double A[3];
#pragma unroll
                for (int x = 0; x < 3; x++) A[x] = __shfl(f.a[x], (int)s);
#pragma unroll
                for (int c = 0; c < CH; c++) {
                    double q[3];
#pragma unroll
                    for (int x = 0; x < 3; x++) {
                        const double2 u = rows(c, x, s & ~1u);
                        q[x] = A[x] * (s & 1 ? u.y : u.x);
                    }
                    const double d = ((q[0] + q[1]) + q[2]) / 3.0 - JJ[c];
                    JJ[c] = JJ[c] + d / (double)(c0 + s + 1);
                }
            }
        }
    };
    Lane f0{}, f1{};
    if (nst) fetch(f0);
    // the rows pass between lanes: neither the stage's reads nor the next
    // stage's stores may move across (the hardware keeps their order, the
    // compiler would not have to)
    for (uint32_t k = 0; k < nst; k += 2) {
        wave_sync_lds();
        stash();
        wave_sync_lds();
        if (k + 1 < nst) fetch(f1);
        stage(k, f0);
        if (k + 1 < nst) {
            wave_sync_lds();
            stash();
            wave_sync_lds();
            if (k + 2 < nst) fetch(f0);
            stage(k + 1, f1);
        }
    }
    const uint32_t np = a.ncur * a.ncur;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const uint32_t it = tile * W + lane + (LAGS ? 64 * c : 0), pair = LAGS ? 0 : ja * NCUR + jb0 + c;
        if (it >= a.leff || (!LAGS && jb0 + c >= NCUR)) continue;
        if (a.segm) {
            a.segm[(((uint64_t)blk * a.n_seg + iseg) * np + pair) * a.leff + it] = JJ[c];
            continue;
        }
        double *o = a.out + blk * a.out_stride + (uint64_t)it * a.narr;
        const double v = iseg ? o[pair] : 0.0;
        o[pair] = v + (JJ[c] - v) / (double)(iseg + 1);  // :230-237
        if (it == 0 && pair == 0)
            for (uint32_t k = np; k < a.narr; k++) o[k] = 0.0;
    }
}

// The same means where a lag has few t0 (gk_plan): a thread holds every pair of
// one lag and takes the segments one after the other, with true divisions.  The
// kernels above would fill their stages for a term or two, in a workgroup per
// segment.
template <int NC>
__global__ __launch_bounds__(64) void gk_few_kernel(const GkArgs a) {
    constexpr int NP = NC * NC;
    const uint32_t it = blockIdx.x * 64 + threadIdx.x, blk = blockIdx.y;
    if (it >= a.leff) return;
    const double *d = a.data + a.bl.primo[blk] * a.ncols;
    const uint32_t seg = a.bl.n[blk] / a.n_seg;
    double v[NP] = {};
    for (uint32_t iseg = 0; iseg < (seg ? a.n_seg : 0); iseg++) {  // empty segments: the mean of zeros
        double JJ[NP] = {};
        uint32_t cont = 0;
        const uint32_t first = seg * iseg + (seg * iseg) % a.skip, end = seg * (iseg + 1);  // :208
        for (uint64_t jm = first; jm < end; jm += a.skip) {
            const double *la = d + jm * a.ncols, *lb = la + (uint64_t)it * a.ncols;
            double A[NC][3], B[NC][3];
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int x = 0; x < 3; x++) A[c][x] = la[a.idx[c] + x], B[c][x] = lb[a.idx[c] + x];
            const double dc = (double)++cont;
#pragma unroll
            for (int k = 0; k < NP; k++) {
                const double q = (A[k / NC][0] * B[k % NC][0] + A[k / NC][1] * B[k % NC][1]) + A[k / NC][2] * B[k % NC][2];
                JJ[k] = JJ[k] + (q / 3.0 - JJ[k]) / dc;  // :200-228
            }
        }
#pragma unroll
        for (int k = 0; k < NP; k++) v[k] = v[k] + (JJ[k] - v[k]) / (double)(iseg + 1);  // :230-237
    }
    double *o = a.out + blk * a.out_stride + (uint64_t)it * a.narr;
#pragma unroll
    for (int k = 0; k < NP; k++) o[k] = v[k];
    if (it == 0)  // the integrals start from zero
        for (uint32_t k = NP; k < a.narr; k++) o[k] = 0.0;
}

// The running mean over the segments (:230-237) of the segment means.
__global__ __launch_bounds__(256) void gk_segments_kernel(const GkArgs a) {
    const uint32_t np = a.ncur * a.ncur, blk = blockIdx.y;
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= np * a.leff) return;
    const uint32_t pair = w / a.leff, it = w - pair * a.leff;
    const double *m = a.segm + ((uint64_t)blk * a.n_seg * np + pair) * a.leff + it;
    double v = 0.0;
    for (uint32_t k = 0; k < a.n_seg; k++) v = v + (m[(uint64_t)k * np * a.leff] - v) / (double)(k + 1);
    double *o = a.out + blk * a.out_stride + (uint64_t)it * a.narr;
    o[pair] = v;
    if (w == 0)
        for (uint32_t k = np; k < a.narr; k++) o[k] = 0.0;
}

// The serial scans over lags below take the reference's order in wave 0 of
// one workgroup per block, a lane per column, NC columns.  Waves 1 to 7 load a
// tile of lags to registers while the tile before it is scanned, and prepare
// its terms in LDS (two buffers, one barrier per tile), so that the scan
// reads one LDS entry per lag, a batch ahead, and does only the operations
// that depend on the lag before.
constexpr uint32_t GK_SCAN = 512, GK_LOAD = GK_SCAN - 64;
constexpr uint32_t gk_scan_tile(uint32_t nc) { return 768 / nc / 16 * 16; }  // lags
constexpr uint32_t gk_scan_regs(uint32_t nc) { return ((gk_scan_tile(nc) + 1) * nc + GK_LOAD - 1) / GK_LOAD; }

// Loader thread t's values C(it0 + e / NC)[e % NC], e = t + GK_LOAD j, of a
// tile of n lags (clamped past the end).
template <uint32_t NC>
struct GkTile {
    double v[gk_scan_regs(NC)];
    __device__ __forceinline__ void load(const double *out, uint32_t narr, uint32_t it0, uint32_t n, uint32_t t) {
#pragma unroll
        for (uint32_t j = 0; j < gk_scan_regs(NC); j++) {
            const uint32_t e = min(t + GK_LOAD * j, n * NC - 1);
            v[j] = out[(uint64_t)(it0 + e / NC) * narr + e % NC];
        }
    }
};

// :259-277 the mean of C over lags [start_mean, leff) as the running mean
// m += (C - m)/c, dividing through 1/c (div_by; a tile whose differences
// leave its range takes true divisions), then subtracted from every lag.
// 1,000 of 5,000 lags, 2 currents: 42 us (77 us with true divisions).
template <uint32_t NC>
__global__ __launch_bounds__(GK_SCAN) void gk_mean_kernel(double *__restrict__ out, uint32_t leff,
                                                          uint32_t start_mean, uint64_t stride,
                                                          const double2 *__restrict__ rec) {
    constexpr uint32_t narr = 3 * NC + 2, TL = gk_scan_tile(NC), B = 8;
    __shared__ __align__(16) double2 ys[2][TL + 2 * B];
    __shared__ double cs[2][(TL + 2 * B) * NC];
    __shared__ double means[NC];
    out += blockIdx.y * stride;
    const uint32_t t = threadIdx.x, nl = start_mean < leff ? leff - start_mean : 0, ntile = (nl + TL - 1) / TL;
    double m = 0.0;
    GkTile<NC> r;
    double2 yr[2];
    static_assert(TL <= 2 * GK_LOAD, "two 1/c per loader thread");
    auto load = [&](uint32_t i) {
        const uint32_t n = min(TL, nl - i * TL);
        r.load(out, narr, start_mean + i * TL, n, t - 64);
#pragma unroll
        for (uint32_t j = 0; j < 2; j++) yr[j] = rec[i * TL + min(t - 64 + GK_LOAD * j, n - 1)];
    };
    if (t >= 64 && ntile) load(0);
    for (uint32_t i = 0; i <= ntile; i++) {  // tile i is stored, tile i - 1 scanned
        if (t >= 64 && i < ntile) {
            const uint32_t n = min(TL, nl - i * TL);
#pragma unroll
            for (uint32_t j = 0; j < gk_scan_regs(NC); j++)
                if (t - 64 + GK_LOAD * j < n * NC) cs[i & 1u][t - 64 + GK_LOAD * j] = r.v[j];
#pragma unroll
            for (uint32_t j = 0; j < 2; j++)
                if (t - 64 + GK_LOAD * j < n) ys[i & 1u][t - 64 + GK_LOAD * j] = yr[j];
            if (i + 1 < ntile) load(i + 1);
        } else if (t < 64 && i > 0) {  // the whole wavefront, for the ballot; lanes past NC repeat the last column
            const uint32_t c0 = (i - 1) * TL, n = min(TL, nl - c0);
            const double *c = cs[(i - 1) & 1u] + min(t, NC - 1);
            const double2 *y = ys[(i - 1) & 1u];
            const double m0 = m;
            double dmin = 1.0, v[B], vn[B];
            double2 w[B], wn[B];
            auto batch = [&](const double (&cv)[B], const double2 (&cw)[B], double (&nv)[B], double2 (&nw)[B],
                             uint32_t k0) {
#pragma unroll
                for (uint32_t j = 0; j < B; j++) {
                    nv[j] = c[(k0 + B + j) * NC];
                    nw[j] = y[k0 + B + j];
                    const double d = cv[j] - m;
                    dmin = fmin(dmin, fabs(d));
                    m = m + div_by(d, cw[j]);
                }
            };
#pragma unroll
            for (uint32_t j = 0; j < B; j++) {
                v[j] = c[j * NC];
                w[j] = y[j];
            }
            uint32_t k = 0;
            for (; k + 2 * B <= n; k += 2 * B) {
                batch(v, w, vn, wn, k);
                batch(vn, wn, v, w, k + B);
            }
            uint32_t k1 = k;
            if (__ballot(!(dmin > GK_TINY) || !(fabs(m) < 0x1p1000))) {
                m = m0;
                k1 = 0;
            }
            for (; k1 < n; k1++) {
                const double d = c[k1 * NC] - m;
                m = m + d / (double)(c0 + k1 + 1);
            }
        }
        __syncthreads();
    }
    if (t < NC) means[t] = m;
    __syncthreads();
#pragma unroll 8
    for (uint32_t e = t; e < leff * NC; e += GK_SCAN) {
        double *v = out + (uint64_t)(e / NC) * narr + e % NC;
        *v = *v - means[e % NC];
    }
}

// :279-288 trapezoid I and Einstein E running integrals, per correlation
// column: I(it) = (I(it-1) + C(it-1)/2) + C(it)/2, E(it) = (E(it-1) +
// C(it-1) it/2) + C(it) it/2, with I(0) = E(0) = 0 as left by the lag loop.
// A lane scans one of the 2 NC sums; its two terms of a lag are one 16-byte
// LDS entry.  5,000 lags, 2 currents: 80 us (210 us with I and E in one lane
// and their terms formed by it).
template <uint32_t NC>
__global__ __launch_bounds__(GK_SCAN) void gk_integral_kernel(double *__restrict__ out, uint32_t leff,
                                                              uint64_t stride) {
    constexpr uint32_t narr = 3 * NC + 2, TL = gk_scan_tile(NC), NS = 2 * NC, B = 8;
    __shared__ __align__(16) double2 terms[2][(TL + 2 * B) * NS];
    __shared__ double res[2][TL * NS];
    if (leff < 2) return;
    out += blockIdx.y * stride;
    const uint32_t t = threadIdx.x;
    const uint32_t ntile = (leff - 1 + TL - 1) / TL;  // tiles of lags 1 .. leff-1
    GkTile<NC> r;
    // tile i reads C of one lag more, it0 - 1: C(it)'s terms belong to lag it
    // (second) and to lag it + 1 (first)
    auto load = [&](uint32_t i) { r.load(out, narr, i * TL, min(TL, leff - 1 - i * TL) + 1, t - 64); };
    double s = t < NS ? out[NC + t] : 0.0;
    if (t >= 64) load(0);
    for (uint32_t i = 0; i <= ntile + 1; i++) {  // tile i is stored, tile i - 1 scanned, tile i - 2 written out
        if (t >= 64) {
            if (i < ntile) {
                const uint32_t n = min(TL, leff - 1 - i * TL);
                double2 *d = terms[i & 1u];
#pragma unroll
                for (uint32_t j = 0; j < gk_scan_regs(NC); j++) {
                    const uint32_t e = t - 64 + GK_LOAD * j, k = e / NC, jj = e % NC, it = i * TL + k;
                    const double v = r.v[j];
                    if (k > 0 && k <= n) {
                        d[(k - 1) * NS + 2 * jj].y = v / 2.0;
                        d[(k - 1) * NS + 2 * jj + 1].y = v * (double)it / 2.0;
                    }
                    if (k < n) {
                        d[k * NS + 2 * jj].x = v / 2.0;
                        d[k * NS + 2 * jj + 1].x = v * (double)(it + 1) / 2.0;
                    }
                }
                if (i + 1 < ntile) load(i + 1);
            }
            if (i >= 2) {
                const uint32_t it0 = 1 + (i - 2) * TL, n = min(TL, leff - it0);
                const double *src = res[i & 1u];
                for (uint32_t e = t - 64; e < n * NS; e += GK_LOAD)
                    out[(uint64_t)(it0 + e / NS) * narr + NC + e % NS] = src[e];
            }
        } else if (t < NS && i > 0 && i <= ntile) {
            const uint32_t n = min(TL, leff - 1 - (i - 1) * TL);
            const double2 *src = terms[(i - 1) & 1u] + t;
            double *dst = res[(i - 1) & 1u] + t;
            double2 v[B], w[B];
            auto batch = [&](const double2 (&c)[B], double2 (&nx)[B], uint32_t k0) {
#pragma unroll
                for (uint32_t j = 0; j < B; j++) {
                    nx[j] = src[(k0 + B + j) * NS];
                    s = (s + c[j].x) + c[j].y;
                    dst[(k0 + j) * NS] = s;
                }
            };
#pragma unroll
            for (uint32_t j = 0; j < B; j++) v[j] = src[j * NS];
            uint32_t k = 0;
            for (; k + 2 * B <= n; k += 2 * B) {
                batch(v, w, k);
                batch(w, v, k + B);
            }
            for (; k < n; k++) {  // tail of the last tile
                const double2 c = src[k * NS];
                s = (s + c.x) + c.y;
                dst[k * NS] = s;
            }
        }
        __syncthreads();
    }
}

// Parallel forms of the two scans, for the MFMA form (whose C(l) already
// differs from the FP64 one by ~1e-7 of its scale): one workgroup of 1024
// threads per block, partial sums combined in a fixed order, so the result
// is deterministic but rounds differently from the serial reference order
// above.
constexpr uint32_t GK_PAR = 1024;

// :259-277 mean of C over lags [start_mean, leff), subtracted from every lag
__global__ __launch_bounds__(GK_PAR) void gk_mean_par_kernel(double *__restrict__ out, uint32_t narr, uint32_t ncorr,
                                                             uint32_t leff, uint32_t start_mean, uint64_t stride) {
    __shared__ double red[GK_PAR];
    if (start_mean >= leff) return;
    out += blockIdx.y * stride;
    const uint32_t t = threadIdx.x, n = leff - start_mean;
    for (uint32_t j = 0; j < ncorr; j++) {
        double s = 0.0;
        for (uint32_t k = start_mean + t; k < leff; k += GK_PAR) s += out[(uint64_t)k * narr + j];  // coalesced
        red[t] = s;
        __syncthreads();
        for (uint32_t w = GK_PAR / 2; w > 0; w >>= 1) {
            if (t < w) red[t] += red[t + w];
            __syncthreads();
        }
        const double m = red[0] / (double)n;
        __syncthreads();
        for (uint32_t k = t; k < leff; k += GK_PAR) out[(uint64_t)k * narr + j] -= m;
    }
}

// Inclusive prefix sum over the 64 lanes of a wavefront (Hillis-Steele,
// fixed order).
__device__ __forceinline__ double wave_inclusive_scan(double v) {
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const double u = __shfl_up(v, off, 64);
        if (lane >= off) v += u;
    }
    return v;
}

// :279-288 I(it) = I(0) + sum_{k<=it} (C(k-1)/2 + C(k)/2), E likewise with
// weights k/2, as prefix sums over the lags.  The lags 1 .. leff-1 of a block
// are cut into gridDim.x segments, one workgroup each.  A workgroup first sums
// the terms of every lag before its segment (all threads, strided, then a
// fixed-order reduction), then each of its 16 wavefronts owns a contiguous
// range of the segment and reads it 64 consecutive lags at a time, all NC
// columns of a lag from one lane (coalesced): pass 1 sums its range, the
// ranges' offsets come from an exclusive scan of those sums, pass 2 scans
// each 64-lag batch across the lanes and carries between batches.
template <int NC>
__global__ __launch_bounds__(GK_PAR) void gk_integral_par_kernel(double *__restrict__ out, uint32_t narr,
                                                                 uint32_t leff, uint64_t stride) {
    constexpr uint32_t NW = GK_PAR / 64;
    __shared__ double tot[2 * NC][NW];
    __shared__ double pre[2 * NC][NW];
    if (leff < 2) return;
    out += blockIdx.y * stride;
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t n = leff - 1;
    const uint32_t seg = ((n + gridDim.x - 1) / gridDim.x + 63) / 64 * 64;
    const uint32_t s0 = 1 + min(n, blockIdx.x * seg), s1 = 1 + min(n, (blockIdx.x + 1) * seg);
    const uint32_t per = ((s1 - s0 + NW - 1) / NW + 63) / 64 * 64;
    const uint32_t k0 = s0 + min(s1 - s0, wv * per), k1 = s0 + min(s1 - s0, (wv + 1) * per);
    // the two trapezoid terms of lag k for every column
    auto terms = [&](uint32_t k, double (&a)[NC], double (&b)[NC]) {
        const double *rp = out + (uint64_t)(k - 1) * narr, *rv = out + (uint64_t)k * narr;
        const double dk = (double)k;
#pragma unroll
        for (int j = 0; j < NC; j++) {
            const double cp = rp[j], v = rv[j];
            a[j] = cp / 2.0 + v / 2.0;
            b[j] = cp * dk / 2.0 + v * dk / 2.0;
        }
    };
    // sums of the terms of lags 1 .. s0-1 (the segments before this one)
    double sa[NC], sb[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) sa[j] = sb[j] = 0.0;
    for (uint32_t k = 1 + threadIdx.x; k < s0; k += GK_PAR) {
        double a[NC], b[NC];
        terms(k, a, b);
#pragma unroll
        for (int j = 0; j < NC; j++) {
            sa[j] += a[j];
            sb[j] += b[j];
        }
    }
#pragma unroll
    for (int j = 0; j < NC; j++) {
        const double ta = wave_inclusive_scan(sa[j]), tb = wave_inclusive_scan(sb[j]);
        if (lane == 63) {
            pre[2 * j][wv] = ta;
            pre[2 * j + 1][wv] = tb;
        }
    }
    // sums of each wavefront's range of the segment
#pragma unroll
    for (int j = 0; j < NC; j++) sa[j] = sb[j] = 0.0;
    for (uint32_t kb = k0; kb < k1; kb += 64) {
        const uint32_t k = kb + lane;
        if (k < k1) {
            double a[NC], b[NC];
            terms(k, a, b);
#pragma unroll
            for (int j = 0; j < NC; j++) {
                sa[j] += a[j];
                sb[j] += b[j];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NC; j++) {
        const double ta = wave_inclusive_scan(sa[j]), tb = wave_inclusive_scan(sb[j]);
        if (lane == 63) {
            tot[2 * j][wv] = ta;
            tot[2 * j + 1][wv] = tb;
        }
    }
    __syncthreads();
    if (threadIdx.x < 2 * NC) {  // earlier segments, then an exclusive scan of the ranges' sums, in order
        double run = 0.0;
        for (uint32_t w = 0; w < NW; w++) run += pre[threadIdx.x][w];
        for (uint32_t w = 0; w < NW; w++) {
            const double t = tot[threadIdx.x][w];
            tot[threadIdx.x][w] = run;
            run += t;
        }
    }
    __syncthreads();
    double ci[NC], ce[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) {
        ci[j] = out[NC + 2 * j] + tot[2 * j][wv];
        ce[j] = out[NC + 2 * j + 1] + tot[2 * j + 1][wv];
    }
    for (uint32_t kb = k0; kb < k1; kb += 64) {
        const uint32_t k = kb + lane;
        double a[NC], b[NC];
        if (k < k1) {
            terms(k, a, b);
        } else {
#pragma unroll
            for (int j = 0; j < NC; j++) a[j] = b[j] = 0.0;
        }
#pragma unroll
        for (int j = 0; j < NC; j++) {
            a[j] = wave_inclusive_scan(a[j]);
            b[j] = wave_inclusive_scan(b[j]);
        }
        if (k < k1) {
            double *row = out + (uint64_t)k * narr + NC;
#pragma unroll
            for (int j = 0; j < NC; j++) {
                row[2 * j] = ci[j] + a[j];
                row[2 * j + 1] = ce[j] + b[j];
            }
        }
#pragma unroll
        for (int j = 0; j < NC; j++) {
            ci[j] += __shfl(a[j], 63, 64);
            ce[j] += __shfl(b[j], 63, 64);
        }
    }
}

// k = c00 - c(0,1:) inv(c(1:,1:)) c(1:,0), c column-major n x n; the inverse
// by LU with partial pivoting (Eigen's dynamic-size inverse); for n == 2 this
// is c00 - (c01 * (1/c11)) * c10.  n is a template argument so that every
// loop has constant bounds and the small arrays stay in registers.
template <int n>
__device__ __forceinline__ double schur00(const double *c) {
    if constexpr (n <= 1) {
        return c[0];
    } else {
        constexpr int m = n - 1;
        double lu[m * m], inv[m * m], tmp[m];
        int perm[m];
        for (int cc = 0; cc < m; cc++)
            for (int r = 0; r < m; r++) lu[cc * m + r] = c[(cc + 1) * n + (r + 1)];
        for (int i = 0; i < m; i++) perm[i] = i;
        for (int k = 0; k < m; k++) {
            int p = k;
            double best = fabs(lu[k * m + k]);
            for (int r = k + 1; r < m; r++)
                if (fabs(lu[k * m + r]) > best) {
                    best = fabs(lu[k * m + r]);
                    p = r;
                }
            if (p != k) {
                for (int cc = 0; cc < m; cc++) {
                    double t = lu[cc * m + k];
                    lu[cc * m + k] = lu[cc * m + p];
                    lu[cc * m + p] = t;
                }
                int t = perm[k];
                perm[k] = perm[p];
                perm[p] = t;
            }
            for (int r = k + 1; r < m; r++) lu[k * m + r] /= lu[k * m + k];
            for (int cc = k + 1; cc < m; cc++)
                for (int r = k + 1; r < m; r++) lu[cc * m + r] -= lu[k * m + r] * lu[cc * m + k];
        }
        for (int col = 0; col < m; col++) {
            double *x = inv + col * m;
            for (int r = 0; r < m; r++) x[r] = (perm[r] == col) ? 1.0 : 0.0;
            for (int r = 0; r < m; r++)
                for (int k = 0; k < r; k++) x[r] -= lu[k * m + r] * x[k];
            for (int r = m - 1; r >= 0; r--) {
                for (int k = r + 1; k < m; k++) x[r] -= lu[k * m + r] * x[k];
                x[r] = x[r] * (1.0 / lu[r * m + r]);
            }
        }
        for (int cc = 0; cc < m; cc++) {
            double s = c[1 * n + 0] * inv[cc * m + 0];
            for (int k = 1; k < m; k++) s += c[(k + 1) * n + 0] * inv[cc * m + k];
            tmp[cc] = s;
        }
        double s = tmp[0] * c[0 * n + 1];
        for (int cc = 1; cc < m; cc++) s += tmp[cc] * c[0 * n + (cc + 1)];
        return c[0] - s;
    }
}

// :289-346 k_gk and k_einst per lag, then :352-356 E /= l
template <int NCUR>
__global__ void gk_schur_kernel(double *__restrict__ out, uint32_t narr, uint32_t leff, uint64_t stride) {
    constexpr uint32_t ncur = NCUR, ncorr = NCUR * NCUR;
    const uint32_t it = blockIdx.x * blockDim.x + threadIdx.x;
    if (it == 0 || it >= leff) return;
    out += blockIdx.y * stride;
    double *cur = out + (uint64_t)it * narr;
    double matr[ncorr];
    for (uint32_t j = 0; j < ncorr; j++) matr[j] = 0.0;
    uint32_t idx = 0;
    for (uint32_t j1 = 0; j1 < ncur; j1++)
        for (uint32_t j2 = 0; j2 < ncur; j2++) {
            matr[j2 * ncur + j1] += cur[ncorr + 2 * idx] / 2.0;
            matr[j1 * ncur + j2] += cur[ncorr + 2 * idx] / 2.0;
            idx++;
        }
    const double kgk = schur00<NCUR>(matr);
    for (uint32_t j = 0; j < ncorr; j++) matr[j] = 0.0;
    idx = 0;
    const double dit = (double)it;
    for (uint32_t j1 = 0; j1 < ncur; j1++)
        for (uint32_t j2 = 0; j2 < ncur; j2++) {
            const double v = cur[ncorr + 2 * idx] - cur[ncorr + 2 * idx + 1] / dit;
            matr[j2 * ncur + j1] += v / 2.0;
            matr[j1 * ncur + j2] += v / 2.0;
            idx++;
        }
    const double kein = schur00<NCUR>(matr);
    cur[3 * ncorr + 0] = kgk;
    cur[3 * ncorr + 1] = kein;
    for (uint32_t j = 0; j < ncorr; j++) cur[ncorr + 2 * j + 1] = cur[ncorr + 2 * j + 1] / dit;
}

static void gk_schur_launch(double *d, uint32_t narr, uint32_t ncur, uint32_t leff, hipStream_t s, uint32_t nblocks,
                            uint64_t stride) {
    const dim3 grid((leff + 255) / 256, nblocks);
    switch (ncur) {
        case 1: hipLaunchKernelGGL(gk_schur_kernel<1>, grid, dim3(256), 0, s, d, narr, leff, stride); break;
        case 2: hipLaunchKernelGGL(gk_schur_kernel<2>, grid, dim3(256), 0, s, d, narr, leff, stride); break;
        case 3: hipLaunchKernelGGL(gk_schur_kernel<3>, grid, dim3(256), 0, s, d, narr, leff, stride); break;
        case 4: hipLaunchKernelGGL(gk_schur_kernel<4>, grid, dim3(256), 0, s, d, narr, leff, stride); break;
        default: fail(ANL_ERR_ARG, "between 1 and 4 currents are supported");
    }
    ANL_HIP(hipGetLastError());
}

void gk_epilogue(double *d, uint32_t narr, uint32_t ncur, uint32_t leff, int subtract_mean, uint32_t start_mean,
                 hipStream_t s, uint32_t nblocks, uint64_t stride, bool serial_scans, const double2 *rec) {
    const uint32_t ncorr = ncur * ncur;
    if (!serial_scans) {
        if (subtract_mean) {
            hipLaunchKernelGGL(gk_mean_par_kernel, dim3(1, nblocks), dim3(GK_PAR), 0, s, d, narr, ncorr, leff,
                               start_mean, stride);
            ANL_HIP(hipGetLastError());
        }
        // segments of about 2,048 lags per workgroup, at most 16 per block
        const uint32_t nseg = std::max(1u, std::min(16u, (leff + 2047) / 2048));
        switch (ncorr) {
#define ANL_GK_PAR(NCV)                                                                                          \
    case NCV:                                                                                                    \
        hipLaunchKernelGGL(gk_integral_par_kernel<NCV>, dim3(nseg, nblocks), dim3(GK_PAR), 0, s, d, narr, leff,    \
                           stride);                                                                            \
        break;
            ANL_GK_PAR(1)
            ANL_GK_PAR(4)
            ANL_GK_PAR(9)
            ANL_GK_PAR(16)
#undef ANL_GK_PAR
            default:
                fail(ANL_ERR_ARG, "between 1 and 4 currents are supported");
        }
        ANL_HIP(hipGetLastError());
        gk_schur_launch(d, narr, ncur, leff, s, nblocks, stride);
        return;
    }
    switch (ncorr) {
#define ANL_GK_SCANS(NC)                                                                                            \
    case NC:                                                                                                        \
        if (subtract_mean)                                                                                          \
            hipLaunchKernelGGL(gk_mean_kernel<NC>, dim3(1, nblocks), dim3(GK_SCAN), 0, s, d, leff, start_mean, stride, \
                               rec);                                                                                \
        hipLaunchKernelGGL(gk_integral_kernel<NC>, dim3(1, nblocks), dim3(GK_SCAN), 0, s, d, leff, stride);          \
        break;
        ANL_GK_SCANS(1)
        ANL_GK_SCANS(4)
        ANL_GK_SCANS(9)
        ANL_GK_SCANS(16)
#undef ANL_GK_SCANS
        default: fail(ANL_ERR_ARG, "between 1 and 4 currents are supported");
    }
    ANL_HIP(hipGetLastError());
    gk_schur_launch(d, narr, ncur, leff, s, nblocks, stride);
}

void gk_reciprocals(double2 *rec, uint64_t n, hipStream_t s) {
    hipLaunchKernelGGL(gk_reciprocal_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, rec, n);
    ANL_HIP(hipGetLastError());
}

// Wavefronts of 64 means from which a stride 1 launch takes gk_dense_kernel:
// gk_chain_kernel's time for 20,000 t0 grows by 0.48 ms per 256 (one
// per CU), the dense kernel's by 0.2-0.3 ms from 1.4 ms on (2.0 against
// 2.7 ms at 1,024 and 2 currents, 2.9 against 2.6 ms at 2,048 and 4).
constexpr uint64_t GK_DENSE_CHAINS = 1792;

static bool gk_can_allocate(hipStream_t st) {
    hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &c) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return c == hipStreamCaptureStatusNone;
}

// How the FP64 form runs a call.
struct GkPlan {
    bool few = false;      // gk_few_kernel
    size_t seg_bytes = 0;  // of the segment means of segments side by side; 0: one segment, or more than the cap
};
constexpr size_t GK_SEG_BYTES = 1ull << 30;

// The smaller of two estimates (us) decides for gk_few_kernel, which takes K
// terms of a lag one after the other (at least one per segment), 0.16 to 1.3 us
// each by the number of currents.  A workgroup of gk_chain_kernel takes 14 ns of
// the chip before its first term, a wavefront of gk_dense_kernel 2; segments side
// by side take a launch and a division each, one after the other a launch each.
// Measured (us a call, chain or dense and few): 2 currents, one segment, 40
// lags, K 4 25 and 23, K 16 25 and 28; 1,500 lags x 16 blocks, K 16 216 and 225,
// K 64 239 and 229; in 16 segments K 16 536 and 225, K 100 580 and 250; 4
// currents, 40 lags, 16 segments, K 16 35 and 57; 6,000 lags x 16 blocks, 64
// segments, K 100 25,700 and 4,400.
static GkPlan gk_plan(uint32_t ncur, uint32_t leff, uint32_t skip, uint32_t n_seg, const uint32_t *n, uint32_t nblocks,
                      bool side_by_side = true) {
    static const double term[GK_MAXC] = {0.16, 0.41, 0.8, 1.3};
    GkPlan P;
    const uint64_t nb = std::min(GK_MAXB, nblocks), pairs = ncur * ncur;
    const uint64_t need = nb * n_seg * pairs * leff * sizeof(double);
    if (side_by_side && n_seg > 1 && n_seg <= 65535 && need <= GK_SEG_BYTES) P.seg_bytes = need;
    uint64_t seg = 0;
    for (uint32_t b = 0; b < nblocks; b++) seg = std::max<uint64_t>(seg, n[b] / n_seg);
    const double terms = (double)((seg + skip - 1) / skip), lags = (leff + 63) / 64;
    const double chains = lags * pairs * n_seg * nb, waves = lags * nb;
    const bool dense = skip == 1 && chains > GK_DENSE_CHAINS;
    const double few = n_seg * terms * term[ncur - 1] * (1 + waves / 4096);
    const double chain = 1.5 + 0.03 * terms + chains * (dense ? 0.002 : 0.0135) +
                         (n_seg > 1 ? (P.seg_bytes ? 2.5 + 0.15 * n_seg : 4.0 * n_seg) : 0.0);
    P.few = few < chain;
    if (P.few) P.seg_bytes = 0;
    return P;
}

// The segments of a block run side by side into segm (GkPlan::seg_bytes) and
// are folded afterwards; without it one launch per segment folds into the
// output.
static void gk_fp64_enqueue_blocks(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t leff,
                                   uint32_t n_seg, const uint64_t *primo, const uint32_t *n, uint32_t nblocks,
                                   double *d, const GkPlan &plan, double *segm, hipStream_t st) {
    const uint32_t narr = 3 * ncur * ncur + 2;
    const uint64_t stride = (uint64_t)leff * narr;
    for (uint32_t b0 = 0; b0 < nblocks; b0 += GK_MAXB) {
        const uint32_t nb = std::min(GK_MAXB, nblocks - b0);
        GkArgs a{};
        a.data = s->data;
        a.rec = s->rec;
        a.nrows = s->nrows;
        a.ncols = s->ncols;
        a.ncur = ncur;
        for (uint32_t c = 0; c < ncur; c++) a.idx[c] = idx_j[c];
        a.n_seg = n_seg;
        a.skip = skip;
        a.leff = leff;
        a.narr = narr;
        a.out_stride = stride;
        a.out = d + b0 * stride;
        a.segm = segm;
        for (uint32_t b = 0; b < nb; b++) {
            a.bl.primo[b] = primo[b0 + b];
            a.bl.n[b] = n[b0 + b];
        }
        if (plan.few) {
            const dim3 grid((leff + 63) / 64, nb);
            switch (ncur) {
                case 1: hipLaunchKernelGGL(gk_few_kernel<1>, grid, dim3(64), 0, st, a); break;
                case 2: hipLaunchKernelGGL(gk_few_kernel<2>, grid, dim3(64), 0, st, a); break;
                case 3: hipLaunchKernelGGL(gk_few_kernel<3>, grid, dim3(64), 0, st, a); break;
                default: hipLaunchKernelGGL(gk_few_kernel<4>, grid, dim3(64), 0, st, a); break;
            }
            ANL_HIP(hipGetLastError());
            continue;
        }
        const dim3 grid((leff + 63) / 64 * ncur * ncur, segm ? n_seg : 1, nb);
        for (uint32_t k = 0; k < (segm ? 1 : n_seg); k++) {
            a.seg0 = k;
            const uint64_t chains = (uint64_t)grid.x * grid.y * grid.z;
            if (skip == 1 && chains > GK_DENSE_CHAINS) {
                const uint32_t nt64 = (leff + 63) / 64, nt128 = (leff + 127) / 128;
                switch (ncur) {
#define ANL_GK_DENSE(N, C, X) hipLaunchKernelGGL((gk_dense_kernel<N, C>), dim3(X, grid.y, grid.z), dim3(64), 0, st, a)
                    case 1: ANL_GK_DENSE(1, 2, nt128); break;
                    case 2: ANL_GK_DENSE(2, 2, nt64 * 2); break;
                    case 3: ANL_GK_DENSE(3, 3, nt64 * 3); break;
                    default: ANL_GK_DENSE(4, 2, nt64 * 8); break;
#undef ANL_GK_DENSE
                }
            } else if (skip == 1) hipLaunchKernelGGL((gk_chain_kernel<48, 1>), grid, dim3(256), 0, st, a);
            else if (skip <= 8) hipLaunchKernelGGL((gk_chain_kernel<32, 8>), grid, dim3(256), 0, st, a);
            else hipLaunchKernelGGL((gk_chain_kernel<16, 64>), grid, dim3(256), 0, st, a);
            ANL_HIP(hipGetLastError());
        }
        if (segm) {
            hipLaunchKernelGGL(gk_segments_kernel, dim3((ncur * ncur * leff + 255) / 256, nb), dim3(256), 0, st, a);
            ANL_HIP(hipGetLastError());
        }
    }
}

uint32_t gk_block_checks(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t tmax, const uint64_t *primo,
                         const uint32_t *n, uint32_t nblocks) {
    if (!s || !idx_j || !primo || !n) fail(ANL_ERR_ARG, "null pointer passed to anl_gk_calculate");
    if (ncur == 0 || ncur > GK_MAXC) fail(ANL_ERR_ARG, "between 1 and 4 currents are supported");
    if (nblocks == 0) fail(ANL_ERR_ARG, "no blocks");
    for (uint32_t c = 0; c < ncur; c++)
        if (idx_j[c] + 3 > s->ncols) fail(ANL_ERR_HEADER, "current column triplet out of range");
    uint32_t leff0 = 0;
    for (uint32_t b = 0; b < nblocks; b++) {
        const uint32_t leff = (n[b] < tmax || tmax == 0) ? n[b] : tmax;  // greenkubo...cpp:123
        if ((uint64_t)leff + primo[b] + n[b] > s->nrows)                 // :168-169
            fail(ANL_ERR_TOO_SHORT,
                 "trajectory is too short for this kind of calculation. Select a different starting timestep or "
                 "lower the size of the average or the lenght of the correlation function");
        if (b == 0) leff0 = leff;
        else if (leff != leff0)
            fail(ANL_ERR_ARG, "blocks with different numbers of lags cannot be averaged together");
    }
    return leff0;
}

static void gk_defaults(uint32_t &n_seg, uint32_t &skip) {
    n_seg = std::max(n_seg, 1u);  // greenkubo...cpp:50-53
    skip = std::max(skip, 1u);
}
static void gk_enqueue_checks(int form, uint32_t nblocks, const double *mean, const double *var) {
    if ((mean || var) && (!mean || !var || nblocks < 2))
        fail(ANL_ERR_ARG, "block mean and variance need both outputs and at least two blocks");
    if (form != ANL_GK_FP64 && form != ANL_GK_MFMA) fail(ANL_ERR_ARG, "unknown Green-Kubo form");
}

// A checked call (gk_block_checks, gk_enqueue_checks, leff > 0; n_seg and skip at
// least 1) on stream st; plan and segm (its segment means, or null) are the
// FP64 form's.
static void gk_enqueue(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t leff, uint32_t n_seg,
                       int subtract_mean, uint32_t start_mean, const uint64_t *primo, const uint32_t *n,
                       uint32_t nblocks, int form, double *out_dev, double *mean_dev, double *var_dev,
                       const GkPlan &plan, double *segm, hipStream_t st) {
    const uint32_t narr = 3 * ncur * ncur + 2;
    const uint64_t stride = (uint64_t)leff * narr;
    if (form == ANL_GK_MFMA) gk_mfma_enqueue_blocks(s, idx_j, ncur, skip, leff, n_seg, primo, n, nblocks, out_dev, st);
    else gk_fp64_enqueue_blocks(s, idx_j, ncur, skip, leff, n_seg, primo, n, nblocks, out_dev, plan, segm, st);
    // the FP64 form keeps the reference's serial scans (bit-identical results)
    gk_epilogue(out_dev, narr, ncur, leff, subtract_mean, start_mean, st, nblocks, stride, form == ANL_GK_FP64, s->rec);
    if (mean_dev) mediavar_blocks(nullptr, out_dev, nullptr, nblocks, stride, mean_dev, var_dev, st);
}

// The series' segment means for one asynchronous call: calls from any threads
// and on any streams take them in turn, each stream waiting for the call
// before.  p is null, and the call folds segment by segment, where they would
// take more than a kept workspace may, where the memory cannot be had, and on
// a stream under capture (a graph would keep an address that a later call may
// free).
struct GkSegments {
    anl_series *s;
    hipStream_t st;
    std::unique_lock<std::mutex> lock;
    double *p = nullptr;
    GkSegments(anl_series *s, size_t need, hipStream_t st) : s(s), st(st) {
        if (need == 0 || need > SCRATCH_KEEP || !gk_can_allocate(st)) return;
        lock = std::unique_lock<std::mutex>(s->seg_mutex);
        if (!s->seg_done) ANL_HIP(hipEventCreateWithFlags(&s->seg_done, hipEventDisableTiming));
        if (need > s->seg_cap) {
            if (s->seg) ANL_HIP(hipEventSynchronize(s->seg_done));
            (void)hipFree(s->seg);
            s->seg = nullptr;
            s->seg_cap = 0;
            if (hipMalloc(&s->seg, need) != hipSuccess) {
                (void)hipGetLastError();
                s->seg = nullptr;
                return;
            }
            s->seg_cap = need;
        } else {
            ANL_HIP(hipStreamWaitEvent(st, s->seg_done, 0));
        }
        p = (double *)s->seg;
    }
    ~GkSegments() {
        // if the record fails the next call must not go on without it
        if (p && hipEventRecord(s->seg_done, st) != hipSuccess) (void)hipStreamSynchronize(st);
    }
    GkSegments(const GkSegments &) = delete;
    GkSegments &operator=(const GkSegments &) = delete;
};

// A pooled workspace of `bytes` for a synchronous call, with room for the
// segment means behind them if that can be had.
struct GkWorkspace {
    std::optional<ScratchLease> w;
    double *segm = nullptr;
    GkWorkspace(anl_series *s, size_t bytes, size_t seg, size_t pin) {
        bytes = (std::max<size_t>(bytes, 8) + 255) / 256 * 256;
        if (seg) {
            try {
                w.emplace(s->scratch, bytes + seg, pin);
                segm = (double *)((char *)w->s.dev + bytes);
                return;
            } catch (const Error &) {
                (void)hipGetLastError();
            }
        }
        w.emplace(s->scratch, bytes, pin);
    }
    double *dev() const { return (double *)w->s.dev; }
};

}  // namespace anl

using namespace anl;

extern "C" {

int anl_gk_calculate_blocks_async(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t tmax,
                                  uint32_t n_seg, int subtract_mean, uint32_t start_mean, const uint64_t *primo,
                                  const uint32_t *n, uint32_t nblocks, int form, double *out_dev, double *mean_dev,
                                  double *var_dev, void *stream) {
    return guard([&] {
        const uint32_t leff = gk_block_checks(s, idx_j, ncur, tmax, primo, n, nblocks);
        if (!out_dev) fail(ANL_ERR_ARG, "null output passed to anl_gk_calculate_blocks_async");
        gk_enqueue_checks(form, nblocks, mean_dev, var_dev);
        if (leff == 0) return;
        ensure_device();
        hipStream_t st = (hipStream_t)stream;
        gk_defaults(n_seg, skip);
        GkPlan plan = form == ANL_GK_FP64 ? gk_plan(ncur, leff, skip, n_seg, n, nblocks) : GkPlan{};
        GkSegments seg(s, plan.seg_bytes, st);
        if (plan.seg_bytes && !seg.p) plan = gk_plan(ncur, leff, skip, n_seg, n, nblocks, false);
        gk_enqueue(s, idx_j, ncur, skip, leff, n_seg, subtract_mean, start_mean, primo, n, nblocks, form, out_dev,
                   mean_dev, var_dev, plan, seg.p, st);
    });
}

// The device memory and a ring of three pinned pieces are the series' pooled
// workspace.  A fresh output array costs a page fault per 4 KiB, more than its
// copy: while the kernels run, up to 8 threads write a byte of each page of
// their share; then they copy their part of every piece that has arrived in
// the ring while the next ones arrive.  16 blocks x 8,000 lags (14 MB), MFMA: a
// call 1,310 us with a plain copy from memory allocated for it, 820 now, of
// which the kernels are 305.
int anl_gk_calculate_blocks(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t tmax,
                            uint32_t n_seg, int subtract_mean, uint32_t start_mean, const uint64_t *primo,
                            const uint32_t *n, uint32_t nblocks, int form, double *out_host, double *mean_host,
                            double *var_host) {
    return guard([&] {
        const uint32_t leff = gk_block_checks(s, idx_j, ncur, tmax, primo, n, nblocks);
        if (!out_host) fail(ANL_ERR_ARG, "null output passed to anl_gk_calculate_blocks");
        gk_enqueue_checks(form, nblocks, mean_host, var_host);
        if (leff == 0) return;
        ensure_device();
        const size_t len = (size_t)leff * (3 * ncur * ncur + 2), all = len * nblocks, total = all * sizeof(double);
        constexpr size_t PIECE = 2u << 20, RING = 3;
        const size_t pieces = (total + PIECE - 1) / PIECE;
        const unsigned nth = pieces < 2 ? 0 : std::min(8u, std::max(1u, std::thread::hardware_concurrency()));
        gk_defaults(n_seg, skip);
        GkPlan plan = form == ANL_GK_FP64 ? gk_plan(ncur, leff, skip, n_seg, n, nblocks) : GkPlan{};
        const GkWorkspace w(s, (all + 2 * len) * sizeof(double), plan.seg_bytes, nth ? RING * PIECE : 0);
        if (plan.seg_bytes && !w.segm) plan = gk_plan(ncur, leff, skip, n_seg, n, nblocks, false);
        double *d = w.dev();
        char *ring = (char *)w.w->s.pin;
        constexpr int64_t NOT_YET = -1, GIVE_UP = -2;  // no kernels yet; there will be no output
        std::atomic<int64_t> arrived{NOT_YET};         // pieces in the ring so far
        std::atomic<uint64_t> copied[RING] = {};       // shares copied out of each of its slots
        std::mutex mu;
        std::condition_variable news;
        auto publish = [&](int64_t v) {
            {
                std::lock_guard<std::mutex> lock(mu);
                arrived.store(v, std::memory_order_release);
            }
            news.notify_all();
        };
        // more than v pieces (false: there will be none).  Pieces follow each
        // other in tens of us, less than a thread takes to wake, so it looks
        // for them for a while before it sleeps; the kernels may take seconds.
        auto await = [&](int64_t v) {
            const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
            int64_t a;
            while ((a = arrived.load(std::memory_order_acquire)) <= v && a != GIVE_UP) {
                if (std::chrono::steady_clock::now() < until) {
                    std::this_thread::yield();
                } else {
                    std::unique_lock<std::mutex> lock(mu);
                    news.wait(lock, [&] { return arrived.load() > v || arrived.load() == GIVE_UP; });
                }
            }
            return a != GIVE_UP;
        };
        // thread k's share of piece p: [first, last) of the output
        auto share = [&](size_t p, unsigned k) {
            return p * PIECE + std::min(PIECE, total - p * PIECE) * k / nth;
        };
        auto work = [&](unsigned k) {
            if (!await(NOT_YET)) return;
            for (size_t p = 0; p < pieces; p++)
                for (size_t b = share(p, k); b < share(p, k + 1); b += 4096) ((volatile char *)out_host)[b] = 0;
            for (size_t p = 0; p < pieces; p++) {
                if (!await((int64_t)p)) return;
                const size_t b0 = share(p, k), b1 = share(p, k + 1);
                std::memcpy((char *)out_host + b0, ring + p % RING * PIECE + (b0 - p * PIECE), b1 - b0);
                copied[p % RING].fetch_add(1, std::memory_order_release);
            }
        };
        std::vector<std::thread> pool;
        hipEvent_t ev[RING] = {};
        auto end = [&] {
            for (auto &t : pool) t.join();
            for (hipEvent_t e : ev)
                if (e) (void)hipEventDestroy(e);
        };
        try {
            gk_enqueue(s, idx_j, ncur, skip, leff, n_seg, subtract_mean, start_mean, primo, n, nblocks, form, d,
                       mean_host ? d + all : nullptr, var_host ? d + all + len : nullptr, plan, w.segm, 0);
            if (nth) {
                pool.reserve(nth);
                for (unsigned k = 0; k < nth; k++) pool.emplace_back(work, k);
                publish(0);
                for (hipEvent_t &e : ev) ANL_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
                for (size_t p = 0; p <= pieces; p++) {
                    if (p < pieces) {
                        // the slot is free once every share of its earlier pieces has left it
                        while (copied[p % RING].load(std::memory_order_acquire) < nth * (p / RING))
                            std::this_thread::yield();
                        ANL_HIP(hipMemcpyAsync(ring + p % RING * PIECE, (const char *)d + p * PIECE,
                                               std::min(PIECE, total - p * PIECE), hipMemcpyDeviceToHost, 0));
                        ANL_HIP(hipEventRecord(ev[p % RING], 0));
                    }
                    if (p) {
                        ANL_HIP(hipEventSynchronize(ev[(p - 1) % RING]));
                        publish((int64_t)p);
                    }
                }
            } else if (total) {
                ANL_HIP(hipMemcpy(out_host, d, total, hipMemcpyDeviceToHost));
            }
            if (mean_host && len) ANL_HIP(hipMemcpy(mean_host, d + all, len * sizeof(double), hipMemcpyDeviceToHost));
            if (var_host && len) ANL_HIP(hipMemcpy(var_host, d + all + len, len * sizeof(double), hipMemcpyDeviceToHost));
        } catch (...) {
            (void)hipStreamSynchronize(0);  // the workspace goes back unused
            publish(GIVE_UP);
            end();
            throw;
        }
        end();
    });
}

int anl_gk_calculate_async(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t tmax,
                           uint32_t n, uint32_t n_seg, int subtract_mean, uint32_t start_mean, uint64_t primo,
                           double *out_dev, void *stream) {
    return anl_gk_calculate_blocks_async(s, idx_j, ncur, skip, tmax, n_seg, subtract_mean, start_mean, &primo, &n, 1,
                                         ANL_GK_FP64, out_dev, nullptr, nullptr, stream);
}

int anl_gk_calculate_mfma_async(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t tmax,
                                uint32_t n, uint32_t n_seg, int subtract_mean, uint32_t start_mean, uint64_t primo,
                                double *out_dev, void *stream) {
    return anl_gk_calculate_blocks_async(s, idx_j, ncur, skip, tmax, n_seg, subtract_mean, start_mean, &primo, &n, 1,
                                         ANL_GK_MFMA, out_dev, nullptr, nullptr, stream);
}

// Synchronous host-output form.
static int gk_calculate_host(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t tmax,
                             uint32_t n, uint32_t n_seg, int subtract_mean, uint32_t start_mean, uint64_t primo,
                             double *out_host, int form) {
    return guard([&] {
        const uint32_t leff = gk_block_checks(s, idx_j, ncur, tmax, &primo, &n, 1);
        if (!out_host) fail(ANL_ERR_ARG, "null output passed to anl_gk_calculate");
        if (leff == 0) return;
        ensure_device();
        const size_t bytes = (size_t)leff * (3 * ncur * ncur + 2) * sizeof(double);
        gk_defaults(n_seg, skip);
        GkPlan plan = form == ANL_GK_FP64 ? gk_plan(ncur, leff, skip, n_seg, &n, 1) : GkPlan{};
        const GkWorkspace w(s, bytes, plan.seg_bytes, 0);
        if (plan.seg_bytes && !w.segm) plan = gk_plan(ncur, leff, skip, n_seg, &n, 1, false);
        try {
            gk_enqueue(s, idx_j, ncur, skip, leff, n_seg, subtract_mean, start_mean, &primo, &n, 1, form,
                       w.dev(), nullptr, nullptr, plan, w.segm, 0);
            ANL_HIP(hipMemcpy(out_host, w.dev(), bytes, hipMemcpyDeviceToHost));
        } catch (...) {
            (void)hipStreamSynchronize(0);  // the workspace goes back unused
            throw;
        }
    });
}

int anl_gk_set_tuning(anl_series *s, uint32_t tiles_per_wave, uint32_t chunk_steps, uint32_t waves_per_group) {
    return guard([&] {
        if (!s) fail(ANL_ERR_ARG, "null series");
        if (!gkm_shape_ok(tiles_per_wave, chunk_steps, waves_per_group))
            fail(ANL_ERR_ARG, "Green-Kubo MFMA shape: tiles per wavefront 4|8, chunk steps 8|16, wavefronts 2|4");
        s->gk_q = tiles_per_wave;
        s->gk_cs = chunk_steps;
        s->gk_wg = waves_per_group;
    });
}

int anl_gk_get_tuning(anl_series *s, uint32_t *tiles_per_wave, uint32_t *chunk_steps, uint32_t *waves_per_group) {
    return guard([&] {
        if (!s) fail(ANL_ERR_ARG, "null series");
        if (tiles_per_wave) *tiles_per_wave = s->gk_q;
        if (chunk_steps) *chunk_steps = s->gk_cs;
        if (waves_per_group) *waves_per_group = s->gk_wg;
    });
}

// Times the MFMA lag products of the given blocks with each candidate shape
// (one untimed and one timed enqueue each, HIP events on the null stream;
// the epilogue does not depend on the shape and is left out) and keeps the
// fastest in the series.
int anl_gk_autotune(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t tmax, uint32_t n_seg,
                    const uint64_t *primo, const uint32_t *n, uint32_t nblocks, const uint32_t *cand, uint32_t ncand,
                    float *ms_out, uint32_t *best_out) {
    return guard([&] {
        const uint32_t leff = gk_block_checks(s, idx_j, ncur, tmax, primo, n, nblocks);
        static const uint32_t defaults[] = {8, 16, 4, 8, 16, 2, 4, 16, 4, 4, 16, 2, 8, 8, 4, 4, 8, 4};
        if (!cand) {
            cand = defaults;
            ncand = sizeof(defaults) / sizeof(defaults[0]) / 3;
        }
        if (ncand == 0) fail(ANL_ERR_ARG, "no candidates");
        for (uint32_t c = 0; c < ncand; c++)
            if (!gkm_shape_ok(cand[3 * c], cand[3 * c + 1], cand[3 * c + 2]))
                fail(ANL_ERR_ARG, "candidate " + std::to_string(c) +
                                      ": tiles per wavefront 4|8, chunk steps 8|16, wavefronts 2|4");
        if (n_seg < 1) n_seg = 1;
        if (skip == 0) skip = 1;
        if (leff == 0) return;
        ensure_device();
        const uint32_t sq = s->gk_q, sc = s->gk_cs, sw = s->gk_wg;
        double *d = nullptr;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        float best = -1.0f;
        uint32_t besti = 0;
        try {
            ANL_HIP(hipMalloc(&d, (size_t)nblocks * leff * (3 * ncur * ncur + 2) * sizeof(double)));
            ANL_HIP(hipEventCreate(&e0));
            ANL_HIP(hipEventCreate(&e1));
            for (uint32_t c = 0; c < ncand; c++) {
                s->gk_q = cand[3 * c];
                s->gk_cs = cand[3 * c + 1];
                s->gk_wg = cand[3 * c + 2];
                // one untimed call, then the fastest of three timed ones: a
                // call takes a few ms, and the candidates are often within a
                // few per cent of each other
                gk_mfma_enqueue_blocks(s, idx_j, ncur, skip, leff, n_seg, primo, n, nblocks, d, 0);
                float ms = -1.0f;
                for (int r = 0; r < 3; ++r) {
                    ANL_HIP(hipEventRecord(e0, 0));
                    gk_mfma_enqueue_blocks(s, idx_j, ncur, skip, leff, n_seg, primo, n, nblocks, d, 0);
                    ANL_HIP(hipEventRecord(e1, 0));
                    ANL_HIP(hipEventSynchronize(e1));
                    float t = 0.0f;
                    ANL_HIP(hipEventElapsedTime(&t, e0, e1));
                    if (ms < 0.0f || t < ms) ms = t;
                }
                if (ms_out) ms_out[c] = ms;
                if (best < 0.0f || ms < best) {
                    best = ms;
                    besti = c;
                }
            }
        } catch (...) {
            s->gk_q = sq;
            s->gk_cs = sc;
            s->gk_wg = sw;
            (void)hipDeviceSynchronize();
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
            (void)hipFree(d);
            throw;
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        (void)hipFree(d);
        s->gk_q = cand[3 * besti];
        s->gk_cs = cand[3 * besti + 1];
        s->gk_wg = cand[3 * besti + 2];
        if (best_out) *best_out = besti;
    });
}

int anl_gk_calculate(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t tmax, uint32_t n,
                     uint32_t n_seg, int subtract_mean, uint32_t start_mean, uint64_t primo, double *out_host) {
    return gk_calculate_host(s, idx_j, ncur, skip, tmax, n, n_seg, subtract_mean, start_mean, primo, out_host,
                             ANL_GK_FP64);
}

int anl_gk_calculate_mfma(anl_series *s, const uint32_t *idx_j, uint32_t ncur, uint32_t skip, uint32_t tmax,
                          uint32_t n, uint32_t n_seg, int subtract_mean, uint32_t start_mean, uint64_t primo,
                          double *out_host) {
    return gk_calculate_host(s, idx_j, ncur, skip, tmax, n, n_seg, subtract_mean, start_mean, primo, out_host,
                             ANL_GK_MFMA);
}

}  // extern "C"
