// kx_spread.hip -- the forward (spread) launches of the Kirchhoff operator
// and their C ABI entry points kx_spread / kx_spread_models
// (include/kirchx.h).  Kernel bodies: kx_device.h.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>

#include "kx_internal.h"
#include "kx_device.h"
#include "kx_slots.h"

namespace {

// h != NULL: y receives the traces convolved with the nh-tap wavelet h
// (the forward operator), otherwise the traces.
template <typename TD, typename TT, bool DYN, bool NEG, int ORD, int RB, bool XS>
__global__ __launch_bounds__(kSpreadBlock) void spread_kernel(KArgs a, const TD *__restrict__ m,
                                                              TD *__restrict__ y,
                                                              const SpreadScale *__restrict__ sc,
                                                              const TD *__restrict__ h, int nh)
{
    const int L = xcd_remap(blockIdx.x, gridDim.x);
    const SpreadScale scale = *sc;
    spread_item<TD, TT, DYN, NEG, ORD, RB, XS>(a, m, y, scale, L % a.ns, (L / a.ns) * RB, h, nh);
}

// Blocks of 8 or 16 receivers, interleaved traces (kx_slots.h).  The first
// nfull workgroups take a whole (source, receiver block) pair each, pair L
// (after the XCD renumbering) = source L mod ns, block L / ns; each of the
// remaining pairs is shared by `parts` workgroups, pair nfull + (L mod nrest),
// part L / nrest of the tiles: neighbours read the same rows of the receiver
// tables.  Every wave turns the np partial statistics of |m| into the
// launch's scale for itself (one launch less than a kernel for it);
// workgroup 0 keeps it in *sc.
struct SlotsLaunch {
    const float *part;
    int np;
    double wamp, wtyp;
    SpreadScale *sc;
    int nfull, parts;
    unsigned long long *sums;  // [parts][nrest][nt][RB]
};

template <typename TT, bool DYN, bool GATE, bool NEG, int RB>
__global__ __launch_bounds__(kSlotsMaxThreads) void slots_kernel(KArgs a,
                                                                 const float *__restrict__ m,
                                                                 float *__restrict__ y,
                                                                 const float *__restrict__ h,
                                                                 int nh, SlotsLaunch g)
{
    float mx;
    double mean;
    stats_wave(g.part, g.np, mx, mean);
    SpreadScale scale = scale_from_stats(mx, mean, g.wamp, g.wtyp);
    scale.e = __builtin_amdgcn_readfirstlane(scale.e);
    scale.fixed = __builtin_amdgcn_readfirstlane(scale.fixed);
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *g.sc = scale;
    int pair, t0 = 0, t1 = a.ntiles;
    SlotsOut out{y, h, nh, nullptr};
    if ((int)blockIdx.x < g.nfull) {
        pair = xcd_remap(blockIdx.x, g.nfull);
    } else {
        const int nrest = (int)(gridDim.x - g.nfull) / g.parts;
        const int L = xcd_remap(blockIdx.x - g.nfull, gridDim.x - g.nfull);
        const int part = L / nrest;
        pair = g.nfull + L % nrest;
        t0 = (int)((int64_t)a.ntiles * part / g.parts);
        t1 = (int)((int64_t)a.ntiles * (part + 1) / g.parts);
        if (g.parts > 1)
            out.sums = g.sums + (size_t)L * a.nt * RB;
    }
    slots_item<TT, DYN, GATE, NEG, RB>(a, m, scale, pair % a.ns, (pair / a.ns) * RB, t0, t1, out);
}

// The parts of a pair added, converted and convolved: workgroup b = four
// slots (b mod (rb / 4)) of pair nfull + b / (rb / 4).
constexpr int kFinalRows = 4;
__global__ __launch_bounds__(kBlock) void slots_final_kernel(KArgs a, int rb, SlotsLaunch g,
                                                             int nrest, float *__restrict__ y,
                                                             const float *__restrict__ h, int nh)
{
    extern __shared__ __align__(16) unsigned char kx_smem[];
    float *win = reinterpret_cast<float *>(kx_smem);
    const SpreadScale scale = *g.sc;
    const int nq = rb / kFinalRows;
    const int j0 = (int)(blockIdx.x % nq) * kFinalRows, rest = (int)blockIdx.x / nq;
    const int pair = g.nfull + rest;
    const int s = pair % a.ns, r0 = (pair / a.ns) * rb + j0;
    const int nrl = min(kFinalRows, a.nr - r0);
    if (nrl <= 0)
        return;  // uniform over the workgroup
    const int S = fused_row(a.nt, nh), Lm = (nh - 1) / 2;
    const size_t block = (size_t)a.nt * rb, stride = (size_t)nrest * block;
    const unsigned long long *p = g.sums + rest * block + j0;
    for (int i = threadIdx.x; i < a.nt * kFinalRows; i += kBlock) {
        const int j = i & (kFinalRows - 1), n = i / kFinalRows;
        const unsigned long long *q = p + (size_t)n * rb + j;
        unsigned long long acc = 0;
        double accd = 0.0;
#pragma unroll 4
        for (int k = 0; k < g.parts; ++k) {
            const unsigned long long v = q[k * stride];
            acc += v;
            accd += __builtin_bit_cast(double, v);
        }
        if (j < nrl)
            win[j * S + Lm + n] =
                scale.fixed ? (float)ldexp((double)(long long)acc, -scale.e) : (float)accd;
    }
    rows_conv_store(win, y, (size_t)s * a.nr + r0, 1, a.nt, nrl, h, nh);
}

// Traces longer than a workgroup's LDS: workgroup L (after the XCD
// renumbering) = segment L mod nseg of the trace of source (L / nseg) mod
// ns and receiver L / (nseg ns), samples [seg tseg, seg tseg + tseg); the
// segments of one trace are neighbours and share its table rows in L2.
template <typename TD, typename TT, bool DYN, bool NEG>
__global__ __launch_bounds__(kSpreadBlock) void spread_seg_kernel(KArgs a,
                                                                  const TD *__restrict__ m,
                                                                  TD *__restrict__ y,
                                                                  const SpreadScale *__restrict__ sc,
                                                                  int tseg, int nseg)
{
    const int L = xcd_remap(blockIdx.x, gridDim.x);
    const int seg = L % nseg, sr = L / nseg;
    a.t0 = seg * tseg;
    a.tlen = min(tseg, a.nt - a.t0);
    const SpreadScale scale = *sc;
    spread_item<TD, TT, DYN, NEG, kOrdNatural, 1, false, true>(a, m, y, scale, sr % a.ns,
                                                               sr / a.ns);
}

// K models of a float32 operator; workgroup L (after the XCD renumbering) =
// source L mod ns, receiver L / ns.  The launch accumulates in fixed point
// when every model's scale allows it, in float64 otherwise.
template <typename TT, bool DYN, bool NEG, int K>
__global__ __launch_bounds__(kSpreadBlock) void spread_models_kernel(
    KArgs a, const float *__restrict__ m, int64_t ni, float *__restrict__ y, int64_t ystride,
    const SpreadScale *__restrict__ sc)
{
    const int L = xcd_remap(blockIdx.x, gridDim.x);
    bool fixed = true;
#pragma unroll
    for (int j = 0; j < K; ++j)
        fixed = fixed && sc[j].fixed;
    if (fixed)
        spread_models_body<TT, DYN, NEG, true, K>(a, m, ni, y, ystride, sc, L % a.ns, L / a.ns);
    else
        spread_models_body<TT, DYN, NEG, false, K>(a, m, ni, y, ystride, sc, L % a.ns, L / a.ns);
}

constexpr int kRblocks[] = {4, 2, 1};

constexpr int kLdsPerCu = 160 * 1024;
constexpr int kMaxWavesPerCu = 32;

// LDS of a workgroup's traces: 8 bytes per sample, rows trace_stride(nt)
// samples apart (the models kernel keeps rows of nt samples)
size_t spread_lds_bytes(int rb, int nt) { return (size_t)rb * trace_stride(nt) * 8; }
size_t models_lds_bytes(int k, int nt) { return (size_t)k * nt * 8; }

template <typename TD, typename TT, bool DYN, bool NEG, bool XS, int ORD, int RB>
int launch_spread_rb(const KArgs &a, const void *m, void *y, const SpreadScale *sc,
                     hipStream_t st, const void *h, int nh)
{
    const size_t lds = spread_lds_bytes(RB, a.nt);
    if (h != nullptr && (sizeof(TD) != 4 || !fused_conv_ok(RB, a.nt, nh, lds, kSpreadBlock)))
        return KX_ENOFUSE;
    const int nrb = (a.nr + RB - 1) / RB;
    const int nblk = a.ns * nrb;
    allow_lds(reinterpret_cast<const void *>(&spread_kernel<TD, TT, DYN, NEG, ORD, RB, XS>),
              lds);
    hipLaunchKernelGGL((spread_kernel<TD, TT, DYN, NEG, ORD, RB, XS>), dim3(nblk),
                       dim3(kSpreadBlock), lds, st, a, reinterpret_cast<const TD *>(m),
                       reinterpret_cast<TD *>(y), sc, reinterpret_cast<const TD *>(h), nh);
    KX_LAUNCHED("spread");
    return KX_OK;
}

template <typename TD, typename TT, bool DYN, bool NEG, bool XS, int ORD>
const void *spread_fn(int rb)
{
    switch (rb) {
    case 4:
        return reinterpret_cast<const void *>(&spread_kernel<TD, TT, DYN, NEG, ORD, 4, XS>);
    case 2:
        return reinterpret_cast<const void *>(&spread_kernel<TD, TT, DYN, NEG, ORD, 2, XS>);
    default:
        return reinterpret_cast<const void *>(
            &spread_kernel<TD, TT, DYN, NEG, kOrdNatural, 1, XS>);
    }
}

// Workgroups of one spread kernel resident per CU (registers, LDS, waves);
// without a device, the LDS and wave limits alone.
int spread_per_cu(const void *fn, int rb, int nt)
{
    const size_t lds = spread_lds_bytes(rb, nt);
    allow_lds(fn, lds);
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, kSpreadBlock, lds) != hipSuccess ||
        n <= 0) {
        (void)hipGetLastError();
        n = std::min((int)(kLdsPerCu / lds), kMaxWavesPerCu / kSpreadWaves);
    }
    return std::max(n, 1);
}

// Receivers per workgroup.  A requested value is rounded down to a supported
// one whose traces fit in LDS.  Automatic: the block that keeps the most
// traces resident per CU, weighted by how far the resident waves (up to 24)
// can hide the latency of the table loads; ties go to the larger block,
// which re-reads the image and the source table less often.
template <typename TD, typename TT, bool DYN, bool NEG, bool XS, int ORD>
int pick_rblock(int requested, int nr, int nt)
{
    auto fits = [&](int rb) { return spread_lds_bytes(rb, nt) <= lds_budget(); };
    if (requested > 0) {
        for (int rb : kRblocks)
            if (rb <= requested && fits(rb))
                return rb;
        return 1;
    }
    int best = 1;
    double best_score = -1.0;
    for (int rb : kRblocks) {
        if (!fits(rb) || (rb > 1 && rb / 2 >= nr))
            continue;
        const int per_cu =
            spread_per_cu(spread_fn<TD, TT, DYN, NEG, XS, ORD>(rb), rb, nt);
        const double waves = std::min(24.0, (double)per_cu * kSpreadWaves);
        const double score = waves / 24.0 * per_cu * std::min(rb, nr);
        if (score > best_score * 1.0001) {
            best = rb;
            best_score = score;
        }
    }
    return best;
}

template <typename TD, typename TT, bool DYN, bool NEG, bool XS, int ORD>
int launch_spread_o(KArgs a, int requested, const void *m, void *y, const SpreadScale *sc,
                     hipStream_t st, const void *h, int nh)
{
    a.rblock = pick_rblock<TD, TT, DYN, NEG, XS, ORD>(requested, a.nr, a.nt);
    switch (a.rblock) {
    case 4:
        return launch_spread_rb<TD, TT, DYN, NEG, XS, ORD, 4>(a, m, y, sc, st, h, nh);
    case 2:
        return launch_spread_rb<TD, TT, DYN, NEG, XS, ORD, 2>(a, m, y, sc, st, h, nh);
    default:
        return launch_spread_rb<TD, TT, DYN, NEG, XS, kOrdNatural, 1>(a, m, y, sc, st, h, nh);
    }
}

// Whether the kernels of 4, 2 and 1 block sources (see launch_spread_d;
// float16 plans keep the two sides' offsets in different types and block
// receivers).
bool blocks_sources(const kx_plan *p)
{
    if (p->dtype != KX_F32 || p->tab_fmt == KX_F16)
        return false;
    return p->sside == KX_SIDE_AUTO ? p->ny == 1 && p->ns < p->nr : p->sside == KX_SIDE_SOURCES;
}

// How a forward runs in slot blocks: rb receivers per workgroup (0: the
// kernels of 4, 2 and 1), the pairs past the first nfull in `parts`
// workgroups each; fused: the wavelet convolved in the same launch.
struct SlotsShape {
    int rb, threads, nfull, parts;
    bool fused;
    size_t lds, sums_bytes;
};

// Estimated times of a forward, in microseconds: sums of terms whose factors
// were fitted to the measured times of 1859 random 2D and 3D operators (2 to
// 13000 tiles, 1 to 61 sources, 2 to 400 receivers, 60 to 2500 samples, 41 to
// 2300 taps; 27800 launches, 80% of them within 15%).
//   fixed   the launches
//   round   a round of workgroups
//   clear   clearing and writing out, per 1000 samples of a CU
//   step    a wave's (tile, receiver), the instructions and LDS operations of
//           all waves of a CU, per 1000
//   chain   the same where one wave's own chain of operations is as long
//   tile    a wave's tile (its loads' latency), per 1000
//   conv    per 10^6 multiply-adds of a CU
struct RowsTime {
    double fixed, clear, step, chain, conv, tile;
};
struct SlotsTime {
    double fixed, round, clear, step, chain, conv;
    double add;       // adding the parts: per 100 dependent loads of a thread
    double bytes;     // ... per MB of sums
    double add_conv;  // ... its convolution, per 1000 four-tap steps of a thread
};
constexpr RowsTime kRowsTime[2] = {  // kinematic, dynamic
    {7.17, 0.329, 8.65, 11.5, 11.2, 228.0},
    {8.05, 0.356, 10.8, 0.0, 11.4, 277.0},
};
constexpr SlotsTime kSlotsTime[2][2][2] = {  // [dynamic][blocks of 16][1024 threads]
    {{{7.81, 2.47, 0.008, 4.65, 72.4, 14.4, 40.2, 0.319, 74.5},
      {5.59, 4.18, 0.369, 11.5, 0.0, 11.5, 39.9, 0.117, 55.9}},
     {{8.66, 1.42, 0.0, 4.33, 42.1, 10.9, 39.2, 0.568, 81.0},
      {4.07, 6.30, 0.209, 7.94, 0.0, 8.39, 36.7, 0.316, 73.7}}},
    {{{6.73, 2.94, 0.104, 7.74, 51.6, 15.3, 40.8, 0.250, 75.0},
      {3.12, 7.32, 0.284, 11.8, 0.0, 10.2, 39.3, 0.069, 57.9}},
     {{8.23, 0.59, 0.085, 6.61, 36.0, 11.7, 42.2, 0.517, 78.7},
      {1.64, 7.18, 0.196, 9.28, 0.0, 9.73, 37.8, 0.335, 72.0}}},
};

// one(w) summed over the rounds of wgs workgroups, `at_once` at a time
template <typename F> double sum_rounds(int64_t wgs, int64_t at_once, F one)
{
    double t = (double)(wgs / at_once) * (wgs >= at_once ? one(at_once) : 0.0);
    return wgs % at_once ? t + one(wgs % at_once) : t;
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// kx_conv of the traces
double conv_time(const kx_plan *p, int nh, int cus)
{
    const double ntr = (double)p->ns * p->nr;
    return 7.2 + 19.3e-9 * ntr * p->nt * nh +
           6.5e-3 * nh * std::ceil(ntr * ceil_div(p->nt, kConvOut) / (4.0 * cus));
}

// the kernels of 4, 2 and 1, in the block that pick_rblock takes (with its
// registers' share of the occupancy as measured); a caller without a second
// launch (kx_forward_noalloc) compares shapes that convolve in their own
double rows_time(const kx_plan *p, int nh, int cus, bool two_launches)
{
    const RowsTime &M = kRowsTime[p->dynamic != 0];
    const bool xs = blocks_sources(p);
    const int64_t n = xs ? p->ns : p->nr, other = xs ? p->nr : p->ns;
    int rb = 1, per_cu = 1;
    double best = -1.0;
    for (int c : kRblocks) {
        if (spread_lds_bytes(c, p->nt) > lds_budget() || (c > 1 && c / 2 >= n))
            continue;
        const int k = std::min((int)(kLdsPerCu / spread_lds_bytes(c, p->nt)), p->dynamic ? 3 : 4);
        const double score = std::min(24.0, (double)k * kSpreadWaves) / 24.0 * k * std::min<int64_t>(c, n);
        if (score > best * 1.0001) {
            best = score;
            rb = c;
            per_cu = k;
        }
    }
    const bool fused =
        nh > 0 && (!two_launches || fused_conv_ok(rb, p->nt, nh, spread_lds_bytes(rb, p->nt),
                                                  kSpreadBlock));
    const double tiles = (double)ceil_div(p->ntiles, kSpreadWaves);
    const double t = sum_rounds(other * ceil_div(n, rb), (int64_t)cus * per_cu, [&](int64_t w) {
        const double k = (double)ceil_div(w, cus);
        return 1e-3 * (k * p->nt * rb * M.clear + tiles * (M.tile + rb * (M.chain + kSpreadWaves * k * M.step))) +
               (fused ? 1e-6 * k * rb * p->nt * nh * M.conv : 0.0);
    });
    return M.fixed + t + (nh > 0 && !fused ? conv_time(p, nh, cus) : 0.0);
}

// a slot shape, convolving with nh taps (0: none)
double slots_time(const kx_plan *p, const SlotsShape &g, int nh, int cus)
{
    const SlotsTime &M =
        kSlotsTime[p->dynamic != 0][g.rb == 16][g.threads == kSlotsMaxThreads];
    const int nw = g.threads / kWave;
    const int64_t at_once = (int64_t)cus * (kSlotsMaxThreads / g.threads);
    const int64_t nrest = p->ns * ceil_div(p->nr, g.rb) - g.nfull;
    auto rounds = [&](int64_t wgs, int64_t tiles, int taps) {
        const double steps = (double)ceil_div(tiles, nw);
        return sum_rounds(wgs, at_once, [&](int64_t w) {
            const double k = (double)ceil_div(w, cus);
            return M.round + 1e-3 * g.rb * (k * p->nt * M.clear + steps * (M.chain + nw * k * M.step)) +
                   1e-6 * k * g.rb * p->nt * taps * M.conv;
        });
    };
    double t = M.fixed + rounds(g.nfull, p->ntiles, nh);
    if (g.parts > 1) {
        const double wgs = (double)nrest * (g.rb / kFinalRows);
        const double loads = (double)ceil_div((int64_t)p->nt * kFinalRows, kBlock) *
                             (g.parts / 4 + g.parts % 4);
        t += rounds(nrest * g.parts, ceil_div(p->ntiles, g.parts), 0) +
             1e-2 * M.add * loads * std::max(1.0, wgs / (4.0 * cus)) +
             1e-6 * M.bytes * (double)g.sums_bytes +
             1e-3 * M.add_conv * (double)ceil_div(p->nt, kBlock) * (conv_taps_padded(nh) / 4) *
                 std::max(1.0, wgs / (2.0 * cus));
    }
    return t;
}

// The shape with the smallest estimated time; a shape replaces a simpler one
// where it is more than 1% faster.  Where the pairs are no multiple of the
// workgroups that run at once, the last ones may be shared by several
// workgroups, in work_bytes of scratch, whose sums a second launch adds (four
// loads of a thread in flight: counts of parts that are no multiple of 4
// wait longer).  Long filters are convolved by a launch of their own
// (unfused, where the caller can: two_launches), with the whole chip instead
// of the workgroups that hold the traces: 201x150 with 21 x 101 traces of
// 1201 samples, 1139 taps, 414 us in LDS and 214 so.  A requested block size
// is an upper bound, without a comparison with smaller ones than 8.
SlotsShape pick_slots(const kx_plan *p, int nh, int64_t work_bytes, bool two_launches)
{
    SlotsShape best{0, 0, 0, 1, false, 0, 0};
    if (!(p->tabs & KX_TAB_SLOTS) || p->dtype != KX_F32 || p->sside == KX_SIDE_SOURCES ||
        (p->rblock > 0 && p->rblock < 8))
        return best;
    const int cus = device_cus();
    double best_t = p->rblock == 0 ? rows_time(p, nh, cus, two_launches) : 1e300;
    auto consider = [&](SlotsShape g) {
        const double t = nh > 0 && !g.fused ? slots_time(p, g, 0, cus) + conv_time(p, nh, cus)
                                            : slots_time(p, g, nh, cus);
        if (t < best_t * 0.99) {
            best_t = t;
            best = g;
        }
    };
    for (int rb : {16, 8}) {
        if (p->rblock > 0 && rb > p->rblock)
            continue;
        const int64_t pairs = p->ns * ceil_div(p->nr, rb);
        if (nh > 0 && two_launches)
            if (const int th = slots_threads(rb, p->nt, 0))
                consider({rb, th, (int)pairs, 1, false, slots_lds_bytes(rb, p->nt, 0), 0});
        const int th = slots_threads(rb, p->nt, nh);
        if (!th)
            continue;
        const size_t lds = slots_lds_bytes(rb, p->nt, nh);
        consider({rb, th, (int)pairs, 1, nh > 0, lds, 0});
        if (nh <= 0)
            continue;
        const int64_t at_once = (int64_t)cus * (kSlotsMaxThreads / th);
        const int64_t nfull = pairs / at_once * at_once, nrest = pairs - nfull;
        for (int parts : {2, 3, 4, 5, 6, 8, 10, 12, 14, 16}) {
            const size_t sums = (size_t)(nrest * parts) * p->nt * rb * 8;
            if (nrest == 0 || (int64_t)sums > work_bytes ||
                p->ntiles < (int64_t)parts * (th / kWave))
                break;
            consider({rb, th, (int)nfull, parts, true, lds, sums});
        }
    }
    return best;
}

template <typename TT, bool DYN, bool GATE, bool NEG, int RB>
int launch_slots_rb(const KArgs &a, const SlotsShape &g, const SlotsLaunch &l, const void *m,
                    void *y, hipStream_t st, const void *h, int nh)
{
    const int nrest = a.ns * ((a.nr + RB - 1) / RB) - g.nfull;
    allow_lds(reinterpret_cast<const void *>(&slots_kernel<TT, DYN, GATE, NEG, RB>), g.lds);
    hipLaunchKernelGGL((slots_kernel<TT, DYN, GATE, NEG, RB>), dim3(g.nfull + nrest * g.parts),
                       dim3(g.threads), g.lds, st, a, reinterpret_cast<const float *>(m),
                       reinterpret_cast<float *>(y), reinterpret_cast<const float *>(h), nh, l);
    KX_LAUNCHED("spread");
    if (g.parts > 1) {
        const size_t lds =
            ((size_t)kFinalRows * fused_row(a.nt, nh) + conv_taps_padded(nh)) * sizeof(float);
        allow_lds(reinterpret_cast<const void *>(&slots_final_kernel), lds);
        hipLaunchKernelGGL(slots_final_kernel, dim3(nrest * (RB / kFinalRows)), dim3(kBlock), lds,
                           st, a, RB, l, nrest, reinterpret_cast<float *>(y),
                           reinterpret_cast<const float *>(h), nh);
        KX_LAUNCHED("spread parts");
    }
    return KX_OK;
}

template <typename TT, bool DYN, bool GATE, bool NEG>
int launch_slots(const KArgs &a, const SlotsShape &g, const SlotsLaunch &l, const void *m,
                 void *y, hipStream_t st, const void *h, int nh)
{
    return g.rb == 16 ? launch_slots_rb<TT, DYN, GATE, NEG, 16>(a, g, l, m, y, st, h, nh)
                      : launch_slots_rb<TT, DYN, GATE, NEG, 8>(a, g, l, m, y, st, h, nh);
}

template <typename TT>
int launch_slots_d(const kx_plan *p, const KArgs &a, const SlotsShape &g, const SlotsLaunch &l,
                   const void *m, void *y, hipStream_t st, const void *h, int nh)
{
    if (p->dynamic == KX_DYNAMIC_NOGATE)
        return p->neg_trav ? launch_slots<TT, true, false, true>(a, g, l, m, y, st, h, nh)
                           : launch_slots<TT, true, false, false>(a, g, l, m, y, st, h, nh);
    if (p->dynamic)
        return p->neg_trav ? launch_slots<TT, true, true, true>(a, g, l, m, y, st, h, nh)
                           : launch_slots<TT, true, true, false>(a, g, l, m, y, st, h, nh);
    return p->neg_trav ? launch_slots<TT, false, false, true>(a, g, l, m, y, st, h, nh)
                       : launch_slots<TT, false, false, false>(a, g, l, m, y, st, h, nh);
}

template <typename TD, typename TT, bool DYN, bool NEG, bool XS>
int launch_spread_t(const KArgs &a, int order, int requested, const void *m, void *y,
                    const SpreadScale *sc, hipStream_t st, const void *h, int nh)
{
    switch (order) {
    case KX_ORDER_ROTATED:
        return launch_spread_o<TD, TT, DYN, NEG, XS, kOrdRotated>(a, requested, m, y, sc, st, h,
                                                                  nh);
    default:
        return launch_spread_o<TD, TT, DYN, NEG, XS, kOrdNatural>(a, requested, m, y, sc, st, h,
                                                                  nh);
    }
}

// h != NULL: the spread and the wavelet convolution in one launch (y
// receives the data), or KX_ENOFUSE when this plan's launch cannot
// convolve in LDS (float64 data, too little LDS).
// Segments of traces that do not fit a workgroup's LDS: the longest
// multiple of 64 samples that does, or 0 if not even 64 fit.
int trace_segment(int nt)
{
    int t = (int)std::min<size_t>((size_t)nt, lds_budget() / 8) & ~63;
    while (t > 0 && spread_lds_bytes(1, t) > lds_budget())
        t -= 64;
    return t;
}

template <typename TD, typename TT, bool DYN, bool NEG>
int launch_spread_seg(const KArgs &a, const void *m, void *y, const SpreadScale *sc,
                      hipStream_t st)
{
    const int tseg = trace_segment(a.nt);
    if (tseg <= 0)
        return kx_failf(KX_ELDS, "nt=%d: not even 64 samples of a trace fit in LDS", a.nt);
    const int nseg = (a.nt + tseg - 1) / tseg;
    const int64_t nblk = (int64_t)a.ns * a.nr * nseg;
    if (nblk > INT32_MAX)
        return kx_failf(KX_ESHAPE, "spread: %lld trace segments exceed the grid",
                        (long long)nblk);
    const size_t lds = spread_lds_bytes(1, tseg);
    allow_lds(reinterpret_cast<const void *>(&spread_seg_kernel<TD, TT, DYN, NEG>), lds);
    hipLaunchKernelGGL((spread_seg_kernel<TD, TT, DYN, NEG>), dim3((unsigned)nblk),
                       dim3(kSpreadBlock), lds, st, a, reinterpret_cast<const TD *>(m),
                       reinterpret_cast<TD *>(y), sc, tseg, nseg);
    KX_LAUNCHED("spread segments");
    return KX_OK;
}

// work: work_bytes of scratch for the parts of slot blocks (0: one part);
// two_launches: whether the caller convolves by itself after KX_ENOFUSE.
template <typename TD, typename TT>
int launch_spread_d(const kx_plan *p, KArgs a, const void *m, void *y, hipStream_t st,
                    const void *h = nullptr, void *work = nullptr, int64_t work_bytes = 0,
                    bool two_launches = false)
{
    const int nh = h != nullptr ? p->nh : 0;
    if (h != nullptr && sizeof(TD) != 4)
        return KX_ENOFUSE;
    // a trace longer than LDS: spread in time segments (the wavelet then
    // convolves the traces in HBM)
    const bool seg = spread_lds_bytes(1, p->nt) > lds_budget();
    if (seg && h != nullptr)
        return KX_ENOFUSE;
    if (sizeof(TD) == 4 && !p->aux)
        return kx_failf(KX_EINVAL, "spread: plan.aux (KX_AUX_BYTES of device scratch) is NULL");
    SpreadScale *sc = reinterpret_cast<SpreadScale *>(p->aux);
    const SlotsShape slots = pick_slots(p, nh, work ? work_bytes : 0, two_launches);
    if (slots.rb && h != nullptr && !slots.fused)
        return KX_ENOFUSE;
    const bool xs = blocks_sources(p);
    if constexpr (sizeof(TD) == 4) {
        // fixed-point scale of this launch from max|m|
        const int64_t ni = (int64_t)p->nx * p->ny * p->nz;
        float *part = reinterpret_cast<float *>(p->aux) + 16;
        const int nb = (int)std::min<int64_t>(kScaleBlocks, (ni + kBlock - 1) / kBlock);
        hipLaunchKernelGGL(absmax_partial_kernel, dim3(nb), dim3(kBlock), 0, st,
                           reinterpret_cast<const float *>(m), ni, part);
        KX_LAUNCHED("spread scale");
        if (slots.rb) {
            const SlotsLaunch l{part, nb, p->wamp, p->wtyp, sc, slots.nfull, slots.parts,
                                static_cast<unsigned long long *>(work)};
            return launch_slots_d<TT>(p, a, slots, l, m, y, st, h, nh);
        }
        hipLaunchKernelGGL(scale_final_kernel, dim3(1), dim3(kWave), 0, st, part, nb, p->wamp,
                           p->wtyp, sc);
        KX_LAUNCHED("spread scale");
    }
    // A workgroup blocking sources (float32 operators) runs the spread with
    // the two sides' tables exchanged and writes its traces to the
    // transposed positions: T = os + or and the integer bases add in either
    // order, and the dynamic kernel (XS) forms the source-side products per
    // step, so the traces are bitwise those of blocks of receivers.
    // Automatic, where the plan takes no slot blocks: a 2D plan blocks the
    // side with fewer members, whose rows then serve many workgroups through
    // L2 (on a 61 x 301 geometry 13% faster kinematic, either way round, and
    // 6% with dynamic weights: 3.68 against 3.91 ms for the forward with its
    // wavelet); 3D plans block receivers (measured slower otherwise:
    // 128x128x120 with 25 x 400, 24.2 against 22.8 ms for the natural order,
    // 17.4 against 15.8 ms rotated).
    if (seg)
        return p->dynamic ? (p->neg_trav ? launch_spread_seg<TD, TT, true, true>(a, m, y, sc, st)
                                         : launch_spread_seg<TD, TT, true, false>(a, m, y, sc, st))
                          : (p->neg_trav ? launch_spread_seg<TD, TT, false, true>(a, m, y, sc, st)
                                         : launch_spread_seg<TD, TT, false, false>(a, m, y, sc,
                                                                                   st));
    if (xs)
        exchange_sides(a);
    // automatic lane order: rotated when a step loads one receiver table,
    // natural when it loads three (dynamic weights), where the scattered
    // loads cost more than the collisions they avoid
    int order = p->sorder;
    if (order == KX_ORDER_AUTO)
        order = p->dynamic ? KX_ORDER_NATURAL : KX_ORDER_ROTATED;
    // exchanged-side dynamic kernels exist for float32 operators only (xs
    // is false otherwise)
    constexpr bool kXS = sizeof(TD) == 4;
    const int rb = p->rblock;
    if (p->dynamic && xs)
        return p->neg_trav
                   ? launch_spread_t<TD, TT, true, true, kXS>(a, order, rb, m, y, sc, st, h, nh)
                   : launch_spread_t<TD, TT, true, false, kXS>(a, order, rb, m, y, sc, st, h, nh);
    if (p->dynamic)
        return p->neg_trav
                   ? launch_spread_t<TD, TT, true, true, false>(a, order, rb, m, y, sc, st, h, nh)
                   : launch_spread_t<TD, TT, true, false, false>(a, order, rb, m, y, sc, st, h, nh);
    return p->neg_trav
               ? launch_spread_t<TD, TT, false, true, false>(a, order, rb, m, y, sc, st, h, nh)
               : launch_spread_t<TD, TT, false, false, false>(a, order, rb, m, y, sc, st, h, nh);
}

}  // namespace

extern "C" int kx_spread(const kx_plan *p, const void *m, void *traces, void *stream)
{
    int rc = kx_plan_check(p);
    if (rc)
        return rc;
    if (!m || !traces)
        return kx_failf(KX_EINVAL, "spread: NULL buffer");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const KArgs a = make_args(p);
    if (p->dtype == KX_F64)
        return launch_spread_d<double, double>(p, a, m, traces, st);
    if (p->tab_fmt == KX_F16)
        return launch_spread_d<float, __half>(p, a, m, traces, st);
    return launch_spread_d<float, float>(p, a, m, traces, st);
}

extern "C" __attribute__((visibility("hidden"))) int kx_spread_wavelet(
    const kx_plan *p, const void *m, void *d, void *work, int64_t work_bytes, bool two_launches,
    void *stream)
{
    int rc = kx_plan_check(p);
    if (rc)
        return rc;
    if (!m || !d || !p->h || p->nh <= 0)
        return kx_failf(KX_EINVAL, "spread_wavelet: NULL buffer or wavelet");
    if (p->dtype != KX_F32)
        return KX_ENOFUSE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const KArgs a = make_args(p);
    if (p->tab_fmt == KX_F16)
        return launch_spread_d<float, __half>(p, a, m, d, st, p->h, work, work_bytes, two_launches);
    return launch_spread_d<float, float>(p, a, m, d, st, p->h, work, work_bytes, two_launches);
}

extern "C" int kx_forward_slots(const kx_plan *p)
{
    if (!p || p->abi_version != KX_ABI_VERSION || p->nx <= 0 || p->ny <= 0 || p->nz <= 0 ||
        p->ntiles <= 0 || p->ns <= 0 || p->nr <= 0 || p->nt < 2)
        return kx_failf(KX_EINVAL, "forward_slots: bad plan");
    kx_plan q = *p;
    q.tabs |= KX_TAB_SLOTS;
    return pick_slots(&q, q.nh, INT64_MAX, true).rb > 0 || pick_slots(&q, 0, 0, false).rb > 0;
}

extern "C" __attribute__((visibility("hidden"))) int64_t kx_spread_sums_bytes(const kx_plan *p)
{
    return (int64_t)pick_slots(p, p->nh, INT64_MAX, true).sums_bytes;
}

namespace {

constexpr int kMaxModels = 64;
constexpr size_t kModelScaleOffset = 2048;  // bytes into plan.aux

template <typename TT, bool DYN, bool NEG, int K>
void launch_models_k(const KArgs &a, const float *m, int64_t ni, float *y, int64_t ystride,
                     const SpreadScale *sc, hipStream_t st)
{
    const size_t lds = models_lds_bytes(K, a.nt);
    hipLaunchKernelGGL((spread_models_kernel<TT, DYN, NEG, K>), dim3(a.ns * a.nr),
                       dim3(kSpreadBlock), lds, st, a, m, ni, y, ystride, sc);
}

template <typename TT, bool DYN, bool NEG>
int launch_models(const kx_plan *p, const KArgs &a, const float *m, float *y, int nmodel,
                  hipStream_t st)
{
    const int64_t ni = (int64_t)p->nx * p->ny * p->nz;
    const int64_t ystride = (int64_t)p->ns * p->nr * p->nt;
    SpreadScale *scs = reinterpret_cast<SpreadScale *>(static_cast<char *>(p->aux) +
                                                       kModelScaleOffset);
    float *part = reinterpret_cast<float *>(p->aux) + 16;
    const int nb = (int)std::min<int64_t>(kScaleBlocks, (ni + kBlock - 1) / kBlock);
    for (int j = 0; j < nmodel; ++j) {
        hipLaunchKernelGGL(absmax_partial_kernel, dim3(nb), dim3(kBlock), 0, st, m + j * ni, ni,
                           part);
        hipLaunchKernelGGL(scale_final_kernel, dim3(1), dim3(kWave), 0, st, part, nb, p->wamp,
                           p->wtyp, scs + j);
    }
    KX_LAUNCHED("spread models scale");
    int j = 0;
    while (j < nmodel) {
        const int left = nmodel - j;
        auto fits = [&](int k) {
            return k <= left && models_lds_bytes(k, a.nt) <= (size_t)kLdsBudget;
        };
        const float *mj = m + j * ni;
        float *yj = y + j * ystride;
        if (fits(8)) {
            launch_models_k<TT, DYN, NEG, 8>(a, mj, ni, yj, ystride, scs + j, st);
            j += 8;
        } else if (fits(4)) {
            launch_models_k<TT, DYN, NEG, 4>(a, mj, ni, yj, ystride, scs + j, st);
            j += 4;
        } else if (fits(2)) {
            launch_models_k<TT, DYN, NEG, 2>(a, mj, ni, yj, ystride, scs + j, st);
            j += 2;
        } else {
            const int rc = launch_spread_d<float, TT>(p, a, mj, yj, st);
            if (rc)
                return rc;
            j += 1;
        }
        KX_LAUNCHED("spread models");
    }
    return KX_OK;
}

}  // namespace

extern "C" int kx_spread_models(const kx_plan *p, const void *m, void *traces, int32_t nmodel,
                                void *stream)
{
    int rc = kx_plan_check(p);
    if (rc)
        return rc;
    if (!m || !traces)
        return kx_failf(KX_EINVAL, "spread_models: NULL buffer");
    if (p->dtype != KX_F32)
        return kx_failf(KX_ETYPE, "spread_models: float32 operators only");
    if (nmodel < 1 || nmodel > kMaxModels)
        return kx_failf(KX_ESHAPE, "spread_models: nmodel=%d outside [1, %d]", nmodel, kMaxModels);
    if (!p->aux)
        return kx_failf(KX_EINVAL, "spread_models: plan.aux (KX_AUX_BYTES of device scratch) is NULL");
    // (traces of a few models per workgroup that do not fit LDS fall back to
    // single spreads, in time segments if need be)
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const KArgs a = make_args(p);
    const float *mf = reinterpret_cast<const float *>(m);
    float *yf = reinterpret_cast<float *>(traces);
    if (p->tab_fmt == KX_F16)
        return p->dynamic ? (p->neg_trav ? launch_models<__half, true, true>(p, a, mf, yf, nmodel, st)
                                         : launch_models<__half, true, false>(p, a, mf, yf, nmodel, st))
                          : (p->neg_trav ? launch_models<__half, false, true>(p, a, mf, yf, nmodel, st)
                                         : launch_models<__half, false, false>(p, a, mf, yf, nmodel, st));
    return p->dynamic ? (p->neg_trav ? launch_models<float, true, true>(p, a, mf, yf, nmodel, st)
                                     : launch_models<float, true, false>(p, a, mf, yf, nmodel, st))
                      : (p->neg_trav ? launch_models<float, false, true>(p, a, mf, yf, nmodel, st)
                                     : launch_models<float, false, false>(p, a, mf, yf, nmodel, st));
}

// ---------------------------------------------------------------------------
// the forward operator without caller memory
// ---------------------------------------------------------------------------
// The one-launch forward keeps only its accumulation scale and the partial
// maxima of |m| in scratch memory (plan.aux for kx_forward).  For callers
// that cannot allocate, that scratch is this device array: every GPU the
// library runs on holds its own copy (KX_AUX_BYTES) until the process ends.
static __device__ __align__(256) unsigned char scratch[KX_AUX_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// The address of scratch on the current device, looked up once per device
// (hipGetSymbolAddress with that device current).
int scratch_address(void **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return kx_failf((int)e, "forward_noalloc: hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices)
        return kx_failf(KX_EINVAL, "forward_noalloc: device %d beyond the %d supported", dev,
                        kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess)
            return kx_failf((int)e, "forward_noalloc: hipGetSymbolAddress(scratch): %s",
                            hipGetErrorString(e));
        if (ptr == nullptr)
            return kx_failf(KX_EINVAL, "forward_noalloc: scratch has no device address");
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return KX_OK;
}

}  // namespace

extern "C" int kx_forward_noalloc(const kx_plan *p, const void *m, void *d, void *stream)
{
    int rc = kx_plan_check(p);
    if (rc)
        return rc;
    if (!m || !d || !p->h || p->nh <= 0)
        return kx_failf(KX_EINVAL, "forward_noalloc: NULL buffer or wavelet");
    if (p->dtype != KX_F32)
        return kx_failf(KX_ETYPE, "forward_noalloc: float32 plans only (a float64 forward "
                                  "needs kx_forward and its workspace)");
    void *s = nullptr;
    rc = scratch_address(&s);
    if (rc)
        return rc;
    // the plan as given, its scale kept in this device's scratch (every
    // launch writes the scale before the spread reads it: nothing needs
    // clearing)
    kx_plan q = *p;
    q.aux = s;
    rc = kx_spread_wavelet(&q, m, d, nullptr, 0, false, stream);
    if (rc == KX_ENOFUSE && q.rblock == 0 && (q.tabs & KX_TAB_SLOTS) && q.nr > 4) {
        // filters too long for the rows of the estimated fastest shape may
        // fit a slot block, whose LDS is not bound to the sums' size (plans
        // that would leave half of it empty stay refused)
        q.rblock = 16;
        rc = kx_spread_wavelet(&q, m, d, nullptr, 0, false, stream);
    }
    if (rc == KX_ENOFUSE)
        return kx_failf(KX_ELDS,
                        "forward_noalloc: this plan's forward cannot convolve in the spread "
                        "launch (nt=%d traces with %d wavelet taps do not fit a workgroup's "
                        "LDS, or float32 atomics were requested); use kx_forward and its "
                        "workspace",
                        p->nt, p->nh);
    return rc;
}
