// kx_fit.h -- the adjoint of plans whose samples all fall inside the staged
// windows (kx_plan.tabs, KX_TAB_FIT*): gather_tiles without the tests for
// samples outside.
#pragma once
#include "kx_device.h"

namespace {

// The gather is bound by vector instruction issue (3D 128x128x120, 25 sources,
// 400 receivers: 84% of its time).  gather_tiles spends on a sample the window
// test (a maximum and a clamp) and two additions for its window index, and on
// a staged window about nine vector instructions; those are shared by NP tiles
// only, so that with NP = 1 they cost as much as the samples.  Here
//   - the table bounds guarantee that every sample lies in its window
//     (kx_table_fit, kFitBound): no test, no second look;
//   - a window starts at the mean source base plus the mean receiver base of
//     the group, so that the index of a sample is floor(T) plus a constant of
//     the source and one of the receiver: one shift-and-add to the LDS
//     address of its pair;
//   - rows and windows are loaded relative to advancing scalar pointers; a
//     window's address takes two instructions, and windows that lie inside
//     the trace (all but the first and last of a trace) are staged without
//     masks, the difference by one DPP subtraction;
//   - receiver bases and gates are loaded 64 receivers at a time, a lane each.
// Seven and a half vector instructions a sample are left with NP = 4
// (gather_tiles: ten), six of them the sample's own.  Measured, gather_tiles
// and this: the 3D above 7.0 and 5.5 ms, 93x77x101 with float16 tables 0.87
// and 0.68 ms, 2D 601x300 dynamic with 61 x 301 traces 1.98 and 1.72 ms,
// 333x187 dynamic with apertures and float16 tables 0.45 and 0.28 ms.
// (Branching to unclamped window addresses saves two more instructions a
// window but costs more scalar work: 2D dynamic 1.88 -> 2.0 ms.)
// The sums are gather_tiles' in gather_tiles' order: the image is bitwise the
// same.
constexpr float kFitBound = 29.5f;  // kWin / 2 less the floor, the pair and a margin

// waves per SIMD asked of the compiler: with two tiles a dynamic group takes
// 91 vector registers, five waves; six (80 registers, a few words of scratch
// outside the receiver loop) measured 1.88 -> 1.72 ms on 2D 601x300
template <typename TD, bool DYN, int NP, int K> struct FitWaves {
    static constexpr int v = (DYN && NP == 2 && K == 1 && sizeof(TD) == 4) ? 6 : 1;
};

// lane l + 1's value minus this lane's (lane 63: its own value's negative)
__device__ __forceinline__ float next_minus(float v)
{
    return __builtin_bit_cast(
               float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true)) -
           v;
}
__device__ __forceinline__ double next_minus(double v) { return lane_next(v) - v; }

// element i of a row at a wave-uniform address
template <typename T> __device__ __forceinline__ T row_at(const T *row, unsigned i)
{
    return scalar_ptr(row)[i];
}
template <> __device__ __forceinline__ __half row_at(const __half *row, unsigned i)
{
    return __ushort_as_half(scalar_ptr(reinterpret_cast<const unsigned short *>(row))[i]);
}

// value at byte offset at (32 bits) of a wave-uniform address
template <typename T> __device__ __forceinline__ T at_byte(const char *p, unsigned at)
{
    return *(GlobalPtr<T>)(scalar_ptr(p) + at);
}

// min(max(x, lo), hi), lo <= hi
__device__ __forceinline__ int clamp_to(int x, int lo, int hi)
{
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(lo), "v"(hi));
    return r;
}

template <typename TD, typename TT, bool DYN, int JW, int P, int NP, int K = 1, bool GATE = true>
__device__ __forceinline__ void gather_fit(const KArgs &a, const TD *__restrict__ d,
                                           TD *__restrict__ m, int L, int64_t dstride = 0,
                                           int64_t mstride = 0)
{
    using TC = typename TimeType<TD>::type;
    using TP = VecN<TD, 2>;               // (d[k], d[k+1] - d[k])
    typedef TD Pair __attribute__((ext_vector_type(2)));
    using LdsPair = const __attribute__((address_space(3))) Pair *;
    constexpr int NG = kGatherWaves / P;  // tile groups per workgroup
    constexpr int SB = JW * P;            // sources per block (all parts)
    constexpr int kFar = -(1 << 26);      // base of a missing source: before every trace
    constexpr int kPairShift = sizeof(TD) == 4 ? 3 : 4;
    __shared__ TP win[kGatherWaves][K][JW][kWin];
    static_assert(K * NP * kGatherBlock * sizeof(TD) <= sizeof(win), "reduction space");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int part = wave / NG;  // this wave sums sources s0 + part + P i
    const int gq = L * NG + wave % NG;
    const bool active = gq < a.ngroups;
    const int g = active ? gq : a.ngroups - 1;
    const int tzi = g % a.ntz;
    const int grest = g / a.ntz;
    const int gx0 = (grest % a.ngx) * a.gx, gy0 = (grest / a.ngx) * a.gy;
    int t[NP];
    bool tok[NP];
    TilePoint pt[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        const int txi = gx0 + j % a.gx, tyi = gy0 + j / a.gx;
        tok[j] = txi < a.ntx && tyi < a.nty;
        // a tile past the grid's edge repeats the group's first tile and
        // stores nothing
        t[j] = tzi + a.ntz * (tok[j] ? txi + a.ntx * tyi : gx0 + a.ntx * gy0);
        pt[j] = tile_point(a, t[j], lane);
    }
    const typename SrcTab<TT>::type *offs =
        reinterpret_cast<const typename SrcTab<TT>::type *>(a.off_s);
    const TT *offr = reinterpret_cast<const TT *>(a.off_r);
    const TD *wps = reinterpret_cast<const TD *>(a.wp_s);
    const TD *wqs = reinterpret_cast<const TD *>(a.wq_s);
    using RW = typename RecW<TD, TT>::type;
    const RW *wpr = reinterpret_cast<const RW *>(a.wp_r);
    const RW *wqr = reinterpret_cast<const RW *>(a.wq_r);
    const unsigned ntm1 = (unsigned)(a.nt - 1);
    const int vz = vgpr_zero();
    TP(&w)[K][JW][kWin] = win[wave];
    const int wbase = __builtin_amdgcn_readfirstlane(
        (int)(unsigned)(uintptr_t)(__attribute__((address_space(3))) TP *)&w[0][0][0]);

    TD acc[K][NP];
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int j = 0; j < NP; ++j)
            acc[k][j] = TD(0);
    // one block of SB sources, JB slots of this wave (as in gather_tiles)
    auto source_block = [&](auto jw, const int s0) __attribute__((always_inline)) {
        constexpr int JB = decltype(jw)::value;
        TC os[JB][NP];
        TD ps[JB][NP], qs[JB][NP];
        int as[JB][NP];  // LDS byte offset of (source, tile): wave-uniform
        int ms[JB];      // mean source base of the group, less half a window
        int lo = 0x7fffffff, hi = -0x7fffffff;
        // byte of the source's first and last sample in round 0, and of lane
        // l's sample of a window at mean receiver base 0
        int row0[JB], row1[JB], rowl[JB];
#pragma unroll
        for (int i = 0; i < JB; ++i) {
            const int js = s0 + part + P * i;
            int b[NP], sum = 0;
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                if (js < a.ns) {
                    const size_t so = (size_t)t[j] * a.ns + js;
                    os[i][j] = (TC)ld_off(offs + so * kWave + lane);
                    b[j] = __builtin_amdgcn_readfirstlane(a.base_s[so + vz]);
                    if constexpr (DYN) {
                        ps[i][j] = wps[so * kWave + lane];
                        qs[i][j] = wqs[so * kWave + lane];
                    }
                } else {  // past the last source: every sample before the trace
                    os[i][j] = TC(0);
                    b[j] = kFar;
                    ps[i][j] = qs[i][j] = TD(0);
                }
                sum += b[j];
            }
            const int mean = sum >> Log2<NP>::v;
            ms[i] = mean - kWin / 2;
            lo = min(lo, ms[i]);
            hi = max(hi, ms[i]);
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                as[i][j] = wbase + (b[j] - mean + kWin / 2) * (int)sizeof(TP);
                // (one addend: the compiler would split it again)
                asm volatile("" : "+s"(as[i][j]));
            }
            row0[i] = (min(js, a.ns - 1) - s0) * a.nr * a.nt * (int)sizeof(TD) + vz;
            row1[i] = row0[i] + (a.nt - 1) * (int)sizeof(TD);
            rowl[i] = row0[i] + (lane + ms[i]) * (int)sizeof(TD);
        }
        // the windows of round R, of the traces from dr on: lane l holds
        // sample ms + mean receiver base + l, or where that is outside the
        // trace its first or last sample
        const char *dr = reinterpret_cast<const char *>(d + (size_t)s0 * a.nr * a.nt);
        TD sv[K][JB];
        int mr_n = 0, ar_n[NP];  // mean receiver base; LDS byte offsets of the tiles
        auto stage = [&](const int(&br)[NP]) __attribute__((always_inline)) {
            int sum = 0;
#pragma unroll
            for (int j = 0; j < NP; ++j)
                sum += br[j];
            mr_n = sum >> Log2<NP>::v;
#pragma unroll
            for (int j = 0; j < NP; ++j)
                ar_n[j] = (br[j] - mr_n) * (int)sizeof(TP);
#pragma unroll
            for (int i = 0; i < JB; ++i) {
                const int e = clamp_to(rowl[i] + mr_n * (int)sizeof(TD), row0[i], row1[i]);
#pragma unroll
                for (int k = 0; k < K; ++k)
                    sv[k][i] = at_byte<TD>(dr + k * dstride * sizeof(TD), e);
            }
        };
        // receiver rows of the tiles, one row further every round
        const TT *ro[NP];
        const RW *rp[NP], *rq[NP];
        TT orr_c[NP];
        RW pr_c[NP], qr_c[NP];
        auto load_rows = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                orr_c[j] = row_at(ro[j], (unsigned)lane);
                pr_c[j] = qr_c[j] = RW(0.0f);
                if constexpr (DYN) {
                    pr_c[j] = row_at(rp[j], (unsigned)lane);
                    qr_c[j] = row_at(rq[j], (unsigned)lane);
                }
            }
        };
        // receiver bases of the tiles and the gates of the block's traces,
        // kWave receivers at a time in the lanes
        int brv[NP], br[NP], izv[JB];
        auto load_bases = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < NP; ++j)
                brv[j] = a.base_r[(size_t)t[j] * a.nr + min(r0 + lane, a.nr - 1)];
            if constexpr (DYN && GATE)
#pragma unroll
                for (int i = 0; i < JB; ++i)
                    izv[i] = a.izmin[(size_t)min(s0 + part + P * i, a.ns - 1) * a.nr +
                                     min(r0 + lane, a.nr - 1)];
        };
        auto bases = [&](int k) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < NP; ++j)
                br[j] = __builtin_amdgcn_readlane(brv[j], k);
        };
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const size_t o = (size_t)t[j] * a.nr * kWave;
            ro[j] = offr + o;
            rp[j] = wpr + o;
            rq[j] = wqr + o;
        }
        load_rows();
        load_bases(0);
        bases(0);
        stage(br);
        for (int rc = 0; rc < a.nr; rc += kWave - 1) {
            if (rc > 0)
                load_bases(rc);
            const int rend = min(rc + kWave - 1, a.nr);
            for (int r = rc; r < rend; ++r) {
                // this round's pairs into the wave's LDS region; outside [0,
                // nt - 2] (the reference's 0 <= it < nt - 1) they are zero
                int ar[NP];
                const int mr = mr_n;
                if (lo + mr >= 0 && hi + mr + kWin <= a.nt) {
#pragma unroll
                    for (int i = 0; i < JB; ++i)
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            TP q;
                            q.v[0] = sv[k][i];
                            q.v[1] = next_minus(sv[k][i]);
                            w[k][i][lane] = q;
                        }
                } else {
#pragma unroll
                    for (int i = 0; i < JB; ++i)
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            const bool ok = (unsigned)(ms[i] + mr + lane) < ntm1;
                            const TD df = next_minus(sv[k][i]);
                            TP q;
                            q.v[0] = ok ? sv[k][i] : TD(0);
                            q.v[1] = ok ? df : TD(0);
                            w[k][i][lane] = q;
                        }
                }
                TC orr[NP];
                TD pr[NP], qr[NP];
#pragma unroll
                for (int j = 0; j < NP; ++j) {
                    orr[j] = (TC)ld_off(&orr_c[j]);
                    ar[j] = ar_n[j];
                    pr[j] = (TD)wv(pr_c[j]);
                    qr[j] = (TD)wv(qr_c[j]);
                }
                // next round's receiver side and samples, in flight meanwhile
                // (the same loads every round, as in gather_tiles: the last
                // round's are those of the last receiver again)
                {
                    const int more = r + 1 < a.nr;
#pragma unroll
                    for (int j = 0; j < NP; ++j) {
                        ro[j] += more * kWave;
                        rp[j] += more * kWave;
                        rq[j] += more * kWave;
                    }
                    dr += (size_t)more * a.nt * sizeof(TD);
                    load_rows();
                    bases(r + more - rc);
                    stage(br);
                    // (keeps the loads here: the compiler would move them to
                    // the top of the next round, where they are used)
                    asm volatile("" ::: "memory");
                }
#pragma unroll
                for (int i = 0; i < JB; ++i) {
#pragma unroll
                    for (int j = 0; j < NP; ++j) {
                        const TC T = os[i][j] + orr[j];
                        TC f;
                        int kf;
                        if constexpr (sizeof(TC) == 4) {
                            f = __builtin_amdgcn_fractf(T);
                            kf = floor_int(T);
                        } else {
                            const TC fl = floor(T);
                            f = T - fl;
                            kf = (int)fl;
                        }
                        const unsigned at = (unsigned)((kf << kPairShift) + (as[i][j] + ar[j]));
                        TD wgt = TD(1);
                        if constexpr (DYN) {
                            wgt = pair_weight(ps[i][j], pr[j], qs[i][j], qr[j]);
                            if (GATE && pt[j].iz < __builtin_amdgcn_readlane(izv[i], r - rc))
                                wgt = TD(0);
                        }
#pragma unroll
                        for (int k = 0; k < K; ++k) {
                            const Pair q =
                                *((LdsPair)(uintptr_t)(at + (unsigned)((k * JW + i) * kWin * sizeof(TP))));
                            TD v = fma((TD)f, q.y, q.x);
                            acc[k][j] = DYN ? fma(v, wgt, acc[k][j]) : acc[k][j] + v;
                        }
                    }
                }
            }
        }
    };
    if (active) {
        for (int s0 = 0; s0 < a.ns; s0 += SB) {
            // slots i with a source s0 + part + P i < ns
            const int nj = (a.ns - s0 - part + P - 1) / P;
            if (nj > JW / 2)
                source_block(IntC<JW>{}, s0);
            else if (nj > 0)
                source_block(IntC<(JW > 1 ? JW / 2 : 1)>{}, s0);
        }
    }
    gather_store<TD, P, NP, K>(a, acc, &win[0][0][0][0], m, mstride, part, wave, lane, active, tok,
                               pt);
}

}  // namespace
