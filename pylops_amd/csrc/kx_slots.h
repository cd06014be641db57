// kx_slots.h -- the forward's slot kernel (float32 operators): blocks of 8
// or 16 receivers whose LDS traces are interleaved, one LDS bank pair (16
// receivers) or two (8 receivers) per receiver.
#pragma once
#include "kx_device.h"

namespace {

// A 64-bit LDS atomic instruction is served in quarters of 16 lanes, each
// taking about max(1.5, L) clocks of its CU, L the most lanes of the quarter
// on one of the 16 bank pairs; lanes of different quarters never collide.
// With the traces of a block one after the other the samples of a quarter
// fall on random bank pairs: 12 clocks per instruction.  Here sample k of
// receiver j lies at (k RB + j) 8 bytes and lane l treats receiver l mod RB
// for every point, so that with RB = 16 the 16 lanes of a quarter hit 16
// different bank pairs whatever the samples are (6 clocks), and with RB = 8
// at most two lanes share one (8 clocks).
//
// The points move instead: lane l holds point l of the tile (its image
// value, source offset and source weights), and step i treats point i of the
// lane's run of RB consecutive points: a DPP row_newbcast hands the value of
// one lane to the 16 lanes of its row inside the instruction that uses it
// (RB = 16), or in two instructions with bank masks to either half of the row
// (RB = 8).  The receiver's entries of the RB points come from the
// slot-ordered copy of the table: 16-byte loads, contiguous over the lanes
// (read from the tiled table, 64 row parts per instruction, the 3D kernel
// took 18.8 ms where this order first took 12.4).  A receiver's base is one value per lane
// and tile.  A step is 11 (kinematic, RB = 16) to 17 (dynamic, RB = 8) vector
// instructions and two atomics, against about 17 and 20 with rows one after
// the other.
// Measured, forward with its wavelet: 3D 128x128x120 with 25 x 400, kinematic
// float32 15.7 to 10.4 ms (16.4 clocks of a CU per step; the vector
// instructions and the atomics take about 12 each, and either alone with the
// loads 13 to 14); 3D 93x77x101 with 12 x 195, float16 tables, 1.89 to 1.12
// ms; 2D 601x300 with 61 x 301, dynamic float32, RB = 8, 3.58 to 3.51 ms:
// bound by its loads (12 bytes per triplet through L1; without them 2.0 ms,
// without the atomics 3.5 ms).
constexpr int kSlotsMaxThreads = 1024;
// samples per thread of the conversion to float rows (held in registers
// between reading the sums and writing the rows over them)
constexpr int kSlotsHold = 20;

template <int N> __device__ __forceinline__ int row_bcast(int v)
{
    return __builtin_amdgcn_mov_dpp(v, 0x150 + N, 0xf, 0xf, true);
}
template <int N> __device__ __forceinline__ float row_bcast(float v)
{
    return __builtin_bit_cast(float, row_bcast<N>(__builtin_bit_cast(int, v)));
}

// Operations with the value of point N of the lane's run of RB points, v held
// by the lane of that point.  RB = 8: lanes 0-7 of a row take lane N, lanes
// 8-15 lane N + 8.  A DPP instruction must not read a register within two
// wait states of a vector instruction that wrote it.  The compiler sees to it
// for the builtin but does not look into the instructions written here, and
// may copy or reload their operands right before them: they wait themselves
// (601x300 with 61 x 301 traces, float32: dynamic 3.50 ms with one wait per
// tile ahead of all of them and 3.50 so, 3.54 with a wait for each of the
// three pairs; kinematic, three waits a step, 2.29 and 2.32).
#define KX_PAIR(OP, R, V, X, LO, HI)                                                           \
    OP "_dpp " R ", " V ", " X " row_newbcast:" LO " row_mask:0xf bank_mask:0x3\n\t" OP          \
       "_dpp " R ", " V ", " X " row_newbcast:" HI " row_mask:0xf bank_mask:0xc"
#define KX_HALF2(OP) "s_nop 1\n\t" KX_PAIR(OP, "%0", "%1", "%2", "%3", "%4")
template <int RB, int N> __device__ __forceinline__ float point_add(float v, float x)
{
    if constexpr (RB == 16)
        return row_bcast<N>(v) + x;
    float r;
    asm(KX_HALF2("v_add_f32") : "=&v"(r) : "v"(v), "v"(x), "n"(N), "n"(N + 8));
    return r;
}
template <int RB, int N> __device__ __forceinline__ float point_mul(float v, float x)
{
    if constexpr (RB == 16)
        return row_bcast<N>(v) * x;
    float r;
    asm(KX_HALF2("v_mul_f32") : "=&v"(r) : "v"(v), "v"(x), "n"(N), "n"(N + 8));
    return r;
}
// T = ov + ox and w = pv px + qv qx, ov, pv and qv those of the point (the
// three pairs share one wait: none writes what another broadcasts)
template <int RB, int N>
__device__ __forceinline__ void point_time_weight(float ov, float ox, float pv, float px, float qv,
                                                  float qx, float &T, float &w)
{
    if constexpr (RB == 16) {
        T = row_bcast<N>(ov) + ox;
        w = fmaf(row_bcast<N>(qv), qx, row_bcast<N>(pv) * px);
    } else {
        asm("s_nop 1\n\t" KX_PAIR("v_add_f32", "%0", "%2", "%3", "%8", "%9") "\n\t"
            KX_PAIR("v_mul_f32", "%1", "%4", "%5", "%8", "%9") "\n\t"
            KX_PAIR("v_fmac_f32", "%1", "%6", "%7", "%8", "%9")
            : "=&v"(T), "=&v"(w)
            : "v"(ov), "v"(ox), "v"(pv), "v"(px), "v"(qv), "v"(qx), "n"(N), "n"(N + 8));
    }
}
template <int RB, int N> __device__ __forceinline__ int point_sub(int v, int x)
{
    if constexpr (RB == 16)
        return row_bcast<N>(v) - x;
    int r;
    asm(KX_HALF2("v_sub_u32") : "=&v"(r) : "v"(v), "v"(x), "n"(N), "n"(N + 8));
    return r;
}
template <int RB, int N> __device__ __forceinline__ int point_value(int v)
{
    if constexpr (RB == 16)
        return row_bcast<N>(v);
    const int lo = __builtin_amdgcn_mov_dpp(v, 0x150 + N, 0xf, 0xf, true);
    return __builtin_amdgcn_update_dpp(lo, v, 0x150 + (N & 7) + 8, 0xf, 0xc, false);
}
#undef KX_HALF2
#undef KX_PAIR

// A chunk of consecutive points' entries of one receiver.
template <typename TT, typename RW, bool DYN> struct SlotChunk {
    static constexpr int n = SlotChunkLen<TT>::v;
    VecN<TT, n> o;
    VecN<RW, DYN ? n : 1> p, q;
};

// A lane's own point of a tile and its receiver's base.
struct SlotPoint {
    float mv, os, ps, qs;
    int bs, br;  // source and receiver base
    int iz;      // depth index of the lane's point
};

typedef unsigned Words4 __attribute__((ext_vector_type(4)));

// What a lane needs to know to load its tiles.
struct SlotLane {
    int lz, lx, ly;     // the lane's point in a tile
    unsigned rel;       // its image offset from the tile's first point
    unsigned lane, r, run;  // run: the lane's first element in a block of 16
    int s, nb16, b16, vz;
};

template <bool DYN>
__device__ __forceinline__ void slot_load_point(const KArgs &a, const TileCursor &c,
                                                const SlotLane &l, const float *__restrict__ m,
                                                SlotPoint &P)
{
    const int z0 = c.tzi * a.tz, x0 = c.txi * a.tx, y0 = c.tyi * a.ty;
    const bool valid = (l.lz < a.nz - z0) & (l.lx < a.nx - x0) & (l.ly < a.ny - y0);
    const float mval = scalar_ptr(m + ((int64_t)(y0 * a.nx + x0) * a.nz + z0))[valid ? l.rel : 0u];
    P.mv = valid ? mval : 0.f;
    const size_t ts = (size_t)c.t * a.ns + l.s;
    P.os = scalar_ptr(reinterpret_cast<const float *>(a.off_s) + ts * kWave)[l.lane];
    if constexpr (DYN) {
        P.ps = scalar_ptr(reinterpret_cast<const float *>(a.wp_s) + ts * kWave)[l.lane];
        P.qs = scalar_ptr(reinterpret_cast<const float *>(a.wq_s) + ts * kWave)[l.lane];
    }
    P.bs = scalar_ptr(a.base_s + ts)[(unsigned)l.vz];
    P.br = scalar_ptr(a.base_r + (size_t)c.t * a.nr)[l.r];
    P.iz = z0 + l.lz;
}

// Chunk C of the lane's run in tile t.
template <typename TT, bool DYN>
__device__ __forceinline__ void slot_load_chunk(const KArgs &a, int t, const SlotLane &l, int C,
                                                SlotChunk<TT, typename RecW<float, TT>::type, DYN> &K)
{
    using RW = typename RecW<float, TT>::type;
    constexpr int n = SlotChunkLen<TT>::v;
    static_assert(sizeof(RW) == sizeof(TT), "weights and offsets share one chunk length");
    // behind the tiled table
    const int64_t at =
        ((int64_t)a.ntiles * a.nr + ((int64_t)t * l.nb16 + l.b16) * kSlotBlock) * kWave;
    const unsigned e = (l.run + C * 64 * n) / n;  // in 16-byte chunks
    auto chunk = [&](const void *p) __attribute__((always_inline)) {
        return scalar_ptr(
            reinterpret_cast<const Words4 *>(reinterpret_cast<const TT *>(p) + at))[e];
    };
    K.o = __builtin_bit_cast(VecN<TT, n>, chunk(a.off_r));
    if constexpr (DYN) {
        K.p = __builtin_bit_cast(VecN<RW, n>, chunk(a.wp_r));
        K.q = __builtin_bit_cast(VecN<RW, n>, chunk(a.wq_r));
    }
}

// Adds w0 and w1 to two neighbouring samples (byte address at of the first)
// of the lanes in `on`; every lane of the wave is active.  As a branch the
// two atomics cost four scalar instructions.  (The compiler does not count
// these LDS operations: slots_body waits for them itself.)
template <int RB>
__device__ __forceinline__ void slot_add(uint64_t on, unsigned at, long long w0, long long w1)
{
    asm volatile("s_mov_b64 exec, %0\n\t"
                 "ds_add_u64 %1, %2\n\t"
                 "ds_add_u64 %1, %3 offset:%4\n\t"
                 "s_mov_b64 exec, -1"
                 :
                 : "s"(on), "v"(at), "v"(w0), "v"(w1), "i"(RB * 8)
                 : "memory");
}

// Point N of the run: its two samples of this lane's receiver.  os, mv (and
// W, its rounding), mps, mqs and iz belong to the lane's own point.
template <typename TT, typename RW, bool DYN, bool GATE, bool NEG, int ACC, int RB, int N>
__device__ __forceinline__ void slot_point(const SlotChunk<TT, RW, DYN> &K, float os, float mv,
                                           int W, float mps, float mqs, int iz, int base,
                                           int izm, unsigned ntm1, int j, int lane_base, void *lds)
{
    constexpr int u = N % SlotChunkLen<TT>::v;
    // (broadcasts outside any branch: a lane switched off hands out nothing)
    float T, w = 0.f, w1;
    if constexpr (DYN)
        point_time_weight<RB, N>(os, ld_off(&K.o.v[u]), mps, wv(K.p.v[u]), mqs, wv(K.q.v[u]), T, w);
    else
        T = point_add<RB, N>(os, ld_off(&K.o.v[u]));
    const int pz = DYN && GATE ? point_value<RB, N>(iz) : 0;
    float f;
    int k;
    if constexpr (!NEG) {
        f = __builtin_amdgcn_fractf(T);
        k = floor_int(T) + base;
    } else {
        const float fl = floorf(T);
        f = T - fl;
        k = (int)fl + base;
        if (k == -1 && f > 0.f) {
            k = 0;
            f -= 1.f;
        }
    }
    if constexpr (DYN) {
        w1 = w * f;
    } else {
        w1 = point_mul<RB, N>(mv, f);
        if constexpr (ACC != kAccFix)
            w = __builtin_bit_cast(float, point_value<RB, N>(__builtin_bit_cast(int, mv)));
    }
    bool on = (unsigned)k < ntm1;
    if constexpr (DYN && GATE)
        on = on && pz >= izm;
    if constexpr (ACC == kAccFix) {
        const int i1 = round_half_up(w1);
        const int i0 = DYN ? round_half_up(w) - i1 : point_sub<RB, N>(W, i1);
        slot_add<RB>(__ballot(on), (unsigned)((k << (RB == 16 ? 7 : 6)) + lane_base),
                     (long long)i0, (long long)i1);
    } else {
        const float w0 = w * (1.f - f);
        if (on && w != 0.f) {
            double *acc = static_cast<double *>(lds) + (k * RB + j);
            atomicAdd(acc, (double)w0);
            atomicAdd(acc + RB, (double)w1);
        }
    }
}

// Where a slot workgroup's sums go: convolved with the nh-tap wavelet h into
// the traces of y, as traces (h NULL), or as they are into `sums` (not NULL;
// slots_final_kernel adds the parts of a block and finishes).
struct SlotsOut {
    float *y;
    const float *h;
    int nh;
    unsigned long long *sums;
};

// Tiles [t0, t1) of source s and receivers [r0, r0 + RB).
template <typename TT, bool DYN, bool GATE, bool NEG, int ACC, int RB>
__device__ __forceinline__ void slots_body(const KArgs &a, const float *__restrict__ m, int e,
                                           int s, int r0, int t0, int t1, const SlotsOut &out)
{
    extern __shared__ __align__(16) unsigned char kx_smem[];
    void *lds = kx_smem;
    using RW = typename RecW<float, TT>::type;
    constexpr int CH = SlotChunkLen<TT>::v;
    constexpr int NC = RB / CH;  // chunks of a run

    const int nrl = min(RB, a.nr - r0);
    const int nsum = a.nt * RB;
    {
        unsigned long long *p = static_cast<unsigned long long *>(lds);
        for (int i = threadIdx.x; i < nsum; i += blockDim.x)
            p[i] = 0ull;
    }
    __syncthreads();

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int nw = blockDim.x / kWave;
    const int j = lane & (RB - 1);
    // slots past the last receiver repeat it and are not written out
    const int r = r0 + min(j, nrl - 1);
    SlotLane l;
    l.lz = lane % a.tz;
    l.lx = (lane / a.tz) % a.tx;
    l.ly = lane / (a.tz * a.tx);
    l.rel = (unsigned)((l.ly * a.nx + l.lx) * a.nz + l.lz);
    l.lane = (unsigned)lane;
    l.r = (unsigned)r;
    // the lane's chunks in a block of 16: row group lane / 16, and with
    // RB = 8 the second half of the chunks for the upper half of a row
    l.run = (unsigned)((((RB == 8 ? ((lane >> 3) & 1) * NC * 4 : 0) + (lane >> 4)) * 16 +
                        (r0 & (kSlotBlock - 1)) + j) *
                       CH);
    l.s = s;
    l.nb16 = slot_blocks(a.nr);
    l.b16 = r0 / kSlotBlock;
    l.vz = vgpr_zero();
    const size_t first = (size_t)s * a.trs + (size_t)r0 * a.trb;  // trace of slot 0
    const int izm = DYN && GATE ? a.izmin[first + (size_t)(r - r0) * a.trb] : 0;
    const unsigned ntm1 = (unsigned)(a.nt - 1);
    const int lane_base =
        (int)(unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)kx_smem + j * 8;

    // Two tile buffers in turn, each chunk loaded again for the tile two
    // steps of the wave ahead as soon as this tile's is used (float16 tables:
    // 3D 93x77x101 with 12 x 195 8% faster than one buffer; float32 dynamic
    // blocks of 16 have registers for one).  Past the last tile the last one
    // loaded is loaded again, unused.
    constexpr int NBUF = DYN && RB == 16 && sizeof(TT) == 4 ? 1 : 2;
    SlotChunk<TT, RW, DYN> K0[NC], K1[NC];
    SlotPoint P0, P1;
    TileCursor c0, c1, cl;
    auto load_all = [&](const TileCursor &c, SlotPoint &P, SlotChunk<TT, RW, DYN>(&K)[NC])
        __attribute__((always_inline)) {
        slot_load_point<DYN>(a, c, l, m, P);
#pragma unroll
        for (int q = 0; q < NC; ++q)
            slot_load_chunk<TT, DYN>(a, c.t, l, q, K[q]);
    };
    // the tile at c in (P, K), then both filled for the tile 2 nw ahead
    auto tile = [&](TileCursor &c, SlotPoint &P, SlotChunk<TT, RW, DYN>(&K)[NC])
        __attribute__((always_inline)) {
        TileCursor cn = c;
        cn.advance(a, NBUF * nw);
        const bool more = cn.t < t1;  // (field by field: a chosen address would go to scratch)
        cl.t = more ? cn.t : cl.t;
        cl.tzi = more ? cn.tzi : cl.tzi;
        cl.txi = more ? cn.txi : cl.txi;
        cl.tyi = more ? cn.tyi : cl.tyi;
        const bool any = c.t < t1 && __ballot(P.mv != 0.f) != 0;
        float mv = P.mv;
        const float os = P.os;
        const int base = P.bs + P.br;
        if constexpr (ACC == kAccFix)
            mv = ldexpf(mv, e);
        const int W = ACC == kAccFix && !DYN ? round_half_up(mv) : 0;
        float mps = 0.f, mqs = 0.f;
        if constexpr (DYN) {
            mps = mv * P.ps;
            mqs = mv * P.qs;
        }
#define KX_SLOT(C, I)                                                                          \
    if constexpr (I < CH)                                                                      \
    slot_point<TT, RW, DYN, GATE, NEG, ACC, RB, CH * C + (I < CH ? I : 0)>(                     \
        K[C], os, mv, W, mps, mqs, P.iz, base, izm, ntm1, j, lane_base, lds)
#define KX_CHUNK(C)                                                                            \
    if constexpr (C < NC) {                                                                    \
        if (any) {                                                                             \
            KX_SLOT(C, 0);                                                                     \
            KX_SLOT(C, 1);                                                                     \
            KX_SLOT(C, 2);                                                                     \
            KX_SLOT(C, 3);                                                                     \
            KX_SLOT(C, 4);                                                                     \
            KX_SLOT(C, 5);                                                                     \
            KX_SLOT(C, 6);                                                                     \
            KX_SLOT(C, 7);                                                                     \
        }                                                                                      \
        slot_load_chunk<TT, DYN>(a, cl.t, l, C, K[C]);                                         \
    }
        KX_CHUNK(0)
        KX_CHUNK(1)
        KX_CHUNK(2)
        KX_CHUNK(3)
#undef KX_CHUNK
#undef KX_SLOT
        slot_load_point<DYN>(a, cl, l, m, P);
        c = cn;
    };
    c0.start(a, t0 + wave);
    if (c0.t < t1) {
        cl = c1 = c0;
        load_all(c0, P0, K0);
        if constexpr (NBUF == 2) {
            c1.advance(a, nw);
            if (c1.t < t1)
                cl = c1;
            load_all(cl, P1, K1);
        }
        while (c0.t < t1) {
            tile(c0, P0, K0);
            if constexpr (NBUF == 2)
                tile(c1, P1, K1);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // slot_add's
    __syncthreads();  // every contribution added

    const unsigned long long *acci = static_cast<const unsigned long long *>(lds);
    const double *accd = static_cast<const double *>(lds);
    auto value = [&](int i) -> float {
        if constexpr (ACC == kAccF64)
            return (float)accd[i];
        else
            return (float)ldexp((double)(long long)acci[i], -e);
    };
    if (out.sums != nullptr) {
        for (int i = threadIdx.x; i < nsum; i += blockDim.x)
            out.sums[i] = acci[i];
    } else if (out.h == nullptr) {
        float *yo = out.y + first * a.nt;
        for (int i = threadIdx.x; i < nrl * a.nt; i += blockDim.x) {
            const int jr = i / a.nt, n = i - jr * a.nt;
            yo[(size_t)jr * a.trb * a.nt + n] = value(n * RB + jr);
        }
    } else {
        // the sums of the whole block into registers, then float rows over
        // them, convolved as the other forward kernels convolve theirs
        float v[kSlotsHold];
        const int S = fused_row(a.nt, out.nh), L = (out.nh - 1) / 2;
        float *win = static_cast<float *>(lds);
#pragma unroll
        for (int q = 0; q < kSlotsHold; ++q) {
            const int i = q * (int)blockDim.x + (int)threadIdx.x;
            if (i < nsum)
                v[q] = value(i);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kSlotsHold; ++q) {
            const int i = q * (int)blockDim.x + (int)threadIdx.x;
            if (i < nsum && (i & (RB - 1)) < nrl)
                win[(i & (RB - 1)) * S + L + i / RB] = v[q];
        }
        rows_conv_store(win, out.y, first, a.trb, a.nt, nrl, out.h, out.nh);
    }
    __syncthreads();  // read out before a next item clears the traces
}

// One item with the launch's accumulation scale.
template <typename TT, bool DYN, bool GATE, bool NEG, int RB>
__device__ __forceinline__ void slots_item(const KArgs &a, const float *__restrict__ m,
                                           const SpreadScale &sc, int s, int r0, int t0, int t1,
                                           const SlotsOut &out)
{
    if (sc.fixed)
        slots_body<TT, DYN, GATE, NEG, kAccFix, RB>(a, m, sc.e, s, r0, t0, t1, out);
    else
        slots_body<TT, DYN, GATE, NEG, kAccF64, RB>(a, m, 0, s, r0, t0, t1, out);
}

// LDS of a slot workgroup: the sums, or the float rows with the filter
inline size_t slots_lds_bytes(int rb, int nt, int nh)
{
    const size_t sums = (size_t)rb * nt * 8;
    const size_t rows = nh > 0 ? ((size_t)rb * fused_row(nt, nh) + conv_taps_padded(nh)) * 4 : 0;
    return sums > rows ? sums : rows;
}
// Threads of a slot workgroup: 8 waves where two workgroups share a CU's
// LDS, 16 where one fills it; 0 when the block does not fit.
inline int slots_threads(int rb, int nt, int nh)
{
    const size_t lds = slots_lds_bytes(rb, nt, nh);
    if (lds > lds_budget())
        return 0;
    const int th = 2 * lds <= lds_budget() ? kSlotsMaxThreads / 2 : kSlotsMaxThreads;
    return (int64_t)rb * nt <= (int64_t)kSlotsHold * th ? th : 0;
}

}  // namespace
