// fused_tiles.hpp -- the row and column tiles of the fused 2D step: what one
// workgroup does to a few rows or columns of one instance (the pipeline and
// its buffers are described in fused.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "fft_core.hpp"
#include "fused.hpp"
#include "philox.hpp"
#include "update_math.hpp"

namespace cupss {

// ------------------------------------------------------------ row tile

// MAXR: real fields a row holds at once (2, 3, or FUSED_MAX_REAL for systems
// with more; those use 4 elements per lane to stay within the registers).
//
// Elements per lane (E) of rows and columns.  On a small grid a wavefront is
// alone on its SIMD and bound by the issue of its own instructions: fewer
// elements a lane, that is more wavefronts, are faster as long as a line
// stays inside one wavefront.  Many instances at once prefer fewer exchanges.
// us per step with 8 -> 4 elements on rows of 64 and 128 complex points and
// columns of 128 and 256 points: CH 256^2 10.2 -> 8.3, KPZ 128^2 16.3 -> 12.5,
// Gray-Scott 256^2 20.2 -> 16.2, model H 256^2 39.7 -> 36.1, 16 of Gray-Scott
// 256^2 26.6 -> 22.1; 64 of them 54 -> 57, 64 of a three-field system 256^2
// 46.8 -> 50, 512 EW/KPZ instances of 64^2 .. 512^2 170 -> 174, CH 256^3
// 156 -> 161.  The elements set the order of a line's stages, so they cannot
// follow the number of instances: a system has the same bits in any batch.  Rows of 256
// complex points stay at 8 (with 4: KPZ 512^2 20.3 -> 17.7, but the 512
// instances 170 -> 183), and so do columns of 512 (with 4, two wavefronts
// each: 18.3 and 188).  Longer lines take 4 over several wavefronts: 1024-point
// columns of 16 in one wavefront take CH 1024^2 from 16.4 to 18.7 and model H
// 1024^2 from 69 to 83.
//
// Tile row stride: at least lds_len(nc), since each row's transform works
// in place, and chosen for the LDS banks (32 of 4 bytes; a store is served
// 16 lanes at a time, a load 32).  A tile copy moves row pairs: the 16
// lanes of a store cover LPB/2 pairs, 32/(LPB/2) dwords of each, and
// successive pairs lie 4*RS dwords apart, so the runs interleave without
// sharing a bank when RS is odd (LPB 16), 2 mod 4 (LPB 8) or 4 mod 8 (LPB 4).
__host__ __device__ constexpr int tile_stride(int nc, int lpb)
{
    int rs = lds_len(nc);
    if (lpb == 16)
        while (rs % 2 != 1) rs++;
    else if (lpb == 8)
        while (rs % 4 != 2) rs++;
    else if (lpb == 4)
        while (rs % 8 != 4) rs++;
    return rs;
}

template <int NC, int LPB, int MAXR = 3, bool SINGLE = false>
struct FRowCfg {
    static constexpr int E = MAXR > 3 ? (NC >= 4 ? 4 : NC) : (NC >= 1024 ? 16 : (NC == 256 ? 8 : (NC >= 4 ? 4 : NC)));
    static constexpr int T = NC / E;
    static constexpr int THREADS = LPB * T;
    static constexpr int RS = tile_stride(NC, LPB);
    // Two fields, and two products, at a time through their transforms: half
    // the barriers of a line over several wavefronts and one line's LDS
    // latency under the other's butterflies.  us per step, Gray-Scott 64^2
    // 16.7 -> 16.3, 128^2 15.9 -> 15.5, 256^2 16.7 -> 16.2, 512^2 24.2 -> 23.5,
    // 1024x512 25.8 -> 25.2, and the same gain in batches of up to 256 of the
    // short rows.  Launches of many long rows take them singly (SINGLE, with
    // the same bits), see frows_n.  Not the wide kernel, whose LDS and
    // registers are the limit of a batch: model H 1024^2 alone 64.7 -> 63.8,
    // but a mixed batch 122 -> 128.  Not 16 elements a lane (registers).
    static constexpr bool PAIR = !SINGLE && MAXR > 1 && MAXR <= 3 && E <= 8;
    static constexpr int LEN = (PAIR ? 2 : 1) * LPB * RS;
    static constexpr bool valid()
    {
        return THREADS >= 16 && THREADS <= 512 && (LEN + 2 * NC + tw_stage_alloc(NC, E)) * 8 <= 150 * 1024;
    }
};

// four floats as one 16-byte access (a native vector: HIP's float4 copies
// through a generic pointer, which would make the access flat)
typedef float vf4 __attribute__((ext_vector_type(4)));

// rows y0 .. y0+LPB-1 of a column-major half spectrum into the tile (row l
// at l*RS, entry k at k); columns k > kmax read as zero.  Pairs of rows are
// moved with one 16-byte access.  issue() starts a thread's loads (all at
// once where it has at most CH), commit() writes them to the tile (and does
// the whole copy in rounds of CH loads where there are more), so that the
// loads are in flight together instead of one round trip each.
template <int NC, int LPB, int RS, int TH, int CH = 4>
struct TileLoad {
    static constexpr int HP = LPB / 2;
    static constexpr int ITEMS = (NC + 1) * (LPB >= 2 ? HP : 1);
    static constexpr int IT = (ITEMS + TH - 1) / TH;
    static constexpr bool ONE = IT <= CH;
    vf4 w[ONE ? IT : 1];
    __device__ __forceinline__ vf4 item(const float2 *__restrict__ src, int sy, int y0, int kmax, int i) const
    {
        vf4 v = {0.f, 0.f, 0.f, 0.f};
        if constexpr (LPB >= 2) {
            const int k = i / HP, yl = 2 * (i % HP);
            if (k <= kmax) v = gload(reinterpret_cast<const vf4 *>(src + (long)k * sy + y0 + yl), 0);
        } else {
            if (i <= kmax) {
                const float2 z = gload(src, (long)i * sy + y0);
                v.x = z.x;
                v.y = z.y;
            }
        }
        return v;
    }
    __device__ __forceinline__ void put(float2 *__restrict__ tile, int i, vf4 v) const
    {
        if constexpr (LPB >= 2) {
            const int k = i / HP, yl = 2 * (i % HP);
            tile[yl * RS + k] = make_float2(v.x, v.y);
            tile[(yl + 1) * RS + k] = make_float2(v.z, v.w);
        } else {
            tile[i] = make_float2(v.x, v.y);
        }
    }
    __device__ __forceinline__ void issue(const float2 *__restrict__ src, int sy, int y0, int kmax)
    {
        if constexpr (ONE) {
#pragma unroll
            for (int p = 0; p < IT; p++) {
                const int i = threadIdx.x + p * TH;
                if (i < ITEMS) w[p] = item(src, sy, y0, kmax, i);
            }
        }
    }
    __device__ __forceinline__ void commit(float2 *__restrict__ tile, const float2 *__restrict__ src, int sy, int y0,
                                           int kmax)
    {
        if constexpr (ONE) {
#pragma unroll
            for (int p = 0; p < IT; p++) {
                const int i = threadIdx.x + p * TH;
                if (i < ITEMS) put(tile, i, w[p]);
            }
        } else {
#pragma unroll
            for (int p0 = 0; p0 < IT; p0 += CH) {
                vf4 v[CH];
#pragma unroll
                for (int q = 0; q < CH; q++) {
                    const int i = threadIdx.x + (p0 + q) * TH;
                    if (p0 + q < IT && i < ITEMS) v[q] = item(src, sy, y0, kmax, i);
                }
#pragma unroll
                for (int q = 0; q < CH; q++) {
                    const int i = threadIdx.x + (p0 + q) * TH;
                    if (p0 + q < IT && i < ITEMS) put(tile, i, v[q]);
                }
            }
        }
    }
};

template <int NC, int LPB, int RS, int TH>
__device__ __forceinline__ void tile_store(float2 *__restrict__ dst, const float2 *__restrict__ tile, int sy, int y0)
{
    if constexpr (LPB >= 2) {
        constexpr int HP = LPB / 2;
        for (int i = threadIdx.x; i < (NC + 1) * HP; i += TH) {
            const int k = i / HP, yl = 2 * (i % HP);
            const float2 a = tile[yl * RS + k], b = tile[(yl + 1) * RS + k];
            const vf4 w = {a.x, a.y, b.x, b.y};
            gstore(reinterpret_cast<vf4 *>(dst + (long)k * sy + y0 + yl), 0, w);
        }
    } else {
        for (int k = threadIdx.x; k <= NC; k += TH) gstore(dst, (long)k * sy + y0, tile[k]);
    }
}

// C2R pre-processing: Z'[k] from X[k] and X[NC-k]; the imaginary parts of
// the self-conjugate bins k = 0, NC are dropped (real-part projection)
template <int NC, int E, int T>
__device__ __forceinline__ void c2r_prep(const float2 (&xa)[E], const float2 (&ya)[E], int t, float2 (&v)[E],
                                         const float2 *tws)
{
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int k = t + e * T;
        float2 X = xa[e], Y = ya[e];
        if (k == 0) {
            X.y = 0.f;
            Y.y = 0.f;
        }
        const float2 Yc = cconj(Y);
        const float2 xe = cadd(X, Yc);
        const float2 xo = cmul(csub(X, Yc), tw_lookup<+1, 2 * NC>(tws, k, 2 * NC));
        v[e] = cadd(xe, mul_i<+1>(xo));
    }
}

// The tiles must give the same bits in every kernel that inlines them (any
// tile shape, one workgroup or many, a run resumed by another kernel), but
// which products the compiler fuses into which additions depends on the code
// around them: values pass opaquely in and out of a transform where that was
// seen to differ (rows of 16 elements a lane; the lean tiles).
template <int E>
__device__ __forceinline__ void opaque(float2 (&v)[E])
{
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int e = 0; e < E; e++) asm("" : "+v"(v[e].x), "+v"(v[e].y));
#endif
}

// R2C of one row whose real values are packed as v[e] = (x[2m], x[2m+1]);
// the NC+1 bins are left in L[0..NC] (unpadded).  Ends with a barrier.
// tws: the 2NC-point table (post-twiddles); the NC-point transform takes
// its twiddles from ftw (TWF = TW_STAGE: the stage tables, else tws).
template <int NC, int E, int T, int TWF>
__device__ __forceinline__ void r2c_tile(float2 (&v)[E], float2 *L, int t, const float2 *tws, const float2 *ftw)
{
    fft_line<NC, E, -1, TWF, true, (T <= 64)>(v, L, t, ftw);
    float2 o[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int k = t + e * T;
        const float2 A = v[e];
        const float2 B = cconj(L[lpad((NC - k) & (NC - 1))]);
        const float2 xe = cscale(cadd(A, B), 0.5f);
        const float2 xo = cscale(mul_i<-1>(csub(A, B)), 0.5f);
        o[e] = k == 0 ? make_float2(xe.x + xo.x, 0.0f) : cadd(xe, cmul(tw_lookup<-1, 2 * NC>(tws, k, 2 * NC), xo));
    }
    const float2 z0 = L[lpad(0)];
    line_sync<(T <= 64)>();  // every read of the transform's LDS line is done
#pragma unroll
    for (int e = 0; e < E; e++) L[t + e * T] = o[e];
    if (t == 0) L[NC] = make_float2(z0.x - z0.y, 0.0f);
    __syncthreads();
}

// r2c_tile of two rows, the second's LDS ls entries behind the first's
template <int NC, int E, int T>
__device__ __forceinline__ void r2c_pair(float2 (&v)[2][E], float2 *L, int ls, int t, const float2 *tws,
                                         const float2 *ftw)
{
    fft_pair<NC, E, -1, true, (T <= 64)>(v, L, ls, t, ftw);
    float2 o[2][E], z0[2];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int k = t + e * T;
        const float2 tw = tw_lookup<-1, 2 * NC>(tws, k, 2 * NC);
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const float2 A = v[m][e];
            const float2 B = cconj(L[m * ls + lpad((NC - k) & (NC - 1))]);
            const float2 xe = cscale(cadd(A, B), 0.5f);
            const float2 xo = cscale(mul_i<-1>(csub(A, B)), 0.5f);
            o[m][e] = k == 0 ? make_float2(xe.x + xo.x, 0.0f) : cadd(xe, cmul(tw, xo));
        }
    }
#pragma unroll
    for (int m = 0; m < 2; m++) z0[m] = L[m * ls + lpad(0)];
    line_sync<(T <= 64)>();  // every read of the transforms' LDS lines is done
#pragma unroll
    for (int m = 0; m < 2; m++) {
#pragma unroll
        for (int e = 0; e < E; e++) L[m * ls + t + e * T] = o[m][e];
        if (t == 0) L[m * ls + NC] = make_float2(z0[m].x - z0[m].y, 0.0f);
    }
    __syncthreads();
}

// Rows y0 .. y0+LPB-1 of one instance (the whole workgroup).  load_tw:
// copy the twiddle tables into tws (2NC points) and tst (the NC-point
// transform's stage tables) first (otherwise they are there already).
// Ends with a workgroup barrier: the tile and the rows written are free.
template <int NC, int LPB, int MAXR, bool SINGLE = false>
__device__ __forceinline__ void frows_tile(const FusedInst &a, int y0, uint32_t step_rel,
                                           const float2 *__restrict__ sets, bool load_tw, float2 *tws, float2 *tst,
                                           float2 *tile)
{
    using C = FRowCfg<NC, LPB, MAXR, SINGLE>;
    constexpr int E = C::E, T = C::T, RS = C::RS, TH = C::THREADS;
    static_assert(T % 2 == 0 && E % 2 == 0, "noise lanes are paired");
    const int sy = a.g.sy;
    const int l = threadIdx.x / T, t = threadIdx.x % T;
    float2 *L = tile + l * RS;
    const int nreal = a.nreal;
    // twiddle loads first, then the first tile's: their stores then wait
    // for the twiddles only
    SizeTwiddles<2 * NC, TH> twl;
    StageTwiddles<NC, E, TH> tsl;
    if (load_tw) {
        twl.load(sets);
        tsl.load(sets);
    }

    // Fields one by one or in pairs (FRowCfg::PAIR).  The next fields' loads
    // are in flight during a transform (model H 1024^2, five fields: 28.1 ->
    // 27.2 us).
    constexpr int P = C::PAIR ? 2 : 1, TS = LPB * RS;
    float2 r[MAXR][E];
    TileLoad<NC, LPB, RS, TH> tl[P];
#pragma unroll
    for (int m = 0; m < P; m++)
        if (m < nreal) tl[m].issue(a.Z[m], sy, y0, a.kmax[m]);
#pragma unroll
    for (int f = 0; f < MAXR; f += P) {
        if (f < nreal) {
            const bool two = P == 2 && f + 1 < MAXR && f + 1 < nreal;
            if (f == 0 && load_tw) {
                twl.store(tws, sets);
                tsl.store(tst, sets);
            }
            tl[0].commit(tile, a.Z[f], sy, y0, a.kmax[f]);
            if constexpr (P == 2)
                if (two) tl[1].commit(tile + TS, a.Z[f + 1], sy, y0, a.kmax[f + 1]);
            __syncthreads();
#pragma unroll
            for (int m = 0; m < P; m++)
                if (f + P + m < MAXR && f + P + m < nreal) tl[m].issue(a.Z[f + P + m], sy, y0, a.kmax[f + P + m]);
            float2 v[P][E];
#pragma unroll
            for (int m = 0; m < P; m++) {
                if (m == 0 || two) {
                    float2 xa[E], ya[E];
#pragma unroll
                    for (int e = 0; e < E; e++) {
                        const int k = t + e * T;
                        xa[e] = L[m * TS + k];
                        ya[e] = L[m * TS + NC - k];
                    }
                    c2r_prep<NC, E, T>(xa, ya, t, v[m], tws);
                }
            }
            // the row's part of the tile becomes its transform's LDS (the
            // row's lanes are the only ones that read or write it from here)
            line_sync<(T <= 64)>();
            if constexpr (E > 8) opaque(v[0]);
            if constexpr (P == 2) {
                if (two)
                    fft_pair<NC, E, +1, false, (T <= 64)>(v, L, TS, t, tst);
                else
                    fft_line<NC, E, +1, TW_STAGE, false, (T <= 64)>(v[0], L, t, tst);
            } else {
                fft_line<NC, E, +1, TW_STAGE, false, (T <= 64)>(v[0], L, t, tst);
            }
#pragma unroll
            for (int m = 0; m < P; m++)
                if (f + m < MAXR && (m == 0 || two)) {
                    if constexpr (E > 8) opaque(v[m]);
#pragma unroll
                    for (int e = 0; e < E; e++) r[f + m < MAXR ? f + m : 0][e] = cscale(v[m][e], a.scale);
                }
            __syncthreads();
        }
    }
    if (nreal == 0) {
        if (load_tw) {
            twl.store(tws, sets);
            tsl.store(tst, sets);
        }
        __syncthreads();  // twiddles
    }
    // v = group gi's products: coef * prod_f r_f^cnt_f (static field index,
    // uniform powers: no dynamic indexing, so r stays in registers)
    auto products = [&](int gi, float2(&v)[E]) {
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = make_float2(0.f, 0.f);
        for (int pi = a.pg0[gi]; pi < a.pg0[gi + 1]; pi++) {
            float2 p[E];
            const float c0 = a.coef[pi];
#pragma unroll
            for (int e = 0; e < E; e++) p[e] = make_float2(c0, c0);
#pragma unroll
            for (int f = 0; f < MAXR; f++)
                for (int c = 0; c < a.cnt[pi][f]; c++) {
#pragma unroll
                    for (int e = 0; e < E; e++) {
                        p[e].x *= r[f][e].x;
                        p[e].y *= r[f][e].y;
                    }
                }
#pragma unroll
            for (int e = 0; e < E; e++) v[e] = cadd(v[e], p[e]);
        }
    };
    int gi = 0;
    if constexpr (P == 2)
        for (; gi + 1 < a.ngroups; gi += 2) {
            float2 v[2][E];
            products(gi, v[0]);
            products(gi + 1, v[1]);
            r2c_pair<NC, E, T>(v, L, TS, t, tws, tst);
            tile_store<NC, LPB, RS, TH>(a.X[gi], tile, sy, y0);
            tile_store<NC, LPB, RS, TH>(a.X[gi + 1], tile + TS, sy, y0);
            __syncthreads();
        }
    for (; gi < a.ngroups; gi++) {
        float2 v[E];
        products(gi, v);
        if constexpr (E > 8) opaque(v);
        r2c_tile<NC, E, T, TW_STAGE>(v, L, t, tws, tst);
        tile_store<NC, LPB, RS, TH>(a.X[gi], tile, sy, y0);
        __syncthreads();
    }
    // real-space noise of phi (source -1) and of the stored dynamic fields
    // that draw it (their own key, stream and buffer)
    for (int src = -1; src < a.ncons; src++) {
        uint32_t stream, key0, key1;
        float2 *eta;
        if (src < 0) {
            if (a.noise_mode != NOISE_REAL) continue;
            stream = a.stream;
            key0 = a.key0;
            key1 = a.key1;
            eta = a.eta;
        } else {
            const FusedTarget &TG = a.tgt[1 + src];
            if (TG.noisy != NOISE_REAL) continue;
            stream = TG.stream;
            key0 = TG.key0;
            key1 = TG.key1;
            eta = TG.eta;
        }
        // Cells 2k, 2k+1 of row y0+l, k = t + e*T.  The Philox call with
        // counter (row*NC + k) >> 1 serves k and k^1, which sits in lane
        // t^1 (T is even): the even lane computes the calls of elements
        // e < E/2, the odd lane those of e >= E/2, and each hands its
        // partner the Box-Muller pair that the partner's cells take.
        const uint64_t step = a.step_base + step_rel + (src < 0 ? 0 : a.tgt[1 + src].step_off);
        const uint32_t rowbase = (uint32_t)((long)(y0 + l) * NC);
        const bool even = (t & 1) == 0;
        float2 v[E];
#pragma unroll
        for (int e2 = 0; e2 < E / 2; e2++) {
            const uint32_t k = (uint32_t)((t & ~1) + (even ? e2 : e2 + E / 2) * T);
            const Philox4 o = philox4x32_10((rowbase + k) >> 1, (uint32_t)step, (uint32_t)(step >> 32), stream,
                                            key0, key1);
            const float2 ze = box_muller(o.x[0], o.x[1]), zo = box_muller(o.x[2], o.x[3]);
            const float2 own = even ? ze : zo, snd = even ? zo : ze;
            const float2 rcv = make_float2(__shfl_xor(snd.x, 1), __shfl_xor(snd.y, 1));
            v[e2] = even ? own : rcv;
            v[e2 + E / 2] = even ? rcv : own;
        }
        if constexpr (E > 8) opaque(v);
        r2c_tile<NC, E, T, TW_STAGE>(v, L, t, tws, tst);
        tile_store<NC, LPB, RS, TH>(eta, tile, sy, y0);
        __syncthreads();  // the tile is the next source's transform LDS
    }
}

// ------------------------------------------------------------ column tile

// v[e] = p[col + t + e*T] for the E bins of a lane's column, or zeros for
// an inactive column (one uniform branch for the column, the pointer read
// once, constant offsets between the elements)
template <int E, int T>
__device__ __forceinline__ void load_col(float2 (&v)[E], const float2 *__restrict__ p, long col, int t, bool active)
{
    if (active) {
        const float2 *__restrict__ q = p + col + t;
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = gload(q, (long)e * T);
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = make_float2(0.f, 0.f);
    }
}

// m[e] = table `slot` of the instance at the E bins of a lane's column
template <int E, int T>
__device__ __forceinline__ void load_tab(float (&m)[E], const FusedInst &a, int slot, long col, int t, bool active)
{
    if (active) {
        const float *__restrict__ q = a.mtab + (long)slot * a.g.nh + col + t;
#pragma unroll
        for (int e = 0; e < E; e++) m[e] = gload(q, (long)e * T);
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) m[e] = 0.f;
    }
}

// c q^(2 q2n) qx^a qy^b of the bins of a column, zero where the projection
// onto real fields drops it (multiplier())
template <int E>
__device__ __forceinline__ void mono_col(const LeanOp &O, const ColBins<E> &cb, float (&m)[E])
{
    float base = O.c;
    for (int i = 0; i < O.a; i++) base *= cb.qx;
    const int parx = O.mult_i + (cb.nyx ? 0 : O.a);
#pragma unroll
    for (int e = 0; e < E; e++) m[e] = base;
    for (int i = 0; i < O.q2n; i++)
#pragma unroll
        for (int e = 0; e < E; e++) m[e] *= cb.q2[e];
    for (int i = 0; i < O.b; i++)
#pragma unroll
        for (int e = 0; e < E; e++) m[e] *= cb.qy[e];
#pragma unroll
    for (int e = 0; e < E; e++) m[e] = ((parx + (cb.nyy[e] ? 0 : O.b)) & 1) ? 0.0f : m[e];
}

// The multiplier of a term at the bins of a lane's column.  A monomial stands
// in the descriptor beside the term and is evaluated; sums of prefactors and
// operators with 1/|q| are read from the instance's table, with the data they
// multiply.  A walk over the prefactors is a chain of dependent scalar loads
// per prefactor (model H 1024^2: 201 scalar loads and 2930 vector
// instructions per wavefront of the column pass; all from tables 158 and
// 2040, but 28 bytes a point more traffic, which many instances at once pay
// for).
template <int E, int T>
__device__ __forceinline__ void op_col(const FusedInst &a, const FusedOp &O, const ColBins<E> &cb, long col, int t,
                                       bool active, float (&m)[E])
{
    if (O.tab < 0)
        mono_col<E>(O.m, cb, m);
    else
        load_tab<E, T>(m, a, O.tab, col, t, active);
}
// the factor of an update (FusedDiv)
template <int E, int T>
__device__ __forceinline__ void div_col(const FusedInst &a, const FusedDiv &D, const ColBins<E> &cb, long col, int t,
                                        bool active, float (&r)[E])
{
    if (D.tab < 0) {
#pragma unroll
        for (int e = 0; e < E; e++) {
            const float q2 = cb.q2[e];
            r[e] = __builtin_amdgcn_rcpf(D.d[0] + q2 * (D.d[1] + q2 * (D.d[2] + q2 * D.d[3])));
        }
    } else {
        load_tab<E, T>(r, a, D.tab, col, t, active);
    }
}

// Sum of the terms of one target field over the E bins of a lane: product
// groups (FFT_y of X_g times the group multiplier) and single-field or
// constant terms.  xv holds X of the first group on entry when `pre`.
template <int N, int E, int T, bool SKIP>
__device__ __forceinline__ void target_sum(const FusedInst &a, const FusedTarget &TG, const ColBins<E> &cb,
                                           const float2 (&old)[E], const float2 (&nw)[E], float2 (&xv)[E],
                                           bool pre, int parity, bool active, long col, float2 *L, int t,
                                           const float2 *tws, float2 (&acc)[E])
{
    float m[E];
#pragma unroll
    for (int e = 0; e < E; e++) acc[e] = make_float2(0.f, 0.f);
    for (int gi = TG.g0; gi < TG.g1; gi++) {
        if (!(pre && gi == TG.g0)) load_col<E, T>(xv, a.X[gi], col, t, active);
        const TermRefDev &GM = a.gmul[gi];
        op_col<E, T>(a, a.gop[gi], cb, col, t, active, m);
        fft_line<N, E, -1, TW_STAGE, !SKIP, (T <= 64)>(xv, L, t, tws);
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] = cadd(acc[e], apply_mult(m[e], GM.mult_i, xv[e]));
        line_sync<(T <= 64)>();
    }
    for (int ti = 0; ti < TG.nterms; ti++) {
        const FusedTerm &TR = TG.term[ti];
        op_col<E, T>(a, TR.op, cb, col, t, active, m);
        float2 X[E];
        if (TR.src == SRC_OLD || TR.src == SRC_NEW) {
#pragma unroll
            for (int e = 0; e < E; e++) X[e] = TR.src == SRC_OLD ? old[e] : nw[e];
        } else if (TR.src == SRC_CONST) {
#pragma unroll
            for (int e = 0; e < E; e++) X[e] = cb.zero[e] ? make_float2((float)a.g.n, 0.f) : make_float2(0.f, 0.f);
        } else if (TR.src == SRC_DERIVED) {
            const TermRefDev &DM = a.dmul[TR.idx];
            float dm[E];
            op_col<E, T>(a, a.dop[TR.idx], cb, col, t, active, dm);
            const int b = a.dbase[TR.idx];
            if (b < 0) {
#pragma unroll
                for (int e = 0; e < E; e++) X[e] = old[e];
            } else {
                const float2 *__restrict__ src = a.cs[b][parity];
                load_col<E, T>(X, src, col, t, active);
            }
#pragma unroll
            for (int e = 0; e < E; e++) X[e] = apply_mult(dm[e], DM.mult_i, X[e]);
        } else {
            // SRC_DYN_NEW: a stored dynamic field's value after the step, which
            // this lane wrote to the other buffer earlier in the same pass
            const float2 *__restrict__ src = a.cs[TR.idx][TR.src == SRC_DYN_NEW ? parity ^ 1 : parity];
            load_col<E, T>(X, src, col, t, active);
        }
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] = cadd(acc[e], apply_mult(m[e], TR.mult_i, X[e]));
    }
}

// Z_f = IFFT_y(mask_f * val) for the columns the mask keeps
template <int N, int E, int T, bool SKIP>
__device__ __forceinline__ void z_out(const FusedInst &a, int f, const Geom &g, const ColBins<E> &cb,
                                      const float2 (&val)[E], bool zero, int line, bool active, long col, float2 *L,
                                      int t, const float2 *tws)
{
    if (line > a.kmax[f]) return;  // uniform: every column of the workgroup is masked
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; e++)
        v[e] = (zero || !keep_mode2(g, a.kmax[f], a.kymax[f], cb.kx, t + e * T)) ? make_float2(0.f, 0.f) : val[e];
    fft_line<N, E, +1, TW_STAGE, !SKIP, (T <= 64)>(v, L, t, tws);
    if (active && cb.kx <= a.kmax[f]) {
        float2 *__restrict__ z = a.Z[f] + col + t;  // read once: the stores could alias the descriptor
#pragma unroll
        for (int e = 0; e < E; e++) gstore(z, (long)e * T, v[e]);
    }
    line_sync<(T <= 64)>();
}

// noise of a stored field over the E bins of a lane, times its amplitude
// (times 1/sqrt(dt) for a constraint): real-space rows transformed along y,
// or drawn in spectral space, at the pass's step + step_off
template <int N, int E, int T, bool SKIP>
__device__ __forceinline__ void stored_noise(const FusedInst &a, const FusedTarget &TG, const ColBins<E> &cb, int kx,
                                             uint64_t step, bool active, long col, float2 *L, int t,
                                             const float2 *tws, float2 (&v)[E])
{
    float2 ue[E];
#pragma unroll
    for (int e = 0; e < E; e++) ue[e] = make_float2(0.f, 0.f);
    if (TG.noisy == NOISE_REAL) {
        load_col<E, T>(ue, TG.eta, col, t, active);
        fft_line<N, E, -1, TW_STAGE, !SKIP, (T <= 64)>(ue, L, t, tws);
        line_sync<(T <= 64)>();
    } else {
        const uint64_t s = step + (uint64_t)TG.step_off;
#pragma unroll
        for (int e = 0; e < E / 2; e++)
            spectral_noise_pair(a.g, kx, t + e * T, 0, (uint32_t)s, (uint32_t)(s >> 32), TG.stream, TG.key0, TG.key1,
                                ue[e], ue[e + E / 2]);
    }
#pragma unroll
    for (int e = 0; e < E; e++) {
        float pn = TG.noise_base;
        if (TG.noise_q2n != 0) pn *= sqrtf(ipow(cb.q2[e], TG.noise_q2n));
        if (TG.noise_invq != 0) pn *= sqrtf(ipow(col_iq(cb, e), TG.noise_invq));
        if (!TG.dyn) pn = TG.sdt * pn;
        v[e].x += pn * ue[e].x;
        v[e].y += pn * ue[e].y;
    }
}

// values of a stored field times its factor: 1/D(q) of a dynamic field, the
// reciprocal of the implicit operator's sum of a constraint where q != 0
// (setNotDynamic_k, src/field_kernels.cu:130-197)
template <int E, int T>
__device__ __forceinline__ void solve_col(const FusedInst &a, const FusedTarget &TG, const ColBins<E> &cb, long col,
                                          int t, bool active, float2 (&v)[E])
{
    if (TG.nimp <= 0) return;
    float r[E];
    div_col<E, T>(a, TG.div, cb, col, t, active, r);
#pragma unroll
    for (int e = 0; e < E; e++) {
        const float f = !TG.dyn && cb.zero[e] ? 1.0f : r[e];
        v[e].x *= f;
        v[e].y *= f;
    }
}

// Z_f = IFFT_y(mask_f * L_f u) of a real field that is a dynamic field u or
// derived from it
template <int N, int E, int T, bool SKIP>
__device__ __forceinline__ void lz_out(const FusedInst &a, int f, const Geom &g, const ColBins<E> &cb,
                                       const float2 (&u)[E], bool zero, int line, bool active, long col, float2 *L,
                                       int t, const float2 *tws)
{
    float2 v[E];
    const TermRefDev &LM = a.lmul[f];
    if (LM.npres > 0) {
        float lm[E];
        op_col<E, T>(a, a.lop[f], cb, col, t, active, lm);
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = apply_mult(lm[e], LM.mult_i, u[e]);
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = u[e];
    }
    z_out<N, E, T, SKIP>(a, f, g, cb, v, zero, line, active, col, L, t, tws);
}

// Hermitian projection of the columns kx = 0 and kx = sx/2 (2D): bin ky
// and its partner N - ky of such a column both become their Hermitian mean,
// as the reference's IFFT / real part / FFT round trip of every field every
// step makes them (src/field.cpp:59-89; the interior columns stand for their
// partners implicitly).  Without it the anti-Hermitian part of these columns
// -- invisible to C2R, fed by rounding -- grows in linearly unstable bands
// until it leaks into the real fields.  v[e] holds bin t + e*T of the lane's
// column; the whole workgroup calls this (barriers), only `edge` lines
// change.
template <int N, int E, int T>
__device__ __forceinline__ void hermitian_col(float2 (&v)[E], float2 *L, int t, bool edge)
{
#pragma unroll
    for (int e = 0; e < E; e++) L[lpad(t + e * T)] = v[e];
    line_sync<(T <= 64)>();
    if (edge) {
#pragma unroll
        for (int e = 0; e < E; e++) {
            const float2 p = L[lpad((N - (t + e * T)) & (N - 1))];
            v[e] = make_float2(0.5f * (v[e].x + p.x), 0.5f * (v[e].y - p.y));
        }
    }
    line_sync<(T <= 64)>();
}

template <int N, int TWD>
struct FColCfg {
    static constexpr int E = N >= 4096 ? 16 : (N >= 1024 || N == 128 || N == 256 ? 4 : (N >= 8 ? 8 : N));
    static constexpr int T = N / E;
    static constexpr int THREADS = TWD * T;
    static constexpr int LL = lds_len(N);
    static constexpr bool valid() { return THREADS >= 16 && THREADS <= 512; }
};

// CONS: the instances may have stored constraint fields (compiled out
// otherwise, which keeps the kernel within 128 VGPRs: 4 waves per SIMD)
// Columns line .. line+TWD-1 of one instance (the whole workgroup); mode
// 0: prologue (the real fields of the current state), 1: step.  load_tw as
// for frows_tile.  Each column's LDS region is used by its own lanes only.
template <int N, int TWD, bool CONS, bool XDYN>
__device__ __forceinline__ void fcols_tile(const FusedInst &a, int line, int parity, uint32_t step_rel, int mode,
                                           const float2 *__restrict__ sets, bool load_tw, float2 *tws,
                                           float2 *lds)
{
    using C = FColCfg<N, TWD>;
    constexpr int E = C::E, T = C::T;
    const FusedBlock blk{0, line};
    const Geom &g = a.g;
    const int c = threadIdx.x / T, t = threadIdx.x % T;
    const int kx = blk.line + c;
    const bool active = kx < g.nc1;
    float2 *L = lds + c * C::LL;
    const long col = (long)kx * N;
    const bool upd = mode == 1;
    // phi has product groups: load the first early (unless fresh constraints,
    // solved first, need the register block)
    const bool pre = upd && a.tgt[0].g1 > a.tgt[0].g0 && !(XDYN && a.nfresh > 0);
    const float2 *__restrict__ sin = a.spec[parity];

    // the twiddle loads first: waiting for them then leaves the state's
    // loads in flight
    StageTwiddles<N, E, C::THREADS> twr;
    if (load_tw) twr.load(sets);
    float2 cur[E], xv[E];
    load_col<E, T>(cur, sin, col, t, active);
    load_col<E, T>(xv, pre ? a.X[a.tgt[0].g0] : sin, col, t, active && pre);

    ColBins<E> cb;
    col_bins<E, T>(g, kx, t, cb);
    const uint64_t step = a.step_base + step_rel;
    // phi's spectral noise, drawn while the state's loads are in flight and
    // added to phi_m at once (no register block held across the transforms)
    // where nothing else reads phi_m: no single-field terms, no stored
    // fields.  phi_{m+1} = (phi_m + pn eta + dt acc) / D then.  ky and
    // ky + N/2 are elements e and e + E/2 of this lane.
    const bool early = upd && a.noise_mode == NOISE_SPECTRAL && a.u.noisy && a.tgt[0].nterms == 0 &&
                       (!CONS || a.ncons == 0);
    if (early) {
        float2 eta[E];
#pragma unroll
        for (int e = 0; e < E / 2; e++)
            spectral_noise_pair(g, kx, t + e * T, 0, (uint32_t)step, (uint32_t)(step >> 32), a.stream, a.key0,
                                a.key1, eta[e], eta[e + E / 2]);
#pragma unroll
        for (int e = 0; e < E; e++) {
            const float pn = noise_amplitude_col<E>(a.u, cb, e);
            cur[e].x += pn * eta[e].x;
            cur[e].y += pn * eta[e].y;
        }
    }
    if (load_tw) {
        twr.store(tws, sets);
        __syncthreads();
    }
    float2 nw[E];  // phi_{m+1}
    // workgroups holding the column kx = 0 or kx = sx/2 (uniform test)
    const bool edge_wg = blk.line == 0 || blk.line + TWD > g.nc;
    const bool edge = active && (kx == 0 || kx == g.nc);
    if (upd) {
        // ---- fresh constraints (setNotDynamic_k of phase A, src/field_kernels.cu:
        // 130-197): their values of step m, from the dynamic fields of step m,
        // into the buffer the dynamic fields' terms read
        if (XDYN && a.nfresh > 0)
            for (int ci = 0; ci < a.ncons; ci++) {
                const FusedTarget &TG = a.tgt[1 + ci];
                if (!TG.fresh) continue;
                float2 v[E];
                target_sum<N, E, T, !CONS>(a, TG, cb, cur, cur, xv, false, parity, active, col, L, t, tws, v);
                if (TG.noisy) stored_noise<N, E, T, !CONS>(a, TG, cb, kx, step, active, col, L, t, tws, v);
                solve_col<E, T>(a, TG, cb, col, t, active, v);
                if (edge_wg) hermitian_col<N, E, T>(v, L, t, edge);
                if (active) {
                    float2 *__restrict__ cout = a.cs[ci][parity];
#pragma unroll
                    for (int e = 0; e < E; e++) gstore(cout, col + t + e * T, v[e]);
                }
            }
        // ---- phi (setDynamic_k, src/field_kernels.cu:199-227)
        float2 acc[E];
        target_sum<N, E, T, !CONS>(a, a.tgt[0], cb, cur, cur, xv, pre, parity, active, col, L, t, tws, acc);
        float2 eta[E];
#pragma unroll
        for (int e = 0; e < E; e++) eta[e] = make_float2(0.f, 0.f);
        if (a.noise_mode == NOISE_REAL) {
            // loaded here rather than with phi: fewer registers live across
            // the transforms of the terms
            load_col<E, T>(eta, a.eta, col, t, active);
            fft_line<N, E, -1, TW_STAGE, !CONS, (T <= 64)>(eta, L, t, tws);
            line_sync<(T <= 64)>();
        } else if (a.noise_mode == NOISE_SPECTRAL && !early) {
#pragma unroll
            for (int e = 0; e < E / 2; e++)
                spectral_noise_pair(g, kx, t + e * T, 0, (uint32_t)step, (uint32_t)(step >> 32), a.stream, a.key0,
                                    a.key1, eta[e], eta[e + E / 2]);
        }
        float rD[E];
        if (a.u.nimp > 0) div_col<E, T>(a, a.udiv, cb, col, t, active, rD);
#pragma unroll
        for (int e = 0; e < E; e++) {
            float2 s = cur[e];
            s.x += a.u.dt * acc[e].x;
            s.y += a.u.dt * acc[e].y;
            if (a.u.noisy && !early) {
                const float pn = noise_amplitude_col<E>(a.u, cb, e);
                s.x += pn * eta[e].x;
                s.y += pn * eta[e].y;
            }
            if (a.u.nimp > 0) {
                s.x *= rD[e];
                s.y *= rD[e];
            }
            nw[e] = s;
        }
        if (edge_wg) hermitian_col<N, E, T>(nw, L, t, edge);
        if (active) {
            float2 *__restrict__ sout = a.spec[parity ^ 1];
#pragma unroll
            for (int e = 0; e < E; e++) gstore(sout, col + t + e * T, nw[e]);
        }
        // ---- stored fields: further dynamic fields (setDynamic_k) from their
        // values before the step, then the constraints (setNotDynamic_k,
        // src/field_kernels.cu:130-197): their values of step m+1, from the
        // pre-step state of step m+1
        for (int ci = 0; ci < (CONS ? a.ncons : 0); ci++) {
            const FusedTarget &TG = a.tgt[1 + ci];
            if (XDYN && TG.fresh) continue;
            float2 v[E];
            target_sum<N, E, T, !CONS>(a, TG, cb, cur, nw, xv, false, parity, active, col, L, t, tws, v);
            if (XDYN && TG.dyn) {
                float2 u0[E];
                load_col<E, T>(u0, a.cs[ci][parity], col, t, active);
                const float dt = a.u.dt;
#pragma unroll
                for (int e = 0; e < E; e++) v[e] = make_float2(u0[e].x + dt * v[e].x, u0[e].y + dt * v[e].y);
                if (TG.noisy) stored_noise<N, E, T, !CONS>(a, TG, cb, kx, step, active, col, L, t, tws, v);
                solve_col<E, T>(a, TG, cb, col, t, active, v);
            } else if (TG.keep) {
                // no terms: setNotDynamic_k leaves the value as it is, then
                // divides it by the implicit operator's sum (if any)
                const float2 *__restrict__ kin = a.cs[ci][parity];
                load_col<E, T>(v, kin, col, t, active);
                solve_col<E, T>(a, TG, cb, col, t, active, v);
            } else {
                if (XDYN && TG.noisy) stored_noise<N, E, T, !CONS>(a, TG, cb, kx, step, active, col, L, t, tws, v);
                solve_col<E, T>(a, TG, cb, col, t, active, v);
            }
            if (edge_wg) hermitian_col<N, E, T>(v, L, t, edge);
            if (active) {
                float2 *__restrict__ cout = a.cs[ci][parity ^ 1];
#pragma unroll
                for (int e = 0; e < E; e++) gstore(cout, col + t + e * T, v[e]);
            }
            if (TG.z >= 0) z_out<N, E, T, !CONS>(a, TG.z, g, cb, v, false, blk.line, active, col, L, t, tws);
            if (XDYN && TG.dyn)
                for (int f = 0; f < a.nreal; f++)
                    if (a.zsrc[f] < 0 && a.lbase[f] == ci)
                        lz_out<N, E, T, !CONS>(a, f, g, cb, v, false, blk.line, active, col, L, t, tws);
        }
    } else {
        // prologue: the real fields of the current state
#pragma unroll
        for (int e = 0; e < E; e++) nw[e] = cur[e];
        for (int ci = 0; ci < (CONS ? a.ncons : 0); ci++) {
            const int z = a.tgt[1 + ci].z;
            const bool dyn = XDYN && a.tgt[1 + ci].dyn != 0;
            if (z < 0 && !dyn) continue;
            float2 v[E];
            load_col<E, T>(v, a.cs[ci][0], col, t, active);
            if (z >= 0) z_out<N, E, T, !CONS>(a, z, g, cb, v, a.zero[z] != 0, blk.line, active, col, L, t, tws);
            if (dyn)
                for (int f = 0; f < a.nreal; f++)
                    if (a.zsrc[f] < 0 && a.lbase[f] == ci)
                        lz_out<N, E, T, !CONS>(a, f, g, cb, v, a.zero[f] != 0, blk.line, active, col, L, t, tws);
        }
    }
    // real fields that are phi or derived from it: L_f phi_{m+1}
    for (int f = 0; f < a.nreal; f++) {
        if (a.zsrc[f] >= 0 || a.lbase[f] >= 0) continue;
        lz_out<N, E, T, !CONS>(a, f, g, cb, nw, !upd && a.zero[f] != 0, blk.line, active, col, L, t, tws);
    }
}

}  // namespace cupss
