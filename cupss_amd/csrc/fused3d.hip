// fused3d.hip -- the fused four-pass step of 3D systems with one dynamic
// field (the systems and descriptors are those of fused.hip).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fft_core.hpp"
#include "fused.hpp"
#include "fused_tiles.hpp"
#include "philox.hpp"
#include "update_math.hpp"

namespace cupss {

// ------------------------------------------------------------ 3D systems
//
// A 3D system runs alone (insts[0]) with every buffer in the natural half-
// spectrum layout, element (kx, ky, kz) at (kz*sy + ky)*nc1 + kx, so no
// transposes are needed: rows are contiguous, and lines along y and z are
// read TWD adjacent kx at a time.  Per step:
//   rows  (k_f3rows): Z_f rows -C2R_x-> real fields -> products -R2C_x-> X_g;
//                     real-space noise -R2C_x-> eta
//   y     (k_f3y):    X_g = FFT_y(X_g), eta = FFT_y(eta), in one launch
//   z     (k_f3z):    X_g, eta -FFT_z-> terms, noise; update of phi
//                     (setDynamic_k); mask_f * L_f * phi_new -IFFT_z-> W_f
//   y     (k_f3y):    Z_f = IFFT_y(W_f), lines kx <= kmax_f, in one launch
// The z pass writes W_f only on the (kx, ky) lines the dealias mask of f
// keeps; the y pass reads the others as zero.  W_f may be Z_f, or eta or a
// product transform, of which the z pass reads no line after writing it.  The systems have no stored constraint
// fields (the host checks).

// Rows of 128 complex points take 8 elements a lane, not the 4 of the 2D tile
// (FRowCfg); shorter ones 4.  us per step with 4 / 8 elements (CH, and model B
// with real-space noise after the comma): rows of 128 points, 256x32x32 22.4 /
// 22.7, 26.8 / 29.0; 256x64x64 28.6 / 29.0, 38.2 / 39.5; 256x128x128 53.7 /
// 52.0, 71.5 / 70.6; 256^3 162 / 156.5, 225 / 218: eight from 256x128x128 on,
// which is where a step costs most.  Rows of 64 points, 128x32x32 21.5 / 22.3,
// 25.0 / 27.7; 128^3 37.6 / 38.1, 48.3 / 50.6; 128x256x256 88.0 / 85.6, 120.2 /
// 120.0: four.  (The elements set the order of a line's stages; one choice per
// length keeps them apart from the other sides of the box.)
template <int NC, int LPB, int MAXR>
struct F3RowCfg {
    static constexpr int E = NC == 128 && MAXR <= 3 ? 8 : FRowCfg<NC, LPB, MAXR>::E;
    static constexpr int T = NC / E;
    static constexpr int THREADS = LPB * T;
    static constexpr int RS = tile_stride(NC, LPB);
    static constexpr bool valid()
    {
        return THREADS >= 16 && THREADS <= 512 && (LPB * RS + 2 * NC + tw_stage_alloc(NC, E)) * 8 <= 150 * 1024;
    }
};

template <int NC, int LPB, int MAXR>
__global__ __launch_bounds__((F3RowCfg<NC, LPB, MAXR>::THREADS)) void k_f3rows(const FusedInst *__restrict__ insts,
                                                                           uint32_t step_rel,
                                                                           const float2 *__restrict__ sets)
{
    using C = F3RowCfg<NC, LPB, MAXR>;
    constexpr int E = C::E, T = C::T, RS = C::RS;
    __shared__ float2 tws[2 * NC];
    __shared__ __align__(16) float2 tst[tw_stage_alloc(NC, E)];
    __shared__ float2 tile[LPB * RS];
    const FusedInst &a = insts[0];
    const int nc1 = a.g.nc1;
    const long nrows = (long)a.g.sy * a.g.sz;
    const int l = threadIdx.x / T, t = threadIdx.x % T;
    const long row = (long)blockIdx.x * LPB + l;
    const bool active = row < nrows;
    float2 *L = tile + l * RS;
    const int nreal = a.nreal;
    load_twiddles<2 * NC>(tws, sets);
    load_stage_twiddles<NC, E>(tst, sets);
    __syncthreads();

    float2 r[MAXR][E];
#pragma unroll
    for (int f = 0; f < MAXR; f++) {
        if (f < nreal) {
            const float2 *__restrict__ z = a.Z[f] + row * nc1;
            const int km = a.kmax[f];
            float2 xa[E], ya[E], v[E];
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int k = t + e * T;
                xa[e] = (active && k <= km) ? gload(z, k) : make_float2(0.f, 0.f);
                ya[e] = (active && NC - k <= km) ? gload(z, NC - k) : make_float2(0.f, 0.f);
            }
            c2r_prep<NC, E, T>(xa, ya, t, v, tws);
            fft_line<NC, E, +1, TW_STAGE, false, (T <= 64)>(v, L, t, tst);
#pragma unroll
            for (int e = 0; e < E; e++) r[f][e] = cscale(v[e], a.scale);
            line_sync<(T <= 64)>();
        }
    }
    for (int gi = 0; gi < a.ngroups; gi++) {
        float2 v[E];
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
        r2c_tile<NC, E, T, TW_STAGE>(v, L, t, tws, tst);
        if (active) {
            float2 *__restrict__ x = a.X[gi] + row * nc1;
            for (int k = t; k <= NC; k += T) gstore(x, k, L[k]);
        }
        __syncthreads();
    }
    if (a.noise_mode == NOISE_REAL) {
        // cells 2k, 2k+1 of the row, k = t + e*T: lanes t, t^1 share Philox
        // calls and swap the pairs (frows_tile)
        const uint64_t step = a.step_base + step_rel;
        const uint32_t rowbase = (uint32_t)(row * NC);
        const bool even = (t & 1) == 0;
        float2 v[E];
#pragma unroll
        for (int e2 = 0; e2 < E / 2; e2++) {
            const uint32_t k = (uint32_t)((t & ~1) + (even ? e2 : e2 + E / 2) * T);
            const Philox4 o = philox4x32_10((rowbase + k) >> 1, (uint32_t)step, (uint32_t)(step >> 32), a.stream,
                                            a.key0, a.key1);
            const float2 ze = box_muller(o.x[0], o.x[1]), zo = box_muller(o.x[2], o.x[3]);
            const float2 own = even ? ze : zo, snd = even ? zo : ze;
            const float2 rcv = make_float2(__shfl_xor(snd.x, 1), __shfl_xor(snd.y, 1));
            v[e2] = even ? own : rcv;
            v[e2 + E / 2] = even ? rcv : own;
        }
        r2c_tile<NC, E, T, TW_STAGE>(v, L, t, tws, tst);
        if (active) {
            float2 *__restrict__ x = a.eta + row * nc1;
            for (int k = t; k <= NC; k += T) gstore(x, k, L[k]);
        }
    }
}

// Lines along y of several buffers at once (blockIdx.y: the buffer): line
// (kx, kz) of a buffer holds in[(kz*sy + y)*nc1 + kx], kx < ncols; TWD
// adjacent kx per workgroup, out may be in.  Bound by memory on large boxes
// (256^3, one buffer forward: 134 MB in 23 us, 5.8 TB/s), by latency on small
// ones, where one launch for all buffers fills the chip: 128^3 with noise,
// the two forward transforms 16.4 us in two launches of the general column
// kernel, 8.8 us here.
template <int N, int TWD>
struct F3yCfg {
    static constexpr int E = N >= 4096 ? 16 : (N >= 8 ? 8 : N);
    static constexpr int T = N / E;
    static constexpr int THREADS = TWD * T;
    static constexpr int LL = lds_len(N);
    static constexpr bool valid() { return THREADS >= 64 && THREADS <= 512; }
};
template <int N, int TWD, int DIR>
__global__ __launch_bounds__((F3yCfg<N, TWD>::THREADS)) void k_f3y(F3yArgs a, const float2 *__restrict__ sets)
{
    using C = F3yCfg<N, TWD>;
    constexpr int E = C::E, T = C::T;
    constexpr bool WL = TWD * T <= 64;
    __shared__ __align__(16) float2 tst[tw_stage_alloc(N, E)];
    __shared__ float2 lds[TWD * C::LL];
    const int nc1 = a.nc1, ncols = a.ncols[blockIdx.y];
    const int ntx = (ncols + TWD - 1) / TWD;
    const long item = xcd_item(blockIdx.x, gridDim.x);
    if (item >= (long)ntx * a.sz) return;  // whole workgroup idle
    const int kz = (int)(item / ntx), kx0 = (int)(item % ntx) * TWD;
    const int c = threadIdx.x % TWD, t = threadIdx.x / TWD;
    const bool active = kx0 + c < ncols;
    const long base = (long)kz * N * nc1 + kx0 + c;
    StageTwiddles<N, E, C::THREADS> twl;
    twl.load(sets);
    const float2 *in = a.in[blockIdx.y];
    const int kymax = a.kymax[blockIdx.y];
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        // dir > 0: only the bins of the dealias mask hold the field; the
        // others load the lane's first bin again, so that one branch covers
        // all loads
        const bool keep = DIR < 0 || min(t + e * T, N - (t + e * T)) <= kymax;
        v[e] = active ? gload(in, base + t * nc1 + (keep ? e * T * nc1 : 0)) : make_float2(0.f, 0.f);
    }
    if constexpr (DIR > 0) {
#pragma unroll
        for (int e = 0; e < E; e++)
            if (min(t + e * T, N - (t + e * T)) > kymax) v[e] = make_float2(0.f, 0.f);
    }
    twl.store(tst, sets);
    __syncthreads();
    fft_line<N, E, DIR, TW_STAGE, false, WL>(v, lds + c * C::LL, t, tst);
    if (!active) return;
    float2 *out = a.out[blockIdx.y];
#pragma unroll
    for (int e = 0; e < E; e++) gstore(out, base + (long)(t + e * T) * nc1, v[e]);
}

// q of the E bins (kx, ky, t + e*T) that one lane of a z-line kernel holds
template <int E>
struct LineBins {
    float qx, qy;
    bool nyx, nyy;
    bool axis;              // kx = ky = 0 (the reference's i = j = 0 line, Q8)
    float qz[E], q2[E];
    bool nyz[E], zero[E];   // Nyquist plane; the q = 0 bin
};

template <int E, int T>
__device__ __forceinline__ void line_bins(const Geom &g, int kx, int ky, int t, LineBins<E> &lb)
{
    lb.qx = (float)(kx < (g.sx + 1) / 2 ? kx : kx - g.sx) * g.sqx;
    lb.qy = (float)(ky < (g.sy + 1) / 2 ? ky : ky - g.sy) * g.sqy;
    lb.nyx = g.sx > 1 && kx == g.sx / 2;
    lb.nyy = g.sy > 1 && ky == g.sy / 2;
    lb.axis = kx == 0 && ky == 0;
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int kz = t + e * T;
        lb.qz[e] = (float)(kz < (g.sz + 1) / 2 ? kz : kz - g.sz) * g.sqz;
        lb.q2[e] = lb.qx * lb.qx + lb.qy * lb.qy + lb.qz[e] * lb.qz[e];
        lb.nyz[e] = g.sz > 1 && kz == g.sz / 2;
        lb.zero[e] = lb.axis && kz == 0;
    }
}

// multiplier() for the E bins of a z line (same operation order)
template <int E>
__device__ __forceinline__ void multiplier_line(const PresDev *__restrict__ pres, int p0, int np, int mult_i,
                                                const LineBins<E> &lb, float (&m)[E])
{
#pragma unroll
    for (int e = 0; e < E; e++) m[e] = 0.0f;
    for (int p = p0; p < p0 + np; p++) {
        const PresDev P = pres[p];
        const int parl = mult_i + (lb.nyx ? 0 : P.a) + (lb.nyy ? 0 : P.b);
        const float qxa = ipow(lb.qx, P.a), qyb = ipow(lb.qy, P.b);
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int par = parl + (lb.nyz[e] ? 0 : P.cz);
            float v = (par & 1) ? 0.0f : P.c;
            if (P.q2n > 0) v *= ipow(lb.q2[e], P.q2n);
            if (P.a > 0) v *= qxa;
            if (P.b > 0) v *= qyb;
            if (P.cz > 0) v *= ipow(lb.qz[e], P.cz);
            if (P.invq > 0) v *= ipow(lb.zero[e] ? 0.0f : __builtin_amdgcn_rsqf(lb.q2[e]), P.invq);
            m[e] += v;
        }
    }
}

template <int N, int TWD>
struct F3zCfg {
    static constexpr int E = N >= 8 ? 8 : N;
    static constexpr int T = N / E;
    static constexpr int THREADS = TWD * T;
    static constexpr int LL = lds_len(N);
    static constexpr bool valid() { return THREADS >= 64 && THREADS <= 512; }
};

// Lines along z of TWD adjacent kx at one ky (thread = t*TWD + c: a row of
// TWD values is one contiguous access).  Workgroups are placed XCD-aware.
// Register budget for 4 waves per SIMD (128 VGPRs): the pass waits on
// strided HBM accesses, which more resident waves hide.
template <int N, int TWD>
__global__ __launch_bounds__((F3zCfg<N, TWD>::THREADS)) __attribute__((amdgpu_waves_per_eu(4))) void k_f3z(const FusedInst *__restrict__ insts, int parity,
                                                                 uint32_t step_rel, int mode, int herm,
                                                                 const float2 *__restrict__ sets,
                                                                 unsigned long long *__restrict__ ts)
{
    using C = F3zCfg<N, TWD>;
    constexpr int E = C::E, T = C::T;
    __shared__ __align__(16) float2 tws[tw_stage_alloc(N, E)];
    __shared__ float2 lds[TWD * C::LL];
    const FusedInst &a = insts[0];
    const Geom &g = a.g;
    const int ntx = (g.nc1 + TWD - 1) / TWD;
    const long item = xcd_item(blockIdx.x, gridDim.x);
    if (item >= (long)ntx * g.sy) return;  // whole workgroup idle
    unsigned long long *slot = ts ? ts + (size_t)(blockIdx.x % FUSED_TS_SLOTS) * FUSED_TS_STRIDE : nullptr;
    if (slot && threadIdx.x == 0) atomicMin(&slot[0], (unsigned long long)wall_clock64());
    // Each XCD takes a contiguous range of items; the lines the dealias masks
    // keep (which also transform W_f) have small |ky|, so ky is dealt with
    // stride 8 over the ranges to give every XCD its share of them.
    const int kr = (int)(item / ntx), yq = g.sy >> 3;
    const int kx0 = (int)(item % ntx) * TWD, ky = (kr % yq) * 8 + kr / yq;
    const int c = threadIdx.x % TWD, t = threadIdx.x / TWD;
    const int kx = kx0 + c;
    const bool active = kx < g.nc1;
    float2 *L = lds + c * C::LL;
    const long plane = (long)g.nc1 * g.sy;
    const long base = (long)ky * g.nc1 + kx;  // + kz * plane
    const bool upd = mode != 0;
    const FusedTarget &TG = a.tgt[0];
    const float2 *__restrict__ sin = a.spec[parity];

    float2 cur[E], xv[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const long i = base + (long)(t + e * T) * plane;
        cur[e] = active ? gload(sin, i) : make_float2(0.f, 0.f);
        xv[e] = (active && upd && TG.g1 > TG.g0) ? gload(a.X[TG.g0], i) : make_float2(0.f, 0.f);
    }
    if (herm && (kx0 == 0 || kx0 + TWD > g.nc)) {
        // The previous step of this launch sequence left the kx = 0 and sx/2
        // planes as it computed them: their Hermitian projection
        // (k_hermitian_planes, the last step's is done by it) as they are
        // read, bin (ky, kz) with its partner (-ky, -kz)
        if (kx == 0 || kx == g.nc) {
            const long pbase = (long)((g.sy - ky) & (g.sy - 1)) * g.nc1 + kx;
#pragma unroll
            for (int e = 0; e < E; e++) {
                const float2 p = gload(sin, pbase + (long)((N - (t + e * T)) & (N - 1)) * plane);
                cur[e] = make_float2(0.5f * (cur[e].x + p.x), 0.5f * (cur[e].y - p.y));
            }
        }
    }
    load_stage_twiddles<N, E>(tws, sets);
    __syncthreads();

    LineBins<E> lb;
    line_bins<E, T>(g, kx, ky, t, lb);
    float2 nw[E];
    if (upd) {
        float m[E];
        float2 acc[E];
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] = make_float2(0.f, 0.f);
        // product groups: FFT_z of X_g times the group multiplier
        for (int gi = TG.g0; gi < TG.g1; gi++) {
            if (gi != TG.g0) {
#pragma unroll
                for (int e = 0; e < E; e++)
                    xv[e] = active ? gload(a.X[gi], base + (long)(t + e * T) * plane) : make_float2(0.f, 0.f);
            }
            fft_line<N, E, -1, TW_STAGE, false, (TWD * T <= 64)>(xv, L, t, tws);
            const TermRefDev &GM = a.gmul[gi];
            multiplier_line<E>(a.pool, GM.pres0, GM.npres, GM.mult_i, lb, m);
#pragma unroll
            for (int e = 0; e < E; e++) acc[e] = cadd(acc[e], apply_mult(m[e], GM.mult_i, xv[e]));
            line_sync<(TWD * T <= 64)>();
        }
        // single-field and constant terms (phi or a derived field of phi)
        for (int ti = 0; ti < TG.nterms; ti++) {
            const FusedTerm &TR = TG.term[ti];
            multiplier_line<E>(a.pool, TR.pres0, TR.npres, TR.mult_i, lb, m);
            float2 X[E];
            if (TR.src == SRC_CONST) {
#pragma unroll
                for (int e = 0; e < E; e++) X[e] = lb.zero[e] ? make_float2((float)g.n, 0.f) : make_float2(0.f, 0.f);
            } else if (TR.src == SRC_DERIVED) {
                const TermRefDev &DM = a.dmul[TR.idx];
                float dm[E];
                multiplier_line<E>(a.pool, DM.pres0, DM.npres, DM.mult_i, lb, dm);
#pragma unroll
                for (int e = 0; e < E; e++) X[e] = apply_mult(dm[e], DM.mult_i, cur[e]);
            } else {
#pragma unroll
                for (int e = 0; e < E; e++) X[e] = cur[e];
            }
#pragma unroll
            for (int e = 0; e < E; e++) acc[e] = cadd(acc[e], apply_mult(m[e], TR.mult_i, X[e]));
        }
        const UpdateArgs &u = a.u;
        const uint64_t step = a.step_base + step_rel;
        const bool real_noise = u.noisy && a.noise_mode == NOISE_REAL;
        if (real_noise) {
#pragma unroll
            for (int e = 0; e < E; e++)
                xv[e] = active ? gload(a.eta, base + (long)(t + e * T) * plane) : make_float2(0.f, 0.f);
            fft_line<N, E, -1, TW_STAGE, false, (TWD * T <= 64)>(xv, L, t, tws);
            line_sync<(TWD * T <= 64)>();
        }
#pragma unroll
        for (int e = 0; e < E; e++) {
            float2 s = cur[e];
            s.x += u.dt * acc[e].x;
            s.y += u.dt * acc[e].y;
            if (u.noisy) {
                const float2 eta = real_noise ? xv[e]
                                   : active   ? spectral_noise(g, kx, ky, t + e * T, (uint32_t)step,
                                                               (uint32_t)(step >> 32), a.stream, a.key0, a.key1)
                                              : make_float2(0.f, 0.f);
                float pn = u.noise_base;
                if (u.noise_q2n != 0) pn *= sqrtf(ipow(lb.q2[e], u.noise_q2n));
                if (u.noise_invq != 0)
                    pn *= sqrtf(ipow(lb.zero[e] ? 0.0f : __builtin_amdgcn_rsqf(lb.q2[e]), u.noise_invq));
                s.x += pn * eta.x;
                s.y += pn * eta.y;
            }
            if (u.nimp > 0) {
                float D = 1.0f;
                for (int i = 0; i < u.nimp; i++) {
                    const PresDev P = u.imp[i];
                    float th = P.c;
                    if (P.q2n != 0) th *= ipow(lb.q2[e], P.q2n);
                    if (P.invq != 0) th *= ipow(lb.axis ? 0.0f : __builtin_amdgcn_rsqf(lb.q2[e]), P.invq);
                    D -= u.dt * th;
                }
                const float rD = __builtin_amdgcn_rcpf(D);
                s.x *= rD;
                s.y *= rD;
            }
            nw[e] = s;
        }
        if (active) {
            float2 *__restrict__ sout = a.spec[parity ^ 1];
#pragma unroll
            for (int e = 0; e < E; e++) gstore(sout, base + (long)(t + e * T) * plane, nw[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) nw[e] = cur[e];
    }
    if (mode != 2) {
        // W_f = IFFT_z(mask_f * L_f * phi) on the lines the mask keeps
        const int ny = ky > g.sy / 2 ? ky - g.sy : ky;
        for (int f = 0; f < a.nreal; f++) {
            if (kx0 > a.kmax[f] || abs(ny) > a.kymax[f]) continue;  // uniform over the workgroup
            const int lz = a.p[f] > 0 ? g.sz / (a.p[f] + 1) : g.sz;
            const bool zero = !upd && a.zero[f] != 0;
            float2 v[E];
            const TermRefDev &LM = a.lmul[f];
            float lm[E];
            if (LM.npres > 0) multiplier_line<E>(a.pool, LM.pres0, LM.npres, LM.mult_i, lb, lm);
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int kz = t + e * T;
                const int nz = kz > g.sz / 2 ? kz - g.sz : kz;
                const bool keep = !zero && kx <= a.kmax[f] && abs(nz) <= lz;
                const float2 w = LM.npres > 0 ? apply_mult(lm[e], LM.mult_i, nw[e]) : nw[e];
                v[e] = keep ? w : make_float2(0.f, 0.f);
            }
            fft_line<N, E, +1, TW_STAGE, false, (TWD * T <= 64)>(v, L, t, tws);
            if (active && kx <= a.kmax[f]) {
                float2 *__restrict__ w = a.W[f];
#pragma unroll
                for (int e = 0; e < E; e++) gstore(w, base + (long)(t + e * T) * plane, v[e]);
            }
            line_sync<(TWD * T <= 64)>();
        }
    }
    if (slot) {
        __syncthreads();
        if (threadIdx.x == 0) atomicMax(&slot[1], (unsigned long long)wall_clock64());
    }
}

// derived fields psi_d = M_d phi from phi's spectrum [parity] (natural layout)
__global__ __launch_bounds__(256) void k_f3der(const FusedInst *__restrict__ insts, int parity)
{
    const FusedInst &a = insts[0];
    const Geom &g = a.g;
    const long h = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= g.nh) return;
    const int kx = (int)(h % g.nc1);
    const long r = h / g.nc1;
    const Bin b = make_bin(g, kx, (int)(r % g.sy), (int)(r / g.sy));
    const float2 X = gload(a.spec[parity], h);
    for (int d = 0; d < a.nder; d++) {
        const TermRefDev &M = a.dmul[d];
        gstore(a.dout[d], h, apply_mult(multiplier(a.pool, M.pres0, M.npres, M.mult_i, b), M.mult_i, X));
    }
}

// ------------------------------------------------------------ dispatch

// wide row kernels (more than 3 real fields) for the sizes such systems use
#define FUSED_WIDE_NC(NC) ((NC) >= 32 && (NC) <= 1024)

template <int NC, int MAXR>
static hipError_t f3rows_n(const FusedInst *inst, long nrows, uint32_t step_rel, hipStream_t s, const float2 *sets)
{
    constexpr int T = F3RowCfg<NC, 1, MAXR>::T;
    constexpr int LPB = T >= 256 ? 1 : 256 / T;  // 256 threads a workgroup
    static_assert(F3RowCfg<NC, LPB, MAXR>::valid(), "3D row tile");
    hipLaunchKernelGGL((k_f3rows<NC, LPB, MAXR>), dim3((unsigned)((nrows + LPB - 1) / LPB)),
                       dim3(F3RowCfg<NC, LPB, MAXR>::THREADS), 0, s, inst, step_rel, sets);
    return hipGetLastError();
}

hipError_t fused3d_rows_launch(int nc, int maxr, const FusedInst *inst, long nrows, uint32_t step_rel, hipStream_t s)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    switch (nc) {
#define X(NC)                                                                 \
    case NC:                                                                  \
        if (maxr > 3) {                                                       \
            if constexpr (FUSED_WIDE_NC(NC))                                  \
                return f3rows_n<NC, FUSED_MAX_REAL>(inst, nrows, step_rel, s, sets); \
            return hipErrorInvalidValue;                                      \
        }                                                                     \
        if (maxr == 1) return f3rows_n<NC, 1>(inst, nrows, step_rel, s, sets); \
        return f3rows_n<NC, 3>(inst, nrows, step_rel, s, sets);
        X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024)
#undef X
    default:
        return hipErrorInvalidValue;
    }
}

#define F3Y_CASES(X) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)
#define F3Y_TWD(X) X(1) X(2) X(4) X(8) X(16) X(32) X(64)

template <int N>
static hipError_t f3y_n(int dir, const F3yArgs &a, hipStream_t s, const float2 *sets)
{
    int most = 1;
    for (int b = 0; b < a.n; b++) most = std::max(most, a.ncols[b]);
    // 16 adjacent lines (128 bytes a row, one cache line) where that still
    // gives two workgroups a CU, else narrower: 128^3, two buffers, 16 lines
    // 8.8 us against 16.4 us for 4 lines of a buffer at a time
    int pick = 0;
#define X(TWD)                                                                                              \
    if constexpr (F3yCfg<N, TWD>::valid())                                                                  \
        if (!pick || (TWD <= 16 && (long)((most + TWD - 1) / TWD) * a.sz * a.n >= 512)) pick = TWD;
    F3Y_TWD(X)
#undef X
#define X(TWD)                                                                                              \
    if constexpr (F3yCfg<N, TWD>::valid())                                                                  \
        if (pick == TWD) {                                                                                  \
            const dim3 grid((unsigned)xcd_blocks((long)((most + TWD - 1) / TWD) * a.sz), (unsigned)a.n);   \
            if (dir < 0)                                                                                    \
                hipLaunchKernelGGL((k_f3y<N, TWD, -1>), grid, dim3(F3yCfg<N, TWD>::THREADS), 0, s, a, sets); \
            else                                                                                            \
                hipLaunchKernelGGL((k_f3y<N, TWD, +1>), grid, dim3(F3yCfg<N, TWD>::THREADS), 0, s, a, sets); \
            return hipGetLastError();                                                                       \
        }
    F3Y_TWD(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t fused3d_y_launch(const Geom &g, int dir, F3yArgs a, hipStream_t s)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    if (a.n <= 0) return hipSuccess;
    if (a.n > F3Y_BUFS) return hipErrorInvalidValue;
    a.nc1 = g.nc1;
    a.sz = g.sz;
    switch (g.sy) {
#define X(N) \
    case N:  \
        return f3y_n<N>(dir, a, s, sets);
        F3Y_CASES(X)
#undef X
    default:
        return hipErrorInvalidValue;
    }
}

#define F3Z_CASES(X) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024)
#define F3Z_TWD(X) X(4) X(8) X(16) X(32) X(64)

template <int N>
static std::vector<int> z_shapes()
{
    std::vector<int> v;
#define X(TWD) \
    if (F3zCfg<N, TWD>::valid()) v.push_back(TWD);
    F3Z_TWD(X)
#undef X
    return v;
}

static std::vector<int> fused3d_z_shapes(int nz)
{
    switch (nz) {
#define X(N) \
    case N:  \
        return z_shapes<N>();
        F3Z_CASES(X)
#undef X
    default:
        return {};
    }
}

// 16 adjacent lines (128 bytes a row, one cache line) where that still gives
// two workgroups a CU and leaves no more than a fifth of the lanes without a
// line (33 bins: 15 of 48), else narrower.  us per step of model B with
// real-space noise, 16 / 8 / 4 lines where a tile allows them: 64^3 (192
// workgroups of 16) 27.5 / 26.9, 32x32x128 27.6 / 26.5 / 25.5, 128x64x64
// 30.0 / 29.6, 128^3 (640) 48.1 / 48.6 / 49.3, 64x256x256 80.5 / 77.1 / 77.6,
// 256x128x128 70.3 / 72.2 / 69.3, 256x256x128 111 / 120 / 114, 256^3
// 219 / 231 / 256.  Timing the widths on each new system finds none better
// than 2 per cent and cost its first run 160 us (32^3) to 850 us (256x256x128),
// more than the first steps themselves.
int fused3d_z_width(int nz, int nc1, int sy)
{
    int pick = 0;
    for (int w : fused3d_z_shapes(nz)) {
        const int tiles = (nc1 + w - 1) / w;
        if (!pick || (w <= 16 && (long)tiles * sy >= 512 && 4 * tiles * w <= 5 * nc1)) pick = w;
    }
    return pick;
}

template <int N>
static hipError_t f3z_n(int twd, const FusedInst *inst, int nc1, int sy, int parity, uint32_t step_rel, int mode,
                        int herm, hipStream_t s, const float2 *sets, unsigned long long *ts)
{
#define X(TWD)                                                                                           \
    if constexpr (F3zCfg<N, TWD>::valid()) {                                                            \
        if (twd == TWD) {                                                                                \
            const long total = (long)((nc1 + TWD - 1) / TWD) * sy;                                       \
            hipLaunchKernelGGL((k_f3z<N, TWD>), dim3((unsigned)xcd_blocks(total)),                      \
                               dim3(F3zCfg<N, TWD>::THREADS), 0, s, inst, parity, step_rel, mode, herm, sets, ts); \
            return hipGetLastError();                                                                    \
        }                                                                                                \
    }
    F3Z_TWD(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t fused3d_z_launch(int nz, int twd, const FusedInst *inst, int nc1, int sy, int parity, uint32_t step_rel,
                            int mode, int herm, hipStream_t s, unsigned long long *ts)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    switch (nz) {
#define X(N) \
    case N:  \
        return f3z_n<N>(twd, inst, nc1, sy, parity, step_rel, mode, herm, s, sets, ts);
        F3Z_CASES(X)
#undef X
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t fused3d_derived_launch(const FusedInst *inst, long nh, int parity, hipStream_t s)
{
    hipLaunchKernelGGL(k_f3der, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, s, inst, parity);
    return hipGetLastError();
}

}  // namespace cupss
