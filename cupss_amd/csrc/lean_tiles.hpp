// lean_tiles.hpp -- the row and column tiles of the fused 2D step for simple
// systems: one field with at most one product group, two real fields and
// monomial operators (FusedLean; Cahn-Hilliard, KPZ and their like).
//
// The general tiles walk the descriptor's lists: every count, pointer and
// prefactor is a scalar load whose address depends on the one before, about
// twenty in a chain of 150 to 200 cycles each, which a wavefront of a small
// grid has nothing to hide behind (CH 1024^2: the column pass waits for 63 %
// of its wavefronts' life and issues vector instructions in 9 % of it).
// These tiles read the whole program of a system in one go, 64-byte scalar
// loads of independent addresses, and keep it in scalar registers; the
// implicit operator is one polynomial in q^2.  Measured, us per step, general
// tiles -> these: CH 256^2 11.9 -> 10.1, CH 1024^2 17.6 -> 16.3, KPZ 512^2
// with real-space noise 22.4 -> 20.1; 512 EW/KPZ instances of 64^2 .. 512^2
// 183 -> 169 (with the elements a lane of FRowCfg and FColCfg, CH 256^2 takes
// 8.2 today).  What bounds them now: one or two wavefronts a SIMD and two
// launches a step on a small grid, vector issue on many instances.
#pragma once
#include <hip/hip_runtime.h>

#include "fused_tiles.hpp"

namespace cupss {

// As the general tiles these must give the same bits in every kernel that
// inlines them; here a*b + c is also fused within one expression only.
#pragma clang fp contract(on)
typedef uint32_t vu16 __attribute__((ext_vector_type(16)));

// the lean program and phi's buffers of instance a, in scalar registers
struct LeanRegs {
    FusedLean p;
    float2 *spec0, *spec1;
    uint64_t step;
};
__device__ __forceinline__ void lean_load(const FusedInst &a, LeanRegs &R)
{
    static_assert(sizeof(FusedLean) % 64 == 0, "whole 64-byte loads");
    constexpr int NV = sizeof(FusedLean) / 64;
    vu16 v[NV];
    const vu16 *src = reinterpret_cast<const vu16 *>(&a.lean);
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = src[i];
    R.spec0 = a.spec[0];
    R.spec1 = a.spec[1];
    R.step = a.step_base;
#if defined(__HIP_DEVICE_COMPILE__)
    // pinned here: the compiler would otherwise sink each load to its use
#pragma unroll
    for (int i = 0; i < NV; i++) asm volatile("" : "+s"(v[i]));
    asm volatile("" : "+s"(R.spec0), "+s"(R.spec1), "+s"(R.step));
#endif
    __builtin_memcpy(&R.p, v, sizeof(FusedLean));
}

// Rows y0 .. y0+LPB-1 of one instance (the whole workgroup), as frows_tile.
template <int NC, int LPB, int MAXR>
__device__ __forceinline__ void lean_rows_tile(const LeanRegs &R, int y0, uint64_t step,
                                               const float2 *__restrict__ sets, bool load_tw, float2 *tws,
                                               float2 *tst, float2 *tile)
{
    using C = FRowCfg<NC, LPB, MAXR>;
    constexpr int E = C::E, T = C::T, RS = C::RS, TH = C::THREADS;
    const FusedLean &P = R.p;
    const int sy = P.sy;
    const int l = threadIdx.x / T, t = threadIdx.x % T;
    float2 *L = tile + l * RS;
    SizeTwiddles<2 * NC, TH> twl;
    StageTwiddles<NC, E, TH> tsl;
    if (load_tw) {
        twl.load(sets);
        tsl.load(sets);
    }
    float2 r[MAXR][E];
#pragma unroll
    for (int f = 0; f < MAXR; f++) {
        if (f < P.nreal) {
            TileLoad<NC, LPB, RS, TH> tl;
            tl.issue(P.Z[f], sy, y0, P.f[f].kmax);
            if (f == 0 && load_tw) {
                twl.store(tws, sets);
                tsl.store(tst, sets);
            }
            tl.commit(tile, P.Z[f], sy, y0, P.f[f].kmax);
            __syncthreads();
            float2 xa[E], ya[E], v[E];
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int k = t + e * T;
                xa[e] = L[k];
                ya[e] = L[NC - k];
            }
            line_sync<(T <= 64)>();
            c2r_prep<NC, E, T>(xa, ya, t, v, tws);
            opaque(v);
            fft_line<NC, E, +1, TW_STAGE, false, (T <= 64)>(v, L, t, tst);
            opaque(v);
#pragma unroll
            for (int e = 0; e < E; e++) r[f][e] = cscale(v[e], P.scale);
            __syncthreads();
        }
    }
    if (P.nreal == 0) {
        if (load_tw) {
            twl.store(tws, sets);
            tsl.store(tst, sets);
        }
        __syncthreads();
    }
    if (P.ngroups > 0) {
        float2 v[E];
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = make_float2(0.f, 0.f);
#pragma unroll
        for (int pi = 0; pi < LEAN_PRODS; pi++) {
            if (pi >= P.nprod) break;
            float2 p[E];
#pragma unroll
            for (int e = 0; e < E; e++) p[e] = make_float2(P.coef[pi], P.coef[pi]);
#pragma unroll
            for (int f = 0; f < MAXR; f++)
                for (int c = (P.power[pi] >> (8 * f)) & 0xff; c > 0; c--) {
#pragma unroll
                    for (int e = 0; e < E; e++) {
                        p[e].x *= r[f][e].x;
                        p[e].y *= r[f][e].y;
                    }
                }
#pragma unroll
            for (int e = 0; e < E; e++) v[e] = cadd(v[e], p[e]);
        }
        opaque(v);
        r2c_tile<NC, E, T, TW_STAGE>(v, L, t, tws, tst);
        tile_store<NC, LPB, RS, TH>(P.X, tile, sy, y0);
        __syncthreads();
    }
    if (P.noise_mode == NOISE_REAL) {
        // as frows_tile: lanes t, t^1 share Philox calls and swap the pairs
        const uint32_t rowbase = (uint32_t)((long)(y0 + l) * NC);
        const bool even = (t & 1) == 0;
        float2 v[E];
#pragma unroll
        for (int e2 = 0; e2 < E / 2; e2++) {
            const uint32_t k = (uint32_t)((t & ~1) + (even ? e2 : e2 + E / 2) * T);
            const Philox4 o = philox4x32_10((rowbase + k) >> 1, (uint32_t)step, (uint32_t)(step >> 32), P.stream,
                                            P.key0, P.key1);
            const float2 ze = box_muller(o.x[0], o.x[1]), zo = box_muller(o.x[2], o.x[3]);
            const float2 own = even ? ze : zo, snd = even ? zo : ze;
            const float2 rcv = make_float2(__shfl_xor(snd.x, 1), __shfl_xor(snd.y, 1));
            v[e2] = even ? own : rcv;
            v[e2 + E / 2] = even ? rcv : own;
        }
        opaque(v);
        r2c_tile<NC, E, T, TW_STAGE>(v, L, t, tws, tst);
        tile_store<NC, LPB, RS, TH>(P.eta, tile, sy, y0);
        __syncthreads();
    }
}

// Columns line .. line+TWD-1 of one instance (the whole workgroup), as
// fcols_tile: mode 0 prologue, 1 step from buffer `parity`.
template <int N, int TWD>
__device__ __forceinline__ void lean_cols_tile(const LeanRegs &R, int line, int parity, uint64_t step, int mode,
                                               const float2 *__restrict__ sets, bool load_tw, float2 *tws,
                                               float2 *lds)
{
    using C = FColCfg<N, TWD>;
    constexpr int E = C::E, T = C::T;
    constexpr bool WL = T <= 64;
    const FusedLean &P = R.p;
    const int c = threadIdx.x / T, t = threadIdx.x % T;
    const int kx = line + c;
    const bool active = kx < P.nc1;
    float2 *L = lds + c * C::LL;
    const long col = (long)kx * N;
    const bool upd = mode == 1;
    StageTwiddles<N, E, C::THREADS> twr;
    if (load_tw) twr.load(sets);
    float2 cur[E], xv[E], eta[E];
    load_col<E, T>(cur, parity ? R.spec1 : R.spec0, col, t, active);
    load_col<E, T>(xv, P.X, col, t, active && upd && P.ngroups > 0);
    load_col<E, T>(eta, P.eta, col, t, active && upd && P.noise_mode == NOISE_REAL);

    Geom g;
    g.sx = 2 * P.nc;
    g.sy = P.sy;
    g.sz = 1;
    g.nc = P.nc;
    g.nc1 = P.nc1;
    g.n = (long)g.sx * g.sy;
    g.sqx = P.sqx;
    g.sqy = P.sqy;
    ColBins<E> cb;
    col_bins<E, T>(g, kx, t, cb);
    if (upd && P.noise_mode == NOISE_SPECTRAL) {
#pragma unroll
        for (int e = 0; e < E / 2; e++)
            spectral_noise_pair(g, kx, t + e * T, 0, (uint32_t)step, (uint32_t)(step >> 32), P.stream, P.key0, P.key1,
                                eta[e], eta[e + E / 2]);
        // added at once: no register block held across the transforms
#pragma unroll
        for (int e = 0; e < E; e++) {
            float pn = P.noise_base;
            if (P.noise_q2n != 0) pn *= sqrtf(ipow(cb.q2[e], P.noise_q2n));
            cur[e].x += pn * eta[e].x;
            cur[e].y += pn * eta[e].y;
        }
    }
    if (load_tw) {
        twr.store(tws, sets);
        __syncthreads();
    }
    float2 nw[E];
    if (upd) {
#pragma unroll
        for (int e = 0; e < E; e++) nw[e] = cur[e];
        if (P.ngroups > 0) {
            fft_line<N, E, -1, TW_STAGE, false, WL>(xv, L, t, tws);
            opaque(xv);
            line_sync<WL>();
            float m[E];
            mono_col<E>(P.g, cb, m);
#pragma unroll
            for (int e = 0; e < E; e++) {
                const float2 v = apply_mult(m[e], P.g.mult_i, xv[e]);
                nw[e].x += P.dt * v.x;
                nw[e].y += P.dt * v.y;
            }
        }
        if (P.cst != 0.0f) {  // constant terms: N at q = 0
#pragma unroll
            for (int e = 0; e < E; e++)
                if (cb.zero[e]) nw[e].x += P.dt * (P.cst * (float)g.n);
        }
        if (P.noise_mode == NOISE_REAL) {
            fft_line<N, E, -1, TW_STAGE, false, WL>(eta, L, t, tws);
            opaque(eta);
            line_sync<WL>();
#pragma unroll
            for (int e = 0; e < E; e++) {
                float pn = P.noise_base;
                if (P.noise_q2n != 0) pn *= sqrtf(ipow(cb.q2[e], P.noise_q2n));
                nw[e].x += pn * eta[e].x;
                nw[e].y += pn * eta[e].y;
            }
        }
        if (P.nimp > 0) {
#pragma unroll
            for (int e = 0; e < E; e++) {
                const float q2 = cb.q2[e];
                const float rD = __builtin_amdgcn_rcpf(P.d[0] + q2 * (P.d[1] + q2 * (P.d[2] + q2 * P.d[3])));
                nw[e].x *= rD;
                nw[e].y *= rD;
            }
        }
        if (line == 0 || line + TWD > P.nc) hermitian_col<N, E, T>(nw, L, t, active && (kx == 0 || kx == P.nc));
        if (active) {
            float2 *__restrict__ sout = (parity ? R.spec0 : R.spec1) + col + t;
#pragma unroll
            for (int e = 0; e < E; e++) gstore(sout, (long)e * T, nw[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) nw[e] = cur[e];
    }
#pragma unroll
    for (int f = 0; f < 2; f++) {
        if (f >= P.nreal || line > P.f[f].kmax) continue;  // uniform
        const bool zero = !upd && P.f[f].zero != 0;
        float2 v[E];
        if (P.f[f].lin) {
            float m[E];
            mono_col<E>(P.f[f].op, cb, m);
#pragma unroll
            for (int e = 0; e < E; e++) v[e] = apply_mult(m[e], P.f[f].op.mult_i, nw[e]);
        } else {
#pragma unroll
            for (int e = 0; e < E; e++) v[e] = nw[e];
        }
#pragma unroll
        for (int e = 0; e < E; e++)
            if (zero || !keep_mode2(g, P.f[f].kmax, P.f[f].kymax, kx, t + e * T)) v[e] = make_float2(0.f, 0.f);
        opaque(v);
        fft_line<N, E, +1, TW_STAGE, false, WL>(v, L, t, tws);
        if (active && kx <= P.f[f].kmax) {
            float2 *__restrict__ z = P.Z[f] + col + t;
#pragma unroll
            for (int e = 0; e < E; e++) gstore(z, (long)e * T, v[e]);
        }
        line_sync<WL>();
    }
}

}  // namespace cupss
