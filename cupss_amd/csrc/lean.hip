// lean.hip -- row and column kernels of the fused 2D step for simple systems
// (lean_tiles.hpp), launched like those of fused.hip.
#include <hip/hip_runtime.h>

#include "lean_tiles.hpp"

namespace cupss {

namespace lean {

template <int NC, int LPB>
__global__ __launch_bounds__((FRowCfg<NC, LPB, 2>::THREADS)) void k_frows(const FusedInst *__restrict__ insts,
                                                                       const FusedBlock *__restrict__ blocks,
                                                                       uint32_t step_rel,
                                                                       const float2 *__restrict__ sets)
{
    using C = FRowCfg<NC, LPB, 2>;
    __shared__ __align__(16) float2 tws[2 * NC];
    __shared__ __align__(16) float2 tst[tw_stage_alloc(NC, C::E)];
    __shared__ float2 tile[LPB * C::RS];
    const FusedBlock blk = blocks[blockIdx.x];
    if (blk.inst < 0) return;
    LeanRegs R;
    lean_load(insts[blk.inst], R);
    lean_rows_tile<NC, LPB, 2>(R, blk.line, R.step + step_rel, sets, true, tws, tst, tile);
}

template <int N, int TWD>
__global__ __launch_bounds__((FColCfg<N, TWD>::THREADS)) void k_fcols(const FusedInst *__restrict__ insts,
                                                                   const FusedBlock *__restrict__ blocks, int parity,
                                                                   uint32_t step_rel, int mode,
                                                                   const float2 *__restrict__ sets,
                                                                   unsigned long long *__restrict__ ts)
{
    using C = FColCfg<N, TWD>;
    __shared__ __align__(16) float2 tws[tw_stage_alloc(N, C::E)];
    __shared__ float2 lds[TWD * C::LL];
    const FusedBlock blk = blocks[blockIdx.x];
    if (blk.inst < 0) return;
    LeanRegs R;
    lean_load(insts[blk.inst], R);
    if (mode == 0 && R.p.resume) return;  // Z_f of this state left by the previous run
    unsigned long long *slot = ts ? ts + (size_t)(blockIdx.x % FUSED_TS_SLOTS) * FUSED_TS_STRIDE : nullptr;
    if (slot && threadIdx.x == 0) atomicMin(&slot[0], (unsigned long long)wall_clock64());
    lean_cols_tile<N, TWD>(R, blk.line, parity, R.step + step_rel, mode, sets, true, tws, lds);
    if (slot) {
        __syncthreads();
        if (threadIdx.x == 0) atomicMax(&slot[1], (unsigned long long)wall_clock64());
    }
}

// Whole steps of a 64^2 instance in one workgroup, as k_fsmall of fused.hip
template <int NC, int N>
struct SmallCfg {
    static constexpr int THREADS = 512;
    static constexpr int LPB = THREADS / FRowCfg<NC, 1, 2>::T;
    static constexpr int TWD = THREADS / FColCfg<N, 1>::T;
    static constexpr int ROW = LPB * FRowCfg<NC, LPB, 2>::RS, COL = TWD * FColCfg<N, TWD>::LL;
    static constexpr int LDSN = ROW > COL ? ROW : COL;
};

template <int NC, int N>
__global__ __launch_bounds__(512) void k_fsmall(const FusedInst *__restrict__ insts, const int *__restrict__ ids,
                                                int n0, int k, int rel0, const float2 *__restrict__ sets,
                                                unsigned long long *__restrict__ ts)
{
    using C = SmallCfg<NC, N>;
    __shared__ float2 twr[2 * NC];
    __shared__ __align__(16) float2 tsr[tw_stage_alloc(NC, FRowCfg<NC, C::LPB, 2>::E)];
    __shared__ __align__(16) float2 twc[tw_stage_alloc(N, FColCfg<N, C::TWD>::E)];
    __shared__ float2 buf[C::LDSN];
    unsigned long long *slot = ts ? ts + (size_t)(blockIdx.x % FUSED_TS_SLOTS) * FUSED_TS_STRIDE : nullptr;
    if (slot && threadIdx.x == 0) atomicMin(&slot[0], (unsigned long long)wall_clock64());
    LeanRegs R;
    lean_load(insts[ids[blockIdx.x]], R);
    load_twiddles<2 * NC>(twr, sets);
    load_stage_twiddles<NC, FRowCfg<NC, C::LPB, 2>::E>(tsr, sets);
    load_stage_twiddles<N, FColCfg<N, C::TWD>::E>(twc, sets);
    __syncthreads();
    for (int n = n0; n < n0 + k; n++) {
        const uint64_t step = R.step + (uint32_t)(n - rel0);
        for (int y0 = 0; y0 < N; y0 += C::LPB) lean_rows_tile<NC, C::LPB, 2>(R, y0, step, sets, false, twr, tsr, buf);
        // rows ended with a barrier: X_g and eta are written, the buffer is free
        for (int x0 = 0; x0 <= NC; x0 += C::TWD) lean_cols_tile<N, C::TWD>(R, x0, n & 1, step, 1, sets, false, twc, buf);
        __syncthreads();  // Z_f and the spectra written; the buffer is free for the rows
    }
    if (slot && threadIdx.x == 0) atomicMax(&slot[1], (unsigned long long)wall_clock64());
}

// Simple instances without transforms (diffusion, Edwards-Wilkinson), as
// k_felem of fused.hip: one thread per pair of bins (kx, j), (kx, j + sy/2)
// takes nsteps steps in registers.  One step of a small grid is a chain of
// three memory latencies (block, program, spectrum); the general kernel's
// walk over the terms and operators adds more (256^2, runs of one step: 4.04
// us in the general kernel, 3.79 here; the launch itself is the rest).
__global__ __launch_bounds__(FUSED_ELEM_BLOCK) void k_felem(const FusedInst *__restrict__ insts,
                                                            const FusedBlock *__restrict__ blocks, int parity,
                                                            uint32_t step_rel, int nsteps)
{
    const FusedBlock blk = blocks[blockIdx.x];
    if (blk.inst < 0) return;
    const FusedInst &a = insts[blk.inst];
    LeanRegs R;
    lean_load(a, R);
    const FusedLean &P = R.p;
    const uint32_t hy = (uint32_t)P.sy / 2, nint = (uint32_t)(P.nc - 1) * hy;
    const uint32_t pidx = (uint32_t)blk.line + threadIdx.x;
    if (pidx >= (uint32_t)P.nc1 * hy) return;  // no barriers below
    // the interior columns first, then those of the kx = 0 and nc planes
    // (k_felem of fused.hip)
    uint32_t j, kx;
    if (pidx < nint) {
        j = pidx / (uint32_t)(P.nc - 1);
        kx = 1 + pidx - j * (uint32_t)(P.nc - 1);
    } else {
        kx = ((pidx - nint) & 1) ? (uint32_t)P.nc : 0;
        j = (pidx - nint) >> 1;
    }
    const float2 *__restrict__ src = parity ? R.spec1 : R.spec0;
    float2 cur[2];
    long h[2];
#pragma unroll
    for (int w = 0; w < 2; w++) {
        h[w] = (long)(j + w * hy) * P.nc1 + kx;
        cur[w] = gload(src, h[w]);
    }
    Geom g;
    g.sx = 2 * P.nc;
    g.sy = P.sy;
    g.sz = 1;
    g.nc = P.nc;
    g.nc1 = P.nc1;
    g.nh = (long)P.nc1 * P.sy;
    g.n = (long)g.sx * g.sy;
    g.sqx = P.sqx;
    g.sqy = P.sqy;
    g.sqz = 0.f;
    const bool noisy = P.noise_mode == NOISE_SPECTRAL;
    const float qx = (float)((int)kx < (g.sx + 1) / 2 ? (int)kx : (int)kx - g.sx) * g.sqx;
    float rD[2], pn[2];
#pragma unroll
    for (int w = 0; w < 2; w++) {
        const int ky = (int)(j + w * hy);
        const float qy = (float)(ky < (g.sy + 1) / 2 ? ky : ky - g.sy) * g.sqy;
        const float q2 = qx * qx + qy * qy;
        rD[w] = P.nimp > 0 ? __builtin_amdgcn_rcpf(P.d[0] + q2 * (P.d[1] + q2 * (P.d[2] + q2 * P.d[3]))) : 1.0f;
        pn[w] = noisy ? P.noise_base : 0.f;
        if (noisy && P.noise_q2n != 0) pn[w] *= sqrtf(ipow(q2, P.noise_q2n));
    }
    const float cst = P.dt * (P.cst * (float)g.n);  // constant terms, at q = 0
    const bool zero = kx == 0 && j == 0;
    for (int n = 0; n < nsteps; n++) {
        if (n == nsteps - 1) {
            // derived fields of the last step's start
            for (int d = 0; d < a.nder; d++) {
                const TermRefDev &M = a.dmul[d];
#pragma unroll
                for (int w = 0; w < 2; w++) {
                    const Bin b = make_bin(g, (int)kx, (int)(j + w * hy), 0);
                    gstore(a.dout[d], h[w],
                           apply_mult(multiplier(a.pool, M.pres0, M.npres, M.mult_i, b), M.mult_i, cur[w]));
                }
            }
        }
        float2 eta[2] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
        if (noisy) {
            const uint64_t step = R.step + step_rel + (uint64_t)n;
            spectral_noise_pair(g, (int)kx, (int)j, 0, (uint32_t)step, (uint32_t)(step >> 32), P.stream, P.key0, P.key1,
                                eta[0], eta[1]);
        }
#pragma unroll
        for (int w = 0; w < 2; w++) {
            if (w == 0 && zero) cur[w].x += cst;
            if (noisy) {
                cur[w].x += pn[w] * eta[w].x;
                cur[w].y += pn[w] * eta[w].y;
            }
            cur[w].x *= rD[w];
            cur[w].y *= rD[w];
        }
    }
    float2 *__restrict__ dst = (parity ^ (nsteps & 1)) ? R.spec1 : R.spec0;
#pragma unroll
    for (int w = 0; w < 2; w++) gstore(dst, h[w], cur[w]);
}

}  // namespace lean

#define LEAN_ROW_CASES(X) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048)
#define LEAN_COL_CASES(X) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)
#define LEAN_TILES(X) X(1) X(2) X(4) X(8) X(16)

template <int NC>
static hipError_t lrows_n(int lpb, const FusedInst *inst, const FusedBlock *blocks, int nblocks, uint32_t step_rel,
                          hipStream_t s, const float2 *sets)
{
#define X(LPB)                                                                                                \
    if constexpr (FRowCfg<NC, LPB, 2>::valid()) {                                                            \
        if (lpb == LPB) {                                                                                     \
            hipLaunchKernelGGL((lean::k_frows<NC, LPB>), dim3(nblocks), dim3(FRowCfg<NC, LPB, 2>::THREADS), 0, \
                               s, inst, blocks, step_rel, sets);                                              \
            return hipGetLastError();                                                                         \
        }                                                                                                     \
    }
    LEAN_TILES(X)
#undef X
    return hipErrorInvalidValue;
}

template <int N>
static hipError_t lcols_n(int twd, const FusedInst *inst, const FusedBlock *blocks, int nblocks, int parity,
                          uint32_t step_rel, int mode, hipStream_t s, const float2 *sets, unsigned long long *ts)
{
#define X(TWD)                                                                                                \
    if constexpr (FColCfg<N, TWD>::valid()) {                                                                \
        if (twd == TWD) {                                                                                     \
            hipLaunchKernelGGL((lean::k_fcols<N, TWD>), dim3(nblocks), dim3(FColCfg<N, TWD>::THREADS), 0, s, inst,  \
                               blocks, parity, step_rel, mode, sets, ts);                                     \
            return hipGetLastError();                                                                         \
        }                                                                                                     \
    }
    LEAN_TILES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t lean_rows_launch(int nc, int lpb, const FusedInst *inst, const FusedBlock *blocks, int nblocks,
                            uint32_t step_rel, hipStream_t s)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    switch (nc) {
#define X(NC) \
    case NC:  \
        return lrows_n<NC>(lpb, inst, blocks, nblocks, step_rel, s, sets);
        LEAN_ROW_CASES(X)
#undef X
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t lean_cols_launch(int ny, int twd, const FusedInst *inst, const FusedBlock *blocks, int nblocks, int parity,
                            uint32_t step_rel, int mode, hipStream_t s, unsigned long long *ts)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    switch (ny) {
#define X(N) \
    case N:  \
        return lcols_n<N>(twd, inst, blocks, nblocks, parity, step_rel, mode, s, sets, ts);
        LEAN_COL_CASES(X)
#undef X
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t lean_small_launch(int nc, int ny, const FusedInst *inst, const int *ids, int nids, int n0, int k, int rel0,
                             hipStream_t s, unsigned long long *ts)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    if (nids <= 0 || k <= 0) return hipSuccess;
    if (nc != 32 || ny != 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL((lean::k_fsmall<32, 64>), dim3(nids), dim3(512), 0, s, inst, ids, n0, k, rel0, sets, ts);
    return hipGetLastError();
}

hipError_t lean_elem_launch(const FusedInst *inst, const FusedBlock *blocks, int nblocks, int parity,
                            uint32_t step_rel, int nsteps, hipStream_t s)
{
    hipLaunchKernelGGL(lean::k_felem, dim3(nblocks), dim3(FUSED_ELEM_BLOCK), 0, s, inst, blocks, parity, step_rel,
                       nsteps);
    return hipGetLastError();
}

}  // namespace cupss
