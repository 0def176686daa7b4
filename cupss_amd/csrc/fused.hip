// fused.hip -- the fused two-kernel step for 2D systems: the first dynamic
// field phi, fields linear in a dynamic field ("derived": psi = M_psi(q) u
// with no implicit operator and no noise, e.g. iqxh = iqx*h) and stored
// fields -- further dynamic fields, constraints of dynamic-field products,
// other constraints and coefficient fields (fused.hpp).  Covers diffusion,
// Cahn-Hilliard, Edwards-Wilkinson, KPZ, model H and reaction-diffusion
// systems.  Every launch serves any number of instances (systems) of one
// size class through a table of instance descriptors (FusedInst) and a
// per-workgroup block table.
//
// Pipeline state between the kernels, all column-major (element (kx, y) at
// kx*sy + y) so that the column kernel streams whole contiguous columns:
//   phi_hat  two spectra, [parity] in and [parity^1] out
//   Z_f  = IFFT_y(mask_f * L_f * phi_hat)   for each real field f needed by a
//          product (f = phi, L = 1; f = psi, L = M_psi); only the columns
//          kx <= sx/(p_f+1) that the dealias mask keeps are stored
//   X_g  = R2C_x(sum of the products of group g)  (rows transformed only)
//   eta  = R2C_x(xi)                        (real-space noise, rows only)
// Per step:
//   row kernel:    a tile of LPB rows of each Z_f is staged through LDS
//                  (runs of LPB*8 contiguous bytes per column), C2R along x
//                  -> real dealiased fields -> products, noise -R2C-> X_g,
//                  eta rows, written back through the same tile
//   column kernel: X_g, eta columns -FFT_y-> spectral terms; constraints of
//                  dynamic-field products; update of phi (setDynamic_k);
//                  the stored fields; mask_f * L_f * u_new -IFFT_y-> Z_f
// Terms with equal prefactor lists form one group: M*FFT(a) + M*FFT(b) =
// M*FFT(a + b).  The order of phases A-D of the reference
// (src/evolver.cpp:199-226) is kept: derived fields are evaluated from phi
// at the start of the step (phase A/B) and used by phi's products in phase
// C; phi's own dealiased copy is zero before its first update (step 0).
//
// A run starts with a tiled transpose of the system's spectrum into the
// column-major buffer and ends with the transpose back (plus the derived
// fields); instances whose step needs no transform advance any number of
// steps per launch in registers (k_felem).
#include <hip/hip_runtime.h>

#include "fft_core.hpp"
#include "fused.hpp"
#include "fused_tiles.hpp"
#include "philox.hpp"
#include "update_math.hpp"

namespace cupss {

// ------------------------------------------------------------ row and column kernels

template <int NC, int LPB, int MAXR, bool SINGLE>
__global__ __launch_bounds__((FRowCfg<NC, LPB, MAXR, SINGLE>::THREADS)) void k_frows(const FusedInst *__restrict__ insts,
                                                                          const FusedBlock *__restrict__ blocks,
                                                                          uint32_t step_rel,
                                                                          const float2 *__restrict__ sets)
{
    using C = FRowCfg<NC, LPB, MAXR, SINGLE>;
    __shared__ __align__(16) float2 tws[2 * NC];
    __shared__ __align__(16) float2 tst[tw_stage_alloc(NC, C::E)];
    __shared__ float2 tile[C::LEN];
    const FusedBlock blk = blocks[blockIdx.x];
    if (blk.inst < 0) return;
    frows_tile<NC, LPB, MAXR, SINGLE>(insts[blk.inst], blk.line, step_rel, sets, true, tws, tst, tile);
}

template <int N, int TWD, bool CONS, bool XDYN>
__global__ __launch_bounds__((FColCfg<N, TWD>::THREADS)) void k_fcols(const FusedInst *__restrict__ insts,
                                                                   const FusedBlock *__restrict__ blocks,
                                                                   int parity, uint32_t step_rel, int mode,
                                                                   const float2 *__restrict__ sets,
                                                                   unsigned long long *__restrict__ ts)
{
    using C = FColCfg<N, TWD>;
    __shared__ __align__(16) float2 tws[tw_stage_alloc(N, C::E)];
    __shared__ float2 lds[TWD * C::LL];
    const FusedBlock blk = blocks[blockIdx.x];
    if (blk.inst < 0) return;
    if (mode == 0 && insts[blk.inst].resume) return;  // Z_f of this state left by the previous run
    // launch timing (ts != null): earliest workgroup start and latest end in
    // ticks of the constant-rate wall clock, spread over FUSED_TS_SLOTS
    // cache lines so that the workgroups' atomics do not contend
    unsigned long long *slot = ts ? ts + (size_t)(blockIdx.x % FUSED_TS_SLOTS) * FUSED_TS_STRIDE : nullptr;
    if (slot && threadIdx.x == 0) atomicMin(&slot[0], (unsigned long long)wall_clock64());
    fcols_tile<N, TWD, CONS, XDYN>(insts[blk.inst], blk.line, parity, step_rel, mode, sets, true, tws, lds);
    if (slot) {
        __syncthreads();
        if (threadIdx.x == 0) atomicMax(&slot[1], (unsigned long long)wall_clock64());
    }
}

// ------------------------------------------------------------ small instances

// Instances small enough for one workgroup (64^2): K steps in one
// launch, one workgroup per instance, each step the same row and column
// tiles as the two-kernel step (so the same results bit for bit) in turn,
// separated by workgroup barriers -- no launch per pass, and the
// instance's buffers stay in the L2 of its workgroup's XCD.
template <int NC, int N, bool CONS, bool XDYN>
struct FSmallCfg {
    static constexpr int THREADS = 512;
    static constexpr int LPB = THREADS / FRowCfg<NC, 1, 3>::T;
    static constexpr int TWD = THREADS / FColCfg<N, 1>::T;
    static constexpr int LDSN = FRowCfg<NC, LPB, 3>::LEN > TWD * FColCfg<N, TWD>::LL
                                    ? FRowCfg<NC, LPB, 3>::LEN
                                    : TWD * FColCfg<N, TWD>::LL;
    static constexpr bool valid()
    {
        return FRowCfg<NC, LPB, 3>::valid() && FColCfg<N, TWD>::valid() && LPB <= N &&
               (2 * NC + tw_stage_alloc(NC, FRowCfg<NC, LPB, 3>::E) + tw_stage_alloc(N, FColCfg<N, TWD>::E) + LDSN) *
                       8 <=
                   150 * 1024;
    }
};

template <int NC, int N, bool CONS, bool XDYN>
__global__ __launch_bounds__(512) void k_fsmall(const FusedInst *__restrict__ insts, const int *__restrict__ ids,
                                                int n0, int k, int rel0, const float2 *__restrict__ sets,
                                                unsigned long long *__restrict__ ts)
{
    using C = FSmallCfg<NC, N, CONS, XDYN>;
    __shared__ float2 twr[2 * NC];
    __shared__ __align__(16) float2 tsr[tw_stage_alloc(NC, FRowCfg<NC, C::LPB, 3>::E)];
    __shared__ __align__(16) float2 twc[tw_stage_alloc(N, FColCfg<N, C::TWD>::E)];
    __shared__ float2 buf[C::LDSN];
    unsigned long long *slot = ts ? ts + (size_t)(blockIdx.x % FUSED_TS_SLOTS) * FUSED_TS_STRIDE : nullptr;
    if (slot && threadIdx.x == 0) atomicMin(&slot[0], (unsigned long long)wall_clock64());
    const FusedInst &a = insts[ids[blockIdx.x]];
    load_twiddles<2 * NC>(twr, sets);
    load_stage_twiddles<NC, FRowCfg<NC, C::LPB, 3>::E>(tsr, sets);
    load_stage_twiddles<N, FColCfg<N, C::TWD>::E>(twc, sets);
    __syncthreads();
    for (int n = n0; n < n0 + k; n++) {
        const uint32_t rel = (uint32_t)(n - rel0);
        for (int y0 = 0; y0 < N; y0 += C::LPB) frows_tile<NC, C::LPB, 3>(a, y0, rel, sets, false, twr, tsr, buf);
        // rows ended with a barrier: X_g and eta are written, the buffer is free
        for (int x0 = 0; x0 <= NC; x0 += C::TWD) fcols_tile<N, C::TWD, CONS, XDYN>(a, x0, n & 1, rel, 1, sets, false, twc, buf);
        __syncthreads();  // Z_f and the spectra written; the buffer is free for the rows
    }
    if (slot && threadIdx.x == 0) atomicMax(&slot[1], (unsigned long long)wall_clock64());
}

// ------------------------------------------------------------ transposes

// tile (tx, ty) of an instance: columns kx in [tx*S, tx*S+S), rows ky in
// [ty*S, ty*S+S) of the half spectrum
__device__ __forceinline__ void tile_origin(const Geom &g, int line, int &x0, int &y0)
{
    const int ntx = (g.nc1 + FUSED_TILE - 1) / FUSED_TILE;
    x0 = (line % ntx) * FUSED_TILE;
    y0 = (line / ntx) * FUSED_TILE;
}

// one tile of a natural half spectrum into a column-major one
__device__ __forceinline__ void tile_to_cm(float2 (&s)[FUSED_TILE][FUSED_TILE + 1], const Geom &g, int x0, int y0,
                                           const float2 *__restrict__ src, float2 *__restrict__ dst)
{
    constexpr int S = FUSED_TILE;
    for (int q = threadIdx.x; q < S * S; q += blockDim.x) {
        const int i = q % S, j = q / S;
        if (x0 + i < g.nc1 && y0 + j < g.sy) s[j][i] = gload(src, (long)(y0 + j) * g.nc1 + x0 + i);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < S * S; q += blockDim.x) {
        const int j = q % S, i = q / S;
        if (x0 + i < g.nc1 && y0 + j < g.sy) gstore(dst, (long)(x0 + i) * g.sy + y0 + j, s[j][i]);
    }
    __syncthreads();
}

// one tile of a column-major half spectrum into a natural one, each value
// times M (npres = 0: copied)
__device__ __forceinline__ void tile_to_nat(float2 (&s)[FUSED_TILE][FUSED_TILE + 1], const FusedInst &a, int x0,
                                            int y0, const float2 *__restrict__ src, float2 *__restrict__ dst,
                                            const TermRefDev &M)
{
    constexpr int S = FUSED_TILE;
    const Geom &g = a.g;
    for (int q = threadIdx.x; q < S * S; q += blockDim.x) {
        const int j = q % S, i = q / S;
        if (x0 + i < g.nc1 && y0 + j < g.sy) s[j][i] = gload(src, (long)(x0 + i) * g.sy + y0 + j);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < S * S; q += blockDim.x) {
        const int i = q % S, j = q / S;
        const int kx = x0 + i, ky = y0 + j;
        if (kx < g.nc1 && ky < g.sy) {
            const long h = (long)ky * g.nc1 + kx;
            if (M.npres == 0) {
                gstore(dst, h, s[j][i]);
            } else {
                const Bin b = make_bin(g, kx, ky, 0);
                gstore(dst, h, apply_mult(multiplier(a.pool, M.pres0, M.npres, M.mult_i, b), M.mult_i, s[j][i]));
            }
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(256) void k_ftrans_in(const FusedInst *__restrict__ insts,
                                                   const FusedBlock *__restrict__ blocks)
{
    __shared__ float2 s[FUSED_TILE][FUSED_TILE + 1];
    const FusedBlock blk = blocks[blockIdx.x];
    if (blk.inst < 0) return;
    const FusedInst &a = insts[blk.inst];
    int x0, y0;
    tile_origin(a.g, blk.line, x0, y0);
    if (!a.resume) tile_to_cm(s, a.g, x0, y0, a.nat, a.spec[0]);
    if (!a.cont)
        for (int c = 0; c < a.ncons; c++) tile_to_cm(s, a.g, x0, y0, a.cnat[c], a.cs[c][0]);
}

// column-major phi and stored dynamic fields [fin] -> natural; stored
// constraints of the last step's start ([fin^1]) -> natural; the derived
// fields of the last step's starting values of their base ([fin^1]) in
// natural layout
__global__ __launch_bounds__(256) void k_fsettle(const FusedInst *__restrict__ insts,
                                                 const FusedBlock *__restrict__ blocks, int fin)
{
    __shared__ float2 s[FUSED_TILE][FUSED_TILE + 1];
    const FusedBlock blk = blocks[blockIdx.x];
    if (blk.inst < 0) return;
    const FusedInst &a = insts[blk.inst];
    int x0, y0;
    tile_origin(a.g, blk.line, x0, y0);
    const TermRefDev copy{nullptr, 0, 0, 0, 0};
    tile_to_nat(s, a, x0, y0, a.spec[fin], a.nat, copy);
    for (int c = 0; c < a.ncons; c++)
        tile_to_nat(s, a, x0, y0, a.cs[c][a.tgt[1 + c].dyn ? fin : fin ^ 1], a.cnat[c], copy);
    for (int d = 0; d < a.nder; d++)
        tile_to_nat(s, a, x0, y0, a.dbase[d] < 0 ? a.spec[fin ^ 1] : a.cs[a.dbase[d]][fin ^ 1], a.dout[d], a.dmul[d]);
}

// ------------------------------------------------------------ operator tables

// every table of one instance, a thread per bin (column-major)
__global__ __launch_bounds__(256) void k_ftables(const FusedInst *__restrict__ insts, int inst)
{
    const FusedInst &a = insts[inst];
    const long h = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= a.g.nh) return;
    ColBins<1> cb;
    col_bins<1, 1>(a.g, (int)(h / a.g.sy), (int)(h % a.g.sy), cb);
    for (int i = 0; i < a.ntab; i++) {
        const FusedTab &T = a.tab[i];
        float m[1];
        if (T.kind == TAB_MULT) {
            multiplier_col<1>(a.pool, T.pres0, T.npres, T.mult_i, cb, m);
        } else {
            float sum = T.kind == TAB_DYNAMIC ? 1.0f : 0.0f;
            for (int k = 0; k < T.npres; k++) {
                const PresDev P = T.pres0 < 0 ? a.u.imp[k] : a.pool[T.pres0 + k];
                float th = P.c;
                for (int j = 0; j < P.q2n; j++) th *= cb.q2[0];
                if (P.invq != 0) {
                    const float iq = col_iq(cb, 0);
                    for (int j = 0; j < P.invq; j++) th *= iq;
                }
                if (T.kind == TAB_DYNAMIC)
                    sum -= a.u.dt * th;
                else
                    sum += th;
            }
            m[0] = T.kind == TAB_CONSTRAINT && cb.zero[0] ? 1.0f : __builtin_amdgcn_rcpf(sum);
        }
        gstore(a.mtab, (long)i * a.g.nh + h, m[0]);
    }
}

// ------------------------------------------------------------ elementwise

// Instances whose step needs no transform (no products, noise drawn in
// spectral space or absent): one thread per pair of bins (kx, j, kz),
// (kx, j + sy/2, kz) -- the pair that shares a noise draw -- advances
// nsteps steps in registers.  The explicit terms are linear in phi or
// constant, so their sum is (ar + i ai) phi_hat + cst; the step is the
// dynamic branch of finish_update with D(q) and the noise amplitude
// evaluated once.
__global__ __launch_bounds__(FUSED_ELEM_BLOCK) void k_felem(const FusedInst *__restrict__ insts,
                                                            const FusedBlock *__restrict__ blocks, int parity,
                                                            uint32_t step_rel, int nsteps)
{
    const FusedBlock blk = blocks[blockIdx.x];
    if (blk.inst < 0) return;
    const FusedInst &a = insts[blk.inst];
    const Geom &g = a.g;
    const int hy = g.sy / 2;  // sy >= 8 for fused instances
    const long pidx = (long)blk.line + threadIdx.x;
    if (pidx >= g.nh / 2) return;  // no barriers below
    // Pairs of the interior columns 1..nc-1 first, then those of the kx = 0
    // and kx = nc planes, whose noise takes two Philox calls (Hermitian
    // partners): only the last waves take that branch, none diverges on it.
    const long prow = (long)hy * g.sz, nint = (long)(g.nc - 1) * prow;
    int kx;
    long r;
    if (pidx < nint) {
        kx = 1 + (int)(pidx % (g.nc - 1));
        r = pidx / (g.nc - 1);
    } else {
        const long q = pidx - nint;
        kx = (q & 1) ? g.nc : 0;
        r = q >> 1;
    }
    const int j = (int)(r % hy), kz = (int)(r / hy);
    const UpdateArgs &u = a.u;
    const bool noisy = u.noisy && a.noise_mode == NOISE_SPECTRAL;
    Bin b[2];
    float ar[2], ai[2], D[2], pn[2];
    float2 cst[2], cur[2];
#pragma unroll
    for (int w = 0; w < 2; w++) {
        b[w] = make_bin(g, kx, j + w * hy, kz);
        ar[w] = 0.f;
        ai[w] = 0.f;
        cst[w] = make_float2(0.f, 0.f);
        for (int ti = 0; ti < u.nterms; ti++) {
            const TermRefDev &TR = u.terms[ti];
            const float m = multiplier(u.pres, TR.pres0, TR.npres, TR.mult_i, b[w]);
            if (TR.kind == TERM_CONST) {
                if (b[w].h == 0) cst[w] = cadd(cst[w], apply_mult(m, TR.mult_i, make_float2((float)g.n, 0.f)));
            } else if (TR.mult_i) {
                ai[w] += m;
            } else {
                ar[w] += m;
            }
        }
        D[w] = 1.0f;
        for (int i = 0; i < u.nimp; i++) {
            const PresDev P = u.imp[i];
            float th = P.c;
            if (P.q2n != 0) th *= ipow(b[w].q2, P.q2n);
            if (P.invq != 0) th *= ipow(b[w].iqd, P.invq);
            D[w] -= u.dt * th;
        }
        D[w] = __builtin_amdgcn_rcpf(D[w]);  // 1/D(q): hardware reciprocal, once per bin
        pn[w] = noisy ? noise_amplitude(u, b[w]) : 0.f;
        cur[w] = gload(a.spec[parity], b[w].h);
    }
    const uint64_t s0 = a.step_base + step_rel;
    for (int n = 0; n < nsteps; n++) {
        if (n == nsteps - 1) {
            for (int d = 0; d < a.nder; d++) {
                const TermRefDev &M = a.dmul[d];
#pragma unroll
                for (int w = 0; w < 2; w++)
                    gstore(a.dout[d], b[w].h,
                           apply_mult(multiplier(a.pool, M.pres0, M.npres, M.mult_i, b[w]), M.mult_i, cur[w]));
            }
        }
        float2 eta[2] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
        if (noisy) {
            const uint64_t step = s0 + (uint64_t)n;
            spectral_noise_pair(g, kx, j, kz, (uint32_t)step, (uint32_t)(step >> 32), a.stream, a.key0, a.key1,
                                eta[0], eta[1]);
        }
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const float2 c = cur[w];
            float2 s = c;
            s.x += u.dt * (ar[w] * c.x - ai[w] * c.y + cst[w].x);
            s.y += u.dt * (ar[w] * c.y + ai[w] * c.x + cst[w].y);
            if (noisy) {
                s.x += pn[w] * eta[w].x;
                s.y += pn[w] * eta[w].y;
            }
            if (u.nimp > 0) {
                s.x *= D[w];
                s.y *= D[w];
            }
            cur[w] = s;
        }
    }
#pragma unroll
    for (int w = 0; w < 2; w++) gstore(a.spec[parity ^ (nsteps & 1)], b[w].h, cur[w]);
}

// ------------------------------------------------------------ dispatch

#define FUSED_ROW_CASES(X) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048)
#define FUSED_COL_CASES(X) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)
#define FUSED_LPB(X) X(1) X(2) X(4) X(8) X(16)
#define FUSED_TWD(X) X(1) X(2) X(4) X(8) X(16)

bool fused_supported(int sx, int sy, int sz)
{
    if (sz > 1) return sz >= 8 && sz <= 1024 && sx >= 16 && sx <= 2048 && sy >= 8 && sy <= 4096;  // 3D
    return sx >= 16 && sx <= 4096 && sy >= 8 && sy <= 4096;
}

// wide row kernels (more than 3 real fields) for the sizes such systems use;
// narrow ones (at most 2: fewer registers, one more wave per SIMD) for the
// sizes of large instances (others run the 3-field kernel)
#define FUSED_WIDE_NC(NC) ((NC) >= 32 && (NC) <= 1024)
#define FUSED_NARROW_NC(NC) ((NC) >= 32 && (NC) <= 1024)

int fused_row_width(int nreal) { return nreal <= 2 ? 2 : (nreal == 3 ? 3 : FUSED_MAX_REAL); }

bool fused_shapes_exist(int sx, int sy, int sz, int nreal)
{
    const int nc = sx / 2;
    if (sz > 1) return nreal <= 3 || (nc >= 32 && nc <= 1024);
    return !fused_row_shapes(nc, sy, fused_row_width(nreal)).empty() && !fused_col_shapes(sy).empty();
}

template <int NC, int MAXR>
static std::vector<int> row_shapes(int ny)
{
    std::vector<int> v;
#define X(LPB) \
    if (FRowCfg<NC, LPB, MAXR>::valid() && LPB <= ny) v.push_back(LPB);
    FUSED_LPB(X)
#undef X
    return v;
}

std::vector<int> fused_row_shapes(int nc, int ny, int width)
{
    switch (nc) {
#define X(NC)                                                                                            \
    case NC:                                                                                             \
        if (width > 3) return FUSED_WIDE_NC(NC) ? row_shapes<NC, FUSED_MAX_REAL>(ny) : std::vector<int>(); \
        if (width == 2 && FUSED_NARROW_NC(NC)) return row_shapes<NC, 2>(ny);                              \
        return row_shapes<NC, 3>(ny);
        FUSED_ROW_CASES(X)
#undef X
    default:
        return {};
    }
}

template <int N>
static std::vector<int> col_shapes()
{
    std::vector<int> v;
#define X(TWD) \
    if (FColCfg<N, TWD>::valid()) v.push_back(TWD);
    FUSED_TWD(X)
#undef X
    return v;
}

std::vector<int> fused_col_shapes(int ny)
{
    switch (ny) {
#define X(N) \
    case N:  \
        return col_shapes<N>();
        FUSED_COL_CASES(X)
#undef X
    default:
        return {};
    }
}

int fused_col_lanes(int ny)
{
    switch (ny) {
#define X(N) \
    case N:  \
        return FColCfg<N, 1>::T;
        FUSED_COL_CASES(X)
#undef X
    default:
        return 0;
    }
}

// Rows of 256 and 512 complex points: pairs (FRowCfg::PAIR) up to 4096 rows a
// launch, beyond that their LDS and registers cost more than the latency they
// hide.  us per step, singly / pairs: Gray-Scott 512^2 x8 (4096 rows) 36.4 /
// 35.6, x16 53.4 / 56.0, x32 97 / 100; a three-field system 512^2 x8 31.5 /
// 31.0, x16 45.1 / 48.1, 1024^2 x4 (4096 rows) 59.7 / 59.8, x8 93 / 100.
constexpr long ROW_PAIRS_MAX = 4096;
template <int NC, int MAXR>
static hipError_t frows_n(int lpb, const FusedInst *inst, const FusedBlock *blocks, int nblocks, uint32_t step_rel,
                          hipStream_t s, const float2 *sets)
{
    constexpr bool BOTH = NC >= 256 && FRowCfg<NC, 1, MAXR>::PAIR;
#define L(LPB, SINGLE)                                                                                    \
    hipLaunchKernelGGL((k_frows<NC, LPB, MAXR, SINGLE>), dim3(nblocks),                                  \
                       dim3(FRowCfg<NC, LPB, MAXR, SINGLE>::THREADS), 0, s, inst, blocks, step_rel, sets)
#define X(LPB)                                                           \
    if constexpr (FRowCfg<NC, LPB, MAXR>::valid()) {                    \
        if (lpb == LPB) {                                                \
            if (BOTH && (long)nblocks * LPB > ROW_PAIRS_MAX)             \
                L(LPB, BOTH);                                            \
            else                                                         \
                L(LPB, false);                                           \
            return hipGetLastError();                                    \
        }                                                                \
    }
    FUSED_LPB(X)
#undef X
#undef L
    return hipErrorInvalidValue;
}

hipError_t fused_rows_launch(int nc, int lpb, int width, const FusedInst *inst, const FusedBlock *blocks,
                             int nblocks, uint32_t step_rel, hipStream_t s)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    switch (nc) {
#define X(NC)                                                                                      \
    case NC:                                                                                       \
        if (width > 3) {                                                                           \
            if constexpr (FUSED_WIDE_NC(NC))                                                       \
                return frows_n<NC, FUSED_MAX_REAL>(lpb, inst, blocks, nblocks, step_rel, s, sets); \
            return hipErrorInvalidValue;                                                           \
        }                                                                                          \
        if constexpr (FUSED_NARROW_NC(NC))                                                         \
            if (width == 2) return frows_n<NC, 2>(lpb, inst, blocks, nblocks, step_rel, s, sets);  \
        return frows_n<NC, 3>(lpb, inst, blocks, nblocks, step_rel, s, sets);
        FUSED_ROW_CASES(X)
#undef X
    default:
        return hipErrorInvalidValue;
    }
}

template <int N>
static hipError_t fcols_n(int twd, int stored, const FusedInst *inst, const FusedBlock *blocks, int nblocks,
                          int parity, uint32_t step_rel, int mode, hipStream_t s, const float2 *sets,
                          unsigned long long *ts)
{
#define L(CONS, XDYN, TWD)                                                                                    \
    hipLaunchKernelGGL((k_fcols<N, TWD, CONS, XDYN>), dim3(nblocks), dim3(FColCfg<N, TWD>::THREADS), 0, s, inst, \
                       blocks, parity, step_rel, mode, sets, ts)
#define X(TWD)                                   \
    if constexpr (FColCfg<N, TWD>::valid()) {   \
        if (twd == TWD) {                        \
            if (stored == 2)                     \
                L(true, true, TWD);              \
            else if (stored == 1)                \
                L(true, false, TWD);             \
            else                                 \
                L(false, false, TWD);            \
            return hipGetLastError();            \
        }                                        \
    }
    FUSED_TWD(X)
#undef X
#undef L
    return hipErrorInvalidValue;
}

hipError_t fused_cols_launch(int ny, int twd, int stored, const FusedInst *inst, const FusedBlock *blocks,
                             int nblocks, int parity, uint32_t step_rel, int mode, hipStream_t s,
                             unsigned long long *ts)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    switch (ny) {
#define X(N) \
    case N:  \
        return fcols_n<N>(twd, stored, inst, blocks, nblocks, parity, step_rel, mode, s, sets, ts);
        FUSED_COL_CASES(X)
#undef X
    default:
        return hipErrorInvalidValue;
    }
}

// 64^2: one workgroup takes the steps in one launch, without a kernel boundary
// per pass; on 128^2 one CU's vector issue is the bound and two launches per
// step over the chip are faster.  us per step, one workgroup / two launches:
// CH 64^2 5.9 / 8.2, KPZ 64^2 11.8 / 12.9, Gray-Scott 64^2 16.6 / 18.0; 128^2:
// KPZ alone 43 / 12.5, 64 of them 43.6 / 18.6, 512 91 / 73; Gray-Scott alone
// 49 / 15.4, 64 50 / 21.6.  Only where the instances just fill the CUs is one
// workgroup each the better choice there: 256 of Gray-Scott 53 / 56, of
// Cahn-Hilliard 25.7 / 26.6, of KPZ 48 / 45.
bool fused_small_class(int nc, int ny, int width) { return width <= 3 && nc == 32 && ny == 64; }

template <int NC, int N>
static hipError_t fsmall_n(int stored, const FusedInst *inst, const int *ids, int nids, int n0, int k, int rel0,
                           hipStream_t s, const float2 *sets, unsigned long long *ts)
{
#define L(CONS, XDYN)                                                                                         \
    static_assert(FSmallCfg<NC, N, CONS, XDYN>::valid(), "small-instance tile");                           \
    hipLaunchKernelGGL((k_fsmall<NC, N, CONS, XDYN>), dim3(nids), dim3(FSmallCfg<NC, N, CONS, XDYN>::THREADS), \
                       0, s, inst, ids, n0, k, rel0, sets, ts)
    if (stored == 2) {
        L(true, true);
    } else if (stored == 1) {
        L(true, false);
    } else {
        L(false, false);
    }
#undef L
    return hipGetLastError();
}

hipError_t fused_small_launch(int nc, int ny, int stored, const FusedInst *inst, const int *ids, int nids, int n0,
                              int k, int rel0, hipStream_t s, unsigned long long *ts)
{
    const float2 *sets = twiddle_sets(s);
    if (!sets) return hipErrorOutOfMemory;
    if (nids <= 0 || k <= 0) return hipSuccess;
    if (nc == 32 && ny == 64) return fsmall_n<32, 64>(stored, inst, ids, nids, n0, k, rel0, s, sets, ts);
    return hipErrorInvalidValue;
}

hipError_t fused_tables_launch(const FusedInst *inst, int i, long nh, hipStream_t s)
{
    hipLaunchKernelGGL(k_ftables, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, s, inst, i);
    return hipGetLastError();
}

hipError_t fused_transpose_in_launch(const FusedInst *inst, const FusedBlock *blocks, int nblocks, hipStream_t s)
{
    hipLaunchKernelGGL(k_ftrans_in, dim3(nblocks), dim3(256), 0, s, inst, blocks);
    return hipGetLastError();
}

hipError_t fused_settle_launch(const FusedInst *inst, const FusedBlock *blocks, int nblocks, int fin, hipStream_t s)
{
    hipLaunchKernelGGL(k_fsettle, dim3(nblocks), dim3(256), 0, s, inst, blocks, fin);
    return hipGetLastError();
}

hipError_t fused_elem_launch(const FusedInst *inst, const FusedBlock *blocks, int nblocks, int parity,
                             uint32_t step_rel, int nsteps, hipStream_t s)
{
    hipLaunchKernelGGL(k_felem, dim3(nblocks), dim3(FUSED_ELEM_BLOCK), 0, s, inst, blocks, parity, step_rel,
                       nsteps);
    return hipGetLastError();
}

__global__ void k_ts_reset(unsigned long long *ts, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n * FUSED_TS_SLOTS) {
        ts[(size_t)i * FUSED_TS_STRIDE] = ~0ull;
        ts[(size_t)i * FUSED_TS_STRIDE + 1] = 0ull;
    }
}

hipError_t fused_ts_reset_launch(unsigned long long *ts, int n, hipStream_t s)
{
    const int m = n * FUSED_TS_SLOTS;
    hipLaunchKernelGGL(k_ts_reset, dim3((m + 255) / 256), dim3(256), 0, s, ts, n);
    return hipGetLastError();
}

}  // namespace cupss
