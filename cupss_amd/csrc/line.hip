// line.hip -- 1D systems (sy = sz = 1): the whole step program of the general
// path (system.hip run_phase: noise, products, updates, dealiased copies, in
// phase order, src/evolver.cpp:199-226) by one workgroup, any number of steps
// per launch.
//
// A 1D grid has at most 4096 points, far too few for a launch per pass: the
// general program takes seven launches for a step of a KPZ line, 27 us of
// which nearly all is launch and first-access latency.  Here every field's
// spectrum, the dealiased copies, the product transforms and the noise stay
// in LDS for the whole run, and the stages of a step are separated by
// workgroup barriers.  Up to 512 complex points one wavefront takes one
// transform (independent transforms run side by side on different wavefronts,
// the draws of the next step on those left over); longer ones take all of the
// workgroup's, one after another (LineCfg).  What bounds it is the chain of a step: an inverse and
// a forward transform of about 1.6 us each and two updates of 0.9 us, mostly
// LDS and scalar-load latency.  Measured, us per step of a KPZ line with
// real-space noise, general program -> here: 64 points 28 -> 3.5, 256 points
// 27 -> 3.4, 1024 points 28 -> 5.2, 2048 points 39 -> 9.9, 4096 points
// 51 -> 13.5.  It is faster over the whole range, so the general program
// serves 1D only where the program does not fit (line_plan).
//
// The multipliers M(q), 1/D(q) and noise amplitudes do not change during a
// run; k_line_tables evaluates them once per program into tables of one float
// per bin (a 1D table is a few KB; a 2D one would cost a pass over memory per
// step, so the 2D kernels evaluate theirs).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "fft_core.hpp"
#include "internal.hpp"
#include "philox.hpp"
#include "system_impl.hpp"
#include "update_math.hpp"

namespace cupss {

constexpr int LINE_MAX_FIELDS = 16;
constexpr int LINE_MAX_TERMS = 48;
constexpr int LINE_LDS = 150 * 1024;
constexpr int LINE_CHUNK = 4096;  // steps per launch

struct LineField {
    int dynamic, noisy, cut;   // cut: largest kx that the dealias mask keeps
    int t0, nterms, nimp;      // its terms [t0, t0 + nterms)
    int dslot, eslot;          // dealiased copy and noise transform (-1: none)
    uint32_t key0, key1;
    float2 *spec[2];
    float *dreal;
};

struct LineTerm {
    int kind;                  // TermKind
    int mult_i, src, srcdyn;   // TERM_FIELD: the field, and whether it is dynamic
    int xslot, nfac;           // TERM_BUFFER: product transform
    int fac[MAX_FACTORS];      // dealiased slots of the factors
};

// transform of one stage: R2C of a product or of a noise field, or the
// dealiased copy of a field
enum LineTask : int { LINE_PRODUCT = 0, LINE_NOISE = 1, LINE_DEALIAS = 2 };
struct LineJob {
    int task, id;
};

struct LineProg {
    Geom g;
    float dt, scale;           // scale: 1/N of the inverse transform
    int nf, nterms, ndreal, nx, neta;
    int spectral;              // noise drawn per bin
    int n[2];                  // fields of each phase (0: constraints, 1: dynamic)
    int field[2][LINE_MAX_FIELDS];
    // jobs of the stages: before each phase's updates, and after them
    int njob[2][2];
    LineJob job[2][2][LINE_MAX_TERMS + 2 * LINE_MAX_FIELDS];
    int draws[LINE_MAX_FIELDS];  // the fields that draw real-space noise
    LineField f[LINE_MAX_FIELDS];
    LineTerm t[LINE_MAX_TERMS];
    const float *mult;         // [nterms][nc1]
    const float *rdiv;         // [nf][nc1]: 1/D (dynamic) or 1/L (constraint)
    const float *amp;          // [nf][nc1]
};

template <int NC>
struct LineCfg {
    // Up to 512 complex points: one wavefront per transform, up to four side
    // by side, and four more wavefronts for the draws and updates.  Longer
    // transforms are bound by the issue of one wavefront, so all four or
    // eight wavefronts take each of them, with workgroup barriers.
    static constexpr bool ONE = NC <= 512;
    static constexpr int E = ONE ? row_elems(NC) : 4;
    static constexpr int T = NC / E;
    static constexpr int GROUP = ONE ? 64 : T;       // lanes of one transform
    static constexpr int G = ONE ? 4 : 1;
    static constexpr int THREADS = ONE ? 512 : T;
    static constexpr int LL = lds_len(NC);
    // twiddles in LDS (table 2*NC, then the stage tables) where they leave
    // room for the fields
    static constexpr bool TWL = ONE;
    static constexpr int TWLEN = TWL ? 2 * NC + tw_stage_alloc(NC, E) : 0;
};

// LDS entries (8 bytes): twiddles, transform lines, then per field, slot and
// noise field the arrays; with `tables` the multiplier tables too
static long line_entries(const LineProg &p, int tw, int lines, bool tables)
{
    const long nc = p.g.nc, nc1 = p.g.nc1;
    return tw + lines + p.nf * 2 * nc1 + p.ndreal * nc + p.nx * nc1 + p.neta * 2 * nc1 +
           (tables ? ((p.nterms + 2 * p.nf) * nc1 + 1) / 2 : 0);
}

// TAB: the multiplier tables are copied to LDS (they stay in memory where the
// fields leave no room)
template <int NC, bool TAB>
__global__ __launch_bounds__(LineCfg<NC>::THREADS) void k_line(const LineProg *__restrict__ prog, uint32_t cur,
                                                               uint64_t step0, int nsteps,
                                                               const float2 *__restrict__ sets)
{
    using C = LineCfg<NC>;
    constexpr int E = C::E, T = C::T, TH = C::THREADS, NC1 = NC + 1;
    constexpr bool WL = C::ONE;
    extern __shared__ __align__(16) float2 lds[];
    const LineProg &P = *prog;
    const float dt = P.dt, scale = P.scale;
    const int neta = P.neta, spectral = P.spectral;
    const int njob00 = P.njob[0][0], njob01 = P.njob[0][1], njob10 = P.njob[1][0], njob11 = P.njob[1][1];
    const int nfield[2] = {P.n[0], P.n[1]};
    // lanes beyond a short transform's T repeat its work on the same line
    // (same values to the same places); grp is uniform over a wavefront
    const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x / C::GROUP);
    const int t = ((int)threadIdx.x % C::GROUP) % T;
    float2 *p = lds + C::TWLEN;
    float2 *L = p + (grp < C::G ? grp : 0) * C::LL;
    p += C::G * C::LL;
    float2 *spec = p;  // [nf][2][NC1]
    p += P.nf * 2 * NC1;
    float2 *dreal = p;  // [ndreal][NC]: pairs of real points
    p += P.ndreal * NC;
    float2 *X = p;  // [nx][NC1]
    p += P.nx * NC1;
    float2 *eta = p;  // [neta][NC1]: noise transforms
    p += P.neta * NC1;
    float2 *xi = p;  // [neta][NC1]: normals, pairs of cells
    p += P.neta * NC1;
    float *tab = reinterpret_cast<float *>(p);  // mult, rdiv, amp
    auto table = [&](const float *g, int row, int h) {
        if constexpr (TAB)
            return tab[(int)(g - P.mult) + row * NC1 + h];
        else
            return gload(g, (long)row * NC1 + h);
    };

    // exp(-2 pi i j / 2NC) for the real transforms' outer pass, and the stage
    // tables of the NC-point transform
    if constexpr (C::TWL) {
        load_twiddles<2 * NC>(lds, sets);
        load_stage_twiddles<NC, E>(lds + 2 * NC, sets);
    }
    const float2 *tw2 = C::TWL ? lds : sets + 2 * NC;
    const float2 *tws = C::TWL ? lds + 2 * NC : sets + tw_stage_offset(NC, E);
    if constexpr (TAB)
        for (int i = threadIdx.x; i < (P.nterms + 2 * P.nf) * NC1; i += TH) tab[i] = gload(P.mult, i);
    for (int i = 0; i < P.nf; i++) {
        const LineField &F = P.f[i];
        const float2 *__restrict__ s = F.spec[(cur >> i) & 1];
        for (int h = threadIdx.x; h < NC1; h += TH) spec[(2 * i) * NC1 + h] = gload(s, h);
        if (F.dslot >= 0)
            for (int m = threadIdx.x; m < NC; m += TH)
                dreal[F.dslot * NC + m] = gload(reinterpret_cast<const float2 *>(F.dreal), m);
    }

    // normals of every real-space noise field of a step, by the lanes
    // lane, lane + lanes, ...: one Philox block gives four cells
    auto draw = [&](int lane, int lanes, uint64_t step) {
        for (int q = 0; q < neta; q++) {
            const int i = P.draws[q];
            const LineField &F = P.f[i];
            float2 *z = xi + F.eslot * NC1;
            for (int b = lane; b < (NC + 1) / 2; b += lanes) {
                const Philox4 o = philox4x32_10((uint32_t)b, (uint32_t)step, (uint32_t)(step >> 32), (uint32_t)i,
                                                F.key0, F.key1);
                z[2 * b] = box_muller(o.x[0], o.x[1]);
                z[2 * b + 1] = box_muller(o.x[2], o.x[3]);
            }
        }
    };
    draw(threadIdx.x, TH, step0);
    __syncthreads();

    // the transforms of a stage, one per group of lanes; par: buffer of the
    // spectra that are current
    auto jobs = [&](int ph, int when, int n, const int (&par)[2]) {
        if (grp >= C::G) return;  // a wavefront without a line
        for (int j0 = 0; j0 < n; j0 += C::G) {
            const bool on = j0 + grp < n;
            const LineJob J = P.job[ph][when][on ? j0 + grp : j0];
            float2 v[E];
            if (J.task == LINE_DEALIAS) {
                const LineField &F = P.f[J.id];
                const float2 *x = spec + (2 * J.id + par[F.dynamic]) * NC1;
                const int cut = F.cut;
#pragma unroll
                for (int e = 0; e < E; e++) {
                    const int k = t + e * T;
                    float2 A = x[k], B = x[NC - k];
                    if (k == 0) {
                        A.y = 0.f;
                        B.y = 0.f;
                    }
                    if (k > cut) A = make_float2(0.f, 0.f);
                    if (NC - k > cut) B = make_float2(0.f, 0.f);
                    const float2 Bc = cconj(B);
                    const float2 xo = cmul(csub(A, Bc), tw_lookup<+1, 2 * NC>(tw2, k, 2 * NC));
                    v[e] = cadd(cadd(A, Bc), mul_i<+1>(xo));
                }
                fft_line<NC, E, +1, TW_STAGE, false, WL>(v, L, t, tws);
                if (on) {
#pragma unroll
                    for (int e = 0; e < E; e++) dreal[F.dslot * NC + t + e * T] = cscale(v[e], scale);
                }
            } else {
                float2 *out;
                if (J.task == LINE_NOISE) {
                    out = eta + P.f[J.id].eslot * NC1;
                    const float2 *z = xi + P.f[J.id].eslot * NC1;
#pragma unroll
                    for (int e = 0; e < E; e++) v[e] = z[t + e * T];
                } else {
                    const LineTerm &TR = P.t[J.id];
                    out = X + TR.xslot * NC1;
#pragma unroll
                    for (int e = 0; e < E; e++) v[e] = make_float2(1.f, 1.f);
                    for (int c = 0; c < TR.nfac; c++) {
                        const float2 *r = dreal + TR.fac[c] * NC;
#pragma unroll
                        for (int e = 0; e < E; e++) {
                            const float2 w = r[t + e * T];
                            v[e].x *= w.x;
                            v[e].y *= w.y;
                        }
                    }
                }
                fft_line<NC, E, -1, TW_STAGE, true, WL>(v, L, t, tws);
                if (on) {
#pragma unroll
                    for (int e = 0; e < E; e++) {
                        const int k = t + e * T;
                        const float2 A = v[e];
                        const float2 B = cconj(L[lpad((NC - k) & (NC - 1))]);
                        const float2 xe = cscale(cadd(A, B), 0.5f);
                        const float2 xo = cscale(mul_i<-1>(csub(A, B)), 0.5f);
                        out[k] = k == 0 ? make_float2(xe.x + xo.x, 0.0f)
                                        : cadd(xe, cmul(tw_lookup<-1, 2 * NC>(tw2, k, 2 * NC), xo));
                    }
                    if (t == 0) {
                        const float2 z0 = L[lpad(0)];
                        out[NC] = make_float2(z0.x - z0.y, 0.0f);
                    }
                }
            }
            line_sync<WL>();  // the group's line is free for its next transform
        }
    };
    // setDynamic_k / setNotDynamic_k of every field of the phase, from the
    // values before the phase; a lane's bins (the Nyquist bin among them) go
    // through it together, so their loads are in flight together
    constexpr int HB = (NC1 + TH - 1) / TH < 3 ? (NC1 + TH - 1) / TH : 3;
    auto update_fields = [&](int ph, const int (&par)[2], uint64_t step) {
        for (int q = 0; q < nfield[ph]; q++) {
            const int i = P.field[ph][q];
            const LineField &F = P.f[i];
            const float2 *old = spec + (2 * i + par[ph]) * NC1;
            float2 *out = spec + (2 * i + (par[ph] ^ 1)) * NC1;
            for (int h0 = threadIdx.x; h0 < NC1; h0 += HB * TH) {
                int h[HB];
                float2 acc[HB], s[HB];
#pragma unroll
                for (int j = 0; j < HB; j++) {
                    h[j] = min(h0 + j * TH, NC);
                    acc[j] = make_float2(0.f, 0.f);
                    s[j] = old[h[j]];
                }
                for (int k = F.t0; k < F.t0 + F.nterms; k++) {
                    const LineTerm &TR = P.t[k];
                    if (TR.kind == TERM_CONST) {
#pragma unroll
                        for (int j = 0; j < HB; j++)
                            if (h[j] == 0)
                                acc[j] = cadd(acc[j], apply_mult(table(P.mult, k, 0), TR.mult_i,
                                                                 make_float2((float)P.g.n, 0.f)));
                        continue;
                    }
                    const float2 *x = TR.kind == TERM_BUFFER
                                          ? X + TR.xslot * NC1
                                          : spec + (2 * TR.src + par[TR.srcdyn]) * NC1;
#pragma unroll
                    for (int j = 0; j < HB; j++)
                        acc[j] = cadd(acc[j], apply_mult(table(P.mult, k, h[j]), TR.mult_i, x[h[j]]));
                }
                if (F.dynamic) {
#pragma unroll
                    for (int j = 0; j < HB; j++) {
                        s[j].x += dt * acc[j].x;
                        s[j].y += dt * acc[j].y;
                    }
                } else if (F.nterms > 0 || F.noisy) {
#pragma unroll
                    for (int j = 0; j < HB; j++) s[j] = acc[j];
                }
                if (F.noisy) {
#pragma unroll
                    for (int j = 0; j < HB; j++) {
                        const float2 z = spectral
                                             ? spectral_noise(P.g, h[j], 0, 0, (uint32_t)step, (uint32_t)(step >> 32),
                                                              (uint32_t)i, F.key0, F.key1)
                                             : eta[F.eslot * NC1 + h[j]];
                        const float a = table(P.amp, i, h[j]);
                        s[j].x += a * z.x;
                        s[j].y += a * z.y;
                    }
                }
                if (F.nimp > 0) {
#pragma unroll
                    for (int j = 0; j < HB; j++)
                        if (F.dynamic || h[j] > 0) {
                            const float r = table(P.rdiv, i, h[j]);
                            s[j].x *= r;
                            s[j].y *= r;
                        }
                }
#pragma unroll
                for (int j = 0; j < HB; j++) {
                    if (h[j] == 0 || h[j] == NC) s[j].y = 0.f;  // self-conjugate bins (hermitian_planes)
                    if (h0 + j * TH < NC1) out[h[j]] = s[j];
                }
            }
        }
    };

    int par[2] = {0, 0};  // current buffer of each phase's fields
    for (int n = 0; n < nsteps; n++) {
        const uint64_t step = step0 + (uint64_t)n;
        // phases A, B: constraints
        if (njob00 > 0) {
            jobs(0, 0, njob00, par);
            __syncthreads();
        }
        if (nfield[0] > 0) {
            update_fields(0, par, step);
            __syncthreads();
        }
        par[0] ^= 1;
        // their dealiased copies, beside the transforms of the dynamic
        // fields' noise
        if (njob01 > 0) {
            jobs(0, 1, njob01, par);
            __syncthreads();
        }
        // phases C, D: dynamic fields; the wavefronts without a transform
        // draw the next step's normals
        jobs(1, 0, njob10, par);
        if (neta > 0) {
            const int busy = min(njob10, TH / C::GROUP - 1);
            if (grp >= busy) draw((int)threadIdx.x - busy * C::GROUP, TH - busy * C::GROUP, step + 1);
        }
        __syncthreads();
        update_fields(1, par, step);
        __syncthreads();
        par[1] ^= 1;
        if (njob11 > 0) {
            jobs(1, 1, njob11, par);
            __syncthreads();
        }
    }
    for (int i = 0; i < P.nf; i++) {
        const LineField &F = P.f[i];
        float2 *__restrict__ s = F.spec[((cur >> i) & 1) ^ (nsteps & 1)];
        const float2 *x = spec + (2 * i + par[F.dynamic]) * NC1;
        for (int h = threadIdx.x; h < NC1; h += TH) gstore(s, h, x[h]);
        if (F.dslot >= 0)
            for (int m = threadIdx.x; m < NC; m += TH)
                gstore(reinterpret_cast<float2 *>(F.dreal), m, dreal[F.dslot * NC + m]);
    }
}

// M(q) of each term of one field, 1/D(q) (constraint: 1/L(q)) and the noise
// amplitude (constraint: times 1/sqrt(dt)), as finish_update evaluates them
__global__ __launch_bounds__(256) void k_line_tables(UpdateArgs a, float *__restrict__ mult, float *__restrict__ rdiv,
                                                     float *__restrict__ amp)
{
    const int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= a.g.nc1) return;
    const Bin b = make_bin(a.g, h, 0, 0);
    for (int t = 0; t < a.nterms; t++)
        mult[(long)t * a.g.nc1 + h] = multiplier(a.pres, a.terms[t].pres0, a.terms[t].npres, a.terms[t].mult_i, b);
    float D = a.dynamic ? 1.0f : 0.0f;
    for (int i = 0; i < a.nimp; i++) {
        const PresDev P = a.imp[i];
        float th = P.c;
        if (P.q2n != 0) th *= ipow(b.q2, P.q2n);
        if (P.invq != 0) th *= ipow(a.dynamic ? b.iqd : b.iq, P.invq);
        if (a.dynamic)
            D -= a.dt * th;
        else
            D += th;
    }
    rdiv[h] = __builtin_amdgcn_rcpf(D);
    amp[h] = a.noisy ? (a.dynamic ? 1.0f : a.sdt) * noise_amplitude(a, b) : 0.0f;
}

// ------------------------------------------------------------ host

struct LineState {
    uint64_t gen = 0, vgen = 0;    // the program and prefactor values the device holds
    uint64_t pgen = 0, pvgen = 0;  // those it was laid out for, whether it fits or not
    bool ok = false;
    long bytes = 0;              // dynamic LDS
    bool tab = false;            // the multiplier tables fit it too
    LineProg prog;
    LineProg *dev = nullptr;
    float *tables = nullptr;
    size_t cap = 0;
    ~LineState()
    {
        (void)hipFree(dev);
        (void)hipFree(tables);
    }
};

size_t line_device_bytes(cupss_system s)
{
    if (s->g.sy != 1 || s->g.sz != 1) return 0;
    size_t terms = 0;
    for (auto &F : s->f) terms += F.terms.size();
    return sizeof(LineProg) + sizeof(float) * (size_t)s->g.nc1 * (terms + 2 * s->f.size());
}

void line_release(cupss_system s)
{
    delete static_cast<LineState *>(s->line);
    s->line = nullptr;
}

#define LINE_CASES(X) X(1) X(2) X(4) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048)

static long line_bytes(const LineProg &p, bool tables)
{
    switch (p.g.nc) {
#define X(NC) \
    case NC:  \
        return 8 * line_entries(p, LineCfg<NC>::TWLEN, LineCfg<NC>::G * LineCfg<NC>::LL, tables);
        LINE_CASES(X)
#undef X
    default:
        return 1L << 40;
    }
}

// The program of a 1D system, or ok = false where it does not fit one
// workgroup: more fields or terms than the descriptor holds, or more LDS than
// one workgroup has.  On 4096 points two fields with one dealiased copy, one
// product and real-space noise (a KPZ line) take 149568 of the 153600 bytes;
// on 2048 twice that fits (140408).
static void line_plan(cupss_system s, LineState &S)
{
    S.ok = false;
    LineProg &P = S.prog;
    std::memset(static_cast<void *>(&P), 0, sizeof(P));
    if (s->f.size() > (size_t)LINE_MAX_FIELDS || s->t.size() > (size_t)LINE_MAX_TERMS) return;
    P.g = s->g;
    P.dt = s->dt;
    P.scale = 1.0f / (float)s->g.n;
    P.nf = (int)s->f.size();
    P.spectral = s->noise_mode == 1;
    for (int i = 0; i < P.nf; i++) {
        const FieldRec &R = s->f[i];
        LineField &F = P.f[i];
        F.dynamic = R.dynamic;
        F.noisy = R.noisy;
        F.cut = s->g.sx / (R.order + 1);
        F.nimp = (int)R.imp.size();
        F.dslot = R.order > 0 ? P.ndreal++ : -1;
        F.eslot = -1;
        if (R.noisy && !P.spectral) {
            P.draws[P.neta] = i;
            F.eslot = P.neta++;
        }
        F.key0 = (uint32_t)R.seed;
        F.key1 = (uint32_t)(R.seed >> 32);
        F.spec[0] = R.spec[0];
        F.spec[1] = R.spec[1];
        F.dreal = R.dreal;
    }
    for (int i = 0; i < P.nf; i++) {
        const FieldRec &R = s->f[i];
        LineField &F = P.f[i];
        const int ph = R.dynamic ? 1 : 0;
        P.field[ph][P.n[ph]++] = i;
        F.t0 = P.nterms;
        F.nterms = (int)R.terms.size();
        for (int ti : R.terms) {
            const TermRec &T = s->t[ti];
            LineTerm &L = P.t[P.nterms];
            L.mult_i = (T.pres[0].iqx + T.pres[0].iqy + T.pres[0].iqz) % 2;
            if (T.fac.size() >= 2) {
                L.kind = TERM_BUFFER;
                L.xslot = P.nx++;
                L.nfac = (int)T.fac.size();
                for (int c = 0; c < L.nfac; c++) L.fac[c] = P.f[T.fac[c]].dslot;
                P.job[ph][0][P.njob[ph][0]++] = LineJob{LINE_PRODUCT, P.nterms};
            } else if (T.fac.size() == 1) {
                L.kind = TERM_FIELD;
                L.src = T.fac[0];
                L.srcdyn = s->f[T.fac[0]].dynamic;
            } else {
                L.kind = TERM_CONST;
            }
            P.nterms++;
        }
        if (F.dslot >= 0) P.job[ph][1][P.njob[ph][1]++] = LineJob{LINE_DEALIAS, i};
    }
    // noise transforms: the constraints' before their update, the dynamic
    // fields' beside the constraints' dealiased copies
    for (int ph = 0; ph < 2; ph++)
        for (int q = 0; q < P.n[ph]; q++)
            if (P.f[P.field[ph][q]].eslot >= 0) {
                const int when = ph == 0 ? 0 : 1;
                P.job[0][when][P.njob[0][when]++] = LineJob{LINE_NOISE, P.field[ph][q]};
            }
    S.bytes = line_bytes(P, true);
    S.tab = S.bytes <= LINE_LDS;
    if (!S.tab) S.bytes = line_bytes(P, false);
    S.ok = S.bytes <= LINE_LDS;
}

bool line_eligible(cupss_system s)
{
    if (s->g.sy != 1 || s->g.sz != 1) return false;
    LineState *S = static_cast<LineState *>(s->line);
    if (!S) {
        S = new LineState();
        s->line = S;
    }
    if (S->pgen != s->gen || S->pvgen != s->vgen) {
        line_plan(s, *S);
        S->pgen = s->gen;
        S->pvgen = s->vgen;
        s->line_plans++;
    }
    if (!S->ok) return false;
    // the upload cannot be recorded into a graph: a caller's capture that
    // starts before the program was uploaded records the general program's
    // launches
    return (S->gen == s->gen && S->vgen == s->vgen) || s->own_stream || !recording(s->stream);
}

template <int NC, bool TAB>
static hipError_t line_launch(const LineState &S, uint32_t cur, uint64_t step, int nsteps, hipStream_t st)
{
    const float2 *sets = twiddle_sets(st);
    if (!sets) return hipErrorOutOfMemory;
    if (S.bytes > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_line<NC, TAB>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, LINE_LDS);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_line<NC, TAB>), dim3(1), dim3(LineCfg<NC>::THREADS), (unsigned)S.bytes, st, S.dev, cur, step,
                       nsteps, sets);
    return hipGetLastError();
}

// tables and descriptor of a new program, in stream order (the copies from
// pageable memory are staged before the call returns)
static int line_upload(cupss_system s, LineState &S)
{
    LineProg &P = S.prog;
    const size_t need = sizeof(float) * (size_t)s->g.nc1 * (size_t)(P.nterms + 2 * P.nf);
    if (!S.dev && hipMalloc(&S.dev, sizeof(LineProg)) != hipSuccess)
        return fail(CUPSS_ERR_NOMEM, "device allocation failed");
    if (S.cap < need) {
        HIP_TRY(hipStreamSynchronize(s->stream));
        (void)hipFree(S.tables);
        S.tables = nullptr;
        S.cap = 0;
        if (hipMalloc(&S.tables, need) != hipSuccess) return fail(CUPSS_ERR_NOMEM, "device allocation failed");
        S.cap = need;
    }
    const long nc1 = s->g.nc1;
    P.mult = S.tables;
    P.rdiv = S.tables + P.nterms * nc1;
    P.amp = P.rdiv + P.nf * nc1;
    for (int i = 0; i < P.nf; i++) {
        UpdateArgs a;
        build_update(s, i, a);
        hipLaunchKernelGGL(k_line_tables, dim3((unsigned)((nc1 + 255) / 256)), dim3(256), 0, s->stream, a,
                           S.tables + P.f[i].t0 * nc1, S.tables + (P.nterms + i) * nc1,
                           S.tables + (P.nterms + P.nf + i) * nc1);
        HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipMemcpyAsync(S.dev, &P, sizeof(LineProg), hipMemcpyHostToDevice, s->stream));
    S.gen = s->gen;
    S.vgen = s->vgen;
    return CUPSS_OK;
}

int line_steps(cupss_system s, int nsteps)
{
    LineState &S = *static_cast<LineState *>(s->line);
    s->cont_step = ~0ull;
    for (int i = 0; i < (int)s->f.size(); i++)
        if (int r = materialize(s, i)) return r;
    if (S.gen != s->gen || S.vgen != s->vgen)
        if (int r = line_upload(s, S)) return r;
    for (int done = 0; done < nsteps;) {
        const int k = std::min(LINE_CHUNK, nsteps - done);
        uint32_t cur = 0;
        for (size_t i = 0; i < s->f.size(); i++) cur |= (uint32_t)s->f[i].cur << i;
        hipError_t e = hipErrorInvalidValue;
        switch (s->g.nc) {
#define X(NC)                                                    \
    case NC:                                                     \
        e = S.tab ? line_launch<NC, true>(S, cur, s->step, k, s->stream)     \
                  : line_launch<NC, false>(S, cur, s->step, k, s->stream);   \
        break;
            LINE_CASES(X)
#undef X
        }
        HIP_TRY(e);
        for (auto &F : s->f) {
            F.cur ^= k & 1;
            if (F.order > 0) F.dstate = 1;
        }
        s->step += (uint64_t)k;
        s->line_steps += k;
        done += k;
    }
    return CUPSS_OK;
}

}  // namespace cupss
