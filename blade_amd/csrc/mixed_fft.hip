// FFT channelizer, optionally with the detector, at rates C <= 8192 made of
// 2, 3, 5 and 7 (two polarizations):
//   out[a, f*C + k, s, p] = fftshift(DFT_C(in[a, f, s*C:(s+1)*C, p]))[k]
// (oracle tests/modules/channelizer/advanced.py:49-65).
//
// C is split into as few Stockham passes as radices up to 16 allow (1000 =
// 10 x 10 x 10, 96 = 12 x 8, 6250 = 10 x 5 x 5 x 5 x 5), each radix compiled
// as straight-line code on registers.  A workgroup transforms `spw` spectra at
// once, both polarizations of a point in one 16-byte LDS entry and in the same
// thread: twiddles and indices serve both.
//   first pass   memory -> registers -> LDS (16-byte loads, lanes along the
//                spectrum);
//   middle       LDS -> registers -> LDS;
//   last         LDS -> registers -> memory, or detected powers into LDS, which
//                are summed over the spectra of an integration and stored.
// With several spectra per (antenna, channel) the bins of neighbouring spectra
// are neighbours in the output: the last pass then deals butterflies to lanes
// spectrum first, so that a store writes runs of spw samples.
// Twiddles come from a table per rate laid out in the order the passes read
// it ([pass][r - 1][j mod Ns]: consecutive lanes, consecutive entries), FP64
// computed.  LDS rows carry one entry of padding per 8, which spreads the
// first pass's stride-R writes over the banks.
// Index divisions are by run-time constants, taken as 32-bit multiplies.
// Bound by latency: a workgroup's load, passes and store follow each other, and
// 16 waves per CU overlap.  400 MB in and out, against the run-time-radix LDS
// kernel before: C = 1000 at 12 spectra per channel 95 us (4.2 TB/s), was 415;
// C = 96 83 us; C = 8000 120 us (one workgroup per CU); detector, 200 MB in,
// C = 1000 73-98 us, was 205-327.  C = 32, 64, 128 77-79 us, where a radix-8
// kernel with C/8 threads per spectrum took 84-97 us.
#include "fft_regs.hh"
#include "mixed_fft.hh"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <map>
#include <memory>
#include <mutex>
#include <type_traits>
#include <vector>

namespace bl {

constexpr int kMixPasses = 6;
constexpr int kMixThreads = 1024;          // 16 waves, 4 per SIMD: 128 VGPRs each
constexpr int kMixMaxC = 8192;
constexpr size_t kMixLds = 160 * 1024;

struct MixPass {
    unsigned R, Ns, nb;                    // radix, product of earlier radices, butterflies C / R
    unsigned m_ns, m_nb;                   // ceil(2^32 / d): n / d = umulhi(n, m) for n d < 2^32
    unsigned tw;                           // first twiddle entry
};

struct MixPlan {
    int C, n;
    MixPass p[kMixPasses];
};

struct MixArgs {
    const float4* in;
    void* out;
    const float2* tw;
    MixPlan pl;
    unsigned CS;                           // LDS row stride, float4
    unsigned spw;                          // spectra per workgroup and step
    unsigned sub, steps, gpw;              // detector: spectra of one integration per step, steps, integrations
    unsigned Sg, groups;                   // detector: spectra per integration, integrations per channel
    unsigned S;                            // spectra per (antenna, channel)
    unsigned m_spw, m_sub, m_per, m_gpw;   // division multipliers of spw, sub, S or groups, spw / sub
    uint64_t n_spec, n_groups;
    int flags;
    union {                                // one word: the arguments stay 248 bytes (past it calls of 4 us take 0.2 us more)
        unsigned sums;                     // detector, KEEP: running sums in LDS from this float on
        unsigned wg0;                      // MODE 0, OPT: first workgroup of this launch
    };
};

// n / d from m = ceil(2^32 / d), d > 1; exact for n d < 2^32.  m = 0 stands
// for d = 1.
__device__ __forceinline__ unsigned mix_div(unsigned n, unsigned m) { return __umulhi(n, m); }
__device__ __forceinline__ unsigned mix_div1(unsigned n, unsigned m) { return m ? __umulhi(n, m) : n; }
// n / d for n < d + 64, any d: past 2^15 (where the multiply may be off) the
// quotient is 0 or 1.
__device__ __forceinline__ unsigned mix_div_wide(unsigned n, unsigned d, unsigned m) {
    return d >= (1u << 15) ? (n >= d ? 1u : 0u) : mix_div1(n, m);
}
__device__ __forceinline__ unsigned mix_pad(unsigned i) { return i + (i >> 3); }

// Butterflies of one thread in a pass of radix R.
template <int R>
constexpr int mix_per_thread() { return R <= 8 ? 2 : 1; }

template <int R>
__device__ __forceinline__ void mix_dft(float2 (&x)[R], float2 (&y)[R]) {
    dft_any<R>(x);
    dft_any<R>(y);
}

// LDS reads and twiddles of butterfly j of the row at `row`.
template <int R>
__device__ __forceinline__ void mix_read(const MixPass& p, const float4* row, const float2* tw, unsigned j,
                                         unsigned jm, float2 (&x)[R], float2 (&y)[R]) {
    const float2* const t = tw + p.tw + jm;
    float2 w[R];
    if constexpr (R <= 10) {
#pragma unroll
        for (int r = 1; r < R; r++) w[r] = t[(r - 1) * p.Ns];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if constexpr (R > 10) {
            if (r > 0) w[r] = t[(r - 1) * p.Ns];
            if (r % 4 == 0) __builtin_amdgcn_sched_barrier(0);
        }
        const float4 q = row[mix_pad(j + r * p.nb)];
        x[r] = make_float2(q.x, q.y);
        y[r] = make_float2(q.z, q.w);
        if (r > 0) {
            x[r] = cmul(x[r], w[r]);
            y[r] = cmul(y[r], w[r]);
        }
    }
}

template <int R>
__device__ __forceinline__ void mix_write(float4* row, unsigned d, unsigned Ns, const float2 (&x)[R],
                                          const float2 (&y)[R]) {
#pragma unroll
    for (int r = 0; r < R; r++) row[mix_pad(d + r * Ns)] = make_float4(x[r].x, x[r].y, y[r].x, y[r].y);
}

// First spectrum of slot `slot` in step `step`, or past the end.
template <int MODE>
__device__ __forceinline__ bool mix_spectrum(const MixArgs& a, uint64_t wg, unsigned slot, unsigned step,
                                             uint64_t* sp) {
    if constexpr (MODE == 0) {
        *sp = wg * a.spw + slot;
        return *sp < a.n_spec;
    } else {
        const unsigned gl = mix_div1(slot, a.m_sub), i = slot - gl * a.sub + step * a.sub;
        const uint64_t g = wg * a.gpw + gl;
        *sp = g * a.Sg + i;
        return g < a.n_groups && i < a.Sg;
    }
}

template <int R, int MODE>
__device__ __forceinline__ void mix_first(const MixArgs& a, unsigned t, uint64_t wg, unsigned step, float4* lds) {
    const MixPass& p = a.pl.p[0];
    constexpr int G = mix_per_thread<R>();
#pragma unroll
    for (int g = 0; g < G; g++) {
        const unsigned bf = t + g * blockDim.x;
        const unsigned slot = mix_div(bf, p.m_nb), j = bf - slot * p.nb;
        uint64_t sp;
        if (slot < a.spw && mix_spectrum<MODE>(a, wg, slot, step, &sp)) {
            const float4* const src = a.in + sp * (unsigned)a.pl.C + j;
            float2 x[R], y[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float4 q = src[r * p.nb];
                x[r] = make_float2(q.x, q.y);
                y[r] = make_float2(q.z, q.w);
            }
            mix_dft<R>(x, y);
            mix_write<R>(lds + slot * a.CS, j * R, 1, x, y);
        }
    }
}

template <int R>
__device__ __forceinline__ void mix_mid(const MixArgs& a, unsigned t, const MixPass& p, float4* lds) {
    constexpr int G = mix_per_thread<R>();
    float2 x[G][R], y[G][R];
#pragma unroll
    for (int g = 0; g < G; g++) {
        const unsigned bf = t + g * blockDim.x;
        const unsigned slot = mix_div(bf, p.m_nb), j = bf - slot * p.nb;
        if (slot < a.spw) {
            mix_read<R>(p, lds + slot * a.CS, a.tw, j, j - mix_div(j, p.m_ns) * p.Ns, x[g], y[g]);
            mix_dft<R>(x[g], y[g]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; g++) {
        const unsigned bf = t + g * blockDim.x;
        const unsigned slot = mix_div(bf, p.m_nb), j = bf - slot * p.nb;
        if (slot < a.spw) {
            const unsigned jm = j - mix_div(j, p.m_ns) * p.Ns;
            mix_write<R>(lds + slot * a.CS, (j - jm) * R + jm, p.Ns, x[g], y[g]);
        }
    }
    __syncthreads();
}

template <int R, int MODE, bool OPT>
__device__ __forceinline__ void mix_last(const MixArgs& a, unsigned t, uint64_t wg, float4* lds) {
    const MixPass& p = a.pl.p[a.pl.n - 1];       // Ns = nb: butterfly j holds bins j + r nb
    constexpr int G = mix_per_thread<R>();
    const unsigned C = (unsigned)a.pl.C, half = C / 2;
    if constexpr (MODE == 0) {
        // The workgroup's first spectrum is number s0 of channel af0.
        const uint64_t sp0 = wg * a.spw, af0 = a.S == 1 ? sp0 : sp0 / a.S;
        const unsigned s0 = (unsigned)(sp0 - af0 * a.S);
        float4* const out = static_cast<float4*>(a.out) + af0 * ((uint64_t)C * a.S);
#pragma unroll
        for (int g = 0; g < G; g++) {
            const unsigned bf = t + g * blockDim.x;
            unsigned slot, j;
            if (a.S > 1) {                        // neighbouring spectra on neighbouring lanes
                j = mix_div1(bf, a.m_spw);
                slot = bf - j * a.spw;
                if (j >= p.nb) slot = a.spw;
            } else {
                slot = mix_div(bf, p.m_nb);
                j = bf - slot * p.nb;
            }
            if (slot < a.spw && sp0 + slot < a.n_spec) {
                float2 x[R], y[R];
                mix_read<R>(p, lds + slot * a.CS, a.tw, j, j, x, y);
                mix_dft<R>(x, y);
                const unsigned q = s0 + slot, af = mix_div_wide(q, a.S, a.m_per), s = q - af * a.S;
                float4* const dst = out + (uint64_t)af * ((uint64_t)C * a.S) + s;
                typedef std::conditional_t<OPT, uint64_t, unsigned> Offset;      // within C S outputs
                unsigned ko = j + half;
                if (ko >= C) ko -= C;
                // Two loops: with the branch inside, the compiler merges both
                // forms into four 4-byte stores.
                if (a.S == 1) {
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        __builtin_nontemporal_store(floatx4{x[r].x, x[r].y, y[r].x, y[r].y},
                                                    reinterpret_cast<floatx4*>(dst + ko));
                        ko += p.nb;
                        if (ko >= C) ko -= C;
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        dst[Offset(ko) * a.S] = make_float4(x[r].x, x[r].y, y[r].x, y[r].y);
                        ko += p.nb;
                        if (ko >= C) ko -= C;
                    }
                }
            }
        }
    } else {
        float pw[G][R][MODE];
#pragma unroll
        for (int g = 0; g < G; g++) {
            const unsigned bf = t + g * blockDim.x;
            const unsigned slot = mix_div(bf, p.m_nb), j = bf - slot * p.nb;
            if (slot < a.spw) {
                float2 x[R], y[R];
                mix_read<R>(p, lds + slot * a.CS, a.tw, j, j, x, y);
                mix_dft<R>(x, y);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const float2 X = x[r], Y = y[r];
                    if constexpr (MODE == 1) {
                        pw[g][r][0] = X.x * X.x + X.y * X.y + Y.x * Y.x + Y.y * Y.y;
                    } else {
                        pw[g][r][0] = X.x * X.x + X.y * X.y;
                        pw[g][r][MODE > 1 ? 1 : 0] = Y.x * Y.x + Y.y * Y.y;
                        pw[g][r][MODE > 2 ? 2 : 0] = X.x * Y.x + X.y * Y.y;
                        pw[g][r][MODE > 3 ? 3 : 0] = X.y * Y.x - X.x * Y.y;
                    }
                }
            }
        }
        __syncthreads();
        // Powers over the rows just read (unpadded, row stride CS entries).
#pragma unroll
        for (int g = 0; g < G; g++) {
            const unsigned bf = t + g * blockDim.x;
            const unsigned slot = mix_div(bf, p.m_nb), j = bf - slot * p.nb;
            if (slot < a.spw) {
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const unsigned o = slot * a.CS + j + r * p.nb;
                    if constexpr (MODE == 1)
                        reinterpret_cast<float*>(lds)[o] = pw[g][r][0];
                    else
                        lds[o] = make_float4(pw[g][r][0], pw[g][r][MODE > 1 ? 1 : 0], pw[g][r][MODE > 2 ? 2 : 0],
                                             pw[g][r][MODE > 3 ? 3 : 0]);
                }
            }
        }
    }
}

// Sum the step's powers of every integration and store them.  The same thread
// owns an output in every step.  Where the integration is added to earlier
// blocks', the steps are summed in LDS first: added one by one, each would round
// at the size of the long sum (64 blocks of 128 spectra at rate 1000: error
// 6.0e-7 against 1.2e-7).  KEEP: in a kernel of its own, its registers and branches
// cost the others up to 7%.
template <int MODE, bool KEEP>
__device__ __forceinline__ void mix_sum(const MixArgs& a, unsigned t, uint64_t wg, unsigned step, float4* lds) {
    const unsigned C = (unsigned)a.pl.C, gpw = a.gpw, half = C / 2;
    const uint64_t g0 = wg * gpw, af0 = a.groups == 1 ? g0 : g0 / a.groups;
    const unsigned r0 = (unsigned)(g0 - af0 * a.groups);
    const unsigned cnt = min(a.sub, a.Sg - step * a.sub);
    const bool add = KEEP || step > 0 || (a.flags & 1), circular = a.flags & 2;
    for (unsigned e = t; e < C * gpw; e += blockDim.x) {
        const unsigned k = mix_div1(e, a.m_gpw), gl = e - k * gpw;
        if (g0 + gl >= a.n_groups) continue;
        float v[MODE];
#pragma unroll
        for (int c = 0; c < MODE; c++) v[c] = 0.f;
        for (unsigned i = 0; i < cnt; i++) {
            const unsigned o = (gl * a.sub + i) * a.CS + k;
            if constexpr (MODE == 1) {
                v[0] += reinterpret_cast<const float*>(lds)[o];
            } else {
                const float4 q = lds[o];
                v[0] += q.x;
                v[MODE > 1 ? 1 : 0] += q.y;
                v[MODE > 2 ? 2 : 0] += q.z;
                v[MODE > 3 ? 3 : 0] += q.w;
            }
        }
        if constexpr (KEEP) {                      // one integration per workgroup: e is its output
            float* const sum = reinterpret_cast<float*>(lds) + a.sums + e * MODE;
            if (step > 0) {
#pragma unroll
                for (int c = 0; c < MODE; c++) v[c] = sum[c] + v[c];
            }
            if (step + 1 < a.steps) {
#pragma unroll
                for (int c = 0; c < MODE; c++) sum[c] = v[c];
                continue;
            }
        }
        if (circular) circular_sums<MODE>(v);
        const unsigned q = r0 + gl, af = mix_div_wide(q, a.groups, a.m_per);
        unsigned ko = k + half;
        if (ko >= C) ko -= C;
        const uint64_t o = ((af0 + af) * C + ko) * a.groups + (q - af * a.groups);
        if constexpr (MODE == 1) {
            float* const p = static_cast<float*>(a.out) + o;
            *p = add ? *p + v[0] : v[0];
        } else {
            float4* const p = static_cast<float4*>(a.out) + o;
            float4 q4 = make_float4(v[0], v[MODE > 1 ? 1 : 0], v[MODE > 2 ? 2 : 0], v[MODE > 3 ? 3 : 0]);
            if (add) {
                const float4 u = *p;
                q4 = make_float4(u.x + q4.x, u.y + q4.y, u.z + q4.z, u.w + q4.w);
            }
            *p = q4;
        }
    }
}

#define MIX_RADICES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(14) X(15) X(16)

// MODE 0: spectra; 1: Stokes I; 4: XX*, YY*, Re XY*, Im XY*.  OPT: channels of
// 2^31 outputs or more and 2^32 threads or more in several launches (MODE 0; the
// 64-bit arithmetic costs small calls 2%); the steps of an integration are summed in LDS (detector, mix_sum).
template <int MODE, bool OPT = false>
__global__ __launch_bounds__(kMixThreads) void mixed_fft_kernel(MixArgs a) {
    extern __shared__ __align__(16) float4 lds[];
    // Outputs of neighbouring workgroups that share lines are written on one XCD.
    const unsigned wgi = (MODE == 0 ? a.S > 1 : a.groups > 1) ? xcd_order(blockIdx.x, gridDim.x) : blockIdx.x;
    const uint64_t wg = MODE == 0 && OPT ? a.wg0 + (uint64_t)wgi : wgi;
    const unsigned steps = MODE == 0 ? 1 : a.steps;
    for (unsigned step = 0; step < steps; step++) {
        // Opaque: keeps every radix's index arithmetic from being hoisted out
        // of the step loop (spilled, it cost more than the data's traffic).
        unsigned t = threadIdx.x;
        asm volatile("" : "+v"(t));
        switch (a.pl.p[0].R) {
#define X(R) case R: mix_first<R, MODE>(a, t, wg, step, lds); break;
            MIX_RADICES(X)
#undef X
        }
        __syncthreads();
        for (int i = 1; i + 1 < a.pl.n; i++) {
            switch (a.pl.p[i].R) {
#define X(R) case R: mix_mid<R>(a, t, a.pl.p[i], lds); break;
                MIX_RADICES(X)
#undef X
            }
        }
        switch (a.pl.p[a.pl.n - 1].R) {
#define X(R) case R: mix_last<R, MODE, OPT>(a, t, wg, lds); break;
            MIX_RADICES(X)
#undef X
        }
        if constexpr (MODE != 0) {
            __syncthreads();
            mix_sum<MODE, OPT>(a, t, wg, step, lds);
            if (step + 1 < steps) __syncthreads();     // LDS is rewritten by the next step
        }
    }
}

__global__ void mixed_twiddle_kernel(float2* tw, MixPlan pl) {
    for (int i = 1; i < pl.n; i++) {
        const MixPass& p = pl.p[i];
        const unsigned n = (p.R - 1) * p.Ns;
        for (unsigned e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
            const unsigned r = e / p.Ns + 1, jm = e - (r - 1) * p.Ns;
            double s, c;
            sincospi(-2.0 * (double)(jm * r) / (double)(p.Ns * p.R), &s, &c);
            tw[p.tw + e] = make_float2((float)c, (float)s);
        }
    }
}

static uint64_t gcd(uint64_t x, uint64_t y) {
    while (y) {
        const uint64_t t = x % y;
        x = y;
        y = t;
    }
    return x;
}

static unsigned mix_magic(uint64_t d) { return d > 1 ? (unsigned)((0x100000000ull + d - 1) / d) : 0; }

static int mix_g(unsigned R) { return R <= 8 ? 2 : 1; }

// Fewest passes; among those the smallest largest radix (registers, idle
// lanes).  Every pass must fit 1024 threads (two butterflies each up to radix
// 8).  Radices descend, so the first pass has the fewest butterflies.
static bool mix_search(int C, int left, int depth, int last, int* cur, int* best, int* best_n) {
    static const int radices[] = {16, 15, 14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    if (left == 1) {
        if (depth < 2) return false;
        if (*best_n == 0 || depth < *best_n || (depth == *best_n && cur[0] < best[0])) {
            std::copy(cur, cur + depth, best);
            *best_n = depth;
        }
        return true;
    }
    if (depth >= kMixPasses || (*best_n && depth >= *best_n)) return false;
    bool any = false;
    for (int R : radices) {
        if (R > last || left % R || C / R > kMixThreads * mix_g(R)) continue;
        cur[depth] = R;
        any |= mix_search(C, left / R, depth + 1, R, cur, best, best_n);
    }
    return any;
}

static bool mix_plan(int C, MixPlan* pl) {
    if (C < 4 || C > kMixMaxC) return false;
    int cur[kMixPasses + 1], best[kMixPasses], n = 0;
    if (!mix_search(C, C, 0, 16, cur, best, &n)) return false;
    pl->C = C;
    pl->n = n;
    unsigned Ns = 1, off = 0;
    for (int i = 0; i < n; i++) {
        MixPass& p = pl->p[i];
        p.R = (unsigned)best[i];
        p.Ns = Ns;
        p.nb = (unsigned)C / p.R;
        p.m_nb = mix_magic(p.nb);
        p.m_ns = mix_magic(Ns);
        p.tw = off;
        if (i > 0) off += (p.R - 1) * Ns;
        Ns *= p.R;
    }
    return true;
}

// The search takes microseconds, as long as a small launch: answered once per
// rate (0: not yet, 1: no, 2: yes).
bool mixed_fft_covers(uint64_t rate) {
    static std::atomic<unsigned char> known[kMixMaxC + 1];
    if (rate > (uint64_t)kMixMaxC) return false;
    unsigned char k = known[rate].load(std::memory_order_relaxed);
    if (!k) {
        MixPlan pl;
        k = mix_plan((int)rate, &pl) ? 2 : 1;
        known[rate].store(k, std::memory_order_relaxed);
    }
    return k == 2;
}

// A launch shape, rated by the lanes its passes keep busy and the points in
// flight per CU (short of ~8000 the loads are not hidden).
struct MixShape {
    unsigned spw, threads;                 // spectra per workgroup and step
    double score;
};

// What a rate keeps per device: it depends on the rate alone.  Found anew on
// each call it cost 5-7 us of host time (6 x 74 channels of one 64-sample
// spectrum 12.7 us a call, 5.1 us so).
struct MixTable {
    MixPlan pl;
    unsigned CS;                           // LDS row stride, float4
    std::vector<MixShape> shapes;
    float2* tw;
};

static std::vector<MixShape> mix_shapes(const MixPlan& pl, unsigned CS) {
    std::vector<MixShape> out;
    for (unsigned s = 1; s <= 64; s++) {
        const size_t lds = (size_t)s * CS * 16;
        if (lds > kMixLds) break;
        unsigned one = 0, two = 0;                   // threads with one butterfly each, and with two where allowed
        for (int i = 0; i < pl.n; i++) {
            const unsigned nb = s * pl.p[i].nb;
            one = std::max(one, nb);
            two = std::max(two, (nb + mix_g(pl.p[i].R) - 1) / mix_g(pl.p[i].R));
        }
        for (unsigned need : {one, two}) {
            const unsigned nt = (need + 63) / 64 * 64;
            if (nt > (unsigned)kMixThreads) continue;
            double busy = 0;
            for (int i = 0; i < pl.n; i++) {
                const unsigned nb = s * pl.p[i].nb;
                busy += (double)nb / (nt * ((nb + nt - 1) / nt)) / pl.n;
            }
            const double wgs = std::min<double>({std::floor(160.0 * 1024 / lds), std::floor(1024.0 / nt), 16.0});
            const double points = wgs * s * pl.C;
            out.push_back({s, nt, busy * std::min(1.0, points / 8192) * (wgs < 2 ? 0.7 : 1.0)});
        }
    }
    return out;
}

static std::mutex g_mix_mutex;
static std::map<std::pair<int, int>, std::unique_ptr<MixTable>> g_mix_tables;

static int mix_table(int C, const MixTable** out, bool* made = nullptr) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return fail("channelizer: hipGetDevice failed");
    std::lock_guard<std::mutex> lock(g_mix_mutex);
    std::unique_ptr<MixTable>& slot = g_mix_tables[{dev, C}];
    if (!slot) {
        std::unique_ptr<MixTable> t(new MixTable);
        if (!mix_plan(C, &t->pl)) return fail("channelizer: no mixed-radix plan");
        t->CS = ((unsigned)C + C / 8 + 1) | 1;
        t->shapes = mix_shapes(t->pl, t->CS);
        void* p = nullptr;                            // sum of (R - 1) Ns = C - R_0 entries
        const int rc = device_table("channelizer twiddles", sizeof(float2) * (size_t)C, &p,
                                    [&](void* tw, hipStream_t ts) {
            hipLaunchKernelGGL(mixed_twiddle_kernel, dim3(8), dim3(256), 0, ts, static_cast<float2*>(tw), t->pl);
        });
        if (rc) return rc;
        t->tw = static_cast<float2*>(p);
        slot = std::move(t);
        if (made) *made = true;
    }
    *out = slot.get();
    return BLADE_SUCCESS;
}

int mixed_fft_plan(int C) {
    const MixTable* t = nullptr;
    return mix_table(C, &t);
}

// Spectra per workgroup (a multiple of `unit`) and threads: the rate's shapes
// rated besides by the run of neighbouring output samples their stores write
// (`run_of`) and whether the grid of `units` fills the chip.
template <typename RunOf>
static void mix_shape(const MixTable& t, uint64_t units, unsigned unit, RunOf run_of, unsigned* spw, unsigned* threads) {
    const double full = 2.0 * device_cus();
    double best = -1;
    for (const MixShape& c : t.shapes) {
        if (c.spw % unit || c.score <= best) continue;
        const unsigned m = c.spw / unit;
        const double grid = (double)((units + m - 1) / m) / full;
        const double score = c.score * run_of(c.spw) * std::min(1.0, 0.25 + 0.75 * grid);
        if (score > best) {
            best = score;
            *spw = c.spw;
            *threads = c.threads;
        }
    }
}

template <int MODE, bool OPT = false>
static int mix_launch(MixArgs& a, uint64_t blocks, unsigned threads, hipStream_t s) {
    const void* fn = reinterpret_cast<const void*>(&mixed_fft_kernel<MODE, OPT>);
    const size_t lds = (size_t)a.spw * a.CS * 16 + (OPT ? (size_t)a.pl.C * MODE * 4 : 0);
    if (lds > 65536 && hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return fail("channelizer: LDS attribute of the mixed-radix FFT");
    const uint64_t most = 0xffffffffull / threads & ~7ull;          // a launch holds less than 2^32 threads
    for (uint64_t wg0 = 0; wg0 < blocks; wg0 += most) {             // once unless MODE 0, OPT
        if (MODE == 0) a.wg0 = (unsigned)wg0;
        void* args[] = {&a};
        (void)hipLaunchKernel(fn, dim3((unsigned)std::min(most, blocks - wg0)), dim3(threads), args, lds, s);
    }
    return check_launch("channelizer");
}

int mixed_fft(int C, const float2* in, float2* out, uint64_t S, uint64_t n_spec, hipStream_t s, bool* made) {
    MixArgs a = {};
    const MixTable* t = nullptr;
    int rc = mix_table(C, &t, made);
    if (rc) return rc;
    a.pl = t->pl;
    a.CS = t->CS;
    a.tw = t->tw;
    unsigned threads = 0;
    mix_shape(*t, n_spec, 1, [&](unsigned w) {
        const uint64_t run = S == 1 ? 16 : gcd(S, w);
        return run >= 8 ? 1.0 : run >= 4 ? 0.9 : run >= 2 ? 0.7 : 0.5;
    }, &a.spw, &threads);
    a.in = reinterpret_cast<const float4*>(in);
    a.out = out;
    a.S = (unsigned)S;
    a.n_spec = n_spec;
    a.m_spw = mix_magic(a.spw);
    a.m_per = mix_magic(S);
    uint64_t blocks = ceil_div(n_spec, a.spw);
    if (S > 1) blocks = ceil_div(blocks, 8) * 8;         // xcd_order needs G % 8 == 0
    const bool wide = (uint64_t)C * S >= (1ull << 31) || blocks * threads >= (1ull << 32);
    return wide ? mix_launch<0, true>(a, blocks, threads, s) : mix_launch<0>(a, blocks, threads, s);
}

bool mixed_fft_detect(int C, const float2* in, float* out, uint64_t Sg, int groups, uint64_t n_groups, int out_pols,
                      int flags, hipStream_t s, int* rc, bool* made) {
    MixArgs a = {};
    const MixTable* t = nullptr;
    *rc = mix_table(C, &t, made);
    if (*rc) return true;
    a.pl = t->pl;
    a.CS = t->CS;
    a.tw = t->tw;
    unsigned threads = 0;
    // Whole integrations per workgroup where they fit, otherwise one
    // integration in steps of (about) equal numbers of spectra.
    auto most_of = [&](size_t keep) {                // spectra a step can hold, two workgroups per CU
        unsigned most = 1;
        for (unsigned w = 2; w <= 32; w++) {
            bool ok = (size_t)w * a.CS * 16 + keep <= kMixLds / 2;
            for (int i = 0; i < a.pl.n; i++)
                ok = ok && w * a.pl.p[i].nb <= (unsigned)(kMixThreads / 2 * mix_g(a.pl.p[i].R));
            if (ok) most = w;
        }
        return most;
    };
    a.steps = (unsigned)ceil_div(Sg, most_of(0));
    const bool keep = a.steps > 1 && (flags & 1);
    const size_t sums = keep ? (size_t)C * out_pols * 4 : 0;
    if (keep) a.steps = (unsigned)ceil_div(Sg, most_of(sums));
    a.sub = (unsigned)ceil_div(Sg, a.steps);
    if (keep) {
        const size_t rows = (size_t)a.sub * a.CS * 16;
        if (rows + sums > kMixLds) return false;
        a.sums = (unsigned)(rows / 4);
    }
    if (a.steps > 1) {
        mix_shape(*t, n_groups, a.sub, [&](unsigned w) { return w == a.sub ? 1.0 : 0.0; }, &a.spw, &threads);
    } else {
        mix_shape(*t, n_groups, a.sub, [&](unsigned w) {
            const uint64_t run = groups == 1 ? 64 : out_pols * gcd((uint64_t)groups, w / a.sub);   // floats
            return run >= 16 ? 1.0 : run >= 8 ? 0.9 : run >= 4 ? 0.75 : 0.6;
        }, &a.spw, &threads);
    }
    a.in = reinterpret_cast<const float4*>(in);
    a.out = out;
    a.Sg = (unsigned)Sg;
    a.groups = (unsigned)groups;
    a.n_groups = n_groups;
    a.flags = flags;
    a.gpw = a.spw / a.sub;
    a.m_sub = mix_magic(a.sub);
    a.m_gpw = mix_magic(a.gpw);
    a.m_per = mix_magic((uint64_t)groups);
    uint64_t blocks = ceil_div(n_groups, a.gpw);
    if (groups > 1) blocks = ceil_div(blocks, 8) * 8;    // xcd_order needs G % 8 == 0
    if (blocks * threads >= (1ull << 32)) return false;
    if (keep)
        *rc = out_pols == 1 ? mix_launch<1, true>(a, blocks, threads, s) : mix_launch<4, true>(a, blocks, threads, s);
    else
        *rc = out_pols == 1 ? mix_launch<1>(a, blocks, threads, s) : mix_launch<4>(a, blocks, threads, s);
    return true;
}

}  // namespace bl
