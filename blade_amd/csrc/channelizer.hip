// FFT channelizer:  out[a, f*C + k, s, p] = fftshift(DFT_C(in[a, f, s*C:(s+1)*C, p]))[k]
// (oracle tests/modules/channelizer/advanced.py:49-65; forward, unnormalised,
// e^{-j 2pi k n / C}).  Written from the Stockham autosort formulation of the
// mixed-radix FFT (each pass reads stride C/R, twiddles by W_{Ns R}^{(j mod Ns) r},
// butterflies, writes to (j/Ns)*Ns*R + j mod Ns + r*Ns), so the output lands
// in natural order without a bit-reversal pass.  fftshift is an index remap on
// the store.  Twiddles come from a per-C table built in FP64 and rounded
// once to FP32.
#include "fft_regs.hh"
#include "mixed_fft.hh"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <vector>

namespace bl {

// ---------------------------------------------------------------------------
// Twiddle tables  W_C^m = exp(-j 2 pi m / C),  m in [0, C), one per (device, C).
// ---------------------------------------------------------------------------

__global__ void twiddle_kernel(float2* tw, int C) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < C) {
        double s, c;
        sincospi(-2.0 * (double)m / (double)C, &s, &c);
        tw[m] = make_float2((float)c, (float)s);
    }
}

// Each table is followed by a small sink that idle lanes of the radix-16
// kernel store into, so that every lane issues the same stores.
constexpr size_t kTwiddleSinkBytes = 512 * sizeof(float4);

// W_C^(n1 k2) as a matrix [n1][k2] with rows of N2 entries: between the two
// passes of the four-step FFT lanes with consecutive k2 read consecutive
// entries.  Stored under the negated rate.
__global__ void twiddle_matrix_kernel(float2* tw, int C, int N2) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < C) {
        double s, c;
        sincospi(-2.0 * (double)((m / N2) * (m % N2)) / (double)C, &s, &c);
        tw[m] = make_float2((float)c, (float)s);
    }
}

static std::mutex g_tw_mutex;
static std::map<std::pair<int, int>, float2*> g_tw;

// The table of rate C, or with N2 > 0 the matrix of C = N1 N2.  `made` is set
// when this call built it.
static int get_twiddles(int C, const float2** out, int N2 = 0, bool* made = nullptr) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return fail("channelizer: hipGetDevice failed");
    std::lock_guard<std::mutex> lock(g_tw_mutex);
    const std::pair<int, int> key(dev, N2 > 0 ? -C : C);
    auto it = g_tw.find(key);
    if (it != g_tw.end()) {
        *out = it->second;
        return BLADE_SUCCESS;
    }
    void* p = nullptr;
    const int rc = device_table("channelizer twiddles", sizeof(float2) * C + kTwiddleSinkBytes, &p,
                                [&](void* t, hipStream_t ts) {
        if (N2 > 0)
            hipLaunchKernelGGL(twiddle_matrix_kernel, dim3((C + 255) / 256), dim3(256), 0, ts, static_cast<float2*>(t), C, N2);
        else
            hipLaunchKernelGGL(twiddle_kernel, dim3((C + 255) / 256), dim3(256), 0, ts, static_cast<float2*>(t), C);
    });
    if (rc) return rc;
    *out = g_tw[key] = static_cast<float2*>(p);
    if (made) *made = true;
    return BLADE_SUCCESS;
}

// The table of rate C, and with it on first use the mixed-radix kernel's: which
// of them a call reads depends on its shape, and a call at any shape prepares
// its rate for captures at every other.  Calls of the mixed-radix kernel build
// this one beside theirs (one lookup per call: 0.2 us of 7).
static int rate_twiddles(int C, const float2** out) {
    bool made = false;
    const int rc = get_twiddles(C, out, 0, &made);
    return !rc && made && mixed_fft_covers((uint64_t)C) ? mixed_fft_plan(C) : rc;
}

// ---------------------------------------------------------------------------
// Small DFT in registers.
// ---------------------------------------------------------------------------

// Constant-twiddle DFT for the register kernel (W computed at compile time
// from the table argument in a small struct).
template <int C>
struct SmallTw {
    float2 w[C];
};

template <int C>
__device__ __forceinline__ void dft_small(float2 (&v)[C], const SmallTw<C>& tw) {
    if constexpr (C == 2 || C == 4 || C == 8) {
        dft_reg<C>(v, nullptr, 0);
    } else {
        float2 r[C];
#pragma unroll
        for (int k = 0; k < C; k++) {
            float2 acc = v[0];
#pragma unroll
            for (int n = 1; n < C; n++) {
                const float2 w = tw.w[(n * k) % C];
                acc.x += v[n].x * w.x - v[n].y * w.y;
                acc.y += v[n].x * w.y + v[n].y * w.x;
            }
            r[k] = acc;
        }
#pragma unroll
        for (int k = 0; k < C; k++) v[k] = r[k];
    }
}

// One lane per C-sample spectrum (all P pols), C <= 16.  Reads C*P contiguous
// complex samples, writes one sample per output row (coalesced across lanes).
template <int C, int P>
__global__ __launch_bounds__(256) void chan_small_kernel(const float2* __restrict__ in,
                                                         float2* __restrict__ out,
                                                         uint64_t n_spec, uint64_t S,
                                                         SmallTw<C> tw) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t sp = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; sp < n_spec; sp += stride) {
        const uint64_t af = sp / S, s = sp - af * S;
        float2 v[P][C];
        const float2* src = in + sp * C * P;
#pragma unroll
        for (int n = 0; n < C; n++) {
            if constexpr (P == 2) {
                const float4 q = reinterpret_cast<const float4*>(src)[n];
                v[0][n] = make_float2(q.x, q.y);
                v[1][n] = make_float2(q.z, q.w);
            } else {
                v[0][n] = src[n];
            }
        }
#pragma unroll
        for (int p = 0; p < P; p++) dft_small<C>(v[p], tw);
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int ko = (k + C / 2) % C;
            const uint64_t o = ((af * C + ko) * S + s) * P;
            if constexpr (P == 2) {
                reinterpret_cast<float4*>(out + o)[0] =
                    make_float4(v[0][k].x, v[0][k].y, v[1][k].x, v[1][k].y);
            } else {
                out[o] = v[0][k];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// LDS Stockham kernel: one workgroup per spectrum (all P pols), C up to 8192
// (P = 2) or 16384 (P = 1).
// ---------------------------------------------------------------------------

struct Radices {
    int r[16];
    int n;
};

constexpr int kMaxLdsComplex = 16384;   // 128 KiB of LDS

template <int R>
constexpr int groups_max() {
    return (kMaxLdsComplex / R + 1023) / 1024;
}

// One radix-R pass over PC / C sequences of C points in LDS, sequence p at
// data + p * pstride (pstride = C by default).
template <int R>
__device__ __forceinline__ void stockham_pass(float2* __restrict__ data, int C, int PC, int Ns,
                                              const float2* __restrict__ tw, int pstride = 0) {
    constexpr int G = groups_max<R>();
    const int nthr = blockDim.x;
    const int per_pol = C / R;
    const int total = PC / R;
    const int twstride = C / (Ns * R);
    if (pstride == 0) pstride = C;
    float2 v[G][R];
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int gi = threadIdx.x + g * nthr;
        if (gi < total) {
            const int p = gi / per_pol, j = gi - p * per_pol;
            const float2* base = data + p * pstride;
            const int jm = j % Ns;
#pragma unroll
            for (int r = 0; r < R; r++) {
                float2 x = base[j + r * per_pol];
                if (r > 0 && jm > 0) {
                    const float2 w = tw[jm * r * twstride];
                    x = cmul(x, w);
                }
                v[g][r] = x;
            }
            dft_reg<R>(v[g], tw, C / R);
        }
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int gi = threadIdx.x + g * nthr;
        if (gi < total) {
            const int p = gi / per_pol, j = gi - p * per_pol;
            float2* base = data + p * pstride;
            const int jm = j % Ns;
            const int d = (j - jm) * R + jm;
#pragma unroll
            for (int r = 0; r < R; r++) base[d + r * Ns] = v[g][r];
        }
    }
    __syncthreads();
}

template <int P>
__global__ __launch_bounds__(1024) void chan_lds_kernel(const float2* __restrict__ in,
                                                        float2* __restrict__ out, int C,
                                                        uint64_t S, uint64_t n_spec,
                                                        const float2* __restrict__ tw,
                                                        Radices rad) {
    extern __shared__ float2 data[];
    const int PC = P * C;
    for (uint64_t sp = blockIdx.x; sp < n_spec; sp += gridDim.x) {
        const uint64_t af = sp / S, s = sp - af * S;
        const float2* src = in + sp * (uint64_t)C * P;
        for (int n = threadIdx.x; n < C; n += blockDim.x) {
            if constexpr (P == 2) {
                const float4 q = reinterpret_cast<const float4*>(src)[n];
                data[n] = make_float2(q.x, q.y);
                data[C + n] = make_float2(q.z, q.w);
            } else {
                data[n] = src[n];
            }
        }
        __syncthreads();
        int Ns = 1;
        for (int i = 0; i < rad.n; i++) {
            const int R = rad.r[i];
            switch (R) {
                case 2: stockham_pass<2>(data, C, PC, Ns, tw); break;
                case 3: stockham_pass<3>(data, C, PC, Ns, tw); break;
                case 4: stockham_pass<4>(data, C, PC, Ns, tw); break;
                case 5: stockham_pass<5>(data, C, PC, Ns, tw); break;
                case 7: stockham_pass<7>(data, C, PC, Ns, tw); break;
                default: stockham_pass<8>(data, C, PC, Ns, tw); break;
            }
            Ns *= R;
        }
        const int half = C / 2;
        for (int k = threadIdx.x; k < C; k += blockDim.x) {
            int ko = k + half;
            if (ko >= C) ko -= C;
            const uint64_t o = ((af * C + ko) * S + s) * P;
            if constexpr (P == 2) {
                reinterpret_cast<float4*>(out + o)[0] =
                    make_float4(data[k].x, data[k].y, data[C + k].x, data[C + k].y);
            } else {
                out[o] = data[k];
            }
        }
        __syncthreads();
    }
}

// All passes of `rad` over PC / N sequences of N points at stride pstride.
__device__ __forceinline__ void stockham_all(float2* data, int N, int PC, const float2* tw, const Radices& rad,
                                             int pstride) {
    int Ns = 1;
    for (int i = 0; i < rad.n; i++) {
        switch (rad.r[i]) {
            case 2: stockham_pass<2>(data, N, PC, Ns, tw, pstride); break;
            case 3: stockham_pass<3>(data, N, PC, Ns, tw, pstride); break;
            case 4: stockham_pass<4>(data, N, PC, Ns, tw, pstride); break;
            case 5: stockham_pass<5>(data, N, PC, Ns, tw, pstride); break;
            case 7: stockham_pass<7>(data, N, PC, Ns, tw, pstride); break;
            default: stockham_pass<8>(data, N, PC, Ns, tw, pstride); break;
        }
        Ns *= rad.r[i];
    }
}

// ---------------------------------------------------------------------------
// Rates past one workgroup's LDS (P * C > 16384): two passes through a
// scratch buffer (the four-step FFT).  With C = N1 * N2, n = n1 + N1 n2 and
// k = k2 + N2 k1:
//   pass 1, each n1:  Y[n1, k2] = W_C^(n1 k2) sum_n2 x[n1 + N1 n2] W_N2^(n2 k2)
//   pass 2, each k2:  X[k2 + N2 k1] = sum_n1 Y[n1, k2] W_N1^(n1 k1)
// and the fftshift of X moves k1 by N1 / 2 (N1 even).  Scratch layout
// [spectrum][pol][n1][k2].  A workgroup (1024 threads) transforms a tile of
// `cols` consecutive n1 (pass 1) or k2 (pass 2) of one spectrum, both pols,
// so every global access moves `cols` consecutive samples; the LDS sequences
// are padded by one sample against bank conflicts.
// ---------------------------------------------------------------------------

template <int P>
__global__ __launch_bounds__(1024) void chan_big_pass1(const float2* __restrict__ in, float2* __restrict__ y,
                                                       int C, int N1, int N2, int cols, uint64_t n_spec,
                                                       const float2* __restrict__ twN2,
                                                       const float2* __restrict__ twC, Radices rad) {
    extern __shared__ float2 data[];
    const int stride = N2 + 1;
    const int L = P * cols;
    const uint64_t tiles = (uint64_t)(N1 / cols);
    for (uint64_t it = blockIdx.x; it < n_spec * tiles; it += gridDim.x) {
        const uint64_t sp = it / tiles;
        const int n1_0 = (int)(it - sp * tiles) * cols;
        const float2* src = in + sp * (uint64_t)C * P;
        for (int e = threadIdx.x; e < cols * N2; e += blockDim.x) {
            const int n2 = e / cols, c = e - n2 * cols;
            const uint64_t n = (uint64_t)(n1_0 + c) + (uint64_t)N1 * n2;
            if constexpr (P == 2) {
                const float4 q = reinterpret_cast<const float4*>(src)[n];
                data[c * stride + n2] = make_float2(q.x, q.y);
                data[(cols + c) * stride + n2] = make_float2(q.z, q.w);
            } else {
                data[c * stride + n2] = src[n];
            }
        }
        __syncthreads();
        stockham_all(data, N2, L * N2, twN2, rad, stride);
        for (int e = threadIdx.x; e < L * N2; e += blockDim.x) {
            const int q = e / N2, k2 = e - q * N2;
            const int pp = q / cols, c = q - pp * cols;
            // n1 k2 < N1 N2 = C: the exponent needs no reduction
            const int n1 = n1_0 + c;
            const float2 w = twC[n1 * k2];
            y[((sp * P + pp) * N1 + n1) * (uint64_t)N2 + k2] = cmul(data[q * stride + k2], w);
        }
        __syncthreads();
    }
}

template <int P>
__global__ __launch_bounds__(1024) void chan_big_pass2(const float2* __restrict__ y, float2* __restrict__ out,
                                                       int C, int N1, int N2, int cols, uint64_t n_spec,
                                                       uint64_t S, const float2* __restrict__ twN1, Radices rad) {
    extern __shared__ float2 data[];
    const int stride = N1 + 1;
    const int L = P * cols;
    const uint64_t tiles = (uint64_t)(N2 / cols);
    const int half1 = N1 / 2;
    for (uint64_t it = blockIdx.x; it < n_spec * tiles; it += gridDim.x) {
        const uint64_t sp = it / tiles;
        const int k2_0 = (int)(it - sp * tiles) * cols;
        for (int e = threadIdx.x; e < L * N1; e += blockDim.x) {
            const int c = e % cols, r = e / cols;
            const int n1 = r % N1, pp = r / N1;
            data[(pp * cols + c) * stride + n1] = y[((sp * P + pp) * N1 + n1) * (uint64_t)N2 + k2_0 + c];
        }
        __syncthreads();
        stockham_all(data, N1, L * N1, twN1, rad, stride);
        const uint64_t af = sp / S, s = sp - af * S;
        for (int e = threadIdx.x; e < cols * N1; e += blockDim.x) {
            const int k1 = e / cols, c = e - k1 * cols;
            int k1o = k1 + half1;
            if (k1o >= N1) k1o -= N1;
            const uint64_t ko = (uint64_t)(k2_0 + c) + (uint64_t)N2 * k1o;
            const uint64_t o = ((af * C + ko) * S + s) * P;
            if constexpr (P == 2) {
                const float2 X = data[c * stride + k1], Y = data[(cols + c) * stride + k1];
                reinterpret_cast<float4*>(out + o)[0] = make_float4(X.x, X.y, Y.x, Y.y);
            } else {
                out[o] = data[c * stride + k1];
            }
        }
        __syncthreads();
    }
}

// Channelizer with the detector fused on the output: one workgroup per
// integration walks its S spectra, transforms both pols in LDS and sums
// |X|^2+|Y|^2 (or XX*, YY*, Re XY*, Im XY*) of every fine channel over them in
// registers, writing (or adding to, with accumulate)
//   out[a, f*C + k', group, q].
// The CF32 spectra never reach HBM.
template <int NPOL, int KPT>
__global__ __launch_bounds__(1024) void chan_detect_kernel(const float2* __restrict__ in,
                                                           float* __restrict__ out, int C,
                                                           uint64_t S, uint64_t groups, uint64_t n_items,
                                                           const float2* __restrict__ tw,
                                                           Radices rad, int flags) {
    extern __shared__ float2 data[];
    const int accumulate = flags & 1;
    const bool circular = flags & 2;
    const int PC = 2 * C;
    const int half = C / 2;
    for (uint64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
        float acc[KPT][NPOL];
#pragma unroll
        for (int j = 0; j < KPT; j++)
#pragma unroll
            for (int q = 0; q < NPOL; q++) acc[j][q] = 0.f;
        for (uint64_t s = 0; s < S; s++) {
            const float4* src = reinterpret_cast<const float4*>(in + ((item * S + s) * (uint64_t)C) * 2);
            for (int n = threadIdx.x; n < C; n += blockDim.x) {
                const float4 q = src[n];
                data[n] = make_float2(q.x, q.y);
                data[C + n] = make_float2(q.z, q.w);
            }
            __syncthreads();
            int Ns = 1;
            for (int i = 0; i < rad.n; i++) {
                const int R = rad.r[i];
                switch (R) {
                    case 2: stockham_pass<2>(data, C, PC, Ns, tw); break;
                    case 3: stockham_pass<3>(data, C, PC, Ns, tw); break;
                    case 4: stockham_pass<4>(data, C, PC, Ns, tw); break;
                    case 5: stockham_pass<5>(data, C, PC, Ns, tw); break;
                    case 7: stockham_pass<7>(data, C, PC, Ns, tw); break;
                    default: stockham_pass<8>(data, C, PC, Ns, tw); break;
                }
                Ns *= R;
            }
#pragma unroll
            for (int j = 0; j < KPT; j++) {
                const int k = threadIdx.x + j * blockDim.x;
                if (k < C) {
                    const float2 X = data[k], Y = data[C + k];
                    acc[j][0] += X.x * X.x + X.y * X.y + (NPOL == 1 ? Y.x * Y.x + Y.y * Y.y : 0.f);
                    if constexpr (NPOL == 4) {
                        acc[j][1] += Y.x * Y.x + Y.y * Y.y;
                        acc[j][2] += X.x * Y.x + X.y * Y.y;
                        acc[j][3] += X.y * Y.x - X.x * Y.y;
                    }
                }
            }
            __syncthreads();
            if (s == S - 1) {
                const uint64_t af = item / groups, grp = item - af * groups;
                if (circular) {
#pragma unroll
                    for (int j = 0; j < KPT; j++) circular_sums<NPOL>(acc[j]);
                }
#pragma unroll
                for (int j = 0; j < KPT; j++) {
                    const int k = threadIdx.x + j * blockDim.x;
                    if (k < C) {
                        int ko = k + half;
                        if (ko >= C) ko -= C;
                        float* o = out + ((af * C + ko) * groups + grp) * NPOL;
#pragma unroll
                        for (int q = 0; q < NPOL; q++) {
                            o[q] = accumulate ? o[q] + acc[j][q] : acc[j][q];
                            acc[j][q] = 0.f;
                        }
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Power-of-two rates 256 <= C <= 8192 with both polarizations, radix 16.
//
// Every thread holds 16 points of each polarization, so a spectrum takes
// C/16 threads and a workgroup of NT threads holds NT*16/C spectra.  The
// passes are radix 16 (floor(log2 C / 4) of them) plus one trailing radix 2,
// 4 or 8 pass when log2 C is not a multiple of 4:
//   first   radix 16 on registers loaded straight from HBM: sixteen 16-byte
//           loads per thread (both pols), issued one spectrum ahead so that
//           they are in flight during the LDS passes of the current one;
//   middle  radix 16, LDS -> LDS;
//   last    LDS -> the fftshifted spectrum in HBM (MODE 0), or detector sums
//           in registers (MODE 1: Stokes I; MODE 4: XX*, YY*, Re XY*, Im XY*).
// LDS holds one plane per polarization with one float2 of padding after every
// 16 points: the 16 consecutive points a lane writes in the first pass, and
// the groups of 16 written in the Ns = 16 pass, then fall on distinct banks.
// Twiddles depend only on the thread's position in its spectrum: W, W^2, W^4
// and W^8 of each pass are read from the table once per launch and the other
// powers are products of these, so the loop's only global loads are the next
// spectrum's samples.
// ---------------------------------------------------------------------------

__device__ __forceinline__ int lpad(int pos) { return pos + (pos >> 4); }

template <int R>
__device__ __forceinline__ void dft_pow2(float2 (&v)[R]) {
    if constexpr (R == 16) dft16(v);
    else dft_reg<R>(v, nullptr, 0);
}

// w[r] = W^r for r < R from b = {W, W^2, W^4, W^8}.
template <int R>
__device__ __forceinline__ void twiddle_powers(const float2 (&b)[4], float2 (&w)[R]) {
    w[0] = make_float2(1.f, 0.f);
    if constexpr (R > 1) w[1] = b[0];
    if constexpr (R > 2) { w[2] = b[1]; w[3] = cmul(b[0], b[1]); }
    if constexpr (R > 4) {
        w[4] = b[2];
#pragma unroll
        for (int r = 5; r < 8; r++) w[r] = cmul(w[r - 4], b[2]);
    }
    if constexpr (R > 8) {
        w[8] = b[3];
#pragma unroll
        for (int r = 9; r < 16; r++) w[r] = cmul(w[r - 8], b[3]);
    }
}

// One radix-16 Stockham pass in LDS, Ns = NS, butterfly j = tl.
template <int C, int NS>
__device__ __forceinline__ void fft16_mid(float2* __restrict__ p0, float2* __restrict__ p1, int tl,
                                          const float2* __restrict__ twl) {
    constexpr int STRIDE = C / 16;
    float2 tb[4];
#pragma unroll
    for (int e = 0; e < 4; e++) tb[e] = twl[e * NS + (tl & (NS - 1))];
    // One polarization's results are written while the other is computed.
    float2 a[16], b[16];
    const int rd = lpad(tl);
#pragma unroll
    for (int r = 0; r < 16; r++) a[r] = p0[rd + r * (STRIDE + STRIDE / 16)];
#pragma unroll
    for (int r = 0; r < 16; r++) b[r] = p1[rd + r * (STRIDE + STRIDE / 16)];
    float2 w[16];
    twiddle_powers<16>(tb, w);
#pragma unroll
    for (int r = 1; r < 16; r++) a[r] = cmul(a[r], w[r]);
    dft16(a);
    __syncthreads();                       // both planes have been read
    const int jm = tl & (NS - 1);
    const int wr = lpad((tl - jm) * 16 + jm);
#pragma unroll
    for (int r = 0; r < 16; r++) p0[wr + r * (NS + NS / 16)] = a[r];
#pragma unroll
    for (int r = 1; r < 16; r++) b[r] = cmul(b[r], w[r]);
    dft16(b);
#pragma unroll
    for (int r = 0; r < 16; r++) p1[wr + r * (NS + NS / 16)] = b[r];
    __syncthreads();
}

// LDS twiddle table of the middle passes: pass i (Ns = 16^(i+1)) holds
// W_{16 Ns}^(e' jm) for e' = 1, 2, 4, 8 and jm < Ns, laid out [e][jm] so that
// lanes with consecutive jm read consecutive entries.
__host__ __device__ constexpr int fft16_twl_offset(int i) { return i == 0 ? 0 : 4 * 16 + (i - 1) * 4 * 256; }

template <int C, int NMID, int I>
__device__ __forceinline__ void fft16_mids(float2* p0, float2* p1, int tl, const float2* twl) {
    if constexpr (I < NMID) {
        constexpr int NS = 1 << (4 * (I + 1));
        fft16_mid<C, NS>(p0, p1, tl, twl + fft16_twl_offset(I));
        fft16_mids<C, NMID, I + 1>(p0, p1, tl, twl);
    }
}

// The last radix-16 pass for C = 16^k * 2 kept in registers: butterfly j
// (Ns = NS) reads LDS and its 16 results stay in a[] and b[], at positions
// (j / NS) * 16 NS + (j mod NS) + r NS.  With lane l of wave w taking
// j = 32 w + (l mod 32) + (l >= 32 ? C/32 : 0), the final radix-2 pass's
// partners (positions p and p + C/2) sit in register r of lanes l and l ^ 32.
template <int C, int NS>
__device__ __forceinline__ void fft16_mid_regs(const float2* __restrict__ p0, const float2* __restrict__ p1,
                                               int j, const float2* __restrict__ twl, float2 (&a)[16],
                                               float2 (&b)[16]) {
    constexpr int STRIDE = C / 16;
    float2 tb[4];
#pragma unroll
    for (int e = 0; e < 4; e++) tb[e] = twl[e * NS + (j & (NS - 1))];
    const int rd = lpad(j);
#pragma unroll
    for (int r = 0; r < 16; r++) {
        a[r] = p0[rd + r * (STRIDE + STRIDE / 16)];
        b[r] = p1[rd + r * (STRIDE + STRIDE / 16)];
    }
    float2 w[16];
    twiddle_powers<16>(tb, w);
#pragma unroll
    for (int r = 1; r < 16; r++) {
        a[r] = cmul(a[r], w[r]);
        b[r] = cmul(b[r], w[r]);
    }
    dft16(a);
    dft16(b);
}

// One polarization's plane of fft16_mid_regs.
template <int C, int NS>
__device__ __forceinline__ void fft16_mid_regs1(const float2* __restrict__ pl, int j, const float2* __restrict__ twl,
                                                float2 (&a)[16]) {
    constexpr int STRIDE = C / 16;
    float2 tb[4];
#pragma unroll
    for (int e = 0; e < 4; e++) tb[e] = twl[e * NS + (j & (NS - 1))];
    const int rd = lpad(j);
#pragma unroll
    for (int r = 0; r < 16; r++) a[r] = pl[rd + r * (STRIDE + STRIDE / 16)];
    float2 w[16];
    twiddle_powers<16>(tb, w);
#pragma unroll
    for (int r = 1; r < 16; r++) a[r] = cmul(a[r], w[r]);
    dft16(a);
}

// W_32^r = exp(-j 2 pi r / 32), r < 16, from cos(k pi / 16).
__device__ __forceinline__ float2 w32(int r) {
    constexpr float c1 = 0.98078528040323044913f, c2 = 0.92387953251128675613f;
    constexpr float c3 = 0.83146961230254523708f, c4 = 0.70710678118654752440f;
    constexpr float c5 = 0.55557023301960222474f, c6 = 0.38268343236508977173f;
    constexpr float c7 = 0.19509032201612826785f;
    constexpr float re[16] = {1.f, c1, c2, c3, c4, c5, c6, c7, 0.f, -c7, -c6, -c5, -c4, -c3, -c2, -c1};
    constexpr float im[16] = {0.f, -c7, -c6, -c5, -c4, -c3, -c2, -c1, -1.f, -c1, -c2, -c3, -c4, -c5, -c6, -c7};
    return make_float2(re[r], im[r]);
}

// x at lanes l < 32 holds u, at lanes l >= 32 holds v (same register):
// returns u and v in every lane.
__device__ __forceinline__ void halves(float x, float& u, float& v) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    u = __uint_as_float(p[0]);
    v = __uint_as_float(p[1]);
}

// SM (MODE 0 stores): 0 strided, 1 nontemporal with one spectrum per
// (antenna, channel), 2 transposed through LDS so that the workgroup's SPW
// consecutive spectra of one (antenna, channel) land as whole lines.
// Detector items: SM 0 one integration each (S spectra, `ng` = integrations per
// channel), SM 3 one (antenna, channel) each (S spectra, `ng` = spectra per
// integration).
template <int LC, int NT, int MODE, int SM>
__global__ __launch_bounds__(NT, 2) void fft16_kernel(const float4* __restrict__ in, void* __restrict__ outv,
                                                      uint64_t S, uint64_t n_items, int ng, int flags,
                                                      const float2* __restrict__ tw, float4* __restrict__ sink) {
    const int accumulate = flags & 1;
    const bool circular = flags & 2;
    constexpr int C = 1 << LC;
    constexpr int TPS = C / 16;                        // threads per spectrum
    static_assert(NT % TPS == 0 && LC >= 8, "workgroup must hold whole spectra");
    constexpr int SPW = NT / TPS;                      // spectra per workgroup
    constexpr int RL = 1 << (LC % 4);                  // trailing radix, 1 = none
    constexpr int NMID = LC / 4 - (RL > 1 ? 1 : 2);    // radix-16 passes in LDS
    constexpr int R = RL > 1 ? RL : 16;                // radix of the last pass
    constexpr int G = 16 / R;                          // last-pass butterflies per thread
    constexpr int NSL = C / R;                         // Ns (and stride) of the last pass
    constexpr int PLANE = C + C / 16;
    constexpr int NPOL = MODE == 0 ? 1 : MODE;
    // Final radix-2 pass across lane halves (whole waves per spectrum); the
    // full-Stokes sums need both polarizations at once and keep the LDS pass.
    constexpr bool SW = RL == 2 && TPS % 64 == 0 && NMID >= 1 && MODE != 4;
    extern __shared__ float2 lds[];
    const int slot = threadIdx.x / TPS;
    const int tl = threadIdx.x % TPS;
    float2* const p0 = lds + slot * 2 * PLANE;
    float2* const p1 = p0 + PLANE;

    // Twiddle bases.  Middle pass i has Ns = 16^(i+1) and uses
    // W_{16 Ns}^(tl mod Ns) = tw[(tl mod Ns) * C / (16 Ns)] and its powers 2,
    // 4, 8, from an LDS table behind the data planes (filled here, first read
    // after the first pass's barrier); the last pass uses W_C^(tl r) W_16^(g r)
    // for butterfly j = tl + g * C/16, from per-thread registers.
    float2* const twl = lds + SPW * 2 * PLANE;
#pragma unroll
    for (int i = 0; i < NMID; i++) {
        const int ns = 1 << (4 * (i + 1));
        for (int idx = threadIdx.x; idx < 4 * ns; idx += NT) {
            const int e = idx / ns, jm = idx - e * ns;
            twl[fft16_twl_offset(i) + idx] = tw[((jm * (C / (16 * ns))) << e) & (C - 1)];
        }
    }
    float2 tb[4];
#pragma unroll
    for (int e = 0; e < 4; e++) tb[e] = tw[(tl << e) & (C - 1)];
    // SW: lane l of wave w handles jlow = 32 w + (l mod 32) in the upper
    // (l >= 32) or lower half; its final-pass twiddle base is W_C^jlow.
    const bool hi = (tl & 63) >= 32;
    const int jlow = (tl >> 6) * 32 + (tl & 31);
    const float2 tsw = SW ? tw[jlow] : make_float2(1.f, 0.f);
    // Output channel (fftshifted) of result i: lane base + per-result offset.
    const int ch0 = SW ? jlow + (hi ? 0 : C / 2) : tl;
    auto kofs = [](int i) -> int {
        if constexpr (SW) return i * (C / 32);
        else return ((i / R) * TPS + (i % R) * NSL + (C >> 1)) & (C - 1);
    };

    // Strided stores: workgroups of consecutive spectra share an XCD.
    const unsigned wgi = (MODE == 0 && SM == 0) ? xcd_order(blockIdx.x, gridDim.x) : blockIdx.x;
    const uint64_t per_round = (uint64_t)gridDim.x * SPW;
    const uint64_t rounds = (n_items + per_round - 1) / per_round;
    const int nspec = MODE == 0 ? 1 : (int)S;

    // The spectra of a workgroup in one round are consecutive (items first ..
    // first + SPW - 1): addresses are a workgroup-uniform base plus a 32-bit
    // lane offset.  Idle slots re-read their workgroup's first spectrum (or
    // spectrum 0) and store nothing.
    const unsigned SC = (unsigned)(MODE == 0 ? 1 : S) * C;      // float4s per item
    float4 q[16];
    auto load = [&](uint64_t round, int s) {
        const uint64_t first = (round * gridDim.x + wgi) * SPW;
        const bool any = first < n_items;
        const uint64_t b0 = any ? (MODE == 0 ? first * C : (first * S + s) * C) : 0;
        const unsigned lo = ((any && first + slot < n_items) ? slot * SC : 0u) + tl;
#pragma unroll
        for (int r = 0; r < 16; r++) q[r] = (in + (b0 + r * TPS))[lo];
    };

    float acc[16][NPOL];
#pragma unroll
    for (int i = 0; i < 16; i++)
#pragma unroll
        for (int c = 0; c < NPOL; c++) acc[i][c] = 0.f;

    // The full-Stokes detector keeps 64 sums per thread, which leaves no
    // room for the next spectrum's registers: it loads at the top instead.
    constexpr bool PF = MODE != 4;
    if constexpr (PF) {
        load(0, 0);
        // Nothing pending at loop entry, so the first pass of every spectrum
        // waits only for its own loads, not for the previous spectrum's stores.
        __builtin_amdgcn_s_waitcnt(0);
    }
    for (uint64_t round = 0; round < rounds; round++) {
        const uint64_t first = (round * gridDim.x + wgi) * SPW;
        const uint64_t item = first + slot;
        const bool valid = item < n_items;
        for (int s = 0; s < nspec; s++) {
            if constexpr (!PF) load(round, s);
            // ---- first pass: radix 16 on registers -> LDS (Ns = 1)
            {
                float2 a[16], b[16];
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    a[r] = make_float2(q[r].x, q[r].y);
                    b[r] = make_float2(q[r].z, q[r].w);
                }
                const int wr = tl * 17;
                dft16(a);
#pragma unroll
                for (int r = 0; r < 16; r++) p0[wr + r] = a[r];
                dft16(b);
#pragma unroll
                for (int r = 0; r < 16; r++) p1[wr + r] = b[r];
                // Next spectrum into the registers just consumed (a fresh set
                // would be copied back at the loop latch behind a full wait).
                // After the last spectrum this re-reads spectrum 0 (an L2 hit)
                // rather than branching, which keeps the waits exact.
                if constexpr (PF) {
                    uint64_t nr = round;
                    int ns = s + 1;
                    if (ns == nspec) { ns = 0; nr++; }
                    load(nr, ns);
                }
            }
            __syncthreads();
            float2 a[16], b[16];
            if constexpr (SW) {
                // ---- last radix-16 pass in registers, then radix 2 across
                // lane halves: X(p) = u + W v in the lower half, X(p + C/2) =
                // u - W v in the upper, W = W_C^(jlow + r C/32).
                fft16_mids<C, NMID - 1, 0>(p0, p1, tl, twl);
                constexpr int NSR = 1 << (4 * NMID);
                const int jr = jlow + (hi ? C / 32 : 0);
                const float2* const twr = twl + fft16_twl_offset(NMID - 1);
                const float sg = hi ? -1.f : 1.f;
                auto radix2 = [&](float2& x, const float2 wr) {
                    float2 u, v;
                    halves(x.x, u.x, v.x);
                    halves(x.y, u.y, v.y);
                    const float2 t = cmul(wr, v);
                    x = make_float2(u.x + sg * t.x, u.y + sg * t.y);
                };
                // W_32^(r + 8) = -j W_32^r: one twiddle product serves
                // results r and r + 8.
                auto negj = [](float2 w) { return make_float2(w.y, -w.x); };
                if constexpr (MODE == 1) {
                    // Stokes I: one polarization at a time (half the registers).
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        fft16_mid_regs1<C, NSR>(q == 0 ? p0 : p1, jr, twr, a);
#pragma unroll
                        for (int r = 0; r < 8; r++) {
                            const float2 wr = cmul(tsw, w32(r));
                            radix2(a[r], wr);
                            radix2(a[r + 8], negj(wr));
                            acc[r][0] += a[r].x * a[r].x + a[r].y * a[r].y;
                            acc[r + 8][0] += a[r + 8].x * a[r + 8].x + a[r + 8].y * a[r + 8].y;
                        }
                    }
                } else {
                    fft16_mid_regs<C, NSR>(p0, p1, jr, twr, a, b);
#pragma unroll
                    for (int r = 0; r < 8; r++) {
                        const float2 wr = cmul(tsw, w32(r)), wr8 = negj(wr);
                        radix2(a[r], wr);
                        radix2(b[r], wr);
                        radix2(a[r + 8], wr8);
                        radix2(b[r + 8], wr8);
                    }
                }
            } else {
            fft16_mids<C, NMID, 0>(p0, p1, tl, twl);
            // ---- last pass: radix R, LDS -> output (Ns = C / R)
            const int rd = lpad(tl);
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const int off = (g * TPS + r * NSL) + (g * TPS + r * NSL) / 16;
                    a[g * R + r] = p0[rd + off];
                    b[g * R + r] = p1[rd + off];
                }
            {
                float2 w[R];
                twiddle_powers<R>(tb, w);
#pragma unroll
                for (int g = 0; g < G; g++) {
#pragma unroll
                    for (int r = 1; r < R; r++) {
                        float2 wr = w[r];
                        switch ((g * r) & 15) {     // W_16^(g r), resolved at compile time
                            case 0: break;
                            case 1: wr = mul_w16<1>(wr); break;
                            case 2: wr = mul_w16<2>(wr); break;
                            case 3: wr = mul_w16<3>(wr); break;
                            case 4: wr = mul_w16<4>(wr); break;
                            case 5: wr = mul_w16<5>(wr); break;
                            case 6: wr = mul_w16<6>(wr); break;
                            case 7: wr = mul_w16<7>(wr); break;
                            case 8: wr = mul_w16<8>(wr); break;
                            case 9: wr = mul_w16<9>(wr); break;
                            case 10: wr = mul_w16<10>(wr); break;
                            case 11: wr = mul_w16<11>(wr); break;
                            case 12: wr = mul_w16<12>(wr); break;
                            case 13: wr = mul_w16<13>(wr); break;
                            case 14: wr = mul_w16<14>(wr); break;
                            default: wr = mul_w16<15>(wr); break;
                        }
                        a[g * R + r] = cmul(a[g * R + r], wr);
                        b[g * R + r] = cmul(b[g * R + r], wr);
                    }
                    float2 xa[R], xb[R];
#pragma unroll
                    for (int r = 0; r < R; r++) { xa[r] = a[g * R + r]; xb[r] = b[g * R + r]; }
                    dft_pow2<R>(xa);
                    dft_pow2<R>(xb);
#pragma unroll
                    for (int r = 0; r < R; r++) { a[g * R + r] = xa[r]; b[g * R + r] = xb[r]; }
                }
            }
            }
            // Channel of result i (fftshifted): ch0 + kofs(i).  Without SW,
            // k = tl + K with K = g C/16 + r C/R and ko = tl + ((K + C/2) mod
            // C), the bracket a multiple of C/16.
            // Idle lanes store into the sink (same store count on every lane
            // and path, so waits on the next spectrum's loads stay exact).
            if constexpr (MODE == 0 && SM == 2) {
                // S is a multiple of SPW: the workgroup's spectra are
                // si0 .. si0 + SPW - 1 of one (antenna, channel), whose outputs
                // interleave at (ko S + si).  Stage them [ko][spectrum] in LDS
                // (one float4 of padding per 16) and store runs of SPW.
                __syncthreads();                    // the last pass's LDS reads are done
                float4* const L = reinterpret_cast<float4*>(lds);
                int base = ch0 * SPW + slot;
                asm volatile("" : "+v"(base));      // not hoisted: see below
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int idx = base + kofs(i) * SPW;
                    L[idx + (idx >> 4)] = make_float4(a[i].x, a[i].y, b[i].x, b[i].y);
                }
                __syncthreads();
                // Thread t stores entries t + i NT, i < 16: spectrum t mod SPW,
                // channel t / SPW + i NT / SPW (NT is a multiple of SPW).
                const bool wg_valid = first < n_items;
                const uint64_t af0 = first / S, si0 = first - af0 * S;
                const int tx = threadIdx.x;
                float4* const lb = wg_valid ? static_cast<float4*>(outv) + af0 * C * S + si0 +
                                                  (uint64_t)(tx / SPW) * S + (tx % SPW)
                                            : sink + tx;
                const uint64_t step = wg_valid ? (uint64_t)(NT / SPW) * S : 0;
                const int rb = tx + (tx >> 4);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float4 v = L[rb + i * (NT + NT / 16)];
                    float* const of = reinterpret_cast<float*>(lb + i * step);
                    __builtin_nontemporal_store(v.x, of);
                    __builtin_nontemporal_store(v.y, of + 1);
                    __builtin_nontemporal_store(v.z, of + 2);
                    __builtin_nontemporal_store(v.w, of + 3);
                }
            } else if constexpr (MODE == 0) {
                const uint64_t af = item / S, si = item - af * S;
                float4* const lb = valid ? static_cast<float4*>(outv) + (af * C * S + si) + (uint64_t)ch0 * S
                                         : sink + threadIdx.x;
                const uint64_t step = valid ? S : 0;
#pragma unroll
                for (int g = 0; g < G; g++)
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const int kb = kofs(g * R + r);
                        const float2 X = a[g * R + r], Y = b[g * R + r];
                        float4* const o = lb + (uint64_t)kb * step;
                        if constexpr (SM == 1) {
                            // Component-wise: merged into one nontemporal
                            // global_store_dwordx4 (a vector operand here is
                            // lowered through private memory).
                            float* const of = reinterpret_cast<float*>(o);
                            __builtin_nontemporal_store(X.x, of);
                            __builtin_nontemporal_store(X.y, of + 1);
                            __builtin_nontemporal_store(Y.x, of + 2);
                            __builtin_nontemporal_store(Y.y, of + 3);
                        } else {
                            *o = make_float4(X.x, X.y, Y.x, Y.y);
                        }
                    }
            } else {
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    if constexpr (SW && MODE == 1) break;     // summed in the register pass
                    const float2 X = a[i], Y = b[i];
                    if constexpr (MODE == 1) {
                        acc[i][0] += X.x * X.x + X.y * X.y + Y.x * Y.x + Y.y * Y.y;
                    } else {
                        acc[i][0] += X.x * X.x + X.y * X.y;
                        acc[i][NPOL > 1 ? 1 : 0] += Y.x * Y.x + Y.y * Y.y;
                        acc[i][NPOL > 2 ? 2 : 0] += X.x * Y.x + X.y * Y.y;
                        acc[i][NPOL > 3 ? 3 : 0] += X.y * Y.x - X.x * Y.y;
                    }
                }
                const bool flush = SM == 3 ? ((ng <= (int)S) ? ((s + 1) % ng == 0) : (s == (int)S - 1)) : s == nspec - 1;
                if (flush) {
                    const int groups = SM == 3 ? ((ng <= (int)S) ? (int)S / ng : 1) : ng;
                    uint64_t af = item;
                    unsigned grp = SM == 3 && ng <= (int)S ? s / ng : 0;
                    if (SM != 3 && groups != 1) {          // items fit 32 bits (host check)
                        af = (unsigned)item / (unsigned)groups;
                        grp = (unsigned)item - (unsigned)af * (unsigned)groups;
                    }
                    if (circular) {
#pragma unroll
                        for (int i = 0; i < 16; i++) circular_sums<NPOL>(acc[i]);
                    }
                    const unsigned gn = (unsigned)groups * NPOL;
                    float* const lb = valid ? static_cast<float*>(outv) + (af * C + ch0) * gn + grp * NPOL
                                            : reinterpret_cast<float*>(sink + threadIdx.x);
                    unsigned step = valid ? gn : 0;
                    // Opaque: keeps the 16 output addresses from being hoisted
                    // out of the spectrum loop (they would pin 32 registers).
                    asm volatile("" : "+v"(step));
                    // All earlier sums are read before any store (idle lanes'
                    // addresses coincide, so the compiler cannot interleave).
                    // The four full-Stokes sums of a channel are one 16-byte
                    // access (the output rows are 16-byte aligned).
                    if (accumulate) {
                        float old[16][NPOL];
#pragma unroll
                        for (int g = 0; g < G; g++)
#pragma unroll
                            for (int r = 0; r < R; r++) {
                                const int kb = kofs(g * R + r);
                                const float* const o = lb + (uint64_t)((unsigned)kb * step);
                                if constexpr (NPOL == 4) {
                                    const float4 v = *reinterpret_cast<const float4*>(o);
                                    old[g * R + r][0] = v.x;
                                    old[g * R + r][NPOL > 1 ? 1 : 0] = v.y;
                                    old[g * R + r][NPOL > 2 ? 2 : 0] = v.z;
                                    old[g * R + r][NPOL > 3 ? 3 : 0] = v.w;
                                } else {
                                    old[g * R + r][0] = o[0];
                                }
                            }
#pragma unroll
                        for (int i = 0; i < 16; i++)
#pragma unroll
                            for (int c = 0; c < NPOL; c++) acc[i][c] += old[i][c];
                    }
#pragma unroll
                    for (int g = 0; g < G; g++)
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            const int kb = kofs(g * R + r);
                            float* const o = lb + (uint64_t)((unsigned)kb * step);
                            const int i = g * R + r;
                            if constexpr (NPOL == 4)
                                *reinterpret_cast<float4*>(o) = make_float4(acc[i][0], acc[i][NPOL > 1 ? 1 : 0],
                                                                            acc[i][NPOL > 2 ? 2 : 0],
                                                                            acc[i][NPOL > 3 ? 3 : 0]);
                            else
                                o[0] = acc[i][0];
                        }
#pragma unroll
                    for (int i = 0; i < 16; i++)
#pragma unroll
                        for (int c = 0; c < NPOL; c++) acc[i][c] = 0.f;
                }
            }
            __syncthreads();   // LDS is rewritten by the next spectrum's first pass
        }
    }
}

// Launch of fft16_kernel for C = 2^LC; NT threads use NT * 272 bytes of LDS
// (one 512-thread workgroup per CU).
template <int LC, int NT, int MODE, int SM>
static int launch_fft16_t(const float2* in, void* out, uint64_t S, uint64_t n_items, int groups, int accumulate,
                          const float2* tw, hipStream_t s) {
    constexpr int C = 1 << LC;
    constexpr int SPW = NT / (C / 16);
    constexpr int NMID = LC / 4 - ((LC % 4) ? 1 : 2);
    constexpr size_t lds = sizeof(float2) * (2 * (size_t)(C + C / 16) * SPW + fft16_twl_offset(NMID));
    const void* fn = reinterpret_cast<const void*>(&fft16_kernel<LC, NT, MODE, SM>);
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            set_error(std::string("channelizer: LDS attribute: ") + hipGetErrorString(e));
            return BLADE_HIP_ERROR;
        }
    }
    const uint64_t nb = ceil_div(n_items, SPW);
    const uint64_t resident = (uint64_t)device_cus() * (NT >= 512 ? 1 : 2);
    const uint64_t rounds = ceil_div(nb, resident);
    uint64_t blocks = ceil_div(nb, rounds);            // equal rounds for every workgroup
    if (MODE == 0 && SM == 0) blocks = ceil_div(blocks, 8) * 8;   // xcd_order needs G % 8 == 0
    float4* sink = reinterpret_cast<float4*>(const_cast<float2*>(tw) + C);
    hipLaunchKernelGGL((fft16_kernel<LC, NT, MODE, SM>), dim3((unsigned)blocks), dim3(NT), lds, s,
                       reinterpret_cast<const float4*>(in), out, S, n_items, groups, accumulate, tw, sink);
    return check_launch("channelizer");
}

// fft16_kernel covers the power-of-two rates 256 <= C <= 8192.
static bool use_fft16(int C) { return C >= 256 && C <= 8192 && !(C & (C - 1)); }

template <int LC, int MODE>
static int launch_fft16_lc(const float2* in, void* out, uint64_t S, uint64_t n_items, int groups, int accumulate,
                           const float2* tw, hipStream_t s) {
    // Nontemporal stores pay off only where the stores are whole lines: one
    // spectrum per (antenna, channel), or several staged through LDS when a
    // workgroup holds whole runs of at least four of them (S a multiple of
    // its SPW spectra, so each row of the staged tile is 64 contiguous
    // bytes); with two per row the LDS round trip costs more than the 32-byte
    // pieces save, and interleaved partial lines with nontemporal stores are
    // much slower than plain stores.
    if constexpr (MODE == 0) {
        constexpr uint64_t SPW = 512 / ((1 << LC) / 16);
        if (S == 1) return launch_fft16_t<LC, 512, MODE, 1>(in, out, S, n_items, groups, accumulate, tw, s);
        if constexpr (SPW >= 4) {
            if (S % SPW == 0) return launch_fft16_t<LC, 512, MODE, 2>(in, out, S, n_items, groups, accumulate, tw, s);
        }
    }
    // Detector, C up to 2048: two workgroups of 256 threads per CU overlap each
    // other's loads and passes.  [8,192,8192,2], 4 pols, against one of 512:
    // C = 256 56 / 60 us, 512 60 / 69, 1024 72 / 90; Stokes I 512 55 / 57,
    // 1024 51 / 57, but 256 53 / 47 and C = 4096 109 / 103 (178 / 155 with 4
    // pols), which keep 512.
    // At C = 8192, Stokes I and one integration per channel: the same items through
    // SM 3, whose flush inside the spectrum loop compiles to a loop 2-5% faster
    // ([8,192,4 C,2] 206 against 212 us, [1,40,8 C,2] 55.5 against 58.4).  With 4
    // polarizations it is 2-3% slower, with several integrations per channel, which
    // it would walk one after the other, up to 20% ([1,300,6 C,2], two spectra each,
    // 107 against 86 us).
    if constexpr (MODE == 1 && LC == 13) {
        if (groups == 1) return launch_fft16_t<LC, 512, MODE, 3>(in, out, S, n_items, (int)S, accumulate, tw, s);
    }
    if constexpr ((MODE == 4 && LC <= 11) || (MODE == 1 && LC >= 9 && LC <= 11))
        return launch_fft16_t<LC, 256, MODE, 0>(in, out, S, n_items, groups, accumulate, tw, s);
    else
        return launch_fft16_t<LC, 512, MODE, 0>(in, out, S, n_items, groups, accumulate, tw, s);
}

// Whether a detector call keeps to fft16_kernel's 32-bit offsets: a lane's
// within its workgroup's items (up to 8192 / C, of S spectra each), and from an item's first output
// (C rows of `groups` integrations).  Spectra have none: items are single
// spectra, outputs are indexed in 64 bits.
static bool fft16_fits(int C, uint64_t S, uint64_t groups, uint64_t out_pols) {
    return (8192 / C + 2) * S * (uint64_t)C < (1ull << 31) && (uint64_t)C * groups * out_pols < (1ull << 32);
}

// Launches fft16_kernel for a rate that use_fft16 admits.
template <int MODE>
static int launch_fft16(int C, const float2* in, void* out, uint64_t S, uint64_t n_items, int groups, int accumulate,
                        const float2* tw, hipStream_t s) {
    switch (C) {
        case 1 << 8: return launch_fft16_lc<8, MODE>(in, out, S, n_items, groups, accumulate, tw, s);
        case 1 << 9: return launch_fft16_lc<9, MODE>(in, out, S, n_items, groups, accumulate, tw, s);
        case 1 << 10: return launch_fft16_lc<10, MODE>(in, out, S, n_items, groups, accumulate, tw, s);
        case 1 << 11: return launch_fft16_lc<11, MODE>(in, out, S, n_items, groups, accumulate, tw, s);
        case 1 << 12: return launch_fft16_lc<12, MODE>(in, out, S, n_items, groups, accumulate, tw, s);
        case 1 << 13: return launch_fft16_lc<13, MODE>(in, out, S, n_items, groups, accumulate, tw, s);
    }
    return fail("channelizer: no radix-16 kernel for this rate");
}

// ---------------------------------------------------------------------------
// Two polarizations at C = 2^14, 2^15 and 2^16: the four-step FFT of
// chan_big_pass1/2 with both passes on registers.  A pass transforms columns
// of N = 128 or 256 points: a thread holds 16 points of both polarizations,
// loaded straight from memory (all 16 loads in flight), takes a radix-16
// butterfly, exchanges with its column through LDS one polarization at a time
// (half the LDS: 4 workgroups per CU hide each other's loads), and finishes
// with a radix-8 or 16 butterfly.  COLS = 16 or 32 neighbouring columns per
// workgroup make every global access a run of 256 or 512 bytes.  Pass 1's
// last butterfly is dealt to lanes along k2 instead of along the columns, so
// that its stores into the scratch rows [n1][k2] are runs too.
// LDS columns are N + N/16 + 2 float2 apart (18 or 10 mod 32): columns land on
// even banks and neighbouring butterflies on odd ones.
// Both passes stream at 5-6 TB/s.  Input and output bypass the caches
// (nontemporal) and the spectra go through the passes in groups of 192 MiB of
// scratch, part of which the 256 MB last-level cache then holds between the
// passes: 376 us on [3,192,65536,2] at C = 65536 (1.2 GB in and out), against
// 398 in one group, 456 with plain accesses, 400 at 128 and 454 at 64 MiB
// (too few workgroups per launch), and 1459 with the runtime-radix passes of
// chan_big_pass1/2.
// ---------------------------------------------------------------------------
template <int LN>
struct FourStep {
    static constexpr int N = 1 << LN;
    static constexpr int TPC = N / 16;                 // threads per column
    static constexpr int COLS = 256 / TPC;             // columns per workgroup of 256
    static constexpr int CS = N + N / 16 + 2;          // LDS column stride, float2
    static constexpr int R2 = N / 16;                  // radix of the second butterfly
    static constexpr int G2 = 16 / R2;                 // second butterflies per thread
    static constexpr size_t LDS = sizeof(float2) * ((size_t)COLS * CS + N);
};

// Columns of N points, points `stride` float4s apart.  FIRST: in = spectra
// [n_spec][C], out = scratch [n_spec][N1][N2], times W_C^(n1 k2) (twm).
// Second: in = scratch, out = fftshifted bins at [af, k2 + N2 k1, s].
template <int LN, bool FIRST, bool NTS>
__global__ __launch_bounds__(256, 4) void four_step_kernel(const float4* __restrict__ in, float4* __restrict__ out,
                                                           int other, uint64_t sp0, uint64_t S,
                                                           const float2* __restrict__ tw,
                                                           const float2* __restrict__ twm) {
    typedef FourStep<LN> K;
    constexpr int N = K::N, TPC = K::TPC, COLS = K::COLS;
    extern __shared__ float2 lds[];
    float2* const twl = lds + COLS * K::CS;
    // blockIdx.x = (spectrum of this group, tile of columns); `other` = the
    // length of the other pass = columns per spectrum.
    const unsigned tiles = (unsigned)other / COLS;
    const unsigned b = (gridDim.x & 7u) ? blockIdx.x : xcd_order(blockIdx.x, gridDim.x);
    // Second pass: neighbouring workgroups take the same tile of neighbouring
    // spectra of one (antenna, channel), whose bins interleave at S.
    const unsigned Su = (unsigned)S;
    unsigned sp, tile;
    if (FIRST || Su == 1) {
        sp = b / tiles;
        tile = b - sp * tiles;
    } else {
        const unsigned af = b / (tiles * Su), r = b - af * (tiles * Su);
        tile = r / Su;
        sp = af * Su + (r - tile * Su);
    }
    const unsigned c0 = tile * COLS;
    const size_t C = (size_t)N * other;
    for (int e = threadIdx.x; e < N; e += 256) twl[e] = tw[e];

    const int c = threadIdx.x % COLS, j = threadIdx.x / COLS;
    float2 v[2][16];
    {
        const float4* const src = in + (FIRST ? sp0 + sp : sp) * C + c0 + c;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const float* const q = reinterpret_cast<const float*>(src + (unsigned)((j + r * TPC) * other));
            v[0][r] = make_float2(__builtin_nontemporal_load(q), __builtin_nontemporal_load(q + 1));
            v[1][r] = make_float2(__builtin_nontemporal_load(q + 2), __builtin_nontemporal_load(q + 3));
        }
    }
    // Second butterflies: column c2, butterflies j2 + g TPC.
    const int c2 = FIRST ? threadIdx.x / TPC : c;
    const int j2 = FIRST ? threadIdx.x % TPC : j;
    float2* const wr = lds + c * K::CS + j * 17;
    const float2* const rd = lds + c2 * K::CS + j2;
#pragma unroll
    for (int p = 0; p < 2; p++) {
        dft16(v[p]);
        if (p) __syncthreads();            // polarization 0 has been read
#pragma unroll
        for (int r = 0; r < 16; r++) wr[r] = v[p][r];
        __syncthreads();
#pragma unroll
        for (int g = 0; g < K::G2; g++) {
            float2 x[K::R2];
#pragma unroll
            for (int r = 0; r < K::R2; r++) {
                x[r] = rd[g * TPC + 17 * r];
                if (r > 0) x[r] = cmul(x[r], twl[(j2 + g * TPC) * r]);
            }
            dft_pow2<K::R2>(x);
#pragma unroll
            for (int r = 0; r < K::R2; r++) v[p][g * K::R2 + r] = x[r];
        }
    }
    if constexpr (FIRST) {
        const unsigned n1 = c0 + c2;
        float4* const dst = out + (size_t)sp * C + (size_t)n1 * N + j2;
        const float2* const w = twm + (size_t)n1 * N + j2;
#pragma unroll
        for (int g = 0; g < K::G2; g++)
#pragma unroll
            for (int r = 0; r < K::R2; r++) {
                const int k = g * TPC + 16 * r;
                const float2 wk = w[k];
                const float2 X = cmul(v[0][g * K::R2 + r], wk), Y = cmul(v[1][g * K::R2 + r], wk);
                dst[k] = make_float4(X.x, X.y, Y.x, Y.y);
            }
    } else {
        const uint64_t spg = sp0 + sp, af = spg / S, s = spg - af * S;
        float4* const dst = out + (af * C + c0 + c) * S + s;
#pragma unroll
        for (int g = 0; g < K::G2; g++)
#pragma unroll
            for (int r = 0; r < K::R2; r++) {
                const unsigned k1 = (unsigned)(j2 + g * TPC + 16 * r) ^ (N / 2);    // fftshift
                const float2 X = v[0][g * K::R2 + r], Y = v[1][g * K::R2 + r];
                float4* const o = dst + (size_t)(k1 * other) * S;
                if constexpr (NTS) {
                    float* const of = reinterpret_cast<float*>(o);
                    __builtin_nontemporal_store(X.x, of);
                    __builtin_nontemporal_store(X.y, of + 1);
                    __builtin_nontemporal_store(Y.x, of + 2);
                    __builtin_nontemporal_store(Y.y, of + 3);
                } else {
                    *o = make_float4(X.x, X.y, Y.x, Y.y);
                }
            }
    }
}

constexpr size_t kFourStepScratch = 192ull << 20;

static bool use_four_step(int C, int P) { return P == 2 && (C == 1 << 14 || C == 1 << 15 || C == 1 << 16); }

// C = N1 N2 = 2^ln1 2^ln2.
static void four_step_lengths(int C, int* ln1, int* ln2) {
    *ln2 = C == 1 << 14 ? 7 : 8;
    *ln1 = C == 1 << 16 ? 8 : 7;
}

static int launch_four_step(int C, const float2* in, float2* out, uint64_t S, uint64_t n_spec, hipStream_t s) {
    int ln1, ln2;
    four_step_lengths(C, &ln1, &ln2);
    int N1 = 1 << ln1, N2 = 1 << ln2;
    const float2 *twm = nullptr, *tw1 = nullptr, *tw2 = nullptr;
    int rc = get_twiddles(C, &twm, N2);
    if (!rc) rc = get_twiddles(N1, &tw1);
    if (!rc) rc = get_twiddles(N2, &tw2);
    if (rc) return rc;
    // Spectra per group.  In place, a group's output must not reach input that
    // is still to be read: whole (antenna, channel)s when input and output are
    // the same, everything at once when they overlap otherwise.  Groups are
    // whole (antenna, channel)s where bins of several spectra interleave.
    const size_t bytes = sizeof(float4) * (size_t)C;
    const char* pi = reinterpret_cast<const char*>(in);
    const char* po = reinterpret_cast<const char*>(out);
    const bool overlap = pi < po + bytes * n_spec && po < pi + bytes * n_spec;
    uint64_t group = std::max<uint64_t>(S, kFourStepScratch / bytes / S * S);
    if (overlap && pi != po) group = n_spec;
    group = std::min<uint64_t>(group, n_spec);
    unsigned char* scratch = nullptr;
    rc = library_workspace(WS_CHANNELIZER_BIG, bytes * group, s, &scratch);
    if (rc) return rc;
    float4* y = reinterpret_cast<float4*>(scratch);
    const float4* in4 = reinterpret_cast<const float4*>(in);
    float4* out4 = reinterpret_cast<float4*>(out);
#define FS_FN(...) reinterpret_cast<const void*>(&four_step_kernel<__VA_ARGS__>)
    const void* first = ln2 == 8 ? FS_FN(8, true, false) : FS_FN(7, true, false);
    const void* second = S == 1 ? (ln1 == 8 ? FS_FN(8, false, true) : FS_FN(7, false, true))
                                : (ln1 == 8 ? FS_FN(8, false, false) : FS_FN(7, false, false));
#undef FS_FN
    for (uint64_t sp = 0; sp < n_spec; sp += group) {
        const uint64_t n = std::min<uint64_t>(group, n_spec - sp);
        const dim3 g1((unsigned)(n * N1 / (ln2 == 8 ? FourStep<8>::COLS : FourStep<7>::COLS)));
        const dim3 g2((unsigned)(n * N2 / (ln1 == 8 ? FourStep<8>::COLS : FourStep<7>::COLS)));
        void* args1[] = {&in4, &y, &N1, &sp, &S, &tw2, &twm};
        void* args2[] = {&y, &out4, &N2, &sp, &S, &tw1, &twm};
        (void)hipLaunchKernel(first, g1, dim3(256), args1, ln2 == 8 ? FourStep<8>::LDS : FourStep<7>::LDS, s);
        (void)hipLaunchKernel(second, g2, dim3(256), args2, ln1 == 8 ? FourStep<8>::LDS : FourStep<7>::LDS, s);
    }
    return check_launch("channelizer");
}

// Direct O(C^2) DFT for rates with prime factors above 7.
template <int P>
__global__ __launch_bounds__(256) void chan_direct_kernel(const float2* __restrict__ in,
                                                          float2* __restrict__ out, int C,
                                                          uint64_t S, uint64_t n_spec,
                                                          const float2* __restrict__ tw) {
    extern __shared__ float2 data[];
    for (uint64_t sp = blockIdx.x; sp < n_spec; sp += gridDim.x) {
        const uint64_t af = sp / S, s = sp - af * S;
        const float2* src = in + sp * (uint64_t)C * P;
        for (int i = threadIdx.x; i < C * P; i += blockDim.x) {
            const int n = i / P, p = i - n * P;
            data[p * C + n] = src[i];
        }
        __syncthreads();
        const int half = C / 2;
        for (int i = threadIdx.x; i < C * P; i += blockDim.x) {
            const int k = i / P, p = i - k * P;
            float2 acc = make_float2(0.f, 0.f);
            int m = 0;
            for (int n = 0; n < C; n++) {
                const float2 x = data[p * C + n], w = tw[m];
                acc.x += x.x * w.x - x.y * w.y;
                acc.y += x.x * w.y + x.y * w.x;
                m += k;
                if (m >= C) m -= C;
            }
            int ko = k + half;
            if (ko >= C) ko -= C;
            out[((af * C + ko) * S + s) * P + p] = acc;
        }
        __syncthreads();
    }
}

static bool factorize(int C, Radices* rad) {
    rad->n = 0;
    int c = C;
    // Prefer radix 8, then 4, then one radix 2; then 3, 5, 7.
    while (c % 8 == 0 && rad->n < 16) { rad->r[rad->n++] = 8; c /= 8; }
    while (c % 4 == 0 && rad->n < 16) { rad->r[rad->n++] = 4; c /= 4; }
    while (c % 2 == 0 && rad->n < 16) { rad->r[rad->n++] = 2; c /= 2; }
    while (c % 3 == 0 && rad->n < 16) { rad->r[rad->n++] = 3; c /= 3; }
    while (c % 5 == 0 && rad->n < 16) { rad->r[rad->n++] = 5; c /= 5; }
    while (c % 7 == 0 && rad->n < 16) { rad->r[rad->n++] = 7; c /= 7; }
    return c == 1;
}

// Split C = N1 * N2 for the two-pass FFT: N2 near sqrt(C), N1 even, each
// tile of the passes within 16384 samples of LDS (with the padding sample);
// tiles of up to 16 consecutive columns that divide the other length.
struct BigPlan {
    int N1, N2, cols1, cols2;
    Radices r1, r2;
};

constexpr int kMaxBigRate = 1 << 20;     // the pass-1 twiddle table: 8 MiB

static int big_cols(int n_other, int P, int len) {
    int cols = 64;
    while (cols > 1 && (P * cols * (len + 1) > kMaxLdsComplex || n_other % cols)) cols /= 2;
    return P * cols * (len + 1) <= kMaxLdsComplex ? cols : 0;
}

static bool big_plan(int C, int P, BigPlan* pl) {
    if (C > kMaxBigRate || C % 2) return false;
    double best = 1e30;
    bool found = false;
    for (int n2 = 2; n2 < C; n2++) {
        if (C % n2) continue;
        const int n1 = C / n2;
        if (n1 % 2) continue;
        const int c1 = big_cols(n1, P, n2), c2 = big_cols(n2, P, n1);
        if (!c1 || !c2) continue;
        BigPlan t;
        if (!factorize(n1, &t.r1) || !factorize(n2, &t.r2)) continue;
        const double score = std::fabs(std::log((double)n2) - 0.5 * std::log((double)C)) - 0.01 * (c1 + c2);
        if (score < best) {
            best = score;
            t.N1 = n1; t.N2 = n2; t.cols1 = c1; t.cols2 = c2;
            *pl = t;
            found = true;
        }
    }
    return found;
}

template <int P>
static int launch_big(const BigPlan& pl, int C, const float2* in, float2* out, uint64_t S, uint64_t n_spec,
                      hipStream_t s) {
    const float2 *twC = nullptr, *tw1 = nullptr, *tw2 = nullptr;
    int rc = get_twiddles(C, &twC);
    if (!rc) rc = get_twiddles(pl.N1, &tw1);
    if (!rc) rc = get_twiddles(pl.N2, &tw2);
    if (rc) return rc;
    unsigned char* scratch = nullptr;
    rc = library_workspace(WS_CHANNELIZER_BIG, sizeof(float2) * (size_t)n_spec * C * P, s, &scratch);
    if (rc) return rc;
    float2* y = reinterpret_cast<float2*>(scratch);
    const size_t lds1 = sizeof(float2) * (size_t)P * pl.cols1 * (pl.N2 + 1);
    const size_t lds2 = sizeof(float2) * (size_t)P * pl.cols2 * (pl.N1 + 1);
    const void* f1 = reinterpret_cast<const void*>(&chan_big_pass1<P>);
    const void* f2 = reinterpret_cast<const void*>(&chan_big_pass2<P>);
    if (hipFuncSetAttribute(f1, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds1) != hipSuccess ||
        hipFuncSetAttribute(f2, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds2) != hipSuccess)
        return fail("channelizer: LDS attribute of the two-pass FFT");
    const uint64_t t1 = n_spec * (uint64_t)(pl.N1 / pl.cols1), t2 = n_spec * (uint64_t)(pl.N2 / pl.cols2);
    const unsigned g1 = (unsigned)std::min<uint64_t>(t1, 256 * 64), g2 = (unsigned)std::min<uint64_t>(t2, 256 * 64);
    hipLaunchKernelGGL((chan_big_pass1<P>), dim3(g1), dim3(1024), lds1, s, in, y, C, pl.N1, pl.N2, pl.cols1,
                       n_spec, tw2, twC, pl.r2);
    rc = check_launch("channelizer pass 1");
    if (rc) return rc;
    hipLaunchKernelGGL((chan_big_pass2<P>), dim3(g2), dim3(1024), lds2, s, y, out, C, pl.N1, pl.N2, pl.cols2,
                       n_spec, S, tw1, pl.r1);
    return check_launch("channelizer pass 2");
}

template <int C, int P>
static void launch_small(const float2* in, float2* out, uint64_t n_spec, uint64_t S, hipStream_t s) {
    SmallTw<C> tw;
    for (int m = 0; m < C; m++) {
        const double a = -2.0 * M_PI * (double)m / (double)C;
        tw.w[m] = make_float2((float)cos(a), (float)sin(a));
    }
    // One workgroup per 256 spectra (a compact front streams faster than a
    // capped grid-stride loop); the loop covers sizes past the cap.
    uint64_t blocks = ceil_div(n_spec, 256);
    if (blocks > 0x7fffffffull / 256) blocks = 0x7fffffffull / 256;
    hipLaunchKernelGGL((chan_small_kernel<C, P>), dim3((unsigned)blocks), dim3(256), 0, s, in, out,
                       n_spec, S, tw);
}

template <int P>
static int dispatch_small(int C, const float2* in, float2* out, uint64_t n_spec, uint64_t S,
                          hipStream_t s) {
    switch (C) {
        case 2: launch_small<2, P>(in, out, n_spec, S, s); return 1;
        case 4: launch_small<4, P>(in, out, n_spec, S, s); return 1;
        case 6: launch_small<6, P>(in, out, n_spec, S, s); return 1;
        case 8: launch_small<8, P>(in, out, n_spec, S, s); return 1;
        case 10: launch_small<10, P>(in, out, n_spec, S, s); return 1;
        case 12: launch_small<12, P>(in, out, n_spec, S, s); return 1;
        case 14: launch_small<14, P>(in, out, n_spec, S, s); return 1;
        case 16: launch_small<16, P>(in, out, n_spec, S, s); return 1;
    }
    return 0;
}

}  // namespace bl

using namespace bl;

extern "C" int blade_channelizer(const void* input, void* output, uint64_t A, uint64_t F,
                                 uint64_t T, uint64_t P, uint64_t rate, blade_stream_t stream) {
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    // Validation mirrors src/modules/channelizer/base.cc:17-42 except that any
    // rate dividing T is accepted (the oracle's general semantics).
    if (rate == 0 || T % rate) return fail("channelizer: the number of time samples should be divisible by the channelizer rate");
    if (rate % 2 && rate != 1) return fail("channelizer: the channelizer rate should be divisible by 2");
    if (P != 1 && P != 2) return fail("channelizer: number of polarizations of the input should be one or two");
    const uint64_t n = A * F * T * P;
    if (n == 0) return BLADE_SUCCESS;
    if (!input || !output) return fail("channelizer: null pointer");
    if ((uintptr_t)input % 16 || (uintptr_t)output % 16) return fail("channelizer: misaligned buffer");
    const int C = (int)rate;
    const uint64_t S = T / rate;
    const uint64_t n_spec = A * F * S;
    if (C == 1) {
        if (input == output) return BLADE_SUCCESS;
        hipError_t e = hipMemcpyAsync(output, input, n * 8, hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) {
            set_error(std::string("channelizer copy: ") + hipGetErrorString(e));
            return BLADE_HIP_ERROR;
        }
        return BLADE_SUCCESS;
    }
    const float2* in = static_cast<const float2*>(input);
    float2* out = static_cast<float2*>(output);
    const float2* tw = nullptr;
    if ((uint64_t)C * P > (uint64_t)kMaxLdsComplex) {
        // Past one workgroup's LDS: two passes through a scratch buffer (which
        // also makes any in-place call safe).
        if (use_four_step(C, (int)P)) {
            const int rc = rate_twiddles(C, &tw);     // one polarization's, at 2^14
            return rc ? rc : launch_four_step(C, in, out, S, n_spec, s);
        }
        BigPlan pl;
        if (!big_plan(C, (int)P, &pl))
            return fail("channelizer: rate must be even, at most 2^20, and factor into 2, 3, 5 and 7");
        return P == 2 ? launch_big<2>(pl, C, in, out, S, n_spec, s) : launch_big<1>(pl, C, in, out, S, n_spec, s);
    }
    if (input == output && S != 1)
        return fail("channelizer: in-place operation needs rate == number of time samples");
    if (C <= 16 && input != output) {
        const int ok = (P == 2) ? dispatch_small<2>(C, in, out, n_spec, S, s)
                                : dispatch_small<1>(C, in, out, n_spec, S, s);
        if (ok) return check_launch("channelizer");
    }
    int rc = BLADE_SUCCESS;
    bool made = false;
    // Mixed-radix kernel: every rate made of 2, 3, 5 and 7 but the powers of two
    // of the radix-16 kernel, and of these C = 4096 where several spectra
    // interleave: its stores write runs of them ([8,.,4 C,2]: 123 us against
    // 156 us at S = 4, 102 against 108 at S = 2; 512 to 2048 are staged there
    // and 10-30% faster, 8192 106 against 129 us).
    // The radix-16 kernel keeps one workgroup of two such spectra on a CU.  Where it
    // needs little more than one round, the mixed-radix kernel's spread of spectra
    // over the chip is worse: 520 to 800 spectra on 256 CUs 1 to 16% in its favour at
    // S = 2 to 8 (800 of S = 4 36.2 against 38.8 us, buffers in turn); up to one round
    // (480 of S = 2: 21.3 against 17.6) and from 1.75 on (896 of S = 4: 47.4 against
    // 42.8) the runs win.
    const uint64_t cus = C == 4096 ? (uint64_t)device_cus() : 0;
    const bool runs4096 = C == 4096 && S > 1 && (n_spec <= 2 * cus || 4 * n_spec > 13 * cus);
    if (P == 2 && (!use_fft16(C) || runs4096) && mixed_fft_covers(rate)) {
        rc = mixed_fft(C, in, out, S, n_spec, s, &made);
        return !rc && made ? get_twiddles(C, &tw) : rc;
    }
    rc = rate_twiddles(C, &tw);
    if (rc) return rc;
    if (P == 2 && use_fft16(C)) return launch_fft16<0>(C, in, out, S, n_spec, 1, 0, tw, s);
    Radices rad;
    const size_t lds = sizeof(float2) * (size_t)C * P;
    uint64_t blocks = n_spec;
    if (blocks > 256 * 64) blocks = 256 * 64;
    const void* fn = nullptr;
    int threads = 256;
    if (factorize(C, &rad)) {
        threads = 64;
        while (threads < 1024 && threads * 8 < C * (int)P) threads *= 2;
        fn = (P == 2) ? reinterpret_cast<const void*>(&chan_lds_kernel<2>)
                      : reinterpret_cast<const void*>(&chan_lds_kernel<1>);
    } else {
        fn = (P == 2) ? reinterpret_cast<const void*>(&chan_direct_kernel<2>)
                      : reinterpret_cast<const void*>(&chan_direct_kernel<1>);
    }
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            set_error(std::string("channelizer: LDS attribute: ") + hipGetErrorString(e));
            return BLADE_HIP_ERROR;
        }
    }
    if (fn == reinterpret_cast<const void*>(&chan_lds_kernel<2>))
        hipLaunchKernelGGL((chan_lds_kernel<2>), dim3((unsigned)blocks), dim3(threads), lds, s,
                           in, out, C, S, n_spec, tw, rad);
    else if (fn == reinterpret_cast<const void*>(&chan_lds_kernel<1>))
        hipLaunchKernelGGL((chan_lds_kernel<1>), dim3((unsigned)blocks), dim3(threads), lds, s,
                           in, out, C, S, n_spec, tw, rad);
    else if (P == 2)
        hipLaunchKernelGGL((chan_direct_kernel<2>), dim3((unsigned)blocks), dim3(256), lds, s,
                           in, out, C, S, n_spec, tw);
    else
        hipLaunchKernelGGL((chan_direct_kernel<1>), dim3((unsigned)blocks), dim3(256), lds, s,
                           in, out, C, S, n_spec, tw);
    return check_launch("channelizer");
}

extern "C" int blade_channelizer_plan(uint64_t rate, blade_stream_t stream) {
    if (rate == 0 || (rate % 2 && rate != 1)) return fail("channelizer: invalid rate");
    if (rate > (uint64_t)kMaxBigRate) return fail("channelizer: rate above 2^20 is not supported");
    (void)stream;                           // the tables are filled on a stream of their own
    // Rates up to 16 too: only the channelizer's register kernels (out of place)
    // carry their twiddles as arguments.
    const float2* tw = nullptr;
    int rc = rate_twiddles((int)rate, &tw);
    if (rc) return rc;
    if (use_four_step((int)rate, 2)) {
        int ln1, ln2;
        four_step_lengths((int)rate, &ln1, &ln2);
        rc = get_twiddles((int)rate, &tw, 1 << ln2);
        if (!rc) rc = get_twiddles(1 << ln1, &tw);
        if (!rc) rc = get_twiddles(1 << ln2, &tw);
        if (rc) return rc;
    }
    BigPlan pl;   // the two-pass FFT's tables (for two polarizations)
    if (rate * 2 > (uint64_t)kMaxLdsComplex && big_plan((int)rate, 2, &pl)) {
        rc = get_twiddles(pl.N1, &tw);
        if (!rc) rc = get_twiddles(pl.N2, &tw);
    }
    return rc;
}

extern "C" int blade_channelizer_detector(const void* input, void* output, uint64_t A, uint64_t F,
                                          uint64_t T, uint64_t rate, uint64_t integration,
                                          uint64_t out_pols, int polarize, int accumulate,
                                          blade_stream_t stream) {
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (rate == 0 || T % rate) return fail("channelizer-detector: T must be divisible by the rate");
    if (rate % 2 && rate != 1) return fail("channelizer-detector: the rate should be divisible by 2");
    if (out_pols != 1 && out_pols != 4) return fail("channelizer-detector: output polarizations must be 1 or 4");
    const uint64_t S = T / rate;
    if (integration == 0) return fail("channelizer-detector: integration size should be more than zero");
    if (2 * rate > (uint64_t)kMaxLdsComplex) return fail("channelizer-detector: rate above 8192 is not supported");
    if (A * F * T == 0) return BLADE_SUCCESS;     // before S is used as a divisor
    if (integration <= S ? (S % integration != 0) : (integration % S != 0))
        return fail("channelizer-detector: integration must divide, or be a multiple of, the spectra per block");
    if (!input || !output) return fail("channelizer-detector: null pointer");
    if ((uintptr_t)input % 16 || (uintptr_t)output % 16) return fail("channelizer-detector: misaligned buffer");
    const int C = (int)rate;
    // bit 0: add into the output (stepped integration); bit 1: XY -> LR first
    const int flags = (accumulate ? 1 : 0) | (polarize ? 2 : 0);
    // An item is one integration: Sg spectra in a row of one (antenna, channel)
    // (all S of the block when the integration spans blocks), whose sums stay
    // in one thread's registers.  Every (antenna, channel) gives `groups`; only
    // the kernels behind `small` may count them in an int.
    const uint64_t Sg = std::min(integration, S);
    const uint64_t groups = S / Sg;
    const uint64_t n_items = A * F * groups;
    Radices rad;
    if (!factorize(C, &rad)) return fail("channelizer-detector: rate must factor into 2, 3, 5 and 7");
    const float2* tw = nullptr;
    int rc = BLADE_SUCCESS;
    bool made = false;
    // Mixed-radix kernel: as for the channelizer, and full Stokes at 2048 and
    // 4096 with several integrations per channel, whose 16-byte outputs it writes
    // in runs (one spectrum each: 117 against 151 and 136 against 190 us for
    // 200 MB; Stokes I 95 against 82 and 109 against 71 us the other way).
    const bool small = n_items < (1ull << 31);      // these kernels count items in 32 bits
    const bool runs = out_pols == 4 && groups > 1 && (C == 2048 || C == 4096);
    const bool fft16 = small && use_fft16(C) && fft16_fits(C, Sg, groups, out_pols);
    if (small && Sg < (1ull << 31) && (!fft16 || runs) && mixed_fft_covers(rate) &&
        mixed_fft_detect(C, static_cast<const float2*>(input), static_cast<float*>(output), Sg, (int)groups, n_items,
                         (int)out_pols, flags, s, &rc, &made))
        return !rc && made ? get_twiddles(C, &tw) : rc;
    rc = rate_twiddles(C, &tw);
    if (rc) return rc;
    if (fft16)
        return out_pols == 1 ? launch_fft16<1>(C, static_cast<const float2*>(input), output, Sg, n_items, (int)groups, flags, tw, s)
                             : launch_fft16<4>(C, static_cast<const float2*>(input), output, Sg, n_items, (int)groups, flags, tw, s);
    int threads = 64;
    while (threads < 1024 && threads * 8 < 2 * C) threads *= 2;
    const size_t lds = sizeof(float2) * 2 * (size_t)C;
    uint64_t blocks = n_items;
    if (blocks > 256 * 64) blocks = 256 * 64;
    const void* fn = out_pols == 1 ? reinterpret_cast<const void*>(&chan_detect_kernel<1, 8>)
                                   : reinterpret_cast<const void*>(&chan_detect_kernel<4, 8>);
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            set_error(std::string("channelizer-detector: LDS attribute: ") + hipGetErrorString(e));
            return BLADE_HIP_ERROR;
        }
    }
    const float2* in = static_cast<const float2*>(input);
    float* out = static_cast<float*>(output);
    if (out_pols == 1)
        hipLaunchKernelGGL((chan_detect_kernel<1, 8>), dim3((unsigned)blocks), dim3(threads), lds, s, in, out, C,
                           Sg, groups, n_items, tw, rad, flags);
    else
        hipLaunchKernelGGL((chan_detect_kernel<4, 8>), dim3((unsigned)blocks), dim3(threads), lds, s, in, out, C,
                           Sg, groups, n_items, tw, rad, flags);
    return check_launch("channelizer-detector");
}
