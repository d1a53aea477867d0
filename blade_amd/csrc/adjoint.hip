// Adjoint of the ATA beamformer on CDNA4 matrix cores, and the fused
// Stokes-I calibration gradient.
//
// For y[b,f,t,p] = sum_a w[b,a,f,p] x[a,f,t,p] (the beamformer of
// reference src/modules/beamformer/beamformer.cu:13-79) and an upstream
// gradient gy = dL/dconj(y), the phasor gradient is the contraction over time
//     gw[b,a,f,p] = dL/dconj(w[b,a,f,p]) = sum_t gy[b,f,t,p] conj(x[a,f,t,p]).
// Per (f, p) this is a (B x T)(T x A) product.
//
// Fused Stokes-I mode (stokes_grad_kernel): L = -sum_b lambda_b
// sum_{f,t,p} |y_b|^2, so gy = -lambda_b y_b, which the kernel recomputes from
// the CI8 voltages, read from memory once.  Both contractions run transposed:
//     y^T[t][(b,c)]  = sum_a x^T[t][a] . w^T[a][(b,c)]
//     gw^T[a][(b,c)] = sum_(t,c') x[a][t] . G[(t,c')][(b,c)],
// so the forward accumulator a lane holds (times 4g..4g+3 of column i) is
// exactly the adjoint's B operand for K = those four times: gy never passes
// through LDS.  G's second component block (c' = imaginary part of x) is the
// neighbouring column's value, one lane swap away.  With at most 4 beams the
// FP32 form runs stokes_grad_b4_kernel instead, on 4x4-block matrix
// instructions whose columns are exactly the beams.
//
// Plain adjoint (adjoint_kernel): gy from memory.
//
// Work split: blockIdx = (time split, f, beam tile of 8).  Partial gradients
// are summed across waves in LDS and across time splits by
// adjoint_reduce_kernel, in a fixed order (deterministic, no global atomics).
#include "common.hh"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace bl {

constexpr int ADJ_TC = 128;        // adjoint_kernel: time samples per step of a workgroup, 32 per wave
constexpr int ADJ_WAVES = 4;
constexpr int ADJ_MAXAT = 8;       // antenna tiles of 16: A <= 128
constexpr int ADJ_MAXB = 64;       // beams of the fused loss
constexpr int SG_BATCH = 8;        // stokes_grad_kernel: phasor loads in flight per thread
constexpr int SG_TC = 64;          // stokes_grad_kernel: time samples per tile, 16 per wave
constexpr int SG_XPAD = 4;         // its LDS voltage row stride is apad + 4 words (see sg_xs)

struct AdjArgs {
    const uint32_t* x;       // [A,F,T] dwords: CI8 (re0, im0, re1, im1)
    const float2* w;         // [B,A,F,1,P] phasors (fused mode)
    const float2* gy;        // [B,F,T,P] upstream gradient (adjoint mode)
    float* partial;          // [nsplit][F][P][btiles][16][apad]
    float* loss_part;        // [nsplit][F][btiles]
    int A, F, T, B;
    int apad, n_at, nsteps;  // padded antennas, antenna tiles, forward K steps
    int tsplit;              // time samples per workgroup (a multiple of ADJ_TC or SG_TC)
    int btiles;
    float lambda[ADJ_MAXB];  // beam weights of the fused loss
};

// The value of lane l ^ 1 (DPP quad permutation [1, 0, 3, 2]).
__device__ __forceinline__ float swap_pairs(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
}

__device__ __forceinline__ floatx4 adj_mfma(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float ci8_component(uint32_t d, int idx) {
    return (float)(int8_t)((d >> (8 * idx)) & 0xFFu);
}

// Eight consecutive times of byte k of a voltage dword as a BF16 operand.
__device__ __forceinline__ uint4 ci8_times_bf16(const uint4& lo, const uint4& hi, int k) {
    auto pr = [k](uint32_t d0, uint32_t d1) {
        return bf16_pair((float)(int8_t)(d0 >> (8 * k)), (float)(int8_t)(d1 >> (8 * k)));
    };
    return make_uint4(pr(lo.x, lo.y), pr(lo.z, lo.w), pr(hi.x, hi.y), pr(hi.z, hi.w));
}

// The workgroup's partial gradient from the waves' real products
// acc[pol][antenna tile][component of x] (rows = antennas, columns =
// (beam, component of gy)): combined, then summed over the four waves in
// order through s_part ([wave][p][col][antenna]).
template <int NAT>
__device__ __forceinline__ void adj_store_partials(const AdjArgs& a, const floatx4 (&acc)[2][NAT][2], float* s_part,
                                                   int sp, int f, int bt) {
    constexpr int APAD = 16 * NAT;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, g = lane >> 4;
    const float sg = (i & 1) ? -1.f : 1.f;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int at = 0; at < NAT; at++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                s_part[((wave * 2 + p) * 16 + i) * APAD + at * 16 + 4 * g + r] =
                    acc[p][at][0][r] + sg * swap_pairs(acc[p][at][1][r]);
    __syncthreads();
    constexpr int NPART = 2 * 16 * APAD;
    float* out = a.partial + ((((size_t)sp * a.F + f) * 2) * a.btiles + bt) * 16 * APAD;
    const size_t pstride = (size_t)a.btiles * 16 * APAD;   // between pols
    for (int e = threadIdx.x; e < NPART; e += 64 * ADJ_WAVES) {
        const float v = ((s_part[e] + s_part[NPART + e]) + s_part[2 * NPART + e]) + s_part[3 * NPART + e];
        const int p = e / (16 * APAD), r = e - p * 16 * APAD;
        out[p * pstride + r] = v;
    }
}

// Plain adjoint of A <= 16 NAT antennas and 8 beams: the real products
//     P[c][co] = sum_t x_c[a][t] gy_co[b][t]   (c, co = re, im)
// with rows = antennas, columns = (beam, co) and K = 32 times per
// instruction, combined at the end: Re gw = P[re][re] + P[im][im],
// Im gw = P[re][im] - P[im][re].  A lane holds antenna row i (lane % 16) and
// column i, times 8g .. 8g + 7 of the wave's 32, so both operands are whole
// 16-byte pieces of memory in their native layout: nothing is staged in LDS
// and the waves run without barriers.  CI8 is exact in BF16 and gy is the
// exact sum of three BF16 parts, so the products are exact and v_mfma_f32_
// 16x16x32_bf16 accumulates them in FP32.  The next 32 times' loads are
// issued into the registers just converted.
// HBM bound: A42 F384 T2048 B4 reads 182 MB (x and gy once); with the sums of
// the splits it took 181 us through LDS tiles and FP32 instructions, 41 us so.
// VEC: 16-byte
// loads (T a multiple of 4, both buffers 16-byte aligned); otherwise single
// dwords and float2.
template <int NAT, bool VEC>
__global__ __launch_bounds__(256, (NAT <= 3 ? 3 : NAT <= 5 ? 2 : 1)) void adjoint_kernel(AdjArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int i = lane & 15;
    const int g = lane >> 4;
    const int sp = blockIdx.x;
    const int f = blockIdx.y;
    const int bt = blockIdx.z;
    const int A = a.A, F = a.F, T = a.T, B = a.B;
    const int t_begin = sp * a.tsplit;
    const int t_end = min(T, t_begin + a.tsplit);
    const bool im = i & 1;
    // Rows past A and columns past B repeat the last one (never stored).
    const float2* const gp = a.gy + ((size_t)min(bt * 8 + (i >> 1), B - 1) * F + f) * T * 2;

    uint4 xq[NAT][2];      // [antenna tile][times 0-3, 4-7 of the lane's 8]
    float4 gq[8];          // one time each: (X re, X im, Y re, Y im)
    auto load_x = [&](int t0, int at) {
        const uint32_t* const xp = a.x + ((size_t)min(at * 16 + i, A - 1) * F + f) * T;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int t = t0 + 8 * g + 4 * h;
            if constexpr (VEC) {
                xq[at][h] = *reinterpret_cast<const uint4*>(xp + min(t, t_end - 4));
            } else {
                xq[at][h] = make_uint4(xp[min(t, t_end - 1)], xp[min(t + 1, t_end - 1)], xp[min(t + 2, t_end - 1)],
                                       xp[min(t + 3, t_end - 1)]);
            }
        }
    };
    auto load_g = [&](int t0) {
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int t = min(t0 + 8 * g + q, t_end - 1);
            if constexpr (VEC) {
                gq[q] = *reinterpret_cast<const float4*>(gp + 2 * t);
            } else {
                const float2 u = gp[2 * t], v = gp[2 * t + 1];
                gq[q] = make_float4(u.x, u.y, v.x, v.y);
            }
        }
    };

    floatx4 acc[2][NAT][2];    // [pol][antenna tile][component of x]
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int at = 0; at < NAT; at++)
#pragma unroll
            for (int c = 0; c < 2; c++) acc[p][at][c] = floatx4{0.f, 0.f, 0.f, 0.f};

    int t0 = t_begin + wave * 32;
    if (t0 < t_end) {          // otherwise there is nothing to read (T = 0 included)
        load_g(t0);
#pragma unroll
        for (int at = 0; at < NAT; at++) load_x(t0, at);
    }
    for (; t0 < t_end; t0 += ADJ_TC) {
        // gy of this lane's component, times past the split zeroed, in parts
        uint4 gb[2][3];
        {
            uint32_t w[2][3][4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const bool ok0 = t0 + 8 * g + 2 * q < t_end, ok1 = t0 + 8 * g + 2 * q + 1 < t_end;
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const float4 u = gq[2 * q], v = gq[2 * q + 1];
                    const float u0 = im ? (p ? u.w : u.y) : (p ? u.z : u.x);
                    const float v0 = im ? (p ? v.w : v.y) : (p ? v.z : v.x);
                    float pu[3], pv[3];
                    split_bf16x3(ok0 ? u0 : 0.f, pu);
                    split_bf16x3(ok1 ? v0 : 0.f, pv);
#pragma unroll
                    for (int k = 0; k < 3; k++) w[p][k][q] = bf16_pair(pu[k], pv[k]);
                }
            }
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int k = 0; k < 3; k++) gb[p][k] = make_uint4(w[p][k][0], w[p][k][1], w[p][k][2], w[p][k][3]);
        }
        const int tn = min(t0 + ADJ_TC, t_end - 1);     // past the split: re-read its end
        load_g(tn);
#pragma unroll
        for (int at = 0; at < NAT; at++) {
            uint4 xo[2][2];
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int c = 0; c < 2; c++) xo[p][c] = ci8_times_bf16(xq[at][0], xq[at][1], 2 * p + c);
            load_x(tn, at);
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int c = 0; c < 2; c++) acc[p][at][c] = mfma_bf16(xo[p][c], gb[p][k], acc[p][at][c]);
        }
    }

    adj_store_partials<NAT>(a, acc, reinterpret_cast<float*>(lds_raw), sp, f, bt);
}

// LDS row stride (words) of stokes_grad_kernel's voltage tile s_x[t][antenna]:
// apad + 4 puts both read patterns on distinct banks, the forward's (16 lanes
// read 16 consecutive times of one antenna; lane groups take adjacent
// antennas) and the adjoint's (16 lanes read 16 consecutive antennas at one
// time; lane groups take times 4 apart).
__host__ __device__ constexpr int sg_xs(int apad) { return apad + SG_XPAD; }

// Adjoint of one wave's 16 times (rows trow .. + 15 of the LDS voltage tile)
// and the gy = gy[pol][time 4g + r] its lanes hold: K = 16 times x (re, im) of
// x, which are the lane's own values and, for Im x, the neighbouring column's
// (re <-> im) with the sign of conj(x).  gy as three BF16 parts, CI8 exact:
// exact products, accumulated in FP32 from the smallest part up.  TILE: the 16
// times are summed by themselves, one rounding into the long sum, as the split
// FP16 form always did (error 1.1e-7 at A42 T2048 B16; 1.7e-7 without).  The
// FP32 form's was one chain of 8 instructions, so 3 are below it without.
template <int NAT, int XS, bool TILE>
__device__ __forceinline__ void sg_adjoint(const uint32_t* rows, const float (&gy)[2][4], float swap_sign, int i, int g,
                                           floatx4 (&acc)[2][NAT]) {
    uint4 gb[2][3];
    float mag = 0.f;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int r = 0; r < 4; r++) mag += fabsf(gy[p][r]);
    auto parts = [&](auto checked) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            uint32_t w[3][4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float u[3], v[3];
                split_bf16x3<decltype(checked)::value>(gy[p][r], u);
#pragma unroll
                for (int m = 0; m < 3; m++) {
                    v[m] = swap_sign * swap_pairs(u[m]);
                    w[m][r] = bf16_pair(u[m], v[m]);
                }
            }
#pragma unroll
            for (int m = 0; m < 3; m++) gb[p][m] = make_uint4(w[m][0], w[m][1], w[m][2], w[m][3]);
        }
    };
    // Infinities and NaN (they show in mag) take the split that keeps them.
    if (__all(mag <= 3.0e38f))
        parts(std::false_type{});
    else
        parts(std::true_type{});
#pragma unroll
    for (int at = 0; at < NAT; at++) {
        uint32_t d[4];
#pragma unroll
        for (int q = 0; q < 4; q++) d[q] = rows[(4 * g + q) * XS + at * 16 + i];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const uint4 xo = make_uint4(ci8_to_bf16(d[0], p), ci8_to_bf16(d[1], p), ci8_to_bf16(d[2], p),
                                        ci8_to_bf16(d[3], p));
            floatx4 t = TILE ? floatx4{0.f, 0.f, 0.f, 0.f} : acc[p][at];
#pragma unroll
            for (int m = 2; m >= 0; m--) t = mfma_bf16(xo, gb[p][m], t);
            acc[p][at] = TILE ? acc[p][at] + t : t;
        }
        __builtin_amdgcn_sched_barrier(0);     // one tile's operands live at a time (7 and 8 tiles spilled)
    }
}

// Fused Stokes-I loss and phasor gradient for A <= 16 NAT antennas.  Each
// wave takes 16 time rows of every SG_TC-sample tile; the next tile's
// voltages are loaded into registers while this one is computed and written
// to the other half of a double-buffered LDS stage: one barrier per tile.
// The forward stays on FP32 instructions: the loss is returned in FP64, and
// callers follow its history.  Bound by them (32 cycles per K = 4): A42 F384
// T2048 B16 213 us with an FP32 adjoint of 8 instructions per antenna tile and
// pol, 167 us with sg_adjoint's 3 of half the length.
template <int NAT>
__global__ __launch_bounds__(256, (NAT <= 4 ? 4 : NAT <= 6 ? 3 : 2)) void stokes_grad_kernel(AdjArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int APAD = 16 * NAT;
    constexpr int XS = sg_xs(APAD);
    constexpr int PER = SG_TC * APAD / (64 * ADJ_WAVES);     // staged dwords per thread
    uint32_t* s_x = reinterpret_cast<uint32_t*>(lds_raw);     // [2][SG_TC][XS]
    float* s_w = reinterpret_cast<float*>(s_x + 2 * SG_TC * XS);   // [2][nsteps][64]
    __shared__ float s_loss[ADJ_WAVES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int i = lane & 15;
    const int g = lane >> 4;
    const int sp = blockIdx.x;
    const int f = blockIdx.y;
    const int bt = blockIdx.z;
    const int b0 = bt * 8;
    const int A = a.A, F = a.F, T = a.T, B = a.B;
    const int nsteps = a.nsteps;
    const int n_ag = nsteps / 2;                              // antenna groups of 4
    const int t_begin = sp * a.tsplit;
    const int t_end = min(T, t_begin + a.tsplit);
    const int ntiles = (t_end - t_begin + SG_TC - 1) / SG_TC;

    // Voltage staging: thread (wave, lane) takes antennas wave + 4k at time
    // lane of the tile (one coalesced 256-byte row per wave and k).
    uint32_t pre[PER];
    bool pre_t_ok = true;
    // Unconditional loads from clamped addresses (no branch per antenna row);
    // padded antennas and samples past the split are zeroed when the tile is
    // written to LDS, so the loads stay in flight until then.
    auto load_tile = [&](int t0) {
        const int tt = t0 + lane;
        pre_t_ok = tt < t_end;
        const int ttc = min(tt, t_end - 1);
        // Opaque stride and a uniform wave number: otherwise the PER row
        // addresses are held in registers across tiles.
        size_t st = (size_t)F * T;
        asm volatile("" : "+s"(st));
        const int w0 = __builtin_amdgcn_readfirstlane(wave);
        const uint32_t* const xf = a.x + (size_t)f * T + ttc;
#pragma unroll
        for (int k = 0; k < PER; k++) pre[k] = xf[min(w0 + ADJ_WAVES * k, A - 1) * st];
    };
    auto store_tile = [&](uint32_t* dst) {
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int an = wave + ADJ_WAVES * k;
            dst[lane * XS + an] = (pre_t_ok && an < A) ? pre[k] : 0u;
        }
    };
    load_tile(t_begin);

    // Forward B operand of beams b0..b0+7, both pols: [p][step][g][col],
    // step = 2 * antenna group + component of x, col = (beam, re/im).
    {
        const int n_w = 2 * nsteps * 64;
        for (int e0 = tid; e0 < n_w; e0 += SG_BATCH * ADJ_WAVES * 64) {
            float2 wv[SG_BATCH];
#pragma unroll
            for (int k = 0; k < SG_BATCH; k++) {
                const int e = e0 + k * ADJ_WAVES * 64;
                const int p = e / (nsteps * 64);
                const int r = e - p * nsteps * 64;
                const int st = r >> 6, kg = (r >> 4) & 3, col = r & 15;
                const int an = (st >> 1) * 4 + kg, b = b0 + (col >> 1);
                wv[k] = (e < n_w && b < B && an < A) ? a.w[(((size_t)b * A + an) * F + f) * 2 + p]
                                                      : make_float2(0.f, 0.f);
            }
#pragma unroll
            for (int k = 0; k < SG_BATCH; k++) {
                const int e = e0 + k * ADJ_WAVES * 64;
                if (e < n_w) {
                    const int r = e % (nsteps * 64);
                    const int c = (r >> 6) & 1, co = r & 1;
                    const float2 w = wv[k];
                    // y_r = x_r w_r - x_i w_i, y_i = x_r w_i + x_i w_r
                    s_w[e] = (co == 0) ? (c == 0 ? w.x : -w.y) : (c == 0 ? w.y : w.x);
                }
            }
        }
    }
    store_tile(s_x);
    if (ntiles > 1) load_tile(t_begin + SG_TC);
    __syncthreads();

    const int bcol = b0 + (i >> 1);
    const float lam = bcol < B ? a.lambda[bcol] : 0.f;
    const float swap_sign = (i & 1) ? -1.f : 1.f;
    floatx4 acc2[2][NAT];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int at = 0; at < NAT; at++) acc2[p][at] = floatx4{0.f, 0.f, 0.f, 0.f};
    float loss = 0.f;

    for (int k = 0; k < ntiles; k++) {
        const uint32_t* sx = s_x + (k & 1) * SG_TC * XS;
        const int trow = wave * 16;
        // Forward: y^T rows = this wave's 16 times, both pols from one dword.
        floatx4 y[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int ag = 0; ag < 4 * NAT; ag++) {
            if (ag < n_ag) {                       // uniform
                const uint32_t d = sx[(trow + i) * XS + ag * 4 + g];
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const float w0 = s_w[(p * nsteps + 2 * ag) * 64 + lane];
                    const float w1 = s_w[(p * nsteps + 2 * ag + 1) * 64 + lane];
                    y[p] = adj_mfma(ci8_component(d, 2 * p), w0, y[p]);
                    y[p] = adj_mfma(ci8_component(d, 2 * p + 1), w1, y[p]);
                }
            }
        }
        // Lane (g, i), register r: y at time trow + 4g + r, column i.
        float gy[2][4];
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float v = y[p][r];
                loss += lam * v * v;
                gy[p][r] = -lam * v;
            }
        sg_adjoint<NAT, XS, false>(sx + trow * XS, gy, swap_sign, i, g, acc2);
        if (k + 1 < ntiles) {
            // Tile k + 1 into the other buffer (last read in iteration k - 1,
            // before the barrier that ended it), then tile k + 2's loads.
            store_tile(s_x + ((k + 1) & 1) * SG_TC * XS);
            if (k + 2 < ntiles) load_tile(t_begin + (k + 2) * SG_TC);
        }
        __syncthreads();
    }

    // Partials of the four waves into LDS (the voltage stage is free now),
    // [wave][p][col][antenna], then summed in wave order.
    float* s_part = reinterpret_cast<float*>(lds_raw);
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int at = 0; at < NAT; at++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                s_part[((wave * 2 + p) * 16 + i) * APAD + at * 16 + 4 * g + r] = acc2[p][at][r];
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0) s_loss[wave] = loss;
    __syncthreads();
    constexpr int NPART = 2 * 16 * APAD;
    float* out = a.partial + ((((size_t)sp * F + f) * 2) * a.btiles + bt) * 16 * APAD;
    const size_t pstride = (size_t)a.btiles * 16 * APAD;   // between pols
    for (int e = tid; e < NPART; e += blockDim.x) {
        const float v = ((s_part[e] + s_part[NPART + e]) + s_part[2 * NPART + e]) + s_part[3 * NPART + e];
        const int p = e / (16 * APAD), r = e - p * 16 * APAD;
        out[p * pstride + r] = v;
    }
    if (tid == 0)
        a.loss_part[((size_t)sp * F + f) * a.btiles + bt] = ((s_loss[0] + s_loss[1]) + s_loss[2]) + s_loss[3];
}

// ---------------------------------------------------------------------------
// Stokes-I loss and gradient for at most 4 beams (FP32), on
// v_mfma_f32_4x4x1_16b_f32: 16 independent 4x4 blocks with K = 1.  Lane
// 4 blk + c holds row c of block blk's A operand, column c of its B operand,
// and column c of its result (register r = row r).  With 4 beams the columns
// are exactly the beams, so no matrix work goes to absent beams (the 16x16
// tiles of stokes_grad_kernel are half empty there).  Complex products take
// three real products (P3 - P1 - P2 form).
//   Forward, blocks = groups of 4 times, K = one antenna per instruction:
//     lane (blk, c) feeds x[a][t0 + 4 blk + c] and w[a][beam c]; register r
//     of the result is y at time t0 + 4 blk + r, beam c.
//   Adjoint: gy, cut into three BF16 parts, passes through a per-wave LDS
//     tile into the operand layout of adjoint_kernel, and so does the rest: the
//     voltages as 16-byte pieces of memory (they were just read, so from L2),
//     K = 32 times per instruction.  On 4x4 FP32 blocks as well it took 384
//     instructions of 8 cycles and 96 LDS reads a tile instead of 24 NAT of 16
//     and 12, and a call 95 us instead of 70 us (A42 F384 T2048 B4; A28 77
//     and 49 us).  One pol at a time, and with 4 antenna tiles the voltages
//     after the forward, keep 3 workgroups per CU; A49-64 still spill 72 bytes,
//     with 2 workgroups none (A64 F384 T1024 B2 56 against 68 us, F128 T2048 B4
//     47 against 42 us).
// Each wave takes 64-time tiles; partial sums are added across waves in LDS
// in wave order and across time splits by adjoint_reduce_kernel, whose
// partial layout this kernel writes (rows 2 b and 2 b + 1, beam tile 0).
// Needs A <= 64, T % 4 == 0, A F T < 2^31 and 16-byte aligned voltages.
// ---------------------------------------------------------------------------
constexpr int SG4_TC = 64;            // times per wave tile
constexpr int SG4_WS = 8;             // LDS floats per (antenna, beam): (wr, wi, wr + wi) per pol, padded
// gy tile rows ([p][part][beam][re/im], SG4_TC BF16 times each) are padded by
// 16 bytes, which puts the rows of a read on different banks.
constexpr int SG4_GS = 2 * SG4_TC + 16;      // bytes
constexpr int SG4_GY = 2 * 3 * 8 * SG4_GS;   // bytes of one wave's gy tile
constexpr int SG4_WGS = 3;            // resident workgroups per CU (launch bounds)

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

template <int NAT>
__global__ __launch_bounds__(256, SG4_WGS) void stokes_grad_b4_kernel(AdjArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int AMAX = 16 * NAT;
    float* const s_w = reinterpret_cast<float*>(lds_raw);            // [A][4][SG4_WS]
    unsigned char* const gyw = lds_raw + (size_t)a.A * 4 * SG4_WS * 4 + (threadIdx.x >> 6) * SG4_GY;   // this wave's gy
    __shared__ float s_loss[ADJ_WAVES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int blk = lane >> 2;
    const int c = lane & 3;
    const int sp = blockIdx.x;
    const int f = blockIdx.y;
    const int A = a.A, F = a.F, T = a.T, B = a.B;
    const int t_begin = sp * a.tsplit;
    const int t_end = min(T, t_begin + a.tsplit);
    const int ntiles = (t_end - t_begin + SG4_TC - 1) / SG4_TC;
    const unsigned ant_stride = (unsigned)F * (unsigned)T;   // A F T < 2^31 (host check)

    // Phasors of (antenna, beam): wr, wi, wr + wi of pol 0, then of pol 1.
    for (int e = tid; e < A * 4; e += blockDim.x) {
        const int an = e >> 2, b = e & 3;
        float v[6];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const float2 w = b < B ? a.w[(((size_t)b * A + an) * F + f) * 2 + p] : make_float2(0.f, 0.f);
            v[3 * p] = w.x;
            v[3 * p + 1] = w.y;
            v[3 * p + 2] = w.x + w.y;
        }
        float4* dst = reinterpret_cast<float4*>(s_w + (size_t)e * SG4_WS);
        dst[0] = make_float4(v[0], v[1], v[2], v[3]);
        dst[1] = make_float4(v[4], v[5], 0.f, 0.f);
    }
    __syncthreads();

    const float lam = c < B ? a.lambda[c] : 0.f;
    const int i = lane & 15, g = lane >> 4;                  // adjoint operand row and K group
    floatx4 acc[2][NAT][2];    // [pol][antenna tile][component of x]
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int at = 0; at < NAT; at++)
#pragma unroll
            for (int k = 0; k < 2; k++) acc[p][at][k] = floatx4{0.f, 0.f, 0.f, 0.f};
    float loss = 0.f;

    // Forward voltages of tile kk at this lane's time, antennas 8 g .. 8 g + 7
    // (group g + 1 is in flight while group g is computed: 3% faster than
    // all antennas at once, with 136 instead of 168 VGPRs).  The stride and
    // count are opaque to the compiler, which would otherwise keep one
    // offset and one guard mask per antenna in scalar registers across tiles
    // (and spill them).
    uint32_t xd[2][8];
    auto load_fwd = [&](int kk, int g, uint32_t (&dst)[8]) {
        const int tl = t_begin + kk * SG4_TC + 4 * blk + c;
        const uint32_t* const xf = a.x + (f * T + min(tl, t_end - 1));
        unsigned st = ant_stride;
        int na = A;
        asm volatile("" : "+s"(st), "+s"(na));
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (8 * g + j < na) dst[j] = xf[(8 * g + j) * st];     // uniform
    };
    // Adjoint voltages: times t + 8 g .. + 7 of this lane's row of tile at
    // (antennas past A repeat the last one, never stored; times past the split
    // its end, their gy is 0).
    uint4 xq[NAT][2];
    auto load_adj = [&](int t, int at) {
        unsigned st = ant_stride;
        asm volatile("" : "+s"(st));
        const uint32_t* const xp = a.x + (min(16 * at + i, A - 1) * st + f * T);
#pragma unroll
        for (int h = 0; h < 2; h++) xq[at][h] = *reinterpret_cast<const uint4*>(xp + min(t + 8 * g + 4 * h, t_end - 4));
    };

    for (int k = wave; k < ntiles; k += ADJ_WAVES) {
        const int t0 = t_begin + k * SG4_TC;
        const int tn = min(SG4_TC, t_end - t0);            // a multiple of 4
        // In flight during the forward (4 tiles: after it).
        if constexpr (NAT < 4) {
#pragma unroll
            for (int at = 0; at < NAT; at++) load_adj(t0, at);
        }
        load_fwd(k, 0, xd[0]);
        // ---- forward: this lane feeds time t0 + 4 blk + c (clamped to the
        // split; results for times past it are zeroed below).  The antenna
        // count is opaque here too: 48 hoisted guard masks would not fit in
        // scalar registers.
        int na = A;
        asm volatile("" : "+s"(na));
        floatx4 y[2][3];
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int m = 0; m < 3; m++) y[p][m] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int an = 0; an < AMAX; an++) {
            if (an % 8 == 0 && an + 8 < AMAX) load_fwd(k, an / 8 + 1, xd[(an / 8 + 1) & 1]);
            if (an < na) {                                        // uniform
                const uint32_t d = xd[(an / 8) & 1][an % 8];
                const float* wv = s_w + (an * 4 + c) * SG4_WS;
                const float4 w0 = *reinterpret_cast<const float4*>(wv);
                const float2 w1 = *reinterpret_cast<const float2*>(wv + 4);
                const float wp[2][3] = {{w0.x, w0.y, w0.z}, {w0.w, w1.x, w1.y}};
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const float xr = ci8_component(d, 2 * p), xi = ci8_component(d, 2 * p + 1);
                    y[p][0] = mfma4(xr, wp[p][0], y[p][0]);
                    y[p][1] = mfma4(xi, wp[p][1], y[p][1]);
                    y[p][2] = mfma4(xr + xi, wp[p][2], y[p][2]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (NAT == 4) {
#pragma unroll
            for (int at = 0; at < NAT; at++) load_adj(t0, at);
        }
        // ---- gy = -lambda y at (time t0 + 4 blk + r, beam c), in parts, into
        // this wave's LDS tile.  Times past the split read clamped voltages:
        // their y, and so gy and the loss, are set to 0.
        float gr[2][4], gi[2][4], mag = 0.f;
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const bool ok = 4 * blk + r < tn;
                const float yr = ok ? y[p][0][r] - y[p][1][r] : 0.f;
                const float yi = ok ? (y[p][2][r] - y[p][0][r]) - y[p][1][r] : 0.f;
                loss += lam * (yr * yr + yi * yi);
                gr[p][r] = -lam * yr;
                gi[p][r] = -lam * yi;
                mag += fabsf(gr[p][r]) + fabsf(gi[p][r]);
            }
        auto parts = [&](auto checked) {
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int co = 0; co < 2; co++) {
                    float v[4][3];
#pragma unroll
                    for (int r = 0; r < 4; r++) split_bf16x3<decltype(checked)::value>(co ? gi[p][r] : gr[p][r], v[r]);
#pragma unroll
                    for (int m = 0; m < 3; m++)
                        *reinterpret_cast<uint2*>(gyw + ((p * 3 + m) * 8 + 2 * c + co) * SG4_GS + 8 * blk) =
                            make_uint2(bf16_pair(v[0][m], v[1][m]), bf16_pair(v[2][m], v[3][m]));
                }
        };
        // Infinities and NaN (they show in mag) take the split that keeps them.
        if (__all(mag <= 3.0e38f))
            parts(std::false_type{});
        else
            parts(std::true_type{});
        // ---- adjoint, 32 times at a time.  The wave reads back its own LDS
        // writes (LDS operations of a wave complete in order); columns 8 to 15
        // repeat 0 to 7 and are not used.
#pragma unroll
        for (int h = 0; h < SG4_TC / 32; h++) {
#pragma unroll
            for (int p = 0; p < 2; p++) {
                uint4 gb[3];
#pragma unroll
                for (int m = 0; m < 3; m++)
                    gb[m] = *reinterpret_cast<const uint4*>(gyw + ((p * 3 + m) * 8 + (i & 7)) * SG4_GS + 64 * h + 16 * g);
#pragma unroll
                for (int at = 0; at < NAT; at++) {
                    uint4 xo[2];
#pragma unroll
                    for (int k2 = 0; k2 < 2; k2++) xo[k2] = ci8_times_bf16(xq[at][0], xq[at][1], 2 * p + k2);
                    if (p == 1 && h + 1 < SG4_TC / 32) load_adj(t0 + 32 * (h + 1), at);
#pragma unroll
                    for (int m = 0; m < 3; m++)
#pragma unroll
                        for (int k2 = 0; k2 < 2; k2++) acc[p][at][k2] = mfma_bf16(xo[k2], gb[m], acc[p][at][k2]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0) s_loss[wave] = loss;
    __syncthreads();                          // every wave is done with the LDS operands
    adj_store_partials<NAT>(a, acc, reinterpret_cast<float*>(lds_raw), sp, f, 0);
    if (tid == 0) a.loss_part[(size_t)sp * F + f] = ((s_loss[0] + s_loss[1]) + s_loss[2]) + s_loss[3];
}

// Power-of-two scale s with m * s in [0.5, 1) for m > 0 (1 for m = 0), and 1/s.
__device__ __forceinline__ void pow2_scale(float m, float& s, float& inv) {
    int ex = 0;
    frexpf(m, &ex);
    s = m > 0.f ? ldexpf(1.0f, -ex) : 1.f;
    inv = m > 0.f ? ldexpf(1.0f, ex) : 1.f;
}

// v (|v| < 1) as hi + lo FP16 halves, into element j of two vectors.
__device__ __forceinline__ void split_f16(float v, halfx8& hi, halfx8& lo, int j) {
    const _Float16 h = (_Float16)v;
    hi[j] = h;
    lo[j] = (_Float16)(v - (float)h);
}

// Split-FP16 form of stokes_grad_kernel: the same transposed contractions and
// tiles on v_mfma_f32_16x16x32_f16 (K = 32 per instruction), FP32
// accumulation.  CI8 voltages are exact in FP16.
//   * Forward B operand: the phasor embedding times a power-of-two scale per
//     pol (every component below 1), as hi + lo FP16 halves; K = 16
//     antennas x (re, im) of x per instruction.
//   * Adjoint: sg_adjoint, where gy needs no scale: as hi + lo FP16 halves it
//     took the wave's largest |gy| over 6 lane exchanges per pol and tile.
//     A42 F384 T2048 B4 67 -> 60 us, A28 56 -> 47 us, A16 B8 44 -> 34 us.
// Error against FP64 is that of FP32 arithmetic (hi + lo carry ~22 bits).
template <int NAT>
__global__ __launch_bounds__(256, (NAT <= 3 ? 3 : 2)) void stokes_grad_f16_kernel(AdjArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int APAD = 16 * NAT;
    constexpr int XS = sg_xs(APAD);
    constexpr int PER = SG_TC * APAD / (64 * ADJ_WAVES);
    uint32_t* s_x = reinterpret_cast<uint32_t*>(lds_raw);                 // [2][SG_TC][XS]
    halfx8* s_wh = reinterpret_cast<halfx8*>(s_x + 2 * SG_TC * XS);       // [p][blk][hl][64]
    __shared__ float s_loss[ADJ_WAVES];
    __shared__ unsigned int s_wmax[2];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int i = lane & 15;
    const int g = lane >> 4;
    const int sp = blockIdx.x;
    const int f = blockIdx.y;
    const int bt = blockIdx.z;
    const int b0 = bt * 8;
    const int A = a.A, F = a.F, T = a.T, B = a.B;
    const int t_begin = sp * a.tsplit;
    const int t_end = min(T, t_begin + a.tsplit);
    const int ntiles = (t_end - t_begin + SG_TC - 1) / SG_TC;

    uint32_t pre[PER];
    bool pre_t_ok = true;
    // Unconditional loads from clamped addresses (no branch per antenna row);
    // padded antennas and samples past the split are zeroed when the tile is
    // written to LDS, so the loads stay in flight until then.
    auto load_tile = [&](int t0) {
        const int tt = t0 + lane;
        pre_t_ok = tt < t_end;
        const int ttc = min(tt, t_end - 1);
        size_t st = (size_t)F * T;
        int w0 = wave;
        if constexpr (NAT == ADJ_MAXAT) {
            // Opaque stride, uniform wave number: otherwise the row addresses
            // are held in registers across tiles, which spilled here (A128 F64
            // T2048 B8 80 -> 64 us; with fewer tiles they fit and cost nothing).
            asm volatile("" : "+s"(st));
            w0 = __builtin_amdgcn_readfirstlane(wave);
        }
        const uint32_t* const xf = a.x + (size_t)f * T + ttc;
#pragma unroll
        for (int k = 0; k < PER; k++) pre[k] = xf[min(w0 + ADJ_WAVES * k, A - 1) * st];
    };
    auto store_tile = [&](uint32_t* dst) {
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int an = wave + ADJ_WAVES * k;
            dst[lane * XS + an] = (pre_t_ok && an < A) ? pre[k] : 0u;
        }
    };
    load_tile(t_begin);

    // Phasor scale per pol: the largest component magnitude of this
    // workgroup's beams (an exact maximum, so the order of the atomics does
    // not matter).
    if (tid < 2) s_wmax[tid] = 0u;
    __syncthreads();
    {
        float mx[2] = {0.f, 0.f};
        for (int e = tid; e < 2 * 8 * A; e += blockDim.x) {
            const int p = e / (8 * A), r = e - p * 8 * A;
            const int bb = r / A, an = r - bb * A, b = b0 + bb;
            if (b < B) {
                const float2 w = a.w[(((size_t)b * A + an) * F + f) * 2 + p];
                mx[p] = fmaxf(mx[p], fmaxf(fabsf(w.x), fabsf(w.y)));
            }
        }
        atomicMax(&s_wmax[0], __float_as_uint(mx[0]));
        atomicMax(&s_wmax[1], __float_as_uint(mx[1]));
    }
    __syncthreads();
    float wsc[2], wuns[2];
    pow2_scale(__uint_as_float(s_wmax[0]), wsc[0], wuns[0]);
    pow2_scale(__uint_as_float(s_wmax[1]), wsc[1], wuns[1]);
    // Forward B operand: lane (g, i) of block blk holds k = 8g + 2q + c ->
    // (antenna 16 blk + 4g + q, component c of x), column i -> (beam
    // b0 + i/2, re/im).  y_r = x_r w_r - x_i w_i, y_i = x_r w_i + x_i w_r.
    for (int e = tid; e < 2 * NAT * 64; e += blockDim.x) {
        const int ln = e & 63, pb = e >> 6;
        const int p = pb / NAT, blk = pb - p * NAT;
        const int li = ln & 15, lg = ln >> 4;
        const int b = b0 + (li >> 1), co = li & 1;
        halfx8 hi, lo;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int an = blk * 16 + 4 * lg + q;
            float2 w = make_float2(0.f, 0.f);
            if (b < B && an < A) w = a.w[(((size_t)b * A + an) * F + f) * 2 + p];
            const float v0 = (co == 0 ? w.x : w.y) * wsc[p];     // multiplies Re x
            const float v1 = (co == 0 ? -w.y : w.x) * wsc[p];    // multiplies Im x
            split_f16(v0, hi, lo, 2 * q);
            split_f16(v1, hi, lo, 2 * q + 1);
        }
        s_wh[(pb * 2 + 0) * 64 + ln] = hi;
        s_wh[(pb * 2 + 1) * 64 + ln] = lo;
    }
    store_tile(s_x);
    if (ntiles > 1) load_tile(t_begin + SG_TC);
    __syncthreads();

    const int bcol = b0 + (i >> 1);
    const float lam = bcol < B ? a.lambda[bcol] : 0.f;
    const float swap_sign = (i & 1) ? -1.f : 1.f;
    floatx4 acc2[2][NAT];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int at = 0; at < NAT; at++) acc2[p][at] = floatx4{0.f, 0.f, 0.f, 0.f};
    float loss = 0.f;
    const floatx4 zero4 = {0.f, 0.f, 0.f, 0.f};

    for (int k = 0; k < ntiles; k++) {
        const uint32_t* sx = s_x + (k & 1) * SG_TC * XS;
        const int trow = wave * 16;
        // Forward: rows = this wave's 16 times; one 16-byte LDS read gives
        // 4 antennas x both pols.  The phasor operands are re-read from LDS
        // every tile (an opaque offset keeps the compiler from holding all
        // 4 NAT of them in registers across the loop).
        int woff = lane;
        asm volatile("" : "+v"(woff));
        const halfx8* wh = s_wh + woff;
        floatx4 y[2] = {zero4, zero4};
#pragma unroll
        for (int blk = 0; blk < NAT; blk++) {
            const uint4 d = *reinterpret_cast<const uint4*>(sx + (trow + i) * XS + blk * 16 + 4 * g);
            halfx8 xa[2];
            const uint32_t dw[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                halfx2 h0, h1;
                ci8_to_half2x2(dw[q], h0, h1);
                xa[0][2 * q] = h0[0]; xa[0][2 * q + 1] = h0[1];
                xa[1][2 * q] = h1[0]; xa[1][2 * q + 1] = h1[1];
            }
#pragma unroll
            for (int p = 0; p < 2; p++) {
                y[p] = mfma_f16(xa[p], wh[((p * NAT + blk) * 2 + 0) * 64], y[p]);
                y[p] = mfma_f16(xa[p], wh[((p * NAT + blk) * 2 + 1) * 64], y[p]);
            }
        }
        float gy[2][4];
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float v = y[p][r] * wuns[p];
                loss += lam * v * v;
                gy[p][r] = -lam * v;
            }
        sg_adjoint<NAT, XS, true>(sx + trow * XS, gy, swap_sign, i, g, acc2);
        if (k + 1 < ntiles) {
            store_tile(s_x + ((k + 1) & 1) * SG_TC * XS);
            if (k + 2 < ntiles) load_tile(t_begin + (k + 2) * SG_TC);
        }
        __syncthreads();
    }

    float* s_part = reinterpret_cast<float*>(lds_raw);
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int at = 0; at < NAT; at++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                s_part[((wave * 2 + p) * 16 + i) * APAD + at * 16 + 4 * g + r] = acc2[p][at][r];
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0) s_loss[wave] = loss;
    __syncthreads();
    constexpr int NPART = 2 * 16 * APAD;
    float* out = a.partial + ((((size_t)sp * F + f) * 2) * a.btiles + bt) * 16 * APAD;
    const size_t pstride = (size_t)a.btiles * 16 * APAD;
    for (int e = tid; e < NPART; e += blockDim.x) {
        const float v = ((s_part[e] + s_part[NPART + e]) + s_part[2 * NPART + e]) + s_part[3 * NPART + e];
        const int p = e / (16 * APAD), r = e - p * 16 * APAD;
        out[p * pstride + r] = v;
    }
    if (tid == 0)
        a.loss_part[((size_t)sp * F + f) * a.btiles + bt] = ((s_loss[0] + s_loss[1]) + s_loss[2]) + s_loss[3];
}

// gw[b,a,f,p] = sum over time splits of the partial rows (b, re) and (b, im).
// Threads follow the partial layout (antenna fastest), so the nsplit x 2
// reads per output coalesce; the writes, one float2 per thread into
// [B,A,F,1,P], are the strided side (8 B per thread, one pass).
// With `loss`, the last workgroup sums the n_loss workgroup partials instead,
// in FP64 and a fixed order: loss = -sum (one launch less, 4 us of a call).
__global__ __launch_bounds__(256) void adjoint_reduce_kernel(AdjArgs a, int nsplit, float2* gw, size_t n_loss,
                                                             double* loss) {
    if (loss && blockIdx.x == gridDim.x - 1) {
        __shared__ double s[256];
        double v = 0.0;
        for (size_t e = threadIdx.x; e < n_loss; e += blockDim.x) v += (double)a.loss_part[e];
        s[threadIdx.x] = v;
        __syncthreads();
        for (int off = 128; off > 0; off >>= 1) {
            if ((int)threadIdx.x < off) s[threadIdx.x] += s[threadIdx.x + off];
            __syncthreads();
        }
        if (threadIdx.x == 0) *loss = -s[0];
        return;
    }
    const size_t n = (size_t)a.F * 2 * a.btiles * 8 * a.A;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    size_t r = idx;
    const int an = (int)(r % a.A);
    r /= a.A;
    const int bb = (int)(r % 8);
    r /= 8;
    const int bt = (int)(r % a.btiles);
    r /= a.btiles;
    const int p = (int)(r & 1);
    const int f = (int)(r >> 1);
    const int b = bt * 8 + bb;
    if (b >= a.B) return;
    float re = 0.f, im = 0.f;
    for (int sp = 0; sp < nsplit; sp++) {
        const float* blk = a.partial + ((((size_t)sp * a.F + f) * 2 + p) * a.btiles + bt) * 16 * a.apad;
        re += blk[(2 * bb) * a.apad + an];
        im += blk[(2 * bb + 1) * a.apad + an];
    }
    gw[(((size_t)b * a.A + an) * a.F + f) * 2 + p] = make_float2(re, im);
}

static int run_adjoint(bool fused, bool f16, const void* input, const void* phasors, const void* grad_out,
                       const float* beam_weights, double* loss, void* grad_phasors, uint64_t A,
                       uint64_t F, uint64_t T, uint64_t P, uint64_t B, hipStream_t s) {
    const char* who = fused ? "stokes-i gradient" : "beamformer adjoint";
    if (P != 2) return fail(std::string(who) + ": number of polarizations must be 2");
    if (A == 0 || B == 0) return fail(std::string(who) + ": need at least one antenna and one beam");
    if (A > 16 * ADJ_MAXAT) return fail(std::string(who) + ": at most 128 antennas");
    if (fused && B > ADJ_MAXB) return fail(std::string(who) + ": at most 64 beams");
    if (B > 4096 || F > 65535 || T > (1u << 30)) return fail(std::string(who) + ": shape too large");
    if (!input || !grad_phasors || (fused ? (!phasors || !loss || !beam_weights) : !grad_out))
        return fail(std::string(who) + ": null pointer");
    if ((uintptr_t)input % 4 || (uintptr_t)grad_phasors % 8 || (phasors && (uintptr_t)phasors % 16) ||
        (grad_out && (uintptr_t)grad_out % 8))
        return fail(std::string(who) + ": misaligned buffer");
    AdjArgs a;
    std::memset(&a, 0, sizeof(a));
    a.x = static_cast<const uint32_t*>(input);
    a.w = static_cast<const float2*>(phasors);
    a.gy = static_cast<const float2*>(grad_out);
    a.A = (int)A; a.F = (int)F; a.T = (int)T; a.B = (int)B;
    a.n_at = (int)ceil_div(A, 16);
    a.apad = 16 * a.n_at;
    a.nsteps = 2 * (int)ceil_div(A, 4);
    a.btiles = (int)ceil_div(B, 8);
    if (fused)
        for (uint64_t b = 0; b < B; b++) a.lambda[b] = beam_weights[b];
    // FP32 loss + gradient with at most 4 beams: the 4x4-block kernel.
    const bool b4 = fused && !f16 && B <= 4 && A <= 64 && T % 4 == 0 && (uintptr_t)input % 16 == 0 &&
                    A * F * T < (1ull << 31);
    // Time splits, each a whole number of tiles.  Fused: the split length that
    // minimises rounds of resident workgroups (per CU: 4 FP32 or 3 split FP16
    // up to 64 or 48 antennas, else 2; the 4x4-block kernel SG4_WGS) x tiles
    // per wave.  Plain adjoint: one or two workgroups fill a CU's SIMDs, so a
    // launch costs its workgroups per CU times the tiles of a wave plus about
    // one tile time to sum the waves; a single workgroup per CU hides its
    // loads worse (1.3x a tile).  Ties take the longest split (fewest partial
    // sums).
    const int tc = b4 ? SG4_TC : fused ? SG_TC : ADJ_TC;
    const long tiles = (long)ceil_div(std::max<uint64_t>(T, 1), (uint64_t)tc);
    const long per_split = (long)F * a.btiles;
    const long cus = device_cus();
    const long slots = !fused ? cus : cus * (b4 ? SG4_WGS : f16 ? (a.n_at <= 3 ? 3 : 2) : (a.n_at <= 4 ? 4 : 2));
    long tiles_per = tiles;
    double best = -1;
    for (long tp = tiles; tp >= 1; tp--) {
        const long rounds = ((tiles + tp - 1) / tp * per_split + slots - 1) / slots;
        const long per_wave = b4 ? (tp + ADJ_WAVES - 1) / ADJ_WAVES : tp;   // b4: waves take tiles in turn
        const double cost = fused ? (double)rounds * per_wave : (double)rounds * (per_wave + 1) * (rounds == 1 ? 1.3 : 1.0);
        if (best < 0 || cost < best) { best = cost; tiles_per = tp; }
    }
    const long nsplit = (tiles + tiles_per - 1) / tiles_per;
    a.tsplit = (int)(tiles_per * tc);

    const size_t part_floats = (size_t)nsplit * F * 2 * a.btiles * 16 * a.apad;
    const size_t n_loss = (size_t)nsplit * F * a.btiles;
    unsigned char* ws = nullptr;
    const size_t ws_bytes = (part_floats + n_loss) * sizeof(float);
    if (F == 0) return BLADE_SUCCESS;
    int rc = library_workspace(WS_ADJOINT, ws_bytes, s, &ws);
    if (rc) return rc;
    a.partial = reinterpret_cast<float*>(ws);
    a.loss_part = a.partial + part_floats;

    const size_t lds_sum = (size_t)ADJ_WAVES * 2 * 16 * a.apad * 4;
    const size_t lds = !fused ? lds_sum
                       : b4    ? std::max(lds_sum, (size_t)a.A * 4 * SG4_WS * 4 + ADJ_WAVES * SG4_GY)
                       : f16   ? (size_t)2 * SG_TC * sg_xs(a.apad) * 4 + (size_t)2 * a.n_at * 2 * 64 * 16
                               : ((size_t)2 * SG_TC * sg_xs(a.apad) + 2 * (size_t)a.nsteps * 64) * 4;
#define ADJ_FN(...) reinterpret_cast<const void*>(&__VA_ARGS__)
    static const void* const fn_adj[2][ADJ_MAXAT] = {
        {ADJ_FN(adjoint_kernel<1, false>), ADJ_FN(adjoint_kernel<2, false>), ADJ_FN(adjoint_kernel<3, false>), ADJ_FN(adjoint_kernel<4, false>), ADJ_FN(adjoint_kernel<5, false>), ADJ_FN(adjoint_kernel<6, false>), ADJ_FN(adjoint_kernel<7, false>), ADJ_FN(adjoint_kernel<8, false>)},
        {ADJ_FN(adjoint_kernel<1, true>), ADJ_FN(adjoint_kernel<2, true>), ADJ_FN(adjoint_kernel<3, true>), ADJ_FN(adjoint_kernel<4, true>), ADJ_FN(adjoint_kernel<5, true>), ADJ_FN(adjoint_kernel<6, true>), ADJ_FN(adjoint_kernel<7, true>), ADJ_FN(adjoint_kernel<8, true>)}};
    static const void* const fn_f32[ADJ_MAXAT] = {ADJ_FN(stokes_grad_kernel<1>), ADJ_FN(stokes_grad_kernel<2>), ADJ_FN(stokes_grad_kernel<3>), ADJ_FN(stokes_grad_kernel<4>), ADJ_FN(stokes_grad_kernel<5>), ADJ_FN(stokes_grad_kernel<6>), ADJ_FN(stokes_grad_kernel<7>), ADJ_FN(stokes_grad_kernel<8>)};
    static const void* const fn_f16[ADJ_MAXAT] = {ADJ_FN(stokes_grad_f16_kernel<1>), ADJ_FN(stokes_grad_f16_kernel<2>), ADJ_FN(stokes_grad_f16_kernel<3>), ADJ_FN(stokes_grad_f16_kernel<4>), ADJ_FN(stokes_grad_f16_kernel<5>), ADJ_FN(stokes_grad_f16_kernel<6>), ADJ_FN(stokes_grad_f16_kernel<7>), ADJ_FN(stokes_grad_f16_kernel<8>)};
    static const void* const fn_b4[4] = {ADJ_FN(stokes_grad_b4_kernel<1>), ADJ_FN(stokes_grad_b4_kernel<2>), ADJ_FN(stokes_grad_b4_kernel<3>), ADJ_FN(stokes_grad_b4_kernel<4>)};
#undef ADJ_FN
    const bool vec = T % 4 == 0 && (uintptr_t)input % 16 == 0 && (uintptr_t)grad_out % 16 == 0;
    const void* fn = b4 ? fn_b4[a.n_at - 1] : !fused ? fn_adj[vec][a.n_at - 1] : (f16 ? fn_f16 : fn_f32)[a.n_at - 1];
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            set_error(std::string(who) + ": LDS attribute: " + hipGetErrorString(e));
            return BLADE_HIP_ERROR;
        }
    }
    const dim3 grid((unsigned)nsplit, (unsigned)F, (unsigned)a.btiles);
    void* args[] = {&a};
    (void)hipLaunchKernel(fn, grid, dim3(64 * ADJ_WAVES), args, lds, s);   // check_launch below reports
    const size_t n = (size_t)F * 2 * a.btiles * 8 * A;
    hipLaunchKernelGGL(adjoint_reduce_kernel, dim3((unsigned)ceil_div(n, 256) + (fused ? 1 : 0)), dim3(256), 0, s, a,
                       (int)nsplit, static_cast<float2*>(grad_phasors), n_loss, loss);
    return check_launch(who);
}

}  // namespace bl

using namespace bl;

extern "C" int blade_beamformer_adjoint(const void* input, const void* grad_output,
                                        void* grad_phasors, uint64_t A, uint64_t F, uint64_t T,
                                        uint64_t P, uint64_t B, blade_stream_t stream) {
    return run_adjoint(false, false, input, nullptr, grad_output, nullptr, nullptr, grad_phasors, A, F, T,
                       P, B, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int blade_beamformer_stokes_i_grad(int precision, const void* input, const void* phasors,
                                              const float* beam_weights, double* loss,
                                              void* grad_phasors, uint64_t A, uint64_t F,
                                              uint64_t T, uint64_t P, uint64_t B,
                                              blade_stream_t stream) {
    if (precision != BLADE_PREC_F32 && precision != BLADE_PREC_F16X2)
        return fail("stokes-i gradient: unknown precision");
    return run_adjoint(true, precision == BLADE_PREC_F16X2, input, phasors, nullptr, beam_weights, loss, grad_phasors, A, F, T, P,
                       B, reinterpret_cast<hipStream_t>(stream));
}
