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
// sum_{f,t,p} |y_b|^2, so gy = -lambda_b y_b.  Each wave recomputes y of 64
// times from the CI8 voltages it holds in registers and runs the adjoint on
// the same voltages: neither beams nor gy pass through memory.
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
constexpr int SG_TC = 64;          // stokes_grad_kernel: time samples per tile of a wave
// Words per LDS voltage row of stokes_grad_kernel: 64 times and 4 of padding,
// which puts the 16 rows a read touches on different banks.
constexpr int SG_XS = SG_TC + 4;

struct AdjArgs {
    const uint32_t* x;       // [A,F,T] dwords: CI8 (re0, im0, re1, im1)
    const float2* w;         // [B,A,F,1,P] phasors (fused mode)
    const float2* gy;        // [B,F,T,P] upstream gradient (adjoint mode)
    float* partial;          // [nsplit][F][P][btiles][16][apad]
    double* loss_part;       // [nsplit][F][btiles]
    int A, F, T, B;
    int apad, n_at;          // padded antennas, antenna tiles
    int tsplit;              // time samples per workgroup (a multiple of ADJ_TC or SG_TC)
    int btiles;
    float lambda[ADJ_MAXB];  // beam weights of the fused loss
};

// The value of lane l ^ 1 (DPP quad permutation [1, 0, 3, 2]).
__device__ __forceinline__ float swap_pairs(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
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

// Fused Stokes-I loss and phasor gradient of A <= 16 NAT antennas and 8 beams,
// for either precision (the FP16 split has nothing to gain on it).  A wave
// takes tiles of 64 times, without barriers:
//   * voltages: lane (g, i) loads times 4i .. 4i + 3 of antennas 4g .. 4g + 3
//     of every group of 16 in 16-byte pieces, one tile ahead;
//   * forward: rows = times (4i + n of four instructions n), K = 16 antennas x
//     (re, im), columns = (beam, re/im); the phasors are three exact BF16
//     parts in LDS;
//   * a lane then holds y of 16 consecutive times of its column, which is, cut
//     into three BF16 parts, the B operand of the adjoint as it stands:
//     real products as in adjoint_kernel, K = 32 times;
//   * the adjoint's A operand (rows = antennas, 8 consecutive times) is the
//     same voltages turned through 4 KiB of LDS per wave, 16 antennas at a time.
// Products are exact and accumulate in FP32.  Bound by VALU work (widening the
// voltages twice, cutting gy) and load latency at 2 waves per SIMD (216 VGPRs
// at A = 42; 3 waves spill).  A42 F384 T2048 B4 per call: 53 us, where FP32
// 4x4 and 16x16 matrix instructions took 97 us (B = 4) and 129 us (B = 8), and
// split FP16 through barriered LDS tiles 69 us; error against FP64 5e-8
// (FP32 1.1e-7).  VEC: 16-byte loads (T a multiple of 4, aligned voltages).
template <int NAT, bool VEC>
__global__ __launch_bounds__(256, (NAT <= 2 ? 3 : NAT <= 4 ? 2 : 1)) void stokes_grad_kernel(AdjArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    uint4* const s_w = reinterpret_cast<uint4*>(lds_raw);                 // [unit][p][part][64]
    __shared__ double s_loss[ADJ_WAVES];

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
    uint32_t* const s_x = reinterpret_cast<uint32_t*>(s_w + NAT * 6 * 64) + wave * 16 * SG_XS;   // this wave's rows

    // Voltages of unit u (antennas 16u + 4g + q, times t0 + 4i .. + 3); rows
    // past A repeat the last antenna (their phasors are zero, their sums not
    // stored), times past the split its end (their gy is zeroed).
    uint4 xd[NAT][4];
    const uint32_t* const xf = a.x + (size_t)f * T;
    auto load_unit = [&](int t0, int u) {
        // Opaque stride: keeps the 4 NAT row addresses from being held in
        // registers across tiles.
        size_t st = (size_t)F * T;
        asm volatile("" : "+s"(st));
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t* const xp = xf + min(16 * u + 4 * g + q, A - 1) * st;
            const int t = t0 + 4 * i;
            if constexpr (VEC)
                xd[u][q] = *reinterpret_cast<const uint4*>(xp + min(t, t_end - 4));
            else
                xd[u][q] = make_uint4(xp[min(t, t_end - 1)], xp[min(t + 1, t_end - 1)], xp[min(t + 2, t_end - 1)],
                                      xp[min(t + 3, t_end - 1)]);
        }
    };
    int t0 = t_begin + wave * SG_TC;
    if (t0 < t_end) {
#pragma unroll
        for (int u = 0; u < NAT; u++) load_unit(t0, u);
    }

    // Forward B operand: lane (g, column) of unit u holds k = 8g + 2q + c ->
    // (antenna 16u + 4g + q, component c of x), column -> (beam, re/im):
    // y_r = x_r w_r - x_i w_i, y_i = x_r w_i + x_i w_r.
    for (int e = threadIdx.x; e < NAT * 64; e += 64 * ADJ_WAVES) {
        const int ln = e & 63, u = e >> 6;
        const int col = ln & 15, lg = ln >> 4;
        const int b = bt * 8 + (col >> 1);
        const bool im = col & 1;
        float4 w[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int an = 16 * u + 4 * lg + q;
            w[q] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (b < B && an < A) w[q] = reinterpret_cast<const float4*>(a.w)[((size_t)b * A + an) * F + f];
        }
#pragma unroll
        for (int p = 0; p < 2; p++) {
            uint32_t h[3][4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float wr = p ? w[q].z : w[q].x, wi = p ? w[q].w : w[q].y;
                float v0[3], v1[3];
                split_bf16x3(im ? wi : wr, v0);
                split_bf16x3(im ? wr : -wi, v1);
#pragma unroll
                for (int k = 0; k < 3; k++) h[k][q] = bf16_pair(v0[k], v1[k]);
            }
#pragma unroll
            for (int k = 0; k < 3; k++)
                s_w[((u * 2 + p) * 3 + k) * 64 + ln] = make_uint4(h[k][0], h[k][1], h[k][2], h[k][3]);
        }
    }
    __syncthreads();

    const int bcol = bt * 8 + (i >> 1);
    const float lam = bcol < B ? a.lambda[bcol] : 0.f;
    const floatx4 zero4 = {0.f, 0.f, 0.f, 0.f};
    floatx4 acc[2][NAT][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int at = 0; at < NAT; at++)
#pragma unroll
            for (int c = 0; c < 2; c++) acc[p][at][c] = zero4;
    double loss = 0.0;      // FP64 past the 32 squares of a lane's tile

    for (; t0 < t_end; t0 += ADJ_WAVES * SG_TC) {
        // ---- forward: y[p][n], register r of lane (g, column): time
        // t0 + 16g + 4r + n.
        floatx4 y[2][4];
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int n = 0; n < 4; n++) y[p][n] = zero4;
#pragma unroll
        for (int u = 0; u < NAT; u++)
#pragma unroll
            for (int p = 0; p < 2; p++) {
                uint4 xo[4];
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    auto dw = [&](int q) { return n == 0 ? xd[u][q].x : n == 1 ? xd[u][q].y : n == 2 ? xd[u][q].z : xd[u][q].w; };
                    xo[n] = make_uint4(ci8_to_bf16(dw(0), p), ci8_to_bf16(dw(1), p), ci8_to_bf16(dw(2), p),
                                       ci8_to_bf16(dw(3), p));
                }
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    const uint4 wk = s_w[((u * 2 + p) * 3 + k) * 64 + lane];
#pragma unroll
                    for (int n = 0; n < 4; n++) y[p][n] = mfma_bf16(xo[n], wk, y[p][n]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        // ---- loss and gy = -lambda y in three parts; the 8 times
        // 16g + 8h + (0 .. 7) are one K = 32 operand.
        if (t0 + SG_TC > t_end) {              // uniform: the split's last tile
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int n = 0; n < 4; n++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (t0 + 16 * g + 4 * r + n >= t_end) y[p][n][r] = 0.f;
        }
        float tl = 0.f;
#pragma unroll
        for (int n = 0; n < 4; n++) {
            float e = 0.f;
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int r = 0; r < 4; r++) e += y[p][n][r] * y[p][n][r];
            tl += e;
        }
        loss += (double)lam * (double)tl;
        // Infinities and NaN (they show in tl) take the split that keeps them.
        const bool plain = __all(fabsf(tl) <= 3.0e38f);
        // ---- adjoint, half of the times at a time (half the operands of gy
        // live): per antenna tile, the unit's rows turned through this wave's
        // LDS rows (LDS operations of a wave complete in order); after the
        // second half the next tile's loads go into the registers just read.
        const bool more = t0 + ADJ_WAVES * SG_TC < t_end;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint4 gb[2][3];
            auto parts = [&](auto checked) {
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    uint32_t w[3][4];
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const int r = 2 * h + (m >> 1), n = 2 * (m & 1);
                        float u0[3], u1[3];
                        split_bf16x3<decltype(checked)::value>(-lam * y[p][n][r], u0);
                        split_bf16x3<decltype(checked)::value>(-lam * y[p][n + 1][r], u1);
#pragma unroll
                        for (int k = 0; k < 3; k++) w[k][m] = bf16_pair(u0[k], u1[k]);
                    }
#pragma unroll
                    for (int k = 0; k < 3; k++) gb[p][k] = make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
                }
            };
            if (plain)
                parts(std::false_type{});
            else
                parts(std::true_type{});
#pragma unroll
            for (int at = 0; at < NAT; at++) {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *reinterpret_cast<uint4*>(s_x + (4 * g + q) * SG_XS + 4 * i) = xd[at][q];
                if (h == 1 && more) load_unit(t0 + ADJ_WAVES * SG_TC, at);
                const uint32_t* const row = s_x + i * SG_XS + 16 * g + 8 * h;
                const uint4 lo = *reinterpret_cast<const uint4*>(row), hi = *reinterpret_cast<const uint4*>(row + 4);
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    uint4 xo[2];
#pragma unroll
                    for (int c = 0; c < 2; c++) xo[c] = ci8_times_bf16(lo, hi, 2 * p + c);
#pragma unroll
                    for (int k = 0; k < 3; k++)
#pragma unroll
                        for (int c = 0; c < 2; c++) acc[p][at][c] = mfma_bf16(xo[c], gb[p][k], acc[p][at][c]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0) s_loss[wave] = loss;
    __syncthreads();                          // every wave is done with the LDS operands
    adj_store_partials<NAT>(a, acc, reinterpret_cast<float*>(lds_raw), sp, f, bt);
    if (threadIdx.x == 0)
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
        for (size_t e = threadIdx.x; e < n_loss; e += blockDim.x) v += a.loss_part[e];
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

static int run_adjoint(bool fused, const void* input, const void* phasors, const void* grad_out,
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
    a.btiles = (int)ceil_div(B, 8);
    if (fused)
        for (uint64_t b = 0; b < B; b++) a.lambda[b] = beam_weights[b];
    // Time splits, each a whole number of tiles.  Both kernels fill a CU's
    // SIMDs with one or two workgroups, so a launch costs its workgroups per
    // CU times the tiles of a wave plus about one tile time of set-up (packing
    // the phasors, summing the waves); a single workgroup per CU hides its
    // loads worse (1.3x a tile).  Ties take the longest split (fewest partial
    // sums).  A42 F384 T2048 B4 (loss + gradient): 2 splits 53 us, 1 or 4
    // splits 56 us, 8 splits 70 us.
    const int tc = fused ? SG_TC : ADJ_TC;
    const long tiles = (long)ceil_div(std::max<uint64_t>(T, 1), (uint64_t)tc);
    const long per_split = (long)F * a.btiles;
    const long cus = device_cus();
    long tiles_per = tiles;
    double best = -1;
    for (long tp = tiles; tp >= 1; tp--) {
        const long rounds = ((tiles + tp - 1) / tp * per_split + cus - 1) / cus;
        const long per_wave = fused ? (tp + ADJ_WAVES - 1) / ADJ_WAVES : tp;   // fused: waves take tiles in turn
        const double cost = (double)rounds * (per_wave + 1) * (rounds == 1 ? 1.3 : 1.0);
        if (best < 0 || cost < best) { best = cost; tiles_per = tp; }
    }
    const long nsplit = (tiles + tiles_per - 1) / tiles_per;
    a.tsplit = (int)(tiles_per * tc);

    const size_t part_floats = (size_t)nsplit * F * 2 * a.btiles * 16 * a.apad;
    const size_t n_loss = (size_t)nsplit * F * a.btiles;
    unsigned char* ws = nullptr;
    const size_t ws_bytes = part_floats * sizeof(float) + n_loss * sizeof(double);
    if (F == 0) return BLADE_SUCCESS;
    int rc = library_workspace(WS_ADJOINT, ws_bytes, s, &ws);
    if (rc) return rc;
    a.partial = reinterpret_cast<float*>(ws);
    a.loss_part = reinterpret_cast<double*>(a.partial + part_floats);     // part_floats is even

    const size_t lds_sum = (size_t)ADJ_WAVES * 2 * 16 * a.apad * 4;
    const size_t lds = fused ? std::max(lds_sum, (size_t)a.n_at * 6 * 64 * 16 + ADJ_WAVES * 16 * SG_XS * 4) : lds_sum;
#define ADJ_FN(...) reinterpret_cast<const void*>(&__VA_ARGS__)
    static const void* const fn_adj[2][ADJ_MAXAT] = {
        {ADJ_FN(adjoint_kernel<1, false>), ADJ_FN(adjoint_kernel<2, false>), ADJ_FN(adjoint_kernel<3, false>), ADJ_FN(adjoint_kernel<4, false>), ADJ_FN(adjoint_kernel<5, false>), ADJ_FN(adjoint_kernel<6, false>), ADJ_FN(adjoint_kernel<7, false>), ADJ_FN(adjoint_kernel<8, false>)},
        {ADJ_FN(adjoint_kernel<1, true>), ADJ_FN(adjoint_kernel<2, true>), ADJ_FN(adjoint_kernel<3, true>), ADJ_FN(adjoint_kernel<4, true>), ADJ_FN(adjoint_kernel<5, true>), ADJ_FN(adjoint_kernel<6, true>), ADJ_FN(adjoint_kernel<7, true>), ADJ_FN(adjoint_kernel<8, true>)}};
    static const void* const fn_grad[2][ADJ_MAXAT] = {
        {ADJ_FN(stokes_grad_kernel<1, false>), ADJ_FN(stokes_grad_kernel<2, false>), ADJ_FN(stokes_grad_kernel<3, false>), ADJ_FN(stokes_grad_kernel<4, false>), ADJ_FN(stokes_grad_kernel<5, false>), ADJ_FN(stokes_grad_kernel<6, false>), ADJ_FN(stokes_grad_kernel<7, false>), ADJ_FN(stokes_grad_kernel<8, false>)},
        {ADJ_FN(stokes_grad_kernel<1, true>), ADJ_FN(stokes_grad_kernel<2, true>), ADJ_FN(stokes_grad_kernel<3, true>), ADJ_FN(stokes_grad_kernel<4, true>), ADJ_FN(stokes_grad_kernel<5, true>), ADJ_FN(stokes_grad_kernel<6, true>), ADJ_FN(stokes_grad_kernel<7, true>), ADJ_FN(stokes_grad_kernel<8, true>)}};
#undef ADJ_FN
    const bool vec = T % 4 == 0 && (uintptr_t)input % 16 == 0 && (uintptr_t)grad_out % 16 == 0;
    const void* fn = fused ? fn_grad[vec][a.n_at - 1] : fn_adj[vec][a.n_at - 1];
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
    return run_adjoint(false, input, nullptr, grad_output, nullptr, nullptr, grad_phasors, A, F, T,
                       P, B, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int blade_beamformer_stokes_i_grad(int precision, const void* input, const void* phasors,
                                              const float* beam_weights, double* loss,
                                              void* grad_phasors, uint64_t A, uint64_t F,
                                              uint64_t T, uint64_t P, uint64_t B,
                                              blade_stream_t stream) {
    if (precision != BLADE_PREC_F32 && precision != BLADE_PREC_F16X2)
        return fail("stokes-i gradient: unknown precision");
    return run_adjoint(true, input, phasors, nullptr, beam_weights, loss, grad_phasors, A, F, T, P,
                       B, reinterpret_cast<hipStream_t>(stream));
}
