// Small DFTs in registers and what the channelizer kernels share: forward,
// unnormalised, natural order in and out.
#pragma once

#include "common.hh"

namespace bl {

__device__ __forceinline__ float2 mul_neg_j(float2 a) { return make_float2(a.y, -a.x); }

template <int R>
__device__ __forceinline__ void dft_reg(float2 (&v)[R], const float2* __restrict__ tw, int twstep) {
    if constexpr (R == 1) {
        return;
    } else if constexpr (R == 2) {
        const float2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 4) {
        const float2 s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
        const float2 s13 = cadd(v[1], v[3]), d13 = mul_neg_j(csub(v[1], v[3]));
        v[0] = cadd(s02, s13);
        v[2] = csub(s02, s13);
        v[1] = cadd(d02, d13);
        v[3] = csub(d02, d13);
    } else if constexpr (R == 8) {
        float2 e[4] = {v[0], v[2], v[4], v[6]};
        float2 o[4] = {v[1], v[3], v[5], v[7]};
        dft_reg<4>(e, tw, 0);
        dft_reg<4>(o, tw, 0);
        const float c = 0.70710678118654752440f;
        const float2 o1 = make_float2(c * (o[1].x + o[1].y), c * (o[1].y - o[1].x));   // * e^{-j pi/4}
        const float2 o2 = mul_neg_j(o[2]);                                            // * e^{-j pi/2}
        const float2 o3 = make_float2(c * (o[3].y - o[3].x), -c * (o[3].x + o[3].y)); // * e^{-j 3pi/4}
        v[0] = cadd(e[0], o[0]); v[4] = csub(e[0], o[0]);
        v[1] = cadd(e[1], o1);   v[5] = csub(e[1], o1);
        v[2] = cadd(e[2], o2);   v[6] = csub(e[2], o2);
        v[3] = cadd(e[3], o3);   v[7] = csub(e[3], o3);
    } else {
        // Direct DFT of size R with W_R^q = tw[q * twstep].
        float2 r[R];
#pragma unroll
        for (int k = 0; k < R; k++) {
            float2 acc = v[0];
#pragma unroll
            for (int n = 1; n < R; n++) {
                const float2 w = tw[((n * k) % R) * twstep];
                acc.x += v[n].x * w.x - v[n].y * w.y;
                acc.y += v[n].x * w.y + v[n].y * w.x;
            }
            r[k] = acc;
        }
#pragma unroll
        for (int k = 0; k < R; k++) v[k] = r[k];
    }
}

// a * W_16^E with W_16 = exp(-j 2 pi / 16); cos(2 pi e / 16) by table,
// -sin(2 pi e / 16) = cos(2 pi (e + 4) / 16).
template <int E>
__device__ __forceinline__ float2 mul_w16(float2 a) {
    constexpr int e = E & 15;
    constexpr float c1 = 0.92387953251128675613f;   // cos(pi/8)
    constexpr float s1 = 0.38268343236508977173f;   // sin(pi/8)
    constexpr float h = 0.70710678118654752440f;    // cos(pi/4)
    constexpr float cs[16] = {1.f, c1, h, s1, 0.f, -s1, -h, -c1, -1.f, -c1, -h, -s1, 0.f, s1, h, c1};
    if constexpr (e == 0) return a;
    else if constexpr (e == 4) return make_float2(a.y, -a.x);
    else if constexpr (e == 8) return make_float2(-a.x, -a.y);
    else if constexpr (e == 12) return make_float2(-a.y, a.x);
    else return cmul(a, make_float2(cs[e], cs[(e + 4) & 15]));
}

// 16-point DFT in natural order: n = 4 n1 + n2, k = k1 + 4 k2,
// X[k1 + 4 k2] = sum_n2 W4^(n2 k2) W16^(n2 k1) sum_n1 W4^(n1 k1) x[4 n1 + n2].
__device__ __forceinline__ void dft16(float2 (&v)[16]) {
    float2 y[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; n2++) {
        float2 t[4] = {v[n2], v[n2 + 4], v[n2 + 8], v[n2 + 12]};
        dft_reg<4>(t, nullptr, 0);
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++) y[n2][k1] = t[k1];
    }
    y[1][1] = mul_w16<1>(y[1][1]); y[1][2] = mul_w16<2>(y[1][2]); y[1][3] = mul_w16<3>(y[1][3]);
    y[2][1] = mul_w16<2>(y[2][1]); y[2][2] = mul_w16<4>(y[2][2]); y[2][3] = mul_w16<6>(y[2][3]);
    y[3][1] = mul_w16<3>(y[3][1]); y[3][2] = mul_w16<6>(y[3][2]); y[3][3] = mul_w16<9>(y[3][3]);
#pragma unroll
    for (int k1 = 0; k1 < 4; k1++) {
        float2 t[4] = {y[0][k1], y[1][k1], y[2][k1], y[3][k1]};
        dft_reg<4>(t, nullptr, 0);
#pragma unroll
        for (int k2 = 0; k2 < 4; k2++) v[k1 + 4 * k2] = t[k2];
    }
}

// Odd R by symmetry: with a_h = x_h + x_(R-h), b_h = x_h - x_(R-h),
//   X_k, X_(R-k) = x_0 + sum_h cos(2 pi h k / R) a_h  -+  j sum_h sin(2 pi h k / R) b_h.
template <int R>
__device__ __forceinline__ void dft_odd(float2 (&v)[R]) {
    static_assert(R == 3 || R == 5 || R == 7, "tabulated sizes");
    constexpr float c3[3] = {1.f, -0.5f, -0.5f};
    constexpr float s3[3] = {0.f, 0.86602540378443864676f, -0.86602540378443864676f};
    constexpr float c5[5] = {1.f, 0.30901699437494742410f, -0.80901699437494742410f, -0.80901699437494742410f,
                             0.30901699437494742410f};
    constexpr float s5[5] = {0.f, 0.95105651629515357212f, 0.58778525229247312917f, -0.58778525229247312917f,
                             -0.95105651629515357212f};
    constexpr float c7[7] = {1.f, 0.62348980185873353053f, -0.22252093395631440429f, -0.90096886790241912624f,
                             -0.90096886790241912624f, -0.22252093395631440429f, 0.62348980185873353053f};
    constexpr float s7[7] = {0.f, 0.78183148246802980871f, 0.97492791218182360702f, 0.43388373911755812048f,
                             -0.43388373911755812048f, -0.97492791218182360702f, -0.78183148246802980871f};
    constexpr int H = R / 2;
    float2 a[H + 1], b[H + 1];
#pragma unroll
    for (int h = 1; h <= H; h++) {
        a[h] = cadd(v[h], v[R - h]);
        b[h] = csub(v[h], v[R - h]);
    }
    float2 x0 = v[0];
#pragma unroll
    for (int h = 1; h <= H; h++) x0 = cadd(x0, a[h]);
#pragma unroll
    for (int k = 1; k <= H; k++) {
        float2 m = v[0], n = make_float2(0.f, 0.f);
#pragma unroll
        for (int h = 1; h <= H; h++) {
            const int q = (h * k) % R;
            const float c = R == 3 ? c3[q % 3] : R == 5 ? c5[q % 5] : c7[q % 7];
            const float s = R == 3 ? s3[q % 3] : R == 5 ? s5[q % 5] : s7[q % 7];
            m.x += c * a[h].x;
            m.y += c * a[h].y;
            n.x += s * b[h].x;
            n.y += s * b[h].y;
        }
        v[k] = make_float2(m.x + n.y, m.y - n.x);          // m - j n
        v[R - k] = make_float2(m.x - n.y, m.y + n.x);      // m + j n
    }
    v[0] = x0;
}

template <int R>
__device__ __forceinline__ void dft_any(float2 (&v)[R]);

// R = N1 N2 with coprime factors (Good-Thomas): no twiddles between them.
template <int N1, int N2>
__device__ __forceinline__ void dft_pfa(float2 (&v)[N1 * N2]) {
    float2 y[N1][N2];
#pragma unroll
    for (int n1 = 0; n1 < N1; n1++) {
        float2 t[N2];
#pragma unroll
        for (int n2 = 0; n2 < N2; n2++) t[n2] = v[(N2 * n1 + N1 * n2) % (N1 * N2)];
        dft_any<N2>(t);
#pragma unroll
        for (int k2 = 0; k2 < N2; k2++) y[n1][k2] = t[k2];
    }
#pragma unroll
    for (int k2 = 0; k2 < N2; k2++) {
        float2 t[N1];
#pragma unroll
        for (int n1 = 0; n1 < N1; n1++) t[n1] = y[n1][k2];
        dft_any<N1>(t);
#pragma unroll
        for (int k = 0; k < N1 * N2; k++)
            if (k % N2 == k2) v[k] = t[k % N1];
    }
}

// Nine points as 3 x 3: n = 3 n1 + n2, k = k1 + 3 k2, twiddles W_9^(n2 k1).
__device__ __forceinline__ void dft9(float2 (&v)[9]) {
    const float2 w1 = make_float2(0.76604444311897803520f, -0.64278760968653932632f);
    const float2 w2 = make_float2(0.17364817766693034885f, -0.98480775301220805937f);
    const float2 w4 = make_float2(-0.93969262078590838405f, -0.34202014332566873304f);
    float2 y[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; n2++) {
        float2 t[3] = {v[n2], v[n2 + 3], v[n2 + 6]};
        dft_odd<3>(t);
#pragma unroll
        for (int k1 = 0; k1 < 3; k1++) y[n2][k1] = t[k1];
    }
    y[1][1] = cmul(y[1][1], w1);
    y[1][2] = cmul(y[1][2], w2);
    y[2][1] = cmul(y[2][1], w2);
    y[2][2] = cmul(y[2][2], w4);
#pragma unroll
    for (int k1 = 0; k1 < 3; k1++) {
        float2 t[3] = {y[0][k1], y[1][k1], y[2][k1]};
        dft_odd<3>(t);
#pragma unroll
        for (int k2 = 0; k2 < 3; k2++) v[k1 + 3 * k2] = t[k2];
    }
}

// Any of the radices 2 - 10, 12, 14, 15, 16 (11 and 13 have no use here).
template <int R>
__device__ __forceinline__ void dft_any(float2 (&v)[R]) {
    if constexpr (R == 2 || R == 4 || R == 8) dft_reg<R>(v, nullptr, 0);
    else if constexpr (R == 3 || R == 5 || R == 7) dft_odd<R>(v);
    else if constexpr (R == 6) dft_pfa<2, 3>(v);
    else if constexpr (R == 9) dft9(v);
    else if constexpr (R == 10) dft_pfa<2, 5>(v);
    else if constexpr (R == 12) dft_pfa<4, 3>(v);
    else if constexpr (R == 14) dft_pfa<2, 7>(v);
    else if constexpr (R == 15) dft_pfa<3, 5>(v);
    else dft16(v);
}

// Detector sums of (X, Y) turned into those of (L, R) = (X + jY, X - jY),
// the polarizer (polarizer.cu:5-25) applied before the detector: sums are
// linear in [XX*, YY*, Re XY*, Im XY*], so the map applies after integration.
//   Stokes I doubles; |L|^2 = XX + YY + 2 Im, |R|^2 = XX + YY - 2 Im,
//   Re LR* = XX - YY, Im LR* = 2 Re.
template <int NPOL>
__device__ inline void circular_sums(float (&a)[NPOL]) {
    if constexpr (NPOL == 1) {
        a[0] *= 2.f;
    } else {
        const float xx = a[0], yy = a[1], re = a[2], im = a[3];
        a[0] = (xx + yy) + 2.f * im;
        a[1] = (xx + yy) - 2.f * im;
        a[2] = xx - yy;
        a[3] = 2.f * re;
    }
}

// Workgroup order with consecutive values on one XCD: the dispatcher deals
// workgroups to the 8 XCDs round-robin (b mod 8), so b -> (b mod 8) G/8 + b/8
// hands workgroups that take consecutive spectra to one XCD, whose L2 then
// merges their interleaved pieces of each output line.  G is a multiple of 8.
__device__ __forceinline__ unsigned xcd_order(unsigned b, unsigned G) { return (b & 7u) * (G >> 3) + (b >> 3); }

}  // namespace bl
