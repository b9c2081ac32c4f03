// Least-squares phase unwrapping by a DCT-II Poisson solve (reference DCT_UWLS_Unwrapped,
// DCT_Unwrapping.cu:10-107, 144-246, 300-312, 336-417), batched over maps, for gfx950.
//
// Maths (N = M, Neumann boundaries):
//   rho   = div of wrapped forward differences (NumericDerivative1 + SumDerivative), or with
//           CTDM_UNWRAP_SINCOS  cos(phi) L[sin phi] - sin(phi) L[cos phi] = sum_nbr sin(phi_n - phi)
//           (the trigonometric right-hand side of FastUnwrapping.cu:37-96 on the same stencil)
//   phi   = IDCT2( DCT2(rho) / lambda ),  lambda_ij = -4 (sin^2(pi i/2N) + sin^2(pi j/2N)), DC := 0
//           (REFCOMPAT_EIG: 2cos(4 pi i/(4N-1)) + 2cos(4 pi j/(4N-1)) - 4, DCT_Unwrapping.cu:310)
//   lambda is formed in FP64 (-> 0 at low frequencies, where any rounding is amplified). The batched path multiplies by
//   its reciprocal in FP32, rounded once (with the reference's IDCT: the hardware reciprocal); the plain path divides in FP64.
// Orthonormal DCT-II along a line via one N-point complex FFT (Makhoul reordering):
//   v[n] = x[2n], v[N-1-n] = x[2n+1];  X[k] = s_k Re(exp(-i pi k / 2N) FFT(v)[k]),
//   s_0 = sqrt(1/N), s_k = sqrt(2/N).
// Orthonormal DCT-III (its inverse):
//   V[k] = exp(i pi k/2N) (C_k - i C_{N-k}), C = X / s, C_N = 0;  v = IFFT(V) / N;
//   x[2n] = Re v[n], x[2n+1] = Re v[N-1-n].
// REFCOMPAT_IDCT reproduces the reference IDCT literally (2N Hermitian completion with the (i+1)
// twiddle on the right half, DCT_Unwrapping.cu:218-246), which needs a 2N-point transform.
//
// Batched path: three kernels per batch, each transforming two real lines as one complex line (line a + i
// line b; the transform of a real line is conjugate-symmetric, so the two are told apart afterwards)
//   1. k_uw_rows_fwd: RHS on the fly + DCT-II along x          -> D1[b][y][kx]
//   2. k_uw_cols:     DCT-II along y, / lambda, DCT-III along y -> D2[b][y][kx]
//   3. k_uw_rows_inv: DCT-III along x (+ congruence)           -> out[b][y][x]
#include "fft_dev.hpp"
#include "internal.hpp"

#include <cmath>
#include <mutex>
#include <tuple>

namespace ctdm {

enum : unsigned { F_SINCOS = CTDM_UNWRAP_SINCOS, F_REF_EIG = CTDM_UNWRAP_REFCOMPAT_EIG,
                  F_REF_IDCT = CTDM_UNWRAP_REFCOMPAT_IDCT, F_CONGRUENT = CTDM_UNWRAP_CONGRUENT,
                  F_REF_FAST = CTDM_UNWRAP_REFCOMPAT_FAST, F_ALL = 0x1fu };

static constexpr float kPI = 3.14159265358979323846f;

// Reference wrap of NumericDerivative1 (DCT_Unwrapping.cu:378-379), s = sign(t):
// t - 2 pi s floor(|pi s + t| / 2 pi). |pi s + t| is u = pi + |t| (0 for t = 0), and floor(u / 2 pi) is 0 below
// 2 pi and 1 below 4 pi also after rounding (a float below 2 pi k, divided by 2 pi, rounds below k), so
// differences of less than three half periods, all that wrapped maps have, need no division; the others (and
// infinities and NaN) take the formula as it stands. Bit-identical to it.
__device__ __forceinline__ float wrapdiff(float t)
{
    const float u = kPI + fabsf(t);
    float r = u >= 2.f * kPI ? t - copysignf(2.f * kPI, t) : t;
    if (!(u < 4.f * kPI)) {
        const float s = (t > 0.f) ? 1.f : ((t < 0.f) ? -1.f : 0.f);
        r = t - 2.f * kPI * s * floorf(fabsf(kPI * s + t) / (2.f * kPI));
    }
    return r;
}

// Sine right-hand side at (i, j) of an N x N map.
__device__ __forceinline__ float sin_rhs_at(const float* __restrict__ p, int N, int i, int j)
{
    const int k = i + N * j;
    const float c = p[k];
    float r = 0.f;
    if (i < N - 1) r += sinf(p[k + 1] - c);
    if (i > 0) r += sinf(p[k - 1] - c);
    if (j < N - 1) r += sinf(p[k + N] - c);
    if (j > 0) r += sinf(p[k - N] - c);
    return r;
}

// Makhoul source index: position n of v holds x[src(n)].
__device__ __forceinline__ int mk_src(int n, int N) { return n < N / 2 ? 2 * n : 2 * (N - 1 - n) + 1; }

// Makhoul position of x[i] in v (the inverse of mk_src).
__device__ __forceinline__ int mk_pos(int i, int N) { return i & 1 ? N - 1 - (i >> 1) : i >> 1; }

// Transform and workgroup of a pair of lines of length N: T threads per pair with a radix plan of their own,
// GP row pairs or CP column pairs per workgroup. More threads per line than Plan<N> has, so that a thread's share
// is short (4 or 8 points): these kernels wait for memory and for their own chains far more than they compute,
// and the workgroups are small so that a few maps still spread over the chip (24 maps of 192^2: right-hand side
// and first transform 13.1 us, with Plan<192>'s 16 threads 17.5 us; 45 of 128^2: 8.1 against 11.8 us).
template <int N, int T_, int GP_, int... R>
struct PairOf {
    static constexpr int T = T_, GP = GP_, CP = 8;
    static constexpr int NT = T * GP, NC = T * CP;       // threads of a row / column workgroup
    static constexpr int R0 = std::get<0>(std::make_tuple(R...)), J = N / T;
    static_assert(N / R0 == T, "the first stage's elements of thread t are t + r T");
    template <int DIR, class TW, class GL, class GS>
    __device__ __forceinline__ static void run(int t, float2* s, const TW& tw, GL& gl, GS& gs)
    {
        Stockham<N, T, DIR, 1, R...>::run(t, s, tw, gl, gs);
    }
};
template <int N>
struct Pair;
template <>
struct Pair<32> : PairOf<32, 8, 8, 4, 8> {};
template <>
struct Pair<64> : PairOf<64, 16, 4, 4, 4, 4> {};
template <>
struct Pair<128> : PairOf<128, 32, 8, 4, 4, 8> {};
template <>
struct Pair<192> : PairOf<192, 24, 8, 8, 8, 3> {};
template <>
struct Pair<256> : PairOf<256, 64, 2, 4, 4, 4, 4> {};  // one map 38.2 us from hologram to phase with 32 threads and 8 pairs, 34.2

// Which of a solve's transforms compute their stages in double (Wide). Two lines in one transform take on each other's
// rounding, and the plans of Pair have more stages than Plan's: the solve's error against 64 bits was 6 to 22 % larger than with
// one real line per transform. The rows' right-hand side matters most, since 1 / lambda raises what its transform adds to the low
// frequencies; then the inverse transforms, whose error is the result's. These are as many as bring it below. Mean relative error
// over 64 maps, in 1e-7, for the wrapped and the sine right-hand side, one line per transform | pairs in floats | now:
// 64^2 1.82 1.91 | 1.91 2.07 | 1.62 1.75, 128^2 1.75 1.82 | 1.97 2.05 | 1.52 1.69, 192^2 2.13 2.24 | 2.56 2.71 | 2.05 2.12,
// 256^2 2.88 2.83 | 3.06 3.15 | 2.50 2.58. At 32^2 and 64^2 leaving the factors s_k out is enough. The cost: 60 maps of 256^2
// 33.8 -> 35.1 us, of 192^2 30.3 -> 32.4, of 128^2 18.6 -> 19.8 (55.5, 39.5 and 22.7 with one line per transform); in
// double throughout 38.5, 34.2, 20.2.
template <int N>
struct InDouble {
    static constexpr bool rhs = N >= 128, cols_inv = N == 128, rows_inv = N == 128 || N == 192;
};
template <bool W, class TW>
__device__ __forceinline__ auto wide(const TW& tw)
{
    if constexpr (W)
        return Wide<TW>{tw};
    else
        return tw;
}

// The solve's transforms leave the DCT's factors s_k out, which cancel between a DCT-II and its inverse, and scale each
// forward transform by 1 / DctScale<N> instead: a power of two near N, so that no rounding comes from it and the
// coefficients keep the magnitude of orthonormal ones. What is left of 1 / N^2 joins the eigenvalue (solve_pair).
template <int N>
struct DctScale {
    static constexpr int value = N == 192 ? 128 : N;
    static constexpr double rest = (double)N * N / ((double)value * value);  // 1 for a power of two
};

// The DCT-II coefficients k of two lines a, b, over s_k DctScale<N>, from Z = FFT(v_a + i v_b):
// V_a = (Z[k] + conj Z[-k]) / 2, V_b = (Z[k] - conj Z[-k]) / 2i, X = s_k Re(w V) with w = exp(-i pi k / 2N).
template <int N>
__device__ __forceinline__ float2 dct2_pair(const float2* s, int k, float2 w)
{
    const float2 z = s[lds_pad(k)], m = s[lds_pad(k == 0 ? 0 : N - k)];
    constexpr float sc = 0.5f / DctScale<N>::value;
    const float ax = z.x + m.x, ay = z.y - m.y, bx = z.y + m.y, by = m.x - z.x;
    return make_float2((ax * w.x - ay * w.y) * sc, (bx * w.x - by * w.y) * sc);
}

// Element k of the DCT-III's transform input of two lines whose coefficients c = (a, b) stand in s:
// V_a + i V_b with V = exp(i pi k / 2N) (C_k - i C_{N-k}), C_N = 0.
template <int N>
__device__ __forceinline__ float2 dct3_pair(const float2* s, int k, float2 w)
{
    const float2 c = s[lds_pad(k)];
    const float2 n = k == 0 ? make_float2(0.f, 0.f) : s[lds_pad(N - k)];
    // (c - i n) (w.x - i w.y) for each line
    const float ar = c.x * w.x - n.x * w.y, ai = -c.x * w.y - n.x * w.x;
    const float br = c.y * w.x - n.y * w.y, bi = -c.y * w.y - n.y * w.x;
    return make_float2(ar - bi, ai + br);
}

// ---------------------------------------------------------------- 1. RHS + DCT-II along x
enum : int { RHS_WRAP = 0, RHS_SIN = 1, RHS_NONE = 2 };  // RHS of a wrapped map, or the input as it is (adjoint)

// Rows y0 .. y0 + GR - 1 of a map's right-hand side as GR / 2 complex lines in Makhoul order, by NT threads: each forms
// blocks of 4 x 4 or 4 x 2 pixels straight from the map (every difference within the block once: 2.5 or 2.75 per pixel
// instead of the 4 of the stencil).
template <int N, int RHS, int GR, int NT>
__device__ __forceinline__ void rhs_lines(const float* __restrict__ map, int y0, float2* lds)
{
    constexpr int Q = N / 4, CR = Q * GR / 4 >= NT ? 4 : 2;  // CR: rows of a thread's block
    static_assert(N % GR == 0 && GR % CR == 0, "a workgroup's rows lie in one map");
    for (int e = threadIdx.x; e < Q * (GR / CR); e += NT) {
        const int x = 4 * (e % Q), r = CR * (e / Q), y = y0 + r;
        const float* p = map + (long long)y * N + x;
        float v[CR + 2][4], l[CR], rt[CR];  // rows y - 1 .. y + CR and the pixels beside the block
#pragma unroll
        for (int k = 0; k < CR + 2; ++k) {
            if (RHS == RHS_NONE && (k == 0 || k == CR + 1)) continue;
            // rows and columns past the map are not used: the border rows and columns stand in for them
            const int yy = min(max(y + k - 1, 0), N - 1);
            const float4 q = *reinterpret_cast<const float4*>(map + (long long)yy * N + x);
            v[k][0] = q.x;
            v[k][1] = q.y;
            v[k][2] = q.z;
            v[k][3] = q.w;
        }
        float rho[CR][4];
        if constexpr (RHS == RHS_NONE) {
#pragma unroll
            for (int k = 0; k < CR; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) rho[k][i] = v[k + 1][i];
        } else {
#pragma unroll
            for (int k = 0; k < CR; ++k) {
                l[k] = p[k * N - (x > 0)];
                rt[k] = p[k * N + (x + 4 < N ? 4 : 3)];
            }
            auto step = [](float d) { return RHS == RHS_SIN ? sinf(d) : wrapdiff(d); };
            float up[4];  // differences to the row above
#pragma unroll
            for (int i = 0; i < 4; ++i) up[i] = y == 0 ? 0.f : step(v[1][i] - v[0][i]);
#pragma unroll
            for (int k = 0; k < CR; ++k) {
                const float* c = v[k + 1];
                float left = x == 0 ? 0.f : step(c[0] - l[k]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float nx = i < 3 ? c[i < 3 ? i + 1 : 3] : rt[k];
                    const float right = i == 3 && x + 4 == N ? 0.f : step(nx - c[i]);
                    const float down = k == CR - 1 && y + CR == N ? 0.f : step(v[k + 2][i] - c[i]);
                    rho[k][i] = RHS == RHS_SIN ? ((right - left) + down) - up[i] : (right - left) + (down - up[i]);
                    left = right;
                    up[i] = down;
                }
            }
        }
#pragma unroll
        for (int h = 0; h < CR / 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                lds[(r / 2 + h) * LdsSize<N>::value + lds_pad(mk_pos(x + i, N))] =
                    make_float2(rho[2 * h][i], rho[2 * h + 1][i]);
    }
}

// A workgroup's 2 GP rows lie in one map: their right-hand side as complex lines of two rows, then the transforms.
// Bound by the chain load - differences - transform of one round of workgroups. 60 maps of
// 256^2: 15.2 us (12.5 with its stages in floats), one map 4.9 us; 26.2 and 15.4 us when each thread evaluated the whole stencil for the 16 pixels
// of its transform, with a division in each difference, in 80 KiB of unrolled code.
template <int N, int RHS>
__global__ __launch_bounds__(Pair<N>::NT) void k_uw_rows_fwd(const float* __restrict__ in,
                                                            const float2* __restrict__ tw_n,
                                                            const float2* __restrict__ tw_4n, float* __restrict__ out)
{
    using PR = Pair<N>;
    constexpr int T = PR::T, GP = PR::GP, NT = PR::NT, GR = 2 * GP;
    __shared__ float2 lds[GP * LdsSize<N>::value];
    __shared__ float2 twl[LdsSize<N>::value];
    TwStager<N, NT> tws;
    tws.fetch(tw_n);
    const int g = threadIdx.x / T, t = threadIdx.x % T;
    const long long row0 = (long long)blockIdx.x * GR;
    const int y0 = (int)(row0 % N);
    const float* map = in + (row0 - y0) * N;
    float2 w[PR::J];
#pragma unroll
    for (int j = 0; j < PR::J; ++j) w[j] = tw_4n[t + j * T];
    rhs_lines<N, RHS, GR, NT>(map, y0, lds);
    tws.put(twl);
    const TwPad twp{twl};
    __syncthreads();
    float2* s = lds + g * LdsSize<N>::value;
    auto gl = [&](int n) -> float2 { return s[lds_pad(n)]; };
    auto gs = [&](int i, float2 v) { s[lds_pad(i)] = v; };
    PR::template run<-1>(t, s, wide<RHS != RHS_NONE && InDouble<N>::rhs>(twp), gl, gs);
    __syncthreads();
    float* dst = out + (row0 + 2 * g) * N;
#pragma unroll
    for (int j = 0; j < PR::J; ++j) {
        const int k = t + j * T;
        const float2 X = dct2_pair<N>(s, k, w[j]);
        dst[k] = X.x;
        dst[N + k] = X.y;
    }
}

// Reference IDCT of one line (countIDCT + inverse 2N FFT + cufft2float), dTemp = 1/sqrt(2N).
template <int N, class Put>
__device__ __forceinline__ void idct_refcompat(int t, const float* X, float2* s, const float2* tw_2n,
                                               const float2* tw_4n, Put& put)
{
    const float dT = 1.f / sqrtf(2.f * N);
    const float r2 = 1.41421356237309515f;
    auto gl = [&](int i) -> float2 {
        if (i < N) {
            const float2 w = tw_4n[i];  // (cos, -sin)(pi i / 2N)
            const float C = w.x, S = -w.y, V = X[i] * dT;
            return i == 0 ? make_float2(C * V * r2, S * V * r2) : make_float2(C * V, S * V);
        }
        const int ii = i - N;
        if (ii == 0) return make_float2(0.f, 0.f);
        const float2 w = tw_4n[ii + 1];  // angle (ii+1) pi / 2N
        const float S2 = -w.y, C2 = -w.x, V2 = X[N - ii] * dT;
        return make_float2(S2 * V2, C2 * V2);
    };
    auto gs = [&](int i, float2 v) {
        if (i < N) put(i, v.x);
    };
    Plan<2 * N>::template run<+1>(t, s, tw_2n, gl, gs);
}

// 1 / l to one rounding: the hardware reciprocal of l's float and a Newton step on what it and the float leave.
__device__ __forceinline__ float reciprocal(double l)
{
    const float hi = (float)l, lo = (float)(l - (double)hi), r = __builtin_amdgcn_rcpf(hi);
    return fmaf(r, fmaf(-lo, r, fmaf(-hi, r, 1.f)), r);
}

// Coefficients ky of columns 2c and 2c + 1 over the eigenvalue, which is formed in double. With `num` (the adjoint)
// also times the stencil's own eigenvalue.
template <int N>
__device__ __forceinline__ float2 solve_pair(float2 X, int c, int ky, bool refeig, double e0, double e1, double ey,
                                             const double* __restrict__ num)
{
    constexpr double F = DctScale<N>::rest;
    const double l0 = refeig ? F * (e0 + ey - 4.0) : -4.0 * F * (e0 + ey);
    const double l1 = refeig ? F * (e1 + ey - 4.0) : -4.0 * F * (e1 + ey);
    float2 v;
    v.x = c == 0 && ky == 0 ? 0.f : X.x * reciprocal(l0);
    v.y = X.y * reciprocal(l1);
    if (num) {
        const double n = num[ky];
        v.x *= (float)(-4.0 * (num[2 * c] + n));
        v.y *= (float)(-4.0 * (num[2 * c + 1] + n));
    }
    return v;
}

// ---------------------------------------------------------------- 2. columns: DCT-II, / lambda, DCT-III
// C pairs of neighbouring columns per workgroup, one float2 per row of a pair (C * 8 bytes of a row side by
// side). 60 maps of 256^2: 14.3 us (22.8 with one real column per transform), one map 6.4 us (9.5). The
// coefficient pairs between the two transforms are held in registers while the area is read, then
// written into it: the DCT-III reads them before its first write. For the adjoint: `num`, the exact sin^2 table,
// also multiplies by the stencil's own eigenvalue (the Laplacian of the solution, without the stencil), and
// `dc` receives each map's mean.
template <int N>
__global__ __launch_bounds__(Pair<N>::NC) void k_uw_cols(const float2* __restrict__ in, unsigned flags,
                                                        const double* __restrict__ eig,
                                                        const float2* __restrict__ tw_n,
                                                        const float2* __restrict__ tw_4n, float2* __restrict__ out,
                                                        const double* __restrict__ num, float* __restrict__ dc)
{
    using PR = Pair<N>;
    constexpr int T = PR::T, C = PR::CP, H = N / 2;
    constexpr int LS = LdsStride<N, C>::value;
    __shared__ float2 lds[C * LS];
    __shared__ float2 twl[LdsSize<N>::value];
    TwStager<N, PR::NC> tws;
    tws.fetch(tw_n);
    const int cidx = threadIdx.x % C, t = threadIdx.x / C;
    constexpr int tiles = H / C;
    const long long b = blockIdx.x / tiles;
    const int c = (blockIdx.x % tiles) * C + cidx;  // columns 2c and 2c + 1
    const float2* col = in + b * N * H + c;
    float2* s = lds + cidx * LS;
    StageRegs<N, T, PR::R0> x;
#pragma unroll
    for (int r = 0; r < PR::R0; ++r) x.v[0][r] = col[mk_src(t + r * T, N) * H];
    float2 w[PR::J];
    double ey[PR::J];
#pragma unroll
    for (int j = 0; j < PR::J; ++j) {
        w[j] = tw_4n[t + j * T];
        ey[j] = eig[t + j * T];
    }
    const double e0 = eig[2 * c], e1 = eig[2 * c + 1];
    __builtin_amdgcn_sched_barrier(0);  // every load is under way before the first wait
    tws.put(twl);
    const TwPad twp{twl};
    auto gs = [&](int i, float2 v) { s[lds_pad(i)] = v; };
    PR::template run<-1>(t, s, twp, x, gs);
    __syncthreads();
    const bool refeig = flags & F_REF_EIG;
    float2 xv[PR::J];
#pragma unroll
    for (int j = 0; j < PR::J; ++j) {
        const int ky = t + j * T;
        const float2 X = dct2_pair<N>(s, ky, w[j]);
        xv[j] = solve_pair<N>(X, c, ky, refeig, e0, e1, ey[j], num);
        if (dc && c == 0 && ky == 0) dc[b] = X.x * (float)(1.0 / DctScale<N>::rest);
    }
    __syncthreads();  // every read of the transform's output precedes the coefficients' writes
#pragma unroll
    for (int j = 0; j < PR::J; ++j) s[lds_pad(t + j * T)] = xv[j];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PR::R0; ++r) x.v[0][r] = dct3_pair<N>(s, t + r * T, w[r]);
    float2* dcol = out + b * N * H + c;
    auto gs2 = [&](int n, float2 v) { dcol[mk_src(n, N) * H] = v; };
    PR::template run<+1>(t, s, wide<InDouble<N>::cols_inv>(twp), x, gs2);
}

// The same for one column per transform with the reference's 2N-point IDCT.
template <int N, int C>
__global__ __launch_bounds__(C* Plan<2 * N>::T) void k_uw_cols_ref(const float* __restrict__ in, unsigned flags,
                                                                  const double* __restrict__ eig,
                                                                  const float2* __restrict__ tw_n,
                                                                  const float2* __restrict__ tw_2n,
                                                                  const float2* __restrict__ tw_4n,
                                                                  float* __restrict__ out)
{
    constexpr int LN = 2 * N, TL = Plan<LN>::T;  // threads per column (sized for the longer transform)
    constexpr int LS = LdsStride<LN, C>::value;
    constexpr int J = (N + TL - 1) / TL;  // coefficients per thread
    __shared__ float2 lds[C * LS];
    const int cidx = threadIdx.x % C, t = threadIdx.x / C;
    const int tiles = N / C;
    const long long b = blockIdx.x / tiles;
    const int kx = (blockIdx.x % tiles) * C + cidx;
    const float* col = in + b * N * N + kx;
    float2* s = lds + cidx * LS;
    float* X = reinterpret_cast<float*>(s);  // valid once the forward transform's output has been read
    auto gl = [&](int n) -> float2 { return make_float2(col[(long long)mk_src(n, N) * N], 0.f); };
    auto gs = [&](int i, float2 v) { s[lds_pad(i)] = v; };
    Plan<N>::template run<-1>(t, s, tw_n, gl, gs);
    __syncthreads();
    // s_kx s_ky and the rows' scale in one factor
    constexpr double u = (double)DctScale<N>::value / N, r2 = 1.41421356237309505;
    const float s0 = (float)(kx == 0 ? u : r2 * u), s1 = (float)(kx == 0 ? r2 * u : 2.0 * u);
    const bool refeig = flags & F_REF_EIG;
    float xv[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int ky = t + j * TL;
        if (t < TL && ky < N) {
            const float2 V = s[lds_pad(ky)];
            const float2 w = tw_4n[ky];
            const float Xv = (V.x * w.x - V.y * w.y) * (ky == 0 ? s0 : s1);
            const double lam = refeig ? eig[kx] + eig[ky] - 4.0 : -4.0 * (eig[kx] + eig[ky]);
            xv[j] = (kx == 0 && ky == 0) ? 0.f : Xv * __builtin_amdgcn_rcpf((float)lam);
        }
    }
    __syncthreads();  // every read of the transform's output precedes the coefficients' writes
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int ky = t + j * TL;
        if (t < TL && ky < N) X[ky] = xv[j];
    }
    __syncthreads();
    float* dcol = out + b * N * N + kx;
    auto put = [&](int y, float v) { dcol[(long long)y * N] = v; };
    idct_refcompat<N>(t, X, s, tw_2n, tw_4n, put);
}

// ---------------------------------------------------------------- 3. rows: DCT-III along x
// Congruence: the value of the class w + 2 pi Z nearest to v.
__device__ __forceinline__ float congruent(float v, float w) { return w + 2.f * kPI * rintf((v - w) / (2.f * kPI)); }

// Coefficients of a workgroup's 2 GP rows (two neighbouring rows per pair) into its LDS areas.
template <int N>
__device__ __forceinline__ void load_row_pairs(const float* __restrict__ rows, float2* lds, int ls)
{
    constexpr int Q = N / 4, E = Q * Pair<N>::GP;
    for (int e = threadIdx.x; e < E; e += Pair<N>::NT) {
        const int g = e / Q, x = 4 * (e % Q);
        const float4 a = *reinterpret_cast<const float4*>(rows + 2 * g * N + x);
        const float4 b = *reinterpret_cast<const float4*>(rows + (2 * g + 1) * N + x);
        float2* s = lds + g * ls;
        s[lds_pad(x)] = make_float2(a.x, b.x);
        s[lds_pad(x + 1)] = make_float2(a.y, b.y);
        s[lds_pad(x + 2)] = make_float2(a.z, b.z);
        s[lds_pad(x + 3)] = make_float2(a.w, b.w);
    }
}

template <int N>
__global__ __launch_bounds__(Pair<N>::NT) void k_uw_rows_inv(const float* __restrict__ in, const float* __restrict__ wrapped,
                                                            const float2* __restrict__ tw_n,
                                                            const float2* __restrict__ tw_4n, float* __restrict__ out)
{
    using PR = Pair<N>;
    constexpr int T = PR::T, GP = PR::GP, Q = N / 4, LS = LdsSize<N>::value;
    __shared__ float2 lds[GP * LS];
    __shared__ float2 twl[LS];
    TwStager<N, PR::NT> tws;
    tws.fetch(tw_n);
    const int g = threadIdx.x / T, t = threadIdx.x % T;
    const long long base = (long long)blockIdx.x * 2 * GP * N;
    float2 w[PR::J];
#pragma unroll
    for (int j = 0; j < PR::J; ++j) w[j] = tw_4n[t + j * T];
    load_row_pairs<N>(in + base, lds, LS);
    tws.put(twl);
    const TwPad twp{twl};
    __syncthreads();
    float2* s = lds + g * LS;
    StageRegs<N, T, PR::R0> x;
#pragma unroll
    for (int r = 0; r < PR::R0; ++r) x.v[0][r] = dct3_pair<N>(s, t + r * T, w[r]);
    auto gs = [&](int n, float2 v) { s[lds_pad(mk_src(n, N))] = v; };
    PR::template run<+1>(t, s, wide<InDouble<N>::rows_inv>(twp), x, gs);
    __syncthreads();
    for (int e = threadIdx.x; e < Q * GP; e += PR::NT) {
        const int gg = e / Q, c = 4 * (e % Q);
        const float2* p = lds + gg * LS;
        const float2 v0 = p[lds_pad(c)], v1 = p[lds_pad(c + 1)], v2 = p[lds_pad(c + 2)], v3 = p[lds_pad(c + 3)];
        const long long o = base + 2 * gg * N + c;
        float4 a = make_float4(v0.x, v1.x, v2.x, v3.x), b = make_float4(v0.y, v1.y, v2.y, v3.y);
        if (wrapped) {
            const float4 wa = *reinterpret_cast<const float4*>(wrapped + o);
            const float4 wb = *reinterpret_cast<const float4*>(wrapped + o + N);
            a = make_float4(congruent(a.x, wa.x), congruent(a.y, wa.y), congruent(a.z, wa.z), congruent(a.w, wa.w));
            b = make_float4(congruent(b.x, wb.x), congruent(b.y, wb.y), congruent(b.z, wb.z), congruent(b.w, wb.w));
        }
        *reinterpret_cast<float4*>(out + o) = a;
        *reinterpret_cast<float4*>(out + o + N) = b;
    }
}

// The same for one row per transform with the reference's 2N-point IDCT.
template <int N, int G>
__global__ __launch_bounds__(G* Plan<2 * N>::T) void k_uw_rows_inv_ref(const float* __restrict__ in, int batch,
                                                                      const float* __restrict__ wrapped,
                                                                      const float2* __restrict__ tw_2n,
                                                                      const float2* __restrict__ tw_4n,
                                                                      float* __restrict__ out)
{
    constexpr int LN = 2 * N, TL = Plan<LN>::T;
    __shared__ float2 lds[G * LdsSize<LN>::value];
    const int g = threadIdx.x / TL, t = threadIdx.x % TL;
    const long long row = (long long)blockIdx.x * G + g;
    const bool valid = row < (long long)batch * N;
    const long long r = valid ? row : 0;
    auto put = [&](int x, float v) {
        if (valid) out[r * N + x] = wrapped ? congruent(v, wrapped[r * N + x]) : v;
    };
    idct_refcompat<N>(t, in + r * N, lds + g * LdsSize<LN>::value, tw_2n, tw_4n, put);
}

// Rows of the last unwrapping pass fused with the row pass of the Rytov spectrum (k_rytov_rows of the
// reconstruction module, same transform and twiddles): the DCT-III's two rows, after the congruence step, go to
// the unwrapped map (when wanted) and stay in LDS as floats, one row in each of the pair's two areas (the
// DCT-III's last stage writes only after its barrier), where the forward row transforms of u = logamp + i phi
// read them. Row spectra: P[r][k].
template <int N>
__global__ __launch_bounds__(Pair<N>::NT) void k_uw_rows_inv_rytov(const float* __restrict__ in,
                                                                  const float* __restrict__ wrapped,
                                                                  const float* __restrict__ la,
                                                                  const float2* __restrict__ tw_n,
                                                                  const float2* __restrict__ tw_4n,
                                                                  float* __restrict__ out, float2* __restrict__ P)
{
    using PR = Pair<N>;
    constexpr int T = PR::T, GP = PR::GP, LS = LdsSize<N>::value;
    __shared__ float2 lds[2 * GP * LS];
    const int g = threadIdx.x / T, t = threadIdx.x % T;
    const long long base = (long long)blockIdx.x * 2 * GP * N;
    float2 w[PR::J];
#pragma unroll
    for (int j = 0; j < PR::J; ++j) w[j] = tw_4n[t + j * T];
    load_row_pairs<N>(in + base, lds, 2 * LS);
    __syncthreads();
    float2* s = lds + g * 2 * LS;
    StageRegs<N, T, PR::R0> x;
#pragma unroll
    for (int r = 0; r < PR::R0; ++r) x.v[0][r] = dct3_pair<N>(s, t + r * T, w[r]);
    const long long ra = base + 2 * g * N;
    float* pa = reinterpret_cast<float*>(s);
    float* pb = reinterpret_cast<float*>(s + LS);
    auto gs = [&](int n, float2 v) {
        const int c = mk_src(n, N);
        float a = v.x, b = v.y;
        if (wrapped) {
            a = congruent(a, wrapped[ra + c]);
            b = congruent(b, wrapped[ra + N + c]);
        }
        pa[c] = a;
        pb[c] = b;
        if (out) {
            out[ra + c] = a;
            out[ra + N + c] = b;
        }
    };
    PR::template run<+1>(t, s, wide<InDouble<N>::rows_inv>(TwTable{tw_n}), x, gs);
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const float* ph = h ? pb : pa;
        const float* l = la + ra + h * N;
        float2* dst = P + ra + h * N;
        auto gl = [&](int c) -> float2 { return make_float2(l[c], ph[c]); };
        auto gs2 = [&](int k, float2 v) { dst[k] = v; };
        PR::template run<-1>(t, s + h * LS, tw_n, gl, gs2);
    }
}

// ---------------------------------------------------------------- the three passes in one workgroup
// A map of 32^2 or 64^2 fits a workgroup: all its row pairs at once, the coefficients as a matrix in LDS, all its column
// pairs, the row pairs again; the same operations in the same order as the three kernels, and the same bits. For a few
// maps the three are launches and latency, for many they write and read the coefficients: 1 map of 64^2 12.4 us in
// three launches, 8.3 in one; 256 17.0 and 9.3; 4096 81 and 62; 32^2 11.8 and 6.5, 30 and 23. One 256^2 hologram pair to an
// unwrapped 64^2 map 28.0 and 21.0.
template <int N, int RHS>
__global__ __launch_bounds__(N / 2 * Pair<N>::T) void k_uw_map(const float* __restrict__ in, const float* __restrict__ wrapped,
                                                            unsigned flags, const double* __restrict__ eig,
                                                            const float2* __restrict__ tw_n,
                                                            const float2* __restrict__ tw_4n, float* __restrict__ out,
                                                            const double* __restrict__ num, float* __restrict__ dc)
{
    using PR = Pair<N>;
    constexpr int T = PR::T, NT = N / 2 * T, LS = LdsSize<N>::value, MS = N + 2, Q = N / 4;
    static_assert(64 % T == 0, "a pair's threads lie in one wave");
    __shared__ float2 lds[N / 2 * LS];
    __shared__ float2 twl[LS];
    __shared__ __align__(8) float mat[N * MS];
    TwStager<N, NT> tws;
    tws.fetch(tw_n);
    const int g = threadIdx.x / T, t = threadIdx.x % T;  // a pair of rows (2g, 2g + 1) or of columns
    const long long base = (long long)blockIdx.x * N * N;
    float2 w[PR::J];
    double ey[PR::J];
#pragma unroll
    for (int j = 0; j < PR::J; ++j) {
        w[j] = tw_4n[t + j * T];
        ey[j] = eig[t + j * T];
    }
    const double e0 = eig[2 * g], e1 = eig[2 * g + 1];
    rhs_lines<N, RHS, N, NT>(in + base, 0, lds);
    tws.put(twl);
    const TwWave twp{{twl}};
    __syncthreads();
    float2* s = lds + g * LS;
    auto gl = [&](int n) -> float2 { return s[lds_pad(n)]; };
    auto gs = [&](int i, float2 v) { s[lds_pad(i)] = v; };
    PR::template run<-1>(t, s, twp, gl, gs);
    stage_sync(twp);
#pragma unroll
    for (int j = 0; j < PR::J; ++j) {
        const int k = t + j * T;
        const float2 X = dct2_pair<N>(s, k, w[j]);
        mat[2 * g * MS + k] = X.x;
        mat[(2 * g + 1) * MS + k] = X.y;
    }
    __syncthreads();
    StageRegs<N, T, PR::R0> x;
    float2* col = reinterpret_cast<float2*>(mat) + g;  // (a column pair's float2 of row y at y MS / 2)
#pragma unroll
    for (int r = 0; r < PR::R0; ++r) x.v[0][r] = col[mk_src(t + r * T, N) * (MS / 2)];
    PR::template run<-1>(t, s, twp, x, gs);
    stage_sync(twp);
    const bool refeig = flags & F_REF_EIG;
    float2 xv[PR::J];
#pragma unroll
    for (int j = 0; j < PR::J; ++j) {
        const int ky = t + j * T;
        const float2 X = dct2_pair<N>(s, ky, w[j]);
        xv[j] = solve_pair<N>(X, g, ky, refeig, e0, e1, ey[j], num);
        if (dc && g == 0 && ky == 0) dc[blockIdx.x] = X.x * (float)(1.0 / DctScale<N>::rest);
    }
    stage_sync(twp);
#pragma unroll
    for (int j = 0; j < PR::J; ++j) s[lds_pad(t + j * T)] = xv[j];
    stage_sync(twp);
#pragma unroll
    for (int r = 0; r < PR::R0; ++r) x.v[0][r] = dct3_pair<N>(s, t + r * T, w[r]);
    auto gc = [&](int n, float2 v) { col[mk_src(n, N) * (MS / 2)] = v; };
    PR::template run<+1>(t, s, twp, x, gc);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PR::J; ++j) {
        const int k = t + j * T;
        s[lds_pad(k)] = make_float2(mat[2 * g * MS + k], mat[(2 * g + 1) * MS + k]);
    }
    stage_sync(twp);
#pragma unroll
    for (int r = 0; r < PR::R0; ++r) x.v[0][r] = dct3_pair<N>(s, t + r * T, w[r]);
    auto gr = [&](int n, float2 v) { s[lds_pad(mk_src(n, N))] = v; };
    PR::template run<+1>(t, s, twp, x, gr);
    stage_sync(twp);
    for (int e = t; e < Q; e += T) {  // both rows of the pair, four pixels at a time
        const int c = 4 * e;
        const float2 v0 = s[lds_pad(c)], v1 = s[lds_pad(c + 1)], v2 = s[lds_pad(c + 2)], v3 = s[lds_pad(c + 3)];
        const long long o = base + 2 * g * N + c;
        float4 a = make_float4(v0.x, v1.x, v2.x, v3.x), b = make_float4(v0.y, v1.y, v2.y, v3.y);
        if (wrapped) {
            const float4 wa = *reinterpret_cast<const float4*>(wrapped + o);
            const float4 wb = *reinterpret_cast<const float4*>(wrapped + o + N);
            a = make_float4(congruent(a.x, wa.x), congruent(a.y, wa.y), congruent(a.z, wa.z), congruent(a.w, wa.w));
            b = make_float4(congruent(b.x, wb.x), congruent(b.y, wb.y), congruent(b.z, wb.z), congruent(b.w, wb.w));
        }
        *reinterpret_cast<float4*>(out + o) = a;
        *reinterpret_cast<float4*>(out + o + N) = b;
    }
}

// Adjoint of the right-hand side at a solution v = P g: the zero-flux stencil sum_nbr w_pn (v_n - v_p) with
// weights cos(phi_n - phi_p). With `g` and `mean` (P exact) the unweighted part is known, as the stencil undoes
// P up to the mean, and only sum (cos - 1) (v_n - v_p) is taken from v: v is smooth and large where g is rough,
// so its differences carry its rounding, here times 1 - cos. Four pixels of a row per thread.
__global__ __launch_bounds__(256) void k_uw_stencil(const float* __restrict__ v, const float* __restrict__ phi, int N,
                                                    long long quads, const float* g, const float* __restrict__ mean,
                                                    float* out)  // out may be g
{
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= quads) return;
    const int Q = N / 4;
    const long long row = e / Q, b = row / N;
    const int x = 4 * (int)(e - row * Q), y = (int)(row - b * N);
    const long long o = row * N + x;
    auto quad = [&](const float* m, long long k, float (&q)[4]) {
        const float4 f = *reinterpret_cast<const float4*>(m + k);
        q[0] = f.x;
        q[1] = f.y;
        q[2] = f.z;
        q[3] = f.w;
    };
    // past the border a pixel stands in for its neighbour: no difference, whatever the weight
    const long long ou = o - (y > 0 ? N : 0), od = o + (y < N - 1 ? N : 0);
    float vc[4], vu[4], vd[4], pc[4], pu[4], pd[4];
    quad(v, o, vc);
    quad(v, ou, vu);
    quad(v, od, vd);
    quad(phi, o, pc);
    quad(phi, ou, pu);
    quad(phi, od, pd);
    const long long ol = o - (x > 0), orr = o + (x + 4 < N ? 4 : 3);
    const float one = g ? 1.f : 0.f;
    auto flux = [&](float dp, float dv) { return (cosf(dp) - one) * dv; };
    float left = flux(pc[0] - phi[ol], vc[0] - v[ol]);  // flux from the left neighbour into pixel 0
    float r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float pn = i < 3 ? pc[i < 3 ? i + 1 : 3] : phi[orr], vn = i < 3 ? vc[i < 3 ? i + 1 : 3] : v[orr];
        const float right = flux(pn - pc[i], vn - vc[i]);
        r[i] = ((right - left) + flux(pd[i] - pc[i], vd[i] - vc[i])) + flux(pu[i] - pc[i], vu[i] - vc[i]);
        left = right;
    }
    if (g) {
        const float m = mean[b];
        float gc[4];
        quad(g, o, gc);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] += gc[i] - m;
    }
    *reinterpret_cast<float4*>(out + o) = make_float4(r[0], r[1], r[2], r[3]);
}

// Each map minus its mean (the sums in double), one workgroup per map of n values.
__global__ __launch_bounds__(1024) void k_uw_sub_mean(const float* in, float* out, int n)  // out may be in
{
    __shared__ double red[16];
    const float* m = in + (size_t)blockIdx.x * n;
    float* o = out + (size_t)blockIdx.x * n;
    double sum = 0.0;
    for (int i = 4 * threadIdx.x; i < n; i += 4096) {
        const float4 f = *reinterpret_cast<const float4*>(m + i);
        sum += ((double)f.x + f.y) + ((double)f.z + f.w);
    }
    for (int w = 32; w > 0; w >>= 1) sum += __shfl_xor(sum, w);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < 16; ++w) tot += red[w];
    const float mean = (float)(tot / n);
    for (int i = 4 * threadIdx.x; i < n; i += 4096) {
        const float4 f = *reinterpret_cast<const float4*>(m + i);
        *reinterpret_cast<float4*>(o + i) = make_float4(f.x - mean, f.y - mean, f.z - mean, f.w - mean);
    }
}

// ---------------------------------------------------------------- FastUnwrapping's map conventions
// One workgroup per map: minimum (and maximum) of its n values, left in mn[0] (mx[0]) for every thread.
template <int T>
__device__ __forceinline__ void map_min_max(const float* __restrict__ m, int n, float* red, float& mn, float& mx)
{
    float lo = INFINITY, hi = -INFINITY;
    for (int i = threadIdx.x; i < n; i += T) {
        const float v = m[i];
        lo = fminf(lo, v);
        hi = fmaxf(hi, v);
    }
    red[threadIdx.x] = lo;
    red[T + threadIdx.x] = hi;
    __syncthreads();
    for (int w = T / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            red[threadIdx.x] = fminf(red[threadIdx.x], red[threadIdx.x + w]);
            red[T + threadIdx.x] = fmaxf(red[T + threadIdx.x], red[T + threadIdx.x + w]);
        }
        __syncthreads();
    }
    mn = red[0];
    mx = red[T];
}

// PhaseNormalize + RescalePhaseMap (FastUnwrapping.cu:119-142): each map rescaled to
// 2 pi (x - min) / (max - min), evaluated in double as the reference's double-precision M_PI promotes it.
__global__ __launch_bounds__(256) void k_uw_normalize(const float* __restrict__ in, float* __restrict__ out, int n)
{
    __shared__ float red[512];
    const float* m = in + (size_t)blockIdx.x * n;
    float* o = out + (size_t)blockIdx.x * n;
    float mn, mx;
    map_min_max<256>(m, n, red, mn, mx);
    const double span = (double)(mx - mn);
    for (int i = threadIdx.x; i < n; i += 256) o[i] = (float)(2.0 * M_PI * (double)(m[i] - mn) / span);
}

// subtractMin + PhaseMapSubMin (FastUnwrapping.cu:346-369): each map minus its own minimum, in place.
__global__ __launch_bounds__(256) void k_uw_sub_min(float* __restrict__ x, int n)
{
    __shared__ float red[512];
    float* m = x + (size_t)blockIdx.x * n;
    float mn, mx;
    map_min_max<256>(m, n, red, mn, mx);
    __syncthreads();  // every thread has read the minimum before any value changes
    for (int i = threadIdx.x; i < n; i += 256) m[i] -= mn;
}

// ---------------------------------------------------------------- host side
static const double* eig_table(Ctx& c, int N, bool refcompat, bool existing = false)
{
    const std::string name = std::string(refcompat ? "uw.eigref." : "uw.eig.") + std::to_string(N);
    auto it = c.scratch.find(name);
    if (it != c.scratch.end() && it->second.ptr) return (const double*)it->second.ptr;
    CTDM_REQUIRE(!existing, "unwrap: eigenvalue table missing (it is built when the context is created)");
    std::vector<double> h(N);
    for (int k = 0; k < N; ++k) {
        if (refcompat)
            h[k] = 2.0 * std::cos(4.0 * M_PI * k / (4.0 * N - 1));
        else {
            const double sv = std::sin(M_PI * k / (2.0 * N));
            h[k] = sv * sv;
        }
    }
    double* d = (double*)c.buf(name, sizeof(double) * N, true);  // one table for both lanes
    CTDM_HIP(hipMemcpy(d, h.data(), sizeof(double) * N, hipMemcpyHostToDevice));
    return d;
}

template <int N>
static void run_rows_fwd(Ctx& c, const float* in, int batch, int rhs, float* out)
{
    using PR = Pair<N>;
    const dim3 grid((unsigned)((long long)batch * N / (2 * PR::GP))), block(PR::NT);
    const float2 *tw = c.tw(N), *tw4 = c.tw(4 * N);
    if (rhs == RHS_WRAP)
        hipLaunchKernelGGL((k_uw_rows_fwd<N, RHS_WRAP>), grid, block, 0, c.stream, in, tw, tw4, out);
    else if (rhs == RHS_SIN)
        hipLaunchKernelGGL((k_uw_rows_fwd<N, RHS_SIN>), grid, block, 0, c.stream, in, tw, tw4, out);
    else if constexpr (N > 64)
        hipLaunchKernelGGL((k_uw_rows_fwd<N, RHS_NONE>), grid, block, 0, c.stream, in, tw, tw4, out);
    else
        fail(CTDM_EUNSUPPORTED, "a right-hand side given as it is takes the one-workgroup solve at this size");
    CTDM_CHECK_LAUNCH("k_uw_rows_fwd");
}

template <int N>
static void run_cols(Ctx& c, const float* in, int batch, unsigned flags, float* out, bool existing,
                     const double* num = nullptr, float* dc = nullptr)
{
    const double* eig = eig_table(c, N, flags & F_REF_EIG, existing);
    if (flags & F_REF_IDCT) {
        constexpr int C = (256 / Plan<2 * N>::T) < N ? (256 / Plan<2 * N>::T) : N;
        hipLaunchKernelGGL((k_uw_cols_ref<N, C>), dim3(batch * (N / C)), dim3(C * Plan<2 * N>::T), 0, c.stream, in,
                           flags, eig, c.tw(N), c.tw(2 * N), c.tw(4 * N), out);
    } else {
        using PR = Pair<N>;
        hipLaunchKernelGGL((k_uw_cols<N>), dim3(batch * (N / 2 / PR::CP)), dim3(PR::NC), 0, c.stream,
                           (const float2*)in, flags, eig, c.tw(N), c.tw(4 * N), (float2*)out, num, dc);
    }
    CTDM_CHECK_LAUNCH("k_uw_cols");
}

// wrapped: the map to be congruent to, or null.
template <int N>
static void run_rows_inv(Ctx& c, const float* in, int batch, unsigned flags, const float* wrapped, float* out)
{
    if (!(flags & F_CONGRUENT)) wrapped = nullptr;
    if (flags & F_REF_IDCT) {
        constexpr int G = 256 / Plan<2 * N>::T;
        hipLaunchKernelGGL((k_uw_rows_inv_ref<N, G>), dim3(grid1d((long long)batch * N, G)), dim3(G * Plan<2 * N>::T),
                           0, c.stream, in, batch, wrapped, c.tw(2 * N), c.tw(4 * N), out);
    } else if constexpr (N > 64) {  // (smaller maps: k_uw_map)
        using PR = Pair<N>;
        hipLaunchKernelGGL((k_uw_rows_inv<N>), dim3((unsigned)((long long)batch * N / (2 * PR::GP))), dim3(PR::NT), 0,
                           c.stream, in, wrapped, c.tw(N), c.tw(4 * N), out);
    } else {
        fail(CTDM_EUNSUPPORTED, "rows of this size are solved with the whole map");
    }
    CTDM_CHECK_LAUNCH("k_uw_rows_inv");
}

// Intermediate spectra of one solve: context scratch, or (allocation-free entry point) the fixed
// device array. `existing` also forbids building a missing table.
struct Work {
    float* D1 = nullptr;
    float* D2 = nullptr;
    bool existing = false;
    const double* num = nullptr;  // adjoint only (k_uw_cols)
    float* dc = nullptr;
};

// Whole solve for one size: mode 0 (wrapped input) or 1 (raw input, adjoint).
template <int N>
static void solve(Ctx& c, const float* in, int batch, unsigned flags, int mode, const float* wrapped,
                  float* out, Work w)
{
    if constexpr (N <= 64) {
        if (!(flags & F_REF_IDCT)) {  // (the reference's IDCT has its own kernels)
            const double* eig = eig_table(c, N, flags & F_REF_EIG, w.existing);
            const dim3 grid(batch), block(N / 2 * Pair<N>::T);
            const float* cong = flags & F_CONGRUENT ? wrapped : nullptr;
            const float2 *tw = c.tw(N), *tw4 = c.tw(4 * N);
            if (mode == 1)
                hipLaunchKernelGGL((k_uw_map<N, RHS_NONE>), grid, block, 0, c.stream, in, cong, flags, eig, tw, tw4, out,
                                   w.num, w.dc);
            else if (flags & F_SINCOS)
                hipLaunchKernelGGL((k_uw_map<N, RHS_SIN>), grid, block, 0, c.stream, in, cong, flags, eig, tw, tw4, out,
                                   w.num, w.dc);
            else
                hipLaunchKernelGGL((k_uw_map<N, RHS_WRAP>), grid, block, 0, c.stream, in, cong, flags, eig, tw, tw4, out,
                                   w.num, w.dc);
            CTDM_CHECK_LAUNCH("k_uw_map");
            return;
        }
    }
    if (!w.D1) {
        w.D1 = (float*)c.buf("uw.D1", sizeof(float) * (size_t)batch * N * N);
        w.D2 = (float*)c.buf("uw.D2", sizeof(float) * (size_t)batch * N * N);
    }
    run_rows_fwd<N>(c, in, batch, mode == 1 ? RHS_NONE : (flags & F_SINCOS ? RHS_SIN : RHS_WRAP), w.D1);
    run_cols<N>(c, w.D1, batch, flags, w.D2, w.existing, w.num, w.dc);
    run_rows_inv<N>(c, w.D2, batch, flags, wrapped, out);
}

static void solve_any(Ctx& c, const float* in, int batch, int N, unsigned flags, int mode,
                      const float* wrapped, float* out, Work w = Work{})
{
    switch (N) {
    case 32: solve<32>(c, in, batch, flags, mode, wrapped, out, w); break;
    case 64: solve<64>(c, in, batch, flags, mode, wrapped, out, w); break;
    case 128: solve<128>(c, in, batch, flags, mode, wrapped, out, w); break;
    case 192: solve<192>(c, in, batch, flags, mode, wrapped, out, w); break;
    case 256: solve<256>(c, in, batch, flags, mode, wrapped, out, w); break;
    default: fail(CTDM_EUNSUPPORTED, "unwrap size " + std::to_string(N) + " has no kernel");
    }
}

// ---------------------------------------------------------------- allocation-free entry point
// The two intermediate spectra of ctdm_unwrap_dct_noalloc, CTDM_NOALLOC_MAX_ELEMS floats each, in one
// file-scope device array. Every device the library runs on holds its own copy until the process ends.
// In host code `scratch` is a host-side stand-in: kernels get the per-device address that
// hipGetSymbolAddress returns (noalloc_setup), never the array's name.
static __device__ __align__(256) float scratch[2 * (size_t)CTDM_NOALLOC_MAX_ELEMS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

void noalloc_setup(Ctx& c)
{
    CTDM_REQUIRE(c.device >= 0 && c.device < kMaxDevices, "device ordinal out of range");
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        if (!g_scratch_ptr[c.device]) {  // once per device, with that device current
            float* ptr = nullptr;
            CTDM_HIP(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
            CTDM_REQUIRE(ptr != nullptr, "scratch symbol has no device address");
            g_scratch_ptr[c.device] = ptr;
        }
        c.noalloc_scratch = g_scratch_ptr[c.device];
    }
    // Every table the unwrap kernels read, built now so that the allocation-free call finds them.
    for (int N : {32, 64, 128, 192, 256}) {
        eig_table(c, N, false);
        eig_table(c, N, true);
        c.tw(N);
        c.tw(2 * N);
        c.tw(4 * N);
    }
}

void unwrap_dct_noalloc(Ctx& c, const float* wrapped, float* unwrapped, int batch, int M, unsigned flags)
{
    CTDM_REQUIRE(wrapped && unwrapped, "unwrap_dct_noalloc: null pointer");
    CTDM_REQUIRE(batch >= 0 && M > 0, "unwrap_dct_noalloc: bad size");
    CTDM_REQUIRE(wrapped != unwrapped, "unwrap_dct_noalloc: in-place call not supported");
    CTDM_REQUIRE((flags & ~0xfu) == 0, "unwrap_dct_noalloc: unknown flag");
    CTDM_REQUIRE((size_t)batch * M * M <= (size_t)CTDM_NOALLOC_MAX_ELEMS,
                 "unwrap_dct_noalloc: batch * M * M = " + std::to_string((size_t)batch * M * M) +
                     " exceeds the fixed scratch of " + std::to_string((size_t)CTDM_NOALLOC_MAX_ELEMS) +
                     " elements");
    CTDM_REQUIRE(c.noalloc_scratch, "unwrap_dct_noalloc: scratch address not set up");
    if (batch == 0) return;
    Work w;
    w.D1 = c.noalloc_scratch;
    w.D2 = c.noalloc_scratch + (size_t)CTDM_NOALLOC_MAX_ELEMS;
    w.existing = true;
    solve_any(c, wrapped, batch, M, flags, 0, wrapped, unwrapped, w);
}

// With CTDM_UNWRAP_REFCOMPAT_FAST the maps are first rescaled to [0, 2 pi] (into scratch `name`) and
// the result of each map is shifted to a zero minimum, FastUnwrapping's conventions.
static const float* normalized_input(Ctx& c, const float* wrapped, int batch, int M, const char* name)
{
    float* norm = (float*)c.buf(name, sizeof(float) * (size_t)batch * M * M);
    hipLaunchKernelGGL(k_uw_normalize, dim3(batch), dim3(256), 0, c.stream, wrapped, norm, M * M);
    CTDM_CHECK_LAUNCH("k_uw_normalize");
    return norm;
}

static void subtract_min(Ctx& c, float* out, int batch, int M)
{
    hipLaunchKernelGGL(k_uw_sub_min, dim3(batch), dim3(256), 0, c.stream, out, M * M);
    CTDM_CHECK_LAUNCH("k_uw_sub_min");
}

void unwrap_dct_batched(Ctx& c, const float* wrapped, float* unwrapped, int batch, int M,
                        unsigned flags)
{
    CTDM_REQUIRE(wrapped && unwrapped, "unwrap_dct: null pointer");
    CTDM_REQUIRE(batch >= 0 && M > 0, "unwrap_dct: bad size");
    CTDM_REQUIRE(wrapped != unwrapped, "unwrap_dct: in-place call not supported");
    CTDM_REQUIRE((flags & ~F_ALL) == 0, "unwrap_dct: unknown flag");
    if (batch == 0) return;
    if (flags & F_REF_FAST) {
        const float* norm = normalized_input(c, wrapped, batch, M, "uw.norm");
        solve_any(c, norm, batch, M, flags & ~F_REF_FAST, 0, norm, unwrapped);
        subtract_min(c, unwrapped, batch, M);
        return;
    }
    solve_any(c, wrapped, batch, M, flags, 0, wrapped, unwrapped);
}

template <int N>
static void uw_rytov(Ctx& c, const float* wrapped, float* unwrapped, const float* logamp, int batch, unsigned flags,
                     float2* P)
{
    using PR = Pair<N>;
    float* D1 = (float*)c.buf("uw.D1", sizeof(float) * (size_t)batch * N * N);
    float* D2 = (float*)c.buf("uw.D2", sizeof(float) * (size_t)batch * N * N);
    run_rows_fwd<N>(c, wrapped, batch, flags & F_SINCOS ? RHS_SIN : RHS_WRAP, D1);
    run_cols<N>(c, D1, batch, flags, D2, false);
    hipLaunchKernelGGL((k_uw_rows_inv_rytov<N>), dim3((unsigned)((long long)batch * N / (2 * PR::GP))), dim3(PR::NT),
                       0, c.stream, D2, flags & F_CONGRUENT ? wrapped : nullptr, logamp, c.tw(N), c.tw(4 * N),
                       unwrapped, P);
    CTDM_CHECK_LAUNCH("k_uw_rows_inv_rytov");
}

void unwrap_dct_rytov_rows(Ctx& c, const float* wrapped, float* unwrapped, const float* logamp, int batch, int M,
                           unsigned flags, float2* P)
{
    CTDM_REQUIRE(wrapped && logamp && P, "unwrap_dct_rytov_rows: null pointer");
    CTDM_REQUIRE(batch >= 0 && M > 0, "unwrap_dct_rytov_rows: bad size");
    CTDM_REQUIRE(wrapped != unwrapped, "unwrap_dct_rytov_rows: in-place call not supported");
    CTDM_REQUIRE((flags & ~F_ALL) == 0 && !(flags & (F_REF_FAST | F_REF_IDCT)),
                 "unwrap_dct_rytov_rows: unsupported flag");
    if (batch == 0) return;
    switch (M) {
    case 32: uw_rytov<32>(c, wrapped, unwrapped, logamp, batch, flags, P); break;
    case 64: uw_rytov<64>(c, wrapped, unwrapped, logamp, batch, flags, P); break;
    case 128: uw_rytov<128>(c, wrapped, unwrapped, logamp, batch, flags, P); break;
    case 192: uw_rytov<192>(c, wrapped, unwrapped, logamp, batch, flags, P); break;
    case 256: uw_rytov<256>(c, wrapped, unwrapped, logamp, batch, flags, P); break;
    default: fail(CTDM_EUNSUPPORTED, "unwrap size " + std::to_string(M) + " has no kernel");
    }
}

void unwrap_dct_adjoint(Ctx& c, const float* wrapped, const float* g_out, float* g_in, int batch,
                        int M, unsigned flags)
{
    CTDM_REQUIRE(wrapped && g_out && g_in, "unwrap_dct_adjoint: null pointer");
    CTDM_REQUIRE(!(flags & (F_REF_IDCT | F_REF_FAST)),
                 "unwrap_dct_adjoint: the reference IDCT and FastUnwrapping's rescaling have no adjoint here");
    if (batch == 0) return;
    const size_t n = (size_t)batch * M * M;
    if (flags & F_CONGRUENT) {  // output = wrapped + 2 pi k with k piecewise constant: J = I
        CTDM_HIP(hipMemcpyAsync(g_in, g_out, sizeof(float) * n, hipMemcpyDeviceToDevice, c.stream));
        return;
    }
    // J = P D with P the (symmetric) Poisson operator and D the (symmetric) linearised RHS stencil, so
    // J^T g = D (P g). Without SINCOS D is the Laplacian, which the DCT diagonalises: with the exact eigenvalues
    // D P is the identity but for the mean, with the reference's it is the ratio of the two eigenvalues. With
    // SINCOS the stencil's weights are cos of the phase differences.
    CTDM_REQUIRE(batch > 0, "unwrap_dct_adjoint: negative batch");
    if (!(M == 32 || M == 64 || M == 128 || M == 192 || M == 256))
        fail(CTDM_EUNSUPPORTED, "unwrap size " + std::to_string(M) + " has no kernel");
    const bool refeig = flags & F_REF_EIG;
    if (!(flags & F_SINCOS)) {
        if (!refeig) {
            hipLaunchKernelGGL(k_uw_sub_mean, dim3(batch), dim3(1024), 0, c.stream, g_out, g_in, M * M);
            CTDM_CHECK_LAUNCH("k_uw_sub_mean");
            return;
        }
        Work w;
        w.num = eig_table(c, M, false);
        solve_any(c, g_out, batch, M, F_REF_EIG, 1, nullptr, g_in, w);
        return;
    }
    float* tmp = (float*)c.buf("uw.adj", sizeof(float) * n);
    Work w;
    if (!refeig) w.dc = (float*)c.buf("uw.dc", sizeof(float) * (size_t)batch);
    solve_any(c, g_out, batch, M, flags & F_REF_EIG, 1, nullptr, tmp, w);
    const long long quads = (long long)n / 4;
    hipLaunchKernelGGL(k_uw_stencil, dim3(grid1d(quads, 256)), dim3(256), 0, c.stream, tmp, wrapped, M, quads,
                       refeig ? nullptr : g_out, (const float*)w.dc, g_in);
    CTDM_CHECK_LAUNCH("k_uw_stencil");
}

// ---------------------------------------------------------------- plain (reference-structured) path
// NumericDerivative1 (DCT_Unwrapping.cu:360-392)
__global__ void k_numeric_derivative(float* __restrict__ ox, float* __restrict__ oy, const float* __restrict__ in,
                                     int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= N || j >= N) return;
    const int k = i + N * j;
    const float tx = (i == N - 1) ? -in[k] : in[k + 1] - in[k];
    const float ty = (j == N - 1) ? -in[k] : in[k + N] - in[k];
    ox[k] = wrapdiff(tx);
    oy[k] = wrapdiff(ty);
}

// SumDerivative (DCT_Unwrapping.cu:394-417)
__global__ void k_sum_derivative(float* __restrict__ o, const float* __restrict__ ox, const float* __restrict__ oy,
                                 int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= N || j >= N) return;
    const int k = i + N * j;
    const float c1 = (i == N - 1) ? 0.f : ox[k];
    const float c2 = (i == 0) ? 0.f : ox[k - 1];
    const float c3 = (j == N - 1) ? 0.f : oy[k];
    const float c4 = (j == 0) ? 0.f : oy[k - N];
    o[k] = (c1 - c2) + (c3 - c4);
}

// sin/cos RHS for the plain path: one stencil kernel.
__global__ void k_sincos_rhs(float* __restrict__ o, const float* __restrict__ in, int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= N || j >= N) return;
    o[i + N * j] = sin_rhs_at(in, N, i, j);
}

// float2cufft (DCT_Unwrapping.cu:144-162): row mirror to length 2N.
__global__ void k_mirror(float2* __restrict__ o, const float* __restrict__ in, int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= N || j >= N) return;
    const float v = in[i + N * j];
    o[i + 2 * N * j] = make_float2(v, 0.f);
    o[(2 * N - 1 - i) + 2 * N * j] = make_float2(v, 0.f);
}

// countFDCT (DCT_Unwrapping.cu:202-216)
__global__ void k_count_fdct(float* __restrict__ o, const float2* __restrict__ in, int N, float dT)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= N || j >= N) return;
    const float2 v = in[i + 2 * N * j];
    const float a = (float)i * kPI / (2.f * N);
    o[i + N * j] = (i == 0) ? v.x * dT / 1.41421356237309515f : (v.x * cosf(a) + v.y * sinf(a)) * dT;
}

// transposeShared (DCT_Unwrapping.cu:179-200), square N x N with 32 x 32 LDS tiles.
__global__ void k_transpose(float* __restrict__ o, const float* __restrict__ in, int N)
{
    __shared__ float tile[32][33];
    const int x = blockIdx.x * 32 + threadIdx.x;
    for (int r = threadIdx.y; r < 32; r += blockDim.y) {
        const int y = blockIdx.y * 32 + r;
        if (x < N && y < N) tile[r][threadIdx.x] = in[x + (long long)N * y];
    }
    __syncthreads();
    const int x2 = blockIdx.y * 32 + threadIdx.x;
    for (int r = threadIdx.y; r < 32; r += blockDim.y) {
        const int y2 = blockIdx.x * 32 + r;
        if (x2 < N && y2 < N) o[x2 + (long long)N * y2] = tile[threadIdx.x][r];
    }
}

// devConstant (DCT_Unwrapping.cu:300-312) with the eigenvalue choice of the batched path.
__global__ void k_dev_constant(float* __restrict__ buf, int N, int refeig, const double* __restrict__ eig)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= N || j >= N) return;
    const int k = i + N * j;
    if (i == 0 && j == 0) {
        buf[k] = 0.f;
        return;
    }
    const double lam = refeig ? eig[i] + eig[j] - 4.0 : -4.0 * (eig[i] + eig[j]);
    buf[k] = (float)((double)buf[k] / lam);
}

// countIDCT (DCT_Unwrapping.cu:218-246); `shift` = 1 reproduces the reference's (i+1) twiddle.
__global__ void k_count_idct(float2* __restrict__ o, const float* __restrict__ in, int N, float dT, int shift)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= N || j >= N) return;
    const float a = (float)i * kPI / (2.f * N);
    const float C = cosf(a), S = sinf(a), V = in[i + N * j] * dT;
    const float a2 = ((float)i + (float)shift) * kPI / (2.f * N);
    const float S2 = sinf(a2), C2 = -cosf(a2);
    const float r2 = 1.41421356237309515f;
    float2 t1 = (i == 0) ? make_float2(C * V * r2, S * V * r2) : make_float2(C * V, S * V);
    const float V2 = (i == 0) ? 0.f : in[(N - i) + N * j] * dT;
    float2 t2 = (i == 0) ? make_float2(0.f, 0.f) : make_float2(S2 * V2, C2 * V2);
    o[i + 2 * N * j] = t1;
    o[i + 2 * N * j + N] = t2;
}

// cufft2float (DCT_Unwrapping.cu:164-177)
__global__ void k_real_part(float* __restrict__ o, const float2* __restrict__ in, int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= N || j >= N) return;
    o[i + N * j] = in[i + 2 * N * j].x;
}

__global__ void k_congruent(float* __restrict__ o, const float* __restrict__ w, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) o[i] = w[i] + 2.f * kPI * rintf((o[i] - w[i]) / (2.f * kPI));
}

void unwrap_dct_plain_one(Ctx& c, const float* wrapped, float* out, int N, unsigned flags)
{
    CTDM_REQUIRE(N == 32 || N == 64 || N == 128 || N == 192 || N == 256, "plain unwrap: N in {32, 64, 128, 192, 256}");
    if (flags & F_REF_FAST) {
        const float* norm = normalized_input(c, wrapped, 1, N, "puw.norm");
        unwrap_dct_plain_one(c, norm, out, N, flags & ~F_REF_FAST);
        subtract_min(c, out, 1, N);
        return;
    }
    const size_t n = (size_t)N * N;
    float* inX = (float*)c.buf("puw.inX", sizeof(float) * n);
    float* inY = (float*)c.buf("puw.inY", sizeof(float) * n);
    float* lap = (float*)c.buf("puw.lap", sizeof(float) * n);
    float* dst = (float*)c.buf("puw.dst", sizeof(float) * n);
    float2* cplx = (float2*)c.buf("puw.cplx", sizeof(float2) * 2 * n);
    const double* eig = eig_table(c, N, flags & F_REF_EIG);
    dim3 blk(32, 8), grd((N + 31) / 32, (N + 7) / 8), tg(N / 32, N / 32);
    const float dT = 1.f / sqrtf(2.f * N);
    if (flags & F_SINCOS) {
        hipLaunchKernelGGL(k_sincos_rhs, grd, blk, 0, c.stream, lap, wrapped, N);
    } else {
        hipLaunchKernelGGL(k_numeric_derivative, grd, blk, 0, c.stream, inX, inY, wrapped, N);
        hipLaunchKernelGGL(k_sum_derivative, grd, blk, 0, c.stream, lap, inX, inY, N);
    }
    // myDCT (DCT_Unwrapping.cu:61-83): two passes of mirror / 2N FFT / countFDCT / transpose
    for (int pass = 0; pass < 2; ++pass) {
        float* src = pass == 0 ? lap : inX;
        hipLaunchKernelGGL(k_mirror, grd, blk, 0, c.stream, cplx, src, N);
        fft_rows(c, cplx, 2 * N, N, -1, 1.f, false);
        hipLaunchKernelGGL(k_count_fdct, grd, blk, 0, c.stream, dst, cplx, N, dT);
        hipLaunchKernelGGL(k_transpose, tg, dim3(32, 8), 0, c.stream, inX, dst, N);
    }
    // devConstant
    hipLaunchKernelGGL(k_dev_constant, grd, blk, 0, c.stream, inX, N, (int)((flags & F_REF_EIG) != 0), eig);
    // myIDCT (DCT_Unwrapping.cu:85-107): two passes of transpose / countIDCT / inverse 2N FFT / Re
    for (int pass = 0; pass < 2; ++pass) {
        float* src = pass == 0 ? inX : inY;
        hipLaunchKernelGGL(k_transpose, tg, dim3(32, 8), 0, c.stream, dst, src, N);
        hipLaunchKernelGGL(k_count_idct, grd, blk, 0, c.stream, cplx, dst, N, dT, (int)((flags & F_REF_IDCT) != 0));
        fft_rows(c, cplx, 2 * N, N, +1, 1.f, false);
        hipLaunchKernelGGL(k_real_part, grd, blk, 0, c.stream, pass == 0 ? inY : out, cplx, N);
    }
    if (flags & F_CONGRUENT)
        hipLaunchKernelGGL(k_congruent, dim3(grid1d((long long)n, 256)), dim3(256), 0, c.stream, out, wrapped, (int)n);
    CTDM_CHECK_LAUNCH("plain unwrap");
}

}  // namespace ctdm
