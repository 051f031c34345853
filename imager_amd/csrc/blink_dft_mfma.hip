// Split-precision DFT-as-GEMM on MFMA for small grids (N <= 512).
//
// The gridded plane G is Hermitian (every visibility lands at (u, v) and its
// conjugate at (-u, -v)), so only rows v = 0 .. H = N/2 are gridded, into
// half[img][v][u] (row-major, N complex per row).  With the fftshift
// permutation p folded into the DFT matrices,
//   stage 1 (complex):  T[v][x] = sum_u  D1[x][u] G[v][u],
//                       D1[x][u] = exp(+2 pi i u p(x) / N),     v = 0 .. H;
//   stage 2 (real):     I[y][x] = sum_v  Re(D2[y][v] T[v][x]),
//                       D2[y][v] = w_v exp(+2 pi i v p(y) / N),
// with w_0 = w_H = 1 and w_v = 2 otherwise: row N - v of D1 G is the conjugate
// of row v, so the pair v, N - v contributes 2 Re(D[y][v] T[v][x]) and the
// image is real.  Stage 2 multiplies by (float)(1 / sum counts) and writes the
// imaginary part as 0.
//
// Both stages fold the symmetry of the matrices: frequency rows j and N - j of
// D hold conjugate values, so only j = 0 .. H is multiplied and every result
// serves the two outputs x = H + j (p(x) = j, j < H) and x = H - j (p(x) =
// N - j, j > 0).  With c, s = cos, sin(2 pi j k / N):
//   stage 1: E[u] = G[u] + G[N - u], O[u] = G[u] - G[N - u] for 0 < u < H
//            (E = G, O = 0 at u = 0 and H);  P = sum c E, Q = sum s O over
//            u = 0 .. H;  T[H + j] = P + iQ, T[H - j] = P - iQ;
//   stage 2: P = sum w c Re T, Q = sum w s Im T over v;  I[H + j] = P - Q,
//            I[H - j] = P + Q.
// That is a quarter (stage 1) and a half (stage 2) of the unfolded products,
// and K = H + 1 in both.
//
// The matrix is the first MFMA operand (rows j), the data the second (columns
// m), so the 32 lanes that hold one j store 32 consecutive m: one 256-byte
// segment.
//   stage 1: m = (img, v): half rows in,  inter[img][x][v] out
//   stage 2: m = (img, x): inter rows in, images[img][y][x] out
//
// Precision: every operand x is split into hi = P(x) and lo = P(x - hi),
// P = bf16 or fp16, and products use hi*hi + hi*lo + lo*hi (lo*lo is below
// the FP32 rounding of the sum) with FP32 accumulation in MFMA.  The matrices
// are built on the host in double and split there; the data are split on the
// fly.  fp16 has 5 exponent bits, so each (folded) data row m is first scaled
// by a power of two 2^e that brings its largest component below 2^15 (exact),
// and the result column m is scaled back by 2^-e.
#include <cmath>
#include <cstring>
#include <vector>

#include "blink_kernels.hpp"

namespace blink {

constexpr int kDftMaxTiles = (512 / 2 + 1 + 31) / 32;  // at N = 512, the largest side

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Planes of a split DFT matrix.  The matrix is stored as MFMA operands, in the
// order in which a wave reads them: [32-row tile][16-column step][plane][lane]
// [8], lane l holding row l % 32 and columns 8 (l / 32) .. + 7 of its step.
enum { kReHi = 0, kReLo, kImHi, kImLo, kDftPlanes };

template <int kPrec>
struct Prec;
template <>
struct Prec<kDftBf16> {
    using V = bf16x8;
    static constexpr bool kScale = false;
    using E = __bf16;
    __device__ static f32x16 mfma(V a, V b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct Prec<kDftFp16> {
    using V = f16x8;
    static constexpr bool kScale = true;
    using E = _Float16;
    __device__ static f32x16 mfma(V a, V b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

struct DftGemmArgs {
    const float2* a;          // data rows [m][lda]
    int64_t lda;              // row stride of a (float2, even)
    int64_t m_rows;           // M
    int n, h;                 // N (even) and N / 2: K = h + 1 columns
    int k_pad;                // K rounded up to 16
    int n_tiles;              // 32-row tiles of the matrix rows j = 0 .. h
    const uint16_t* planes;   // split matrix (see kDftPlanes)
    int R;                    // m -> (img = m / R, r = m % R)
    int64_t img_stride, n_stride;  // C[n][m] at out[img * img_stride + n * n_stride + r]
    float2* out;
    const uint32_t* isums;    // stage 2: per-image count sums (set-relative), else null
    double* count_sums;       // stage 2: optional, isums as doubles
    int64_t img0;             // set-relative index of the first image
};

// The 8 folded values u = kb .. kb + 7 of a row of N: E into xs[0..7], O into
// xs[8..15], zero beyond u = h.  `wide`: every octet lies within the row, so
// its two ranges are loaded 16 bytes at a time (rows are 16-byte aligned, N is
// even): u .. u + 7 forwards, and N - u - 8 .. N - u - 1 with N - u by itself.
__device__ __forceinline__ void load_folded(const float2* row, int kb, int n, int h, bool wide,
                                            float2 (&xs)[16]) {
    float2 f[8], b[8];  // G[u], G[N - u] (0 < u < h)
    if (wide) {
        const float4* f4 = (const float4*)(row + kb);
        const float4* b4 = (const float4*)(row + (n - kb - 8));
        b[0] = kb ? row[n - kb] : make_float2(0.f, 0.f);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4 t = f4[q], w = b4[q];
            f[2 * q] = make_float2(t.x, t.y);
            f[2 * q + 1] = make_float2(t.z, t.w);
            // w = G[N - kb - 8 + 2q], G[N - kb - 7 + 2q]
            if (q > 0) b[8 - 2 * q] = make_float2(w.x, w.y);
            b[7 - 2 * q] = make_float2(w.z, w.w);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int u = kb + e;
            f[e] = u <= h ? row[u] : make_float2(0.f, 0.f);
            b[e] = (u > 0 && u < h) ? row[n - u] : make_float2(0.f, 0.f);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int u = kb + e;
        const bool in = u <= h, pair = u > 0 && u < h;
        xs[e].x = pair ? f[e].x + b[e].x : (in ? f[e].x : 0.f);
        xs[e].y = pair ? f[e].y + b[e].y : (in ? f[e].y : 0.f);
        xs[8 + e].x = pair ? f[e].x - b[e].x : 0.f;
        xs[8 + e].y = pair ? f[e].y - b[e].y : 0.f;
    }
}

// The 8 values v = kb .. kb + 7 of a stage-1 row, zero beyond v = h (the row's
// storage reaches k_pad).
__device__ __forceinline__ void load_row8(const float2* row, int kb, int h, float2 (&xs)[8]) {
    const float4* p4 = (const float4*)(row + kb);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4 t = p4[q];
        const bool a = kb + 2 * q <= h, b = kb + 2 * q + 1 <= h;
        xs[2 * q] = make_float2(a ? t.x : 0.f, a ? t.y : 0.f);
        xs[2 * q + 1] = make_float2(b ? t.z : 0.f, b ? t.w : 0.f);
    }
}

constexpr int kOctetStride = 512 + 16;  // bytes: 32 rows x 16, and one bank group of padding

// 8 complex values -> hi and lo of the real and the imaginary parts.
template <int kPrec>
__device__ __forceinline__ void split8(const float2* x, float sc,
                                       typename Prec<kPrec>::V (&v)[4]) {
    using S = Prec<kPrec>;
    using E = typename S::E;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float re = S::kScale ? x[e].x * sc : x[e].x;
        const float im = S::kScale ? x[e].y * sc : x[e].y;
        const E rh = (E)re, ih = (E)im;
        v[0][e] = rh;
        v[1][e] = (E)(re - (float)rh);
        v[2][e] = ih;
        v[3][e] = (E)(im - (float)ih);
    }
}

// A workgroup takes 32 * kTiles data rows: its threads read them once, 8
// columns of a row at a time (coalesced, every load of a batch in flight
// together), and leave them in LDS as split MFMA operands, plane by plane:
// 16 bytes per (row, octet).  Each wave then multiplies them by the 32-row
// matrix tiles t = wave, wave + waves, ..., which come from L2 in operand
// order (1 KB per load, the next step's under the current step's MFMAs): the
// whole matrix is 4 k_pad bytes x 2 per row, 74 KB at N = 180, and every
// workgroup reads the same.  fp16 first needs the largest component of each
// row: the values wait in LDS as FP32, in the bytes of their own later
// operands, for one barrier.
//
// Bound by HBM: at N = 180 the two stages of 768 images move 207 and 305 MB
// and take 53 and 90 us (fp16), 3.9 and 3.4 TB/s; with the unfolded matrix in
// LDS in slices of 64 rows, each of which read all the data (twice, for the
// row maxima), they took 194 and 181 us.
// Whole calls in us, before -> after: 768 x 180^2 fp16 575 -> 357, 100 x 256^2
// fp16 197 -> 132, 40 x 512^2 fp16 373 -> 165, bf16 247 -> 164, 3 x 180^2 fp16
// 82 -> 60.
template <int kPrec, bool kComplex>
__global__ void __launch_bounds__(64 * kDftMaxTiles) k_dft_gemm(DftGemmArgs g) {
    using S = Prec<kPrec>;
    using V = typename S::V;
    constexpr int kTiles = kComplex ? 1 : 2;   // 32-row data tiles
    constexpr int kHalves = kComplex ? 2 : 1;  // E and O, or T: 4 planes each
    constexpr int kRows = 32 * kTiles;
    constexpr int kBatch = kComplex ? 2 : 4;   // octets a thread loads together
    extern __shared__ float4 dft_lds4[];
    char* lds = (char*)dft_lds4;  // [8 planes][k_pad / 8 octets][kOctetStride]
    __shared__ unsigned rmax[kRows];
    const int n_oct = g.k_pad >> 3;
    const int plane = n_oct * kOctetStride;
    const int64_t m0 = (int64_t)xcd_order(blockIdx.x, gridDim.x) * kRows;
    const int n_thr = (int)blockDim.x;
    const int items = kRows * n_oct;
    if (S::kScale) {
        for (int i = (int)threadIdx.x; i < kRows; i += n_thr) rmax[i] = 0;
        __syncthreads();
    }

    const bool wide = g.k_pad <= g.n;
    for (int base = (int)threadIdx.x; base < items; base += kBatch * n_thr) {
        float2 xs[kBatch][8 * kHalves];
        int row[kBatch], oct[kBatch];
#pragma unroll
        for (int b = 0; b < kBatch; b++) {
            // past the end: the last item again, not kept
            const int i = min(base + b * n_thr, items - 1);
            row[b] = i / n_oct;
            oct[b] = i - row[b] * n_oct;
            // rows past M repeat the last one; their results are not stored
            const float2* a = g.a + min(m0 + row[b], g.m_rows - 1) * g.lda;
            if constexpr (kComplex) load_folded(a, 8 * oct[b], g.n, g.h, wide, xs[b]);
            else load_row8(a, 8 * oct[b], g.h, xs[b]);
        }
#pragma unroll
        for (int b = 0; b < kBatch; b++) {
            if (base + b * n_thr >= items) break;
            char* at = lds + (row[b] >> 5) * 4 * plane + oct[b] * kOctetStride + (row[b] & 31) * 16;
            if constexpr (S::kScale) {
                float mx = 0.f;
#pragma unroll
                for (int e = 0; e < 8 * kHalves; e++)
                    mx = fmaxf(mx, fmaxf(fabsf(xs[b][e].x), fabsf(xs[b][e].y)));
                atomicMax(&rmax[row[b]], __float_as_uint(mx));
#pragma unroll
                for (int c = 0; c < 4 * kHalves; c++)
                    *(float4*)(at + c * plane) = make_float4(xs[b][2 * c].x, xs[b][2 * c].y,
                                                             xs[b][2 * c + 1].x, xs[b][2 * c + 1].y);
            } else {
#pragma unroll
                for (int p = 0; p < kHalves; p++) {
                    V v[4];
                    split8<kPrec>(&xs[b][8 * p], 1.f, v);
#pragma unroll
                    for (int c = 0; c < 4; c++) *(V*)(at + (4 * p + c) * plane) = v[c];
                }
            }
        }
    }
    __syncthreads();
    // fp16: power-of-two scale of a row from its largest component
    auto row_exp = [&](int r) {
        const float mx = __uint_as_float(rmax[r]);
        int e = 0;
        if (mx > 0.f && mx < INFINITY) {
            int ex;
            (void)frexpf(mx, &ex);               // mx < 2^ex
            e = max(-126, min(126, 15 - ex));    // mx * 2^e < 2^15
        }
        return e;
    };
    if constexpr (S::kScale) {
        for (int i = (int)threadIdx.x; i < items; i += n_thr) {
            const int r = i / n_oct, o = i - r * n_oct;
            const float sc = __int_as_float((127 + row_exp(r)) << 23);
            char* at = lds + (r >> 5) * 4 * plane + o * kOctetStride + (r & 31) * 16;
#pragma unroll
            for (int p = 0; p < kHalves; p++) {
                float2 x[8];
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float4 t = *(const float4*)(at + (4 * p + c) * plane);
                    x[2 * c] = make_float2(t.x, t.y);
                    x[2 * c + 1] = make_float2(t.z, t.w);
                }
                V v[4];
                split8<kPrec>(x, sc, v);
#pragma unroll
                for (int c = 0; c < 4; c++) *(V*)(at + (4 * p + c) * plane) = v[c];
            }
        }
        __syncthreads();
    }

    const int lane = (int)threadIdx.x & 63;
    const int wave = (int)threadIdx.x >> 6, waves = n_thr >> 6;
    const int n_ks = g.k_pad >> 4;
    const char* dlane = lds + (lane >> 5) * kOctetStride + (lane & 31) * 16;
    for (int t = wave; t < g.n_tiles; t += waves) {
        const V* dp = (const V*)g.planes + (size_t)t * n_ks * (kDftPlanes * 64) + lane;
        // complex: P = p0 + i p1, Q = q0 + i q1; real: P, Q of data tile 0 and 1
        f32x16 p0{}, p1{}, q0{}, q1{};
        V d[kDftPlanes];
#pragma unroll
        for (int c = 0; c < kDftPlanes; c++) d[c] = dp[64 * c];
        for (int ks = 0; ks < n_ks; ks++) {
            V x[8], nd[kDftPlanes];
            const V* dn = dp + (ks + 1 < n_ks ? ks + 1 : ks) * (kDftPlanes * 64);
#pragma unroll
            for (int c = 0; c < kDftPlanes; c++) nd[c] = dn[64 * c];
#pragma unroll
            for (int c = 0; c < 8; c++)
                x[c] = *(const V*)(dlane + c * plane + ks * (2 * kOctetStride));
            // complex: x = Er, Ei, Or, Oi (hi, lo); real: Re, Im of tile 0, then of tile 1
            constexpr int kP1 = kComplex ? 2 : 4, kQ0 = kComplex ? 4 : 2;
            auto mac = [&](const V& hi, const V& lo, int c, f32x16& acc) {
                acc = S::mfma(hi, x[c], acc);
                acc = S::mfma(hi, x[c + 1], acc);
                acc = S::mfma(lo, x[c], acc);
            };
            mac(d[kReHi], d[kReLo], 0, p0);
            mac(d[kReHi], d[kReLo], kP1, p1);
            mac(d[kImHi], d[kImLo], kQ0, q0);
            mac(d[kImHi], d[kImLo], 6, q1);
#pragma unroll
            for (int c = 0; c < kDftPlanes; c++) d[c] = nd[c];
        }

        // acc[i] holds row j = 32 t + 8(i/4) + 4(lane/32) + i%4 of column m
#pragma unroll
        for (int mt = 0; mt < kTiles; mt++) {
            const int64_t m = m0 + 32 * mt + (lane & 31);
            if (m >= g.m_rows) continue;
            const int64_t img = m / g.R;
            const int r = (int)(m - img * g.R);
            float scale = 1.f;
            if constexpr (S::kScale)
                scale = __int_as_float((127 - row_exp(32 * mt + (lane & 31))) << 23);
            if (!kComplex) {
                const uint32_t count = g.isums[g.img0 + img];
                scale *= (float)(1.0 / (double)count);
                if (g.count_sums && r == 0 && t == 0 && lane < 32)
                    g.count_sums[g.img0 + img] = (double)count;
            }
            float2* ob = g.out + img * g.img_stride + r;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int j = 32 * t + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                float2 up, dn;  // outputs h + j, h - j
                if constexpr (kComplex) {
                    up = make_float2((p0[i] - q1[i]) * scale, (p1[i] + q0[i]) * scale);
                    dn = make_float2((p0[i] + q1[i]) * scale, (p1[i] - q0[i]) * scale);
                } else {
                    const float p = mt ? p1[i] : p0[i], q = mt ? q1[i] : q0[i];
                    up = make_float2((p - q) * scale, 0.f);
                    dn = make_float2((p + q) * scale, 0.f);
                }
                float2* pu = &ob[(int64_t)(g.h + j) * g.n_stride];
                float2* pd = &ob[(int64_t)(g.h - j) * g.n_stride];
                if constexpr (kComplex) {
                    if (j < g.h) *pu = up;
                    if (j > 0 && j <= g.h) *pd = dn;
                } else {
                    if (j < g.h) store_stream(pu, up);
                    if (j > 0 && j <= g.h) store_stream(pd, dn);
                }
            }
        }
    }
}

static int pad16(int k) { return (k + 15) / 16 * 16; }
static int dft_tiles(int n) { return (n / 2 + 1 + 31) / 32; }

int dft_inter_stride(int n) { return pad16(n / 2 + 1); }

constexpr int kGemmLdsMax = 160 * 1024 - 1024;  // beside the row maxima

static size_t gemm_lds(int k_pad) { return (size_t)8 * (k_pad / 8) * kOctetStride; }

hipError_t set_dft_kernel_attributes() {
    const void* ks[] = {(const void*)k_dft_gemm<kDftBf16, true>,
                        (const void*)k_dft_gemm<kDftBf16, false>,
                        (const void*)k_dft_gemm<kDftFp16, true>,
                        (const void*)k_dft_gemm<kDftFp16, false>};
    for (const void* k : ks) {
        const hipError_t e =
            hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kGemmLdsMax);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// One wave per 32-row matrix tile: 3 at N = 180, and 9, with 144 KB of LDS, at
// the largest side.
template <bool kComplex>
static hipError_t launch_gemm(const DftGemmArgs& g, int prec, hipStream_t stream) {
    if (g.m_rows == 0) return hipSuccess;
    const size_t lds = gemm_lds(g.k_pad);
    constexpr int kRows = kComplex ? 32 : 64;
    const int64_t blocks = (g.m_rows + kRows - 1) / kRows;
    if (lds > (size_t)kGemmLdsMax || g.n_tiles > kDftMaxTiles || blocks > 0x7fffffff)
        return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)blocks), block(64 * std::max(2, g.n_tiles));
    if (prec == kDftFp16)
        hipLaunchKernelGGL((k_dft_gemm<kDftFp16, kComplex>), grid, block, lds, stream, g);
    else
        hipLaunchKernelGGL((k_dft_gemm<kDftBf16, kComplex>), grid, block, lds, stream, g);
    return hipGetLastError();
}

hipError_t launch_dft_rows(const float* half, const uint16_t* planes1, float* inter, int n,
                           int64_t n_img, int prec, hipStream_t stream) {
    const int h = n / 2;
    DftGemmArgs g{};
    g.a = (const float2*)half;
    g.lda = n;
    g.m_rows = n_img * (h + 1);
    g.n = n;
    g.h = h;
    g.k_pad = pad16(h + 1);
    g.n_tiles = dft_tiles(n);
    g.planes = planes1;
    g.R = h + 1;
    g.n_stride = dft_inter_stride(n);
    g.img_stride = (int64_t)n * g.n_stride;
    g.out = (float2*)inter;
    return launch_gemm<true>(g, prec, stream);
}

hipError_t launch_dft_cols(const float* inter, const uint16_t* planes2, float* images, int n,
                           int64_t n_img, int64_t img0, const uint32_t* isums,
                           double* count_sums, int prec, hipStream_t stream) {
    const int h = n / 2;
    DftGemmArgs g{};
    g.a = (const float2*)inter;
    g.lda = dft_inter_stride(n);
    g.m_rows = n_img * n;
    g.n = n;
    g.h = h;
    g.k_pad = pad16(h + 1);
    g.n_tiles = dft_tiles(n);
    g.planes = planes2;
    g.R = n;
    g.n_stride = n;
    g.img_stride = (int64_t)n * n;
    g.out = (float2*)images + img0 * (int64_t)n * n;
    g.isums = isums;
    g.count_sums = count_sums;
    g.img0 = img0;
    return launch_gemm<false>(g, prec, stream);
}

// Host: rows j = 0 .. H of the matrix exp(+2 pi i j k / N), k = 0 .. H, times
// w_k in stage 2, in double, rounded to nearest even; zero in the padding.
static uint16_t bf16_bits(double v) {
    float f = (float)v;
    uint32_t u;
    memcpy(&u, &f, 4);
    const uint32_t lsb = (u >> 16) & 1u;
    u += 0x7fffu + lsb;
    return (uint16_t)(u >> 16);
}
static double bf16_value(uint16_t b) {
    uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}
static uint16_t fp16_bits(double v) {
    const _Float16 h = (_Float16)v;
    uint16_t b;
    memcpy(&b, &h, 2);
    return b;
}
static double fp16_value(uint16_t b) {
    _Float16 h;
    memcpy(&h, &b, 2);
    return (double)h;
}

void make_dft_planes(int n, int stage, int prec, std::vector<uint16_t>& planes) {
    const int h = n / 2;
    const int n_ks = pad16(h + 1) / 16;
    planes.assign((size_t)dft_tiles(n) * n_ks * kDftPlanes * 512, 0);
    auto bits = [&](double v) { return prec == kDftFp16 ? fp16_bits(v) : bf16_bits(v); };
    auto value = [&](uint16_t b) { return prec == kDftFp16 ? fp16_value(b) : bf16_value(b); };
    for (int j = 0; j <= h; j++) {
        for (int k = 0; k <= h; k++) {
            const long long idx = ((long long)k * j) % n;
            const double a = 2.0 * M_PI * (double)idx / (double)n;
            const double w = (stage == 1 || k == 0 || k == h) ? 1.0 : 2.0;
            const double c = w * std::cos(a), s = w * std::sin(a);
            const uint16_t ch = bits(c), sh = bits(s);
            const int lane = j % 32 + 32 * (k % 16 / 8);
            uint16_t* at = planes.data() +
                           ((size_t)(j / 32) * n_ks + k / 16) * (kDftPlanes * 512) + lane * 8 + k % 8;
            at[kReHi * 512] = ch;
            at[kReLo * 512] = bits(c - value(ch));
            at[kImHi * 512] = sh;
            at[kImLo * 512] = bits(s - value(sh));
        }
    }
}

}  // namespace blink
