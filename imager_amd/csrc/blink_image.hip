// gfx950 kernels of the stage path's 2-D transform: blink_fft2d_c2c and
// blink_image (FFT of the grids, sum of the counts, normalisation, fft_shift,
// grids and counts cleared).
//
// Two passes, row-major throughout:
//   rows     each team of lanes reads one grid row, transforms it and writes
//            it to the image buffer at its shifted columns; with kImage it
//            also sums the counts of the row (one FP64 partial per workgroup),
//            clears the cells of grid and counts that were not zero, and
//            marks the rows that hold anything (the others are not written);
//   columns  each workgroup owns kW adjacent columns of one image, in place:
//            reads the marked rows, transforms, scales by 1 / (sum of the
//            partials) and writes the rows shifted.
// Shifting the columns in the row pass leaves the column pass without a
// partner column to keep, so any side takes the two passes, odd ones too, and
// no second buffer is needed.
//
// Both passes are bound by memory: the necessary traffic of blink_image is 12
// bytes per cell read, 8 written, and the intermediate's 16, of which rows
// without visibilities (40 % at an oversampling of 2) need none.  The
// transforms stay in registers (RegFft) at N = 128 .. 4096; the exchanges
// between passes go through LDS as one FP32 plane at a time (re, then im),
// which halves the LDS and leaves room for two 1024-thread workgroups per CU
// in the column pass, one loading while the other transforms.
#include "blink_fft_reg.hpp"
#include "blink_kernels.hpp"

#include <algorithm>

namespace blink {

namespace {

constexpr int kMaxStageRows = 64;  // rows per workgroup of the generic row pass

// Stockham exchange of RegFft through one FP32 plane: slot(i) is the LDS
// address of element i.
template <class F, int P, bool kBlock, class Slot>
__device__ __forceinline__ void exchange_planes(float2 (&v)[F::V], float* buf, int lane, Slot slot) {
    constexpr int N = F::kN, L = F::kL;
    constexpr int R1 = F::RAD.r[P], NS1 = reg_span(F::RAD, P), B1 = N / R1 / L;
    constexpr int R2 = F::RAD.r[P + 1], NB2 = N / R2, B2 = NB2 / L;
#pragma unroll
    for (int half = 0; half < 2; half++) {
#pragma unroll
        for (int b = 0; b < B1; b++) {
            const int j = lane + L * b, k = j % NS1, base = (j - k) * R1 + k;
#pragma unroll
            for (int r = 0; r < R1; r++)
                buf[slot(base + r * NS1)] = half ? v[b * R1 + r].y : v[b * R1 + r].x;
        }
        team_sync<kBlock>();
#pragma unroll
        for (int b = 0; b < B2; b++)
#pragma unroll
            for (int r = 0; r < R2; r++) {
                const float x = buf[slot(lane + L * b + r * NB2)];
                if (half) v[b * R2 + r].y = x;
                else v[b * R2 + r].x = x;
            }
        team_sync<kBlock>();
    }
}

// The first half of a twiddle table: w(m + N / 2) = -w(m).
template <int N>
struct TwHalf {
    const float2* t;
    __device__ __forceinline__ float2 operator()(int m) const {
        const float2 w = t[m & (N / 2 - 1)];
        return m & (N / 2) ? make_float2(-w.x, -w.y) : w;
    }
};

template <class F, int S, bool kBlock, int P = 0, class TW, class Slot>
__device__ __forceinline__ void run_planes(float2 (&v)[F::V], float* buf, int lane, const TW& tw,
                                           Slot slot) {
    F::template pass<S, P>(v, lane, tw);
    if constexpr (P + 1 < F::RAD.n_pass) {
        exchange_planes<F, P, kBlock>(v, buf, lane, slot);
        run_planes<F, S, kBlock, P + 1>(v, buf, lane, tw, slot);
    }
}

// Lanes per row, threads per workgroup.  One team per workgroup where a row needs
// several wavefronts, so that the workgroups of a CU drift apart and one loads
// while another transforms (4 x 4096^2: 759 -> 723 us per stage call).
template <int N>
struct RowShape;
template <> struct RowShape<128> { static constexpr int L = 16, NT = 256; };
template <> struct RowShape<256> { static constexpr int L = 32, NT = 256; };
template <> struct RowShape<512> { static constexpr int L = 64, NT = 256; };
template <> struct RowShape<1024> { static constexpr int L = 64, NT = 256; };
template <> struct RowShape<2048> { static constexpr int L = 128, NT = 128; };
template <> struct RowShape<4096> { static constexpr int L = 256, NT = 256; };

// Columns and lanes per column of a workgroup: 64- or 128-byte runs, two or more
// workgroups per CU up to 2048 (1024^2: 8 columns 251, 16 columns 260 us per
// stage call of 24 images; 4096^2: 4 columns, two workgroups per CU, 752 against
// 723 us).
template <int N>
struct ColShape;
template <> struct ColShape<128> { static constexpr int W = 16, L = 16; };
template <> struct ColShape<256> { static constexpr int W = 16, L = 32; };
template <> struct ColShape<512> { static constexpr int W = 16, L = 32; };
template <> struct ColShape<1024> { static constexpr int W = 8, L = 64; };
template <> struct ColShape<2048> { static constexpr int W = 8, L = 128; };
template <> struct ColShape<4096> { static constexpr int W = 8, L = 128; };

// Sum over the workgroup, valid in thread 0 (scratch: a double per wavefront).
__device__ __forceinline__ double block_sum_double(double x, double* scratch) {
    for (int o = 32; o > 0; o >>= 1) x += __shfl_down(x, o, 64);
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = x;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x + 63) / 64; w++) t += scratch[w];
    return t;
}

// (float)(1 / sum of an image's partial count sums), in every lane.
__device__ __forceinline__ float scale_of(const double* __restrict__ part, int n_part) {
    double t = 0.0;
    for (int i = threadIdx.x & 63; i < n_part; i += 64) t += part[i];
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    return (float)(1.0 / t);
}

__device__ __forceinline__ bool any_bits(float2 v) {
    return (__float_as_uint(v.x) | __float_as_uint(v.y)) != 0u;
}

}  // namespace

// Rows.  A workgroup takes `iters` groups of NT / L consecutive rows (of one
// image: iters * NT / L divides N), so that the twiddle table is copied to LDS
// once for all of them.  Cells are cleared in runs of 16 lanes (128 bytes of
// grid) that hold a non-zero bit: the gridded cells of a sparse array are a
// few lines of each row.
template <int N, int S, bool kImage>
__global__ void __launch_bounds__(RowShape<N>::NT)
k_stage_rows(StageFftArgs a, int iters, const float2* __restrict__ tw) {
    constexpr int L = RowShape<N>::L, NT = RowShape<N>::NT, TEAMS = NT / L;
    constexpr bool kBlock = L > 64;
    constexpr int PL = padded_len(N);
    using F = RegFft<N, L>;
    extern __shared__ float stage_rows_lds[];
    float2* twl = (float2*)stage_rows_lds;  // [N / 2]
    float* plane = stage_rows_lds + N;      // [TEAMS][PL]
    __shared__ double red[NT / 64];
    const int tid = threadIdx.x, team = tid / L, lane = tid % L;
    for (int i = tid; i < N / 2; i += NT) twl[i] = tw[i];
    __syncthreads();
    float* buf = plane + team * PL;
    double sum = 0.0;
    for (int it = 0; it < iters; it++) {
        const int64_t row = ((int64_t)blockIdx.x * iters + it) * TEAMS + team;
        const float2* src = a.in + row * N;
        float2 v[F::V];
        F::load(v, lane, [&](int i) { return src[i]; });
        if constexpr (kImage) {
            float* crow = a.counts + row * N;
            float c[F::V];
            constexpr int NB = N / F::RAD.r[0];
            // element of v[q]: lane + L b + r NB, q = b R0 + r (RegFft::load)
            auto elem = [&](int q) {
                return lane + L * (q / F::RAD.r[0]) + (q % F::RAD.r[0]) * NB;
            };
#pragma unroll
            for (int q = 0; q < F::V; q++) c[q] = crow[elem(q)];
            bool any = false;
            float2* grow = a.grids + row * N;
            const int run = (int)(threadIdx.x & 48);  // first lane of the run of 16
#pragma unroll
            for (int q = 0; q < F::V; q++) {
                const bool g = any_bits(v[q]), k = __float_as_uint(c[q]) != 0u;
                any |= g;
                sum += (double)c[q];
                if (a.clear) {
                    if ((__ballot(g) >> run) & 0xffffu) grow[elem(q)] = make_float2(0.f, 0.f);
                    if ((__ballot(k) >> run) & 0xffffu) crow[elem(q)] = 0.f;
                }
            }
            bool used;
            if constexpr (kBlock) used = __syncthreads_or(any ? 1 : 0);
            else used = ((__ballot(any) >> (tid & 63 & ~(L - 1))) &
                         (L == 64 ? ~0ull : (1ull << (L & 63)) - 1)) != 0;
            if (lane == 0) a.used[row] = used ? 1 : 0;
            if (!used) continue;  // uniform per team (per workgroup with kBlock)
        }
        run_planes<F, S, kBlock>(v, buf, lane, TwHalf<N>{twl}, [](int i) { return pad_index(i); });
        float2* dst = a.out + row * N;
        F::store(v, lane, [&](int i, float2 x) {
            dst[kImage ? (i < N / 2 ? i + N / 2 : i - N / 2) : i] = x;
        });
    }
    if constexpr (kImage) {
        const double t = block_sum_double(sum, red);
        if (tid == 0) a.part[blockIdx.x] = t;
    }
}

// Columns, in place.  Thread = (column tid % W, lane tid / W), so that global
// accesses are runs of W columns straight from and to registers, and the
// lanes of a wavefront that share a twiddle are W neighbours: the table is
// read through the cache, not copied to LDS.
template <int N, int S, bool kImage>
__global__ void __launch_bounds__(ColShape<N>::W* ColShape<N>::L)
k_stage_cols(StageFftArgs a, int n_part, const float2* __restrict__ tw) {
    constexpr int W = ColShape<N>::W, L = ColShape<N>::L;
    using F = RegFft<N, L>;
    extern __shared__ float stage_cols_lds[];  // [padded_len(N)][W]
    const unsigned bid = xcd_order(blockIdx.x, gridDim.x);
    const int64_t img = bid / (N / W);
    const int col = threadIdx.x % W, lane = threadIdx.x / W;
    float2* base = a.out + img * N * N + (int64_t)(bid % (N / W)) * W + col;
    float2 v[F::V];
    if constexpr (kImage) {
        const unsigned char* used = a.used + img * N;
        unsigned char u[F::V];
        constexpr int R = F::RAD.r[0], NB = N / R;
#pragma unroll
        for (int q = 0; q < F::V; q++) u[q] = used[lane + L * (q / R) + (q % R) * NB];
#pragma unroll
        for (int q = 0; q < F::V; q++) {
            v[q] = make_float2(0.f, 0.f);
            if (u[q]) v[q] = base[(int64_t)(lane + L * (q / R) + (q % R) * NB) * N];
        }
    } else {
        F::load(v, lane, [&](int i) { return base[(int64_t)i * N]; });
    }
    float scale = 1.f;
    if constexpr (kImage) scale = scale_of(a.part + img * n_part, n_part);
    run_planes<F, S, true>(v, stage_cols_lds + col, lane, TwTable{tw},
                           [](int i) { return pad_index(i) * W; });
    F::store(v, lane, [&](int i, float2 x) {
        if constexpr (kImage)
            base[(int64_t)(i < N / 2 ? i + N / 2 : i - N / 2) * N] = cscale(x, scale);
        else
            base[(int64_t)i * N] = x;
    });
}

// Any other side: LDS Stockham passes over a tile of rows (fft_tile).  `rows` rows
// per workgroup, all of one image.
template <int S, bool kImage>
__global__ void __launch_bounds__(1024)
k_stage_rows_any(StageFftArgs a, FftPlan plan, int rows, const float2* __restrict__ tw) {
    extern __shared__ float4 stage_any_lds4[];
    __shared__ double red[16];
    __shared__ int used[kMaxStageRows];
    const int n = plan.n, nt = (int)blockDim.x, tid = threadIdx.x;
    float2* tile = (float2*)stage_any_lds4;       // [rows][n]
    float2* twl = tile + (size_t)rows * n;        // twiddle table copy [n]
    load_twiddles(twl, tw, n);
    const int wg_per_img = (n + rows - 1) / rows;
    const int64_t img = blockIdx.x / wg_per_img;
    const int r0 = (int)(blockIdx.x % wg_per_img) * rows, nr = min(rows, n - r0);
    const int64_t at = (img * n + r0) * n;
    if (kImage && tid < rows) used[tid] = 0;
    __syncthreads();
    double sum = 0.0;
    for (int i0 = tid; i0 < nr * n; i0 += 4 * nt) {  // four loads in flight
        float2 v[4];
        float c[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = i0 + k * nt;
            v[k] = make_float2(0.f, 0.f);
            c[k] = 0.f;
            if (i >= nr * n) continue;
            v[k] = a.in[at + i];
            if constexpr (kImage) c[k] = a.counts[at + i];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = i0 + k * nt;
            if (i >= nr * n) break;
            tile[i] = v[k];
            if constexpr (kImage) {
                sum += (double)c[k];
                if (any_bits(v[k])) {
                    used[i / n] = 1;
                    if (a.clear) a.grids[at + i] = make_float2(0.f, 0.f);
                }
                if (a.clear && __float_as_uint(c[k]) != 0u) a.counts[at + i] = 0.f;
            }
        }
    }
    if constexpr (kImage) {
        const double t = block_sum_double(sum, red);
        if (tid == 0) a.part[blockIdx.x] = t;
    }
    __syncthreads();
    if constexpr (kImage) {
        if (tid < nr) a.used[img * n + r0 + tid] = used[tid] ? 1 : 0;
        int any = 0;
        for (int r = 0; r < nr; r++) any |= used[r];
        if (!any) return;  // uniform
    }
    fft_tile<S>(tile, nr, n, plan, twl);
    for (int i = tid; i < nr * n; i += nt) {
        const int r = i / n;
        if constexpr (kImage) {
            if (used[r]) a.out[at + r * n + shift_index(i - r * n, n)] = tile[i];
        } else {
            a.out[at + i] = tile[i];
        }
    }
}

// Columns in place, w = 2^lw of them per workgroup (fewer in the last one).
template <int S, bool kImage>
__global__ void __launch_bounds__(1024)
k_stage_cols_any(StageFftArgs a, FftPlan plan, int lw, int n_part, const float2* __restrict__ tw) {
    extern __shared__ float4 stage_any_cols_lds4[];
    const int n = plan.n, ld = n + 1, w = 1 << lw;  // padded LDS rows
    float2* tile = (float2*)stage_any_cols_lds4;    // [w][ld]
    float2* twl = tile + (size_t)w * ld;            // twiddle table copy [n]
    load_twiddles(twl, tw, n);
    const int n_cb = (n + w - 1) >> lw;
    const unsigned bid = xcd_order(blockIdx.x, gridDim.x);
    const int64_t img = bid / n_cb;
    const int c0 = (int)(bid % n_cb) << lw;
    const int w_here = min(w, n - c0);
    float2* base = a.out + img * n * n + c0;
    const unsigned char* used = a.used + img * n;
    const int total = n << lw, nt = (int)blockDim.x;
    for (int i0 = threadIdx.x; i0 < total; i0 += 4 * nt) {
        float2 p[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = i0 + k * nt, r = i >> lw, c = i & (w - 1);
            p[k] = make_float2(0.f, 0.f);
            if (i < total && c < w_here && (!kImage || used[r])) p[k] = base[(int64_t)r * n + c];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = i0 + k * nt;
            if (i < total) tile[(size_t)(i & (w - 1)) * ld + (i >> lw)] = p[k];
        }
    }
    float scale = 1.f;
    if constexpr (kImage) scale = scale_of(a.part + img * n_part, n_part);
    __syncthreads();
    fft_tile<S>(tile, w_here, ld, plan, twl);
    for (int i = threadIdx.x; i < total; i += nt) {
        const int r = i >> lw, c = i & (w - 1);
        if (c >= w_here) continue;
        const float2 x = tile[(size_t)c * ld + r];
        if constexpr (kImage) base[(int64_t)shift_index(r, n) * n + c] = cscale(x, scale);
        else base[(int64_t)r * n + c] = x;
    }
}

// ------------------------------------------------------------ launchers

// Rows per workgroup of the generic row pass: what 512 threads hold at about
// 12 values each, fewer while the launch has under 512 workgroups.
static int any_rows(int n, int64_t n_img) {
    int rows = std::max(1, std::min(kMaxStageRows, 6144 / n));
    while (rows > 1 && n_img * ((n + rows - 1) / rows) < 512) rows = (rows + 1) / 2;
    return rows;
}

static int any_threads(const FftPlan& plan, int64_t values) {
    int nt = 256;
    while (nt < 1024 && ((int64_t)nt * plan.cap < values || nt * plan.cap < plan.n)) nt *= 2;
    return nt;
}

// Row groups per workgroup: up to 4 while 1024 workgroups remain (4 per CU).
template <int N>
static int row_iters(int64_t n_img) {
    constexpr int TEAMS = RowShape<N>::NT / RowShape<N>::L;
    int it = 4;
    while (it > 1 && n_img * N / (TEAMS * it) < 1024) it /= 2;
    return it;
}

// N / (rows per workgroup): partial count sums per image.
int stage_fft_parts(int n, int64_t n_img) {
    switch (n) {
#define X(NN) \
    case NN: return NN / (RowShape<NN>::NT / RowShape<NN>::L * row_iters<NN>(n_img));
        X(128) X(256) X(512) X(1024) X(2048) X(4096)
#undef X
        default: return (n + any_rows(n, n_img) - 1) / any_rows(n, n_img);
    }
}

template <int N, int S, bool kImage>
static hipError_t rows_n(const StageFftArgs& a, int64_t n_img, const float2* tw, hipStream_t s) {
    constexpr int TEAMS = RowShape<N>::NT / RowShape<N>::L;
    const int it = row_iters<N>(n_img);
    const size_t lds = sizeof(float) * (N + (size_t)TEAMS * padded_len(N));
    const int64_t blocks = n_img * N / (TEAMS * it);
    if (blocks > 0x7fffffff || (int64_t)lds > g_lds_limit) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((k_stage_rows<N, S, kImage>), dim3((unsigned)blocks),
                       dim3(RowShape<N>::NT), lds, s, a, it, tw);
    return hipGetLastError();
}

template <int N, int S, bool kImage>
static hipError_t cols_n(const StageFftArgs& a, int64_t n_img, int n_part, const float2* tw,
                         hipStream_t s) {
    constexpr int W = ColShape<N>::W, L = ColShape<N>::L;
    const size_t lds = sizeof(float) * (size_t)padded_len(N) * W;
    const int64_t blocks = n_img * (N / W);
    if (blocks > 0x7fffffff || (int64_t)lds > g_lds_limit) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((k_stage_cols<N, S, kImage>), dim3((unsigned)blocks), dim3(W * L), lds, s,
                       a, n_part, tw);
    return hipGetLastError();
}

template <int S, bool kImage>
static hipError_t rows_any(const StageFftArgs& a, const FftPlan& plan, int64_t n_img,
                           const float2* tw, hipStream_t s) {
    const int n = plan.n, rows = any_rows(n, n_img);
    const size_t lds = sizeof(float2) * ((size_t)n * rows + n);
    const int64_t blocks = n_img * ((n + rows - 1) / rows);
    if (blocks > 0x7fffffff || (int64_t)lds > g_lds_limit) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((k_stage_rows_any<S, kImage>), dim3((unsigned)blocks),
                       dim3(any_threads(plan, (int64_t)n * rows)), lds, s, a, plan, rows, tw);
    return hipGetLastError();
}

template <int S, bool kImage>
static hipError_t cols_any(const StageFftArgs& a, const FftPlan& plan, int64_t n_img, int n_part,
                           const float2* tw, hipStream_t s) {
    const int n = plan.n;
    auto lds_for = [&](int lw) { return sizeof(float2) * (((size_t)(n + 1) << lw) + n); };
    // 16 columns (128-byte runs), fewer while the threads do not hold them, two
    // workgroups (from 4 columns on, one) do not fit in LDS, or the launch has
    // under 512 workgroups (two per CU)
    int lw = 4;
    while (lw > 0 && (((int64_t)n << lw) > 1024 * plan.cap || (int64_t)lds_for(lw) > g_lds_limit ||
                      (lw > 2 && 2 * (int64_t)lds_for(lw) > g_lds_limit) ||
                      (lw > 1 && n_img * ((n + (1 << lw) - 1) >> lw) < 512)))
        lw--;
    const size_t lds = lds_for(lw);
    const int64_t blocks = n_img * ((n + (1 << lw) - 1) >> lw);
    if (blocks > 0x7fffffff || (int64_t)lds > g_lds_limit) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((k_stage_cols_any<S, kImage>), dim3((unsigned)blocks),
                       dim3(any_threads(plan, (int64_t)n << lw)), lds, s, a, plan, lw, n_part, tw);
    return hipGetLastError();
}

template <int S, bool kImage>
static hipError_t stage_pass(bool rows, const StageFftArgs& a, const FftPlan& plan, int64_t n_img,
                             int n_part, const float2* tw, hipStream_t s) {
    switch (plan.n) {
#define X(NN)                                                             \
    case NN:                                                              \
        return rows ? rows_n<NN, S, kImage>(a, n_img, tw, s)              \
                    : cols_n<NN, S, kImage>(a, n_img, n_part, tw, s);
        X(128) X(256) X(512) X(1024) X(2048) X(4096)
#undef X
        default:
            return rows ? rows_any<S, kImage>(a, plan, n_img, tw, s)
                        : cols_any<S, kImage>(a, plan, n_img, n_part, tw, s);
    }
}

hipError_t launch_stage_pass(bool rows, const StageFftArgs& a, const FftPlan& plan, int64_t n_img,
                             int sign, const float* tw, hipStream_t stream) {
    if (n_img == 0) return hipSuccess;
    const float2* t = (const float2*)tw;
    if (a.counts) {
        if (sign < 0 || !a.used || !a.part || !a.grids) return hipErrorInvalidValue;
        return stage_pass<1, true>(rows, a, plan, n_img, stage_fft_parts(plan.n, n_img), t, stream);
    }
    return sign > 0 ? stage_pass<1, false>(rows, a, plan, n_img, 0, t, stream)
                    : stage_pass<-1, false>(rows, a, plan, n_img, 0, t, stream);
}

hipError_t set_stage_kernel_attributes() {
    const int max_lds = (int)g_lds_limit;
    hipError_t e = hipSuccess;
    auto set = [&](const void* f) {
        hipError_t r = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
        if (r != hipSuccess && e == hipSuccess) e = r;
    };
#define Y(NN, S, I)                                  \
    set((const void*)k_stage_rows<NN, S, I>);        \
    set((const void*)k_stage_cols<NN, S, I>);
#define X(NN) Y(NN, 1, true) Y(NN, 1, false) Y(NN, -1, false)
    X(128) X(256) X(512) X(1024) X(2048) X(4096)
#undef X
#undef Y
#define X(S, I)                                   \
    set((const void*)k_stage_rows_any<S, I>);     \
    set((const void*)k_stage_cols_any<S, I>);
    X(1, true) X(1, false) X(-1, false)
#undef X
    return e;
}

}  // namespace blink
