// gfx950 kernels of the visibility -> dirty-image path, with their host-side
// launchers.  Every launcher validates the shape it is given against what the
// kernel and its grid assume before it enqueues anything.
#include "blink_kernels.hpp"
#include "blink_gather.hpp"

#include <algorithm>
#include <type_traits>

namespace blink {

int64_t g_lds_limit = 64 * 1024;
int64_t g_lds_budget = 48 * 1024;

int device_cu_count() {
    static const int n_cu = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            n <= 0)
            n = 256;
        return n;
    }();
    return n_cu;
}

// Launch-time guard: a kernel whose LDS request exceeds the device limit is
// not launched.
static bool lds_fits(size_t bytes) { return (int64_t)bytes <= g_lds_limit; }

// Workgroup of the generic direct row passes (one per image).
constexpr int kDirectThreads = 1024;

// ------------------------------------------------------------------ helpers

static unsigned grid_for(int64_t work, int block, int max_blocks) {
    int64_t b = (work + block - 1) / block;
    if (b < 1) b = 1;
    if (b > max_blocks) b = max_blocks;
    return (unsigned)b;
}

// ----------------------------------------------------- (a) phase corrections

// One thread per (t, ch, bl) record: the 4 pol products (32 bytes) are
// rotated by exp(i 2 pi turns) in place.
__global__ void k_phase_correct(float4* __restrict__ vis, int n_bl, int n_ch, int64_t n_rec,
                                const float* __restrict__ w_m, const double* __restrict__ cable_m,
                                const double* __restrict__ freq_hz, unsigned which) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_rec; i += stride) {
        const unsigned bl = (unsigned)(i % n_bl);
        const int ch = (int)((i / n_bl) % n_ch);
        const double nu = freq_hz[ch];
        double turns = 0.0;
        if (which & 1u) turns += reduce_turns(geometric_turns(w_m[bl], nu));
        if (which & 2u) {
            unsigned a1, a2;
            baseline_antennas(bl, a1, a2);
            turns += reduce_turns(cable_turns(cable_m[a2] - cable_m[a1], nu));
        }
        const float2 ph = unit_phasor(turns);
        float4 a = vis[2 * i], b = vis[2 * i + 1];
        float4 ra, rb;
        ra.x = a.x * ph.x - a.y * ph.y;  ra.y = a.y * ph.x + a.x * ph.y;
        ra.z = a.z * ph.x - a.w * ph.y;  ra.w = a.w * ph.x + a.z * ph.y;
        rb.x = b.x * ph.x - b.y * ph.y;  rb.y = b.y * ph.x + b.x * ph.y;
        rb.z = b.z * ph.x - b.w * ph.y;  rb.w = b.w * ph.x + b.z * ph.y;
        vis[2 * i] = ra;
        vis[2 * i + 1] = rb;
    }
}

hipError_t launch_phase_correct(float* vis, int n_ant, int n_ch, int n_t, const float* w_m,
                                const double* cable_m, const double* freq_hz, unsigned which,
                                hipStream_t stream) {
    const int n_bl = n_ant * (n_ant + 1) / 2;
    const int64_t n_rec = (int64_t)n_bl * n_ch * n_t;
    if (n_rec == 0) return hipSuccess;
    hipLaunchKernelGGL(k_phase_correct, dim3(grid_for(n_rec, 256, 65536)), dim3(256), 0, stream,
                       (float4*)vis, n_bl, n_ch, n_rec, w_m, cable_m, freq_hz, which);
    return hipGetLastError();
}

// ----------------------------------------------------------- cell indices

__global__ void k_uv_cells(const float* __restrict__ u_m, const float* __restrict__ v_m,
                           const int* __restrict__ flags, int n_bl,
                           const double* __restrict__ freq_hz, int n_ch, double du, double dv,
                           double min_uv, int n_pixels, int4* __restrict__ cells) {
    const int64_t n = (int64_t)n_bl * n_ch;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const int bl = (int)(i % n_bl);
        const int ch = (int)(i / n_bl);
        int4 c = make_int4(-1, -1, -1, -1);
        int up, vp;
        if (!flags[bl] &&
            cell_of(u_m[bl], v_m[bl], wavelength_of(freq_hz[ch]), du, dv, min_uv, n_pixels, up, vp)) {
            c = make_int4(wrap_index(up, n_pixels), wrap_index(vp, n_pixels),
                          wrap_index(-up, n_pixels), wrap_index(-vp, n_pixels));
        }
        cells[i] = c;
    }
}

hipError_t launch_uv_cells(const float* u_m, const float* v_m, const int* flags, int n_bl,
                           const double* freq_hz, int n_ch, double du, double dv, double min_uv,
                           int n_pixels, int* cells, hipStream_t stream) {
    const int64_t n = (int64_t)n_bl * n_ch;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_uv_cells, dim3(grid_for(n, 256, 65536)), dim3(256), 0, stream, u_m, v_m,
                       flags, n_bl, freq_hz, n_ch, du, dv, min_uv, n_pixels, (int4*)cells);
    return hipGetLastError();
}

// ------------------------------------------------------------ array geometry

__global__ void k_zenith_uvw(const double* __restrict__ x, const double* __restrict__ y,
                             const double* __restrict__ z, int n_bl, float* __restrict__ u_m,
                             float* __restrict__ v_m, float* __restrict__ w_m) {
    const int bl = blockIdx.x * blockDim.x + threadIdx.x;
    if (bl >= n_bl) return;
    unsigned a1, a2;
    baseline_antennas((unsigned)bl, a1, a2);
    u_m[bl] = (float)(-(x[a1] - x[a2]));
    v_m[bl] = (float)(-(y[a1] - y[a2]));
    w_m[bl] = (float)(-(z[a1] - z[a2]));
}

__global__ void k_baseline_flags(const int* __restrict__ ant_flags, int n_bl,
                                 int* __restrict__ bl_flags) {
    const int bl = blockIdx.x * blockDim.x + threadIdx.x;
    if (bl >= n_bl) return;
    unsigned a1, a2;
    baseline_antennas((unsigned)bl, a1, a2);
    bl_flags[bl] = (a1 == a2 || ant_flags[a1] || ant_flags[a2]) ? 1 : 0;
}

// One workgroup: max |u|, |v| over unflagged baselines (exact in double).
__global__ void __launch_bounds__(1024)
k_uv_max(const float* __restrict__ u_m, const float* __restrict__ v_m,
         const int* __restrict__ flags, int n_bl, double* __restrict__ uv_max) {
    __shared__ double red[2][16];
    double um = -INFINITY, vm = -INFINITY;
    for (int i = threadIdx.x; i < n_bl; i += blockDim.x) {
        if (flags[i]) continue;
        um = fmax(um, fabs((double)u_m[i]));
        vm = fmax(vm, fabs((double)v_m[i]));
    }
    for (int o = 32; o > 0; o >>= 1) {
        um = fmax(um, __shfl_down(um, o, 64));
        vm = fmax(vm, __shfl_down(vm, o, 64));
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        red[0][wid] = um;
        red[1][wid] = vm;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) {
            um = fmax(um, red[0][w]);
            vm = fmax(vm, red[1][w]);
        }
        uv_max[0] = um;
        uv_max[1] = vm;
    }
}

hipError_t launch_zenith_uvw(const double* x, const double* y, const double* z, int n_ant,
                             float* u_m, float* v_m, float* w_m, hipStream_t stream) {
    const int n_bl = n_ant * (n_ant + 1) / 2;
    if (n_bl == 0) return hipSuccess;
    hipLaunchKernelGGL(k_zenith_uvw, dim3((n_bl + 255) / 256), dim3(256), 0, stream, x, y, z,
                       n_bl, u_m, v_m, w_m);
    return hipGetLastError();
}

hipError_t launch_baseline_flags(const int* ant_flags, int n_ant, int* bl_flags,
                                 hipStream_t stream) {
    const int n_bl = n_ant * (n_ant + 1) / 2;
    if (n_bl == 0) return hipSuccess;
    hipLaunchKernelGGL(k_baseline_flags, dim3((n_bl + 255) / 256), dim3(256), 0, stream,
                       ant_flags, n_bl, bl_flags);
    return hipGetLastError();
}

hipError_t launch_uv_max(const float* u_m, const float* v_m, const int* flags, int n_bl,
                         double* uv_max, hipStream_t stream) {
    hipLaunchKernelGGL(k_uv_max, dim3(1), dim3(1024), 0, stream, u_m, v_m, flags, n_bl, uv_max);
    return hipGetLastError();
}

// ------------------------------------------------ (b) gridding, plain atomic

// Inputs of the stage gridding kernels.
struct StageGrid {
    const float2* vis;  // [img][bl][4]
    const float* u_m;
    const float* v_m;
    const int* flags;
    const double* freq_hz;
    double du, dv, min_uv;
    int n_bl, n_ch, n_pixels, pol;
    float2* grids;
    float* counts;
};

// The selected polarisation of record (img, bl).
__device__ __forceinline__ float2 stage_value(const StageGrid& g, int64_t img, int bl) {
    const float2* rec = g.vis + 4 * (img * g.n_bl + bl);
    const int p0 = g.pol == 1 ? 3 : (g.pol == 3 ? 1 : 0);
    const float2 x0 = rec[p0];
    const float2 x1 = g.pol >= 2 ? rec[g.pol == 3 ? 2 : 3] : make_float2(0.f, 0.f);
    return select_pol2(x0, x1, g.pol);
}

// FP32 global atomics, one baseline per thread and image blockIdx.y (per-image
// counts as the CPU path keeps them, src/pacer_imager.cpp:387,408).  The
// two components of a cell are added by neighbouring lanes of one instruction,
// so that a cell is one request of the memory side that performs the atomics.
__global__ void __launch_bounds__(256)
k_grid_atomic(StageGrid g, int64_t n_img) {
    const int bl = (int)(blockIdx.x * 256 + threadIdx.x), n = g.n_pixels;
    const int lane = threadIdx.x & 63;
    for (int64_t img = blockIdx.y; img < n_img; img += gridDim.y) {
        const double nu = g.freq_hz[img % g.n_ch];
        float2 val = make_float2(0.f, 0.f);
        int64_t p = -1, q = -1;
        if (bl < g.n_bl && !g.flags[bl]) {
            val = stage_value(g, img, bl);
            int up, vp;
            if (vis_ok(val) && plan_cell(g.u_m[bl], g.v_m[bl], CellUnit(nu, g), g, up, vp)) {
                const int64_t base = img * (int64_t)n * n;
                p = base + (int64_t)wrap_index(vp, n) * n + wrap_index(up, n);
                q = base + (int64_t)wrap_index(-vp, n) * n + wrap_index(-up, n);
            }
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {  // lanes 2 j, 2 j + 1 add cell j + 32 k of the wave
            const int from = (lane >> 1) + 32 * k;
            const float re = __shfl(val.x, from, 64), im = __shfl(val.y, from, 64);
            const int64_t pc = __shfl(p, from, 64), qc = __shfl(q, from, 64);
            if (pc < 0) continue;
            const int odd = lane & 1;
            unsafeAtomicAdd((float*)g.grids + 2 * pc + odd, odd ? im : re);
            unsafeAtomicAdd((float*)g.grids + 2 * qc + odd, odd ? -im : re);
        }
        if (p >= 0) {
            unsafeAtomicAdd(&g.counts[p], 1.0f);
            unsafeAtomicAdd(&g.counts[q], 1.0f);
        }
    }
}

// Cells per thread of the cell kernels.
constexpr int kCellsPer = 4;
static unsigned cell_blocks(int stride) { return (unsigned)((stride + 256 * kCellsPer - 1) / (256 * kCellsPer)); }

// Cells of every (channel, baseline), packed row << 16 | column (kNoCell where
// not gridded), channels `stride` apart (a multiple of 4; the tail is kNoCell).
__global__ void __launch_bounds__(256)
k_stage_cells(StageGrid g, int stride, uint32_t* __restrict__ cells) {
    for (int ch = blockIdx.y; ch < g.n_ch; ch += gridDim.y) {
        const CellUnit cu(g.freq_hz[ch], g);  // (its divisions cost several cells)
#pragma unroll
        for (int k = 0; k < kCellsPer; k++) {
            const int bl = (int)(blockIdx.x * kCellsPer + k) * 256 + (int)threadIdx.x;
            if (bl >= stride) break;
            uint32_t packed = kNoCell;
            int up, vp;
            if (bl < g.n_bl && !g.flags[bl] && plan_cell(g.u_m[bl], g.v_m[bl], cu, g, up, vp))
                packed = ((uint32_t)wrap_index(vp, g.n_pixels) << 16) |
                         (uint32_t)wrap_index(up, g.n_pixels);
            cells[(int64_t)ch * stride + bl] = packed;
        }
    }
}

// Slabs of the Hermitian half plane in LDS.  Workgroup (slab, image) owns the
// rows r = slab, slab + S, .. of 0 .. N/2 (interleaved, so that the rows the
// array reaches are spread evenly).  It walks the cells of
// its channel, kSlabChunk at a time, and queues in LDS the baselines whose
// cell or mirrored cell falls in its rows; then the queue is gridded with full
// wavefronts (a slab's records are 1 / S of all: reading them where they are
// found left most lanes waiting for a few).  At the end it adds its non-empty
// cells, and their conjugates at the mirrored cells, to the global grid (no
// other workgroup touches either).
constexpr int kSlabThreads = 1024, kSlabVec = 3;
constexpr int kSlabChunk = kSlabThreads * 4 * kSlabVec;  // (256 antennas: 3 chunks)
static_assert(kSlabChunk <= 65536, "queue entries are 16-bit offsets");
__global__ void __launch_bounds__(kSlabThreads)
k_grid_slabs(StageGrid g, int S, int rows, int stride, const uint32_t* __restrict__ cells) {
    extern __shared__ float4 slabs_lds4[];
    const int n = g.n_pixels, h = n / 2;
    float2* tile = (float2*)slabs_lds4;                      // [rows][n]
    unsigned* cnt = (unsigned*)(tile + (size_t)rows * n);    // [rows][n]
    unsigned short* queue = (unsigned short*)(cnt + (size_t)rows * n);  // [kSlabChunk]
    __shared__ int n_queued;
    const int slab = (int)(blockIdx.x % (unsigned)S);
    const int64_t img = blockIdx.x / (unsigned)S;
    // r / S of a row r < 2^13 (exact: r and S are below 2^13)
    const unsigned inv = ((1u << 26) + (unsigned)S - 1) / (unsigned)S;
    auto div_s = [&](int r) { return (int)(((uint64_t)r * inv) >> 26); };
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t* cl = cells + (img % g.n_ch) * stride;
    auto load = [&](int base, uint4(&p)[kSlabVec]) {
#pragma unroll
        for (int k = 0; k < kSlabVec; k++) {
            const int b = base + 4 * (tid + k * kSlabThreads);
            p[k] = b < stride ? *(const uint4*)&cl[b]
                              : make_uint4(kNoCell, kNoCell, kNoCell, kNoCell);
        }
    };
    uint4 p[kSlabVec];
    load(0, p);
    for (int i = tid; i < rows * n; i += kSlabThreads) {
        tile[i] = make_float2(0.f, 0.f);
        cnt[i] = 0u;
    }
    for (int base = 0; base < stride; base += kSlabChunk) {
        if (tid == 0) n_queued = 0;
        __syncthreads();
        unsigned keep = 0;
#pragma unroll
        for (int k = 0; k < kSlabVec; k++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t c = j == 0 ? p[k].x : j == 1 ? p[k].y : j == 2 ? p[k].z : p[k].w;
                const int r0 = (int)(c >> 16), r = r0 <= h ? r0 : n - r0;
                if (c != kNoCell && r - S * div_s(r) == slab) keep |= 1u << (4 * k + j);
            }
        int before = __popc(keep);
        const int own = before;
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(before, o, 64);
            if (lane >= o) before += t;
        }
        int at = 0;
        if (lane == 63) at = atomicAdd(&n_queued, before);
        at = __shfl(at, 63, 64) + before - own;
#pragma unroll
        for (int k = 0; k < kSlabVec; k++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                if ((keep >> (4 * k + j)) & 1u)
                    queue[at++] = (unsigned short)(4 * (tid + k * kSlabThreads) + j);
        __syncthreads();
        load(base + kSlabChunk, p);  // the next chunk, while the queue is gridded
        const int nq = n_queued;
        for (int i = tid; i < nq; i += kSlabThreads) {
            const int bl = base + queue[i];
            const uint32_t cell = cl[bl];
            const float2 v = stage_value(g, img, bl);
            if (!vis_ok(v)) continue;
            const int r = (int)(cell >> 16), c = (int)(cell & 0xffffu);
            const int r2 = r == 0 ? 0 : n - r, c2 = c == 0 ? 0 : n - c;
            if (r <= h) {
                const int j = div_s(r) * n + c;
                lds_add(&tile[j], v.x, v.y);
                atomicAdd(&cnt[j], 1u);
            }
            if (r2 <= h) {  // both in the self-conjugate rows 0 and N/2
                const int j = div_s(r2) * n + c2;
                lds_add(&tile[j], v.x, -v.y);
                atomicAdd(&cnt[j], 1u);
            }
        }
        __syncthreads();
    }
    float2* grid = g.grids + img * (int64_t)n * n;
    float* counts = g.counts + img * (int64_t)n * n;
    for (int i = tid; i < rows * n; i += kSlabThreads) {
        const unsigned k = cnt[i];
        if (!k) continue;  // (rows past N/2 hold nothing)
        const int lr = i / n, c = i - lr * n, r = lr * S + slab;
        const float2 t = tile[i];
        // the cell and its mirror (the same twice over in rows 0 and N/2: one write)
        const bool twice = r != 0 && 2 * r != n;
        const int64_t p = (int64_t)r * n + c;
        const int64_t q = twice ? (int64_t)(n - r) * n + (c == 0 ? 0 : n - c) : p;
        const float2 o = grid[p], oq = grid[q];
        const float kp = counts[p], kq = counts[q];
        grid[p] = make_float2(o.x + t.x, o.y + t.y);
        counts[p] = kp + (float)k;
        if (twice) {
            grid[q] = make_float2(oq.x + t.x, oq.y - t.y);
            counts[q] = kq + (float)k;
        }
    }
}

static size_t slab_lds(int n, int rows) { return (size_t)12 * n * rows + 2 * kSlabChunk; }

// Slabs per image: as few as leave two workgroups per CU in LDS (one row at
// the least), more while the images do not give every CU a workgroup.
static int stage_slabs(int n, int64_t n_img) {
    const int h1 = n / 2 + 1;
    const int64_t room = (g_lds_limit / 2 - 2 * kSlabChunk) / (12 * (int64_t)n);
    const int rows = (int)std::max<int64_t>(1, std::min<int64_t>(room, h1));
    const int64_t fill = (device_cu_count() + n_img - 1) / n_img;
    return (int)std::min<int64_t>(h1, std::max<int64_t>((h1 + rows - 1) / rows, fill));
}

// Slabs pay a pass over the channel's cells per slab, atomics pay per
// visibility; slabs win on dense grids of small sides, atomics on sparse or
// large ones and on a single image.  The line compares the two costs fitted to
// measurements (us): slabs 13 + rounds of two workgroups per CU x (2.7 +
// 0.44 per 1000 baselines), atomics 7 + 0.18 per 1000 visibilities.  Measured,
// slabs / atomics, 32896 baselines: 1 x 180^2 18 / 15.5, 3 x 256^2 17 / 26,
// 32 x 225^2 41 / 239, 32 x 512^2 52 / 204, 16 x 1024^2 80 / 102, 16 x 2048^2
// 245 / 102; 8256 baselines: 24 x 512^2 21 / 40, 32 x 800^2 42 / 54, 24 x
// 1024^2 49 / 40, 4 x 4096^2 94 / 9.3.  (Row plans and row tiles before, which
// both replace: 188, -, 224, 327, -, -; 124, -, 170, 381.)
bool stage_grid_slabs(int n, int n_bl, int64_t n_img) {
    if (n > kMaxPixels || n_img == 0) return false;
    const double rounds = (double)n_img * stage_slabs(n, n_img) / (2.0 * device_cu_count());
    return 13.0 + rounds * (2.7 + 0.44e-3 * n_bl) < 7.0 + 0.18e-3 * (double)n_img * n_bl;
}

hipError_t launch_stage_grid(const float* vis, int n_ant, int n_ch, int n_t, const float* u_m,
                             const float* v_m, const int* flags, const double* freq_hz, double du,
                             double dv, double min_uv, int n_pixels, int pol, uint32_t* cells,
                             float* grids, float* counts, hipStream_t stream) {
    const int n_bl = n_ant * (n_ant + 1) / 2;
    const int64_t n_img = (int64_t)n_ch * n_t;
    if (n_img == 0 || n_bl == 0) return hipSuccess;
    const StageGrid g{(const float2*)vis, u_m, v_m, flags, freq_hz, du, dv, min_uv,
                      n_bl, n_ch, n_pixels, pol, (float2*)grids, counts};
    if (!cells) {
        hipLaunchKernelGGL(k_grid_atomic,
                           dim3((unsigned)((n_bl + 255) / 256), (unsigned)std::min<int64_t>(n_img, 65535)),
                           dim3(256), 0, stream, g, n_img);
        return hipGetLastError();
    }
    const int S = stage_slabs(n_pixels, n_img), rows = (n_pixels / 2 + S) / S;
    const size_t lds = slab_lds(n_pixels, rows);
    const int64_t blocks = n_img * S;
    if (!lds_fits(lds) || blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    const int stride = (int)stage_cell_stride(n_bl);
    hipLaunchKernelGGL(k_stage_cells, dim3(cell_blocks(stride), (unsigned)std::min(n_ch, 65535)),
                       dim3(256), 0, stream, g, stride, cells);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_grid_slabs, dim3((unsigned)blocks), dim3(kSlabThreads), lds, stream, g, S,
                       rows, stride, cells);
    return hipGetLastError();
}

// --------------------------------------- (b) convolutional (Kaiser-Bessel) gridding

// Nearest cell and kernel rows of one visibility, as convolve_with_kernel
// chooses them from the 1023-times oversampled fractional cell position
// (src/pacer_imager.cpp:654-714).
struct KbSpot {
    int up, vp;        // nearest cell
    const double* xk;  // K weights along u
    const double* yk;  // K weights along v
};
__device__ __forceinline__ bool kb_spot(const StageGrid& g, double wl, int bl, int K,
                                        const double* __restrict__ kt, KbSpot& sp) {
#pragma clang fp contract(off)
    if (!cell_of(g.u_m[bl], g.v_m[bl], wl, g.du, g.dv, g.min_uv, g.n_pixels, sp.up, sp.vp)) return false;
    const double ue = (double)g.u_m[bl] / wl / g.du;
    const double ve = (double)g.v_m[bl] / wl / g.dv;
    int kx = (int)round((ue - (double)sp.up) * 1023.0);
    int ky = (int)round((ve - (double)sp.vp) * 1023.0);
    kx = (kx + 1534) % 1023;
    ky = (ky + 1534) % 1023;
    sp.xk = kt + (int64_t)kx * K;
    sp.yk = kt + (int64_t)ky * K;
    return true;
}

// Sparse grids of large sides (see kb_grid_slabs): one thread per (image,
// baseline), FP32 global atomics.  The visibility and its conjugate
// are spread over K x K cells with weights kt[ky][j] * kt[kx][i] in FP64; counts
// go to the nearest cells (:387,408).
__global__ void __launch_bounds__(256)
k_grid_kb(StageGrid g, int64_t n_rec, int K, const double* __restrict__ kt) {
#pragma clang fp contract(off)
    const int n = g.n_pixels, mid = K / 2;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x, gs = (int64_t)n * n;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_rec; i += stride) {
        const int bl = (int)(i % g.n_bl);
        const int64_t img = i / g.n_bl;
        if (g.flags[bl]) continue;
        const float2 val = stage_value(g, img, bl);
        KbSpot sp;
        if (!vis_ok(val) || !kb_spot(g, wavelength_of(g.freq_hz[img % g.n_ch]), bl, K, kt, sp)) continue;
        float* grid = (float*)(g.grids + img * gs);
        for (int s = 1; s >= -1; s -= 2) {
            for (int j = 0; j < K; j++) {
                int y;
                if (!kb_cell(sp.vp - mid + j, s, n, y)) continue;
                const double wy = sp.yk[j];
                for (int c = 0; c < K; c++) {
                    int x;
                    if (!kb_cell(sp.up - mid + c, s, n, x)) continue;
                    const double w = wy * sp.xk[c];
                    const int64_t p = (int64_t)y * n + x;
                    unsafeAtomicAdd(&grid[2 * p], (float)((double)val.x * w));
                    unsafeAtomicAdd(&grid[2 * p + 1], (float)((double)s * (double)val.y * w));
                }
            }
            unsafeAtomicAdd(&g.counts[img * gs + (int64_t)wrap_index(s * sp.vp, n) * n +
                                      wrap_index(s * sp.up, n)], 1.0f);
        }
    }
}

// Footprints of the rows r0 .. r0 + nr - 1 (grid rows v, or with kSwap grid columns
// u) accumulated in LDS planes re, im [nr][n].  Each wavefront walks its share of
// the cells of a channel (packed row << 16 | position, `stride` of them), queues
// (baseline, sign) in LDS wherever the nearest row of that footprint lies
// within K / 2 rows (cyclically: a superset of the footprints that reach the
// rows), and whenever 64 are queued each lane spreads one over those of its
// rows that are here (a mask, so that the lanes of a wavefront take few
// turns).  The queues are the wavefronts' own: no barrier until the cells are
// through, so that one wavefront's loads and set-up lie under the others'
// updates.  value(bl) gives the visibility; count(row, position) is called once
// per gridded nearest cell in the rows.
// The work is the K x K updates of every footprint.  The cells are FP64 planes:
// ds_add_f64 costs 21 clocks per wavefront instruction at random cells, also where a
// third of them fall in a dense core (9 at consecutive ones), where compare-and-swaps
// of FP32 cells retry.
// kX: largest K whose weights along a row stay in registers; each weight read in
// the inner loop would be a gather of 64 cache lines per wavefront.
// With a queue and barriers for the whole workgroup, chunk by chunk, 64 x 180^2,
// K = 7 took 335 us (now 313), 32 x 1024^2 284 (270), 4 x 4096^2 846 (568).
// `mirror` (slabs that also write the mirror rows, see k_grid_kb_slabs):
// kb_cell keeps the coordinate -N of a footprint, at cell 0, and drops +N, so where a
// position is +-N only one of a visibility's two footprints has the cell.  Those
// cells stay out of the planes: edge[0 .. nr), [nr .. 2 nr) sum the real and imaginary
// parts of position 0 of the rows, and [2 nr .. 4 nr) those of the mirror rows.
// kHerm (rows 0 .. N / 2 of a plane that is imaged as a Hermitian one, for the real part of
// its image): the Hermitian part of the plane, so that such a cell counts half, at its
// place and, conjugated, at the mirror cell.  A footprint takes its share of both: half
// wherever it or the other one has the cell, nothing where neither has.
// Both in a second walk, if the first one met a footprint that may reach +-N: in
// the first one's loop the cases cost all footprints 1 to 4 %.
// The planes must be cleared and visible before, and are complete after the next
// barrier.  Returns the number of footprints that the wavefront queued.
constexpr int kKbQueue = 64 + 2 * 2 * 64;  // entries of a wavefront: two cells per lane and walk
constexpr size_t kb_queue_bytes(int nt) { return sizeof(uint32_t) * (size_t)(nt / 64) * kKbQueue; }
template <int NT, int kX, bool kSwap, bool kHerm, class Value, class Count>
__device__ __forceinline__ int kb_accumulate(const StageGrid& g, double wl, int K,
                                              const double* __restrict__ kt,
                                              const uint32_t* __restrict__ cl, int stride, int r0,
                                              int nr, double* re, double* im, double* edge,
                                              bool mirror, uint32_t* queues, Value value, Count count) {
#pragma clang fp contract(off)
    const int n = g.n_pixels, mid = K / 2, lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    uint32_t* queue = queues + wave * kKbQueue;
    // rows r0 - reach .. r0 + nr - 1 + reach (kb_cell places the negative rows of
    // an odd side one lower than wrap_index does)
    const int reach = mid + (n & 1), span = nr + 2 * reach;
    const int far = kHerm || mirror ? n - mid : INT_MAX;  // from here on a footprint may reach +-N
    auto near = [&](uint32_t r) {
        int d = (int)r - (r0 - reach);
        d = d < 0 ? d + n : (d >= n ? d - n : d);
        return d < span || span >= n;
    };
    auto load = [&](int base) {  // (stride is a multiple of 4)
        const int b = base + 2 * lane;
        return b < stride ? *(const uint2*)&cl[b] : make_uint2(kNoCell, kNoCell);
    };
    int total = 0, nq = 0, seen_far = 0;
    int base = wave * 128;
    uint2 cur = load(base);
    for (bool more = true; more; base += 2 * NT) {
        more = base < stride;
        if (more) {
            const uint2 nxt = load(base + 2 * NT);
            // an entry: baseline * 2, plus 1 for its conjugate's footprint
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t c = j < 2 ? cur.x : cur.y, r = c >> 16;
                const bool keep = c != kNoCell && near((j & 1) && r ? n - r : r);
                const unsigned long long m = __ballot(keep);
                if (keep)
                    queue[nq + __builtin_amdgcn_mbcnt_hi(
                                   (unsigned)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                        4u * (unsigned)lane + 2u * (unsigned)base + (unsigned)j;
                nq += __popcll(m);
            }
            cur = nxt;
        }
        team_sync<false>();
        while (nq >= 64 || (!more && nq)) {
            const int m = min(nq, 64);
            nq -= m;
            total += m;
            if (lane >= m) continue;
            const uint32_t q = queue[nq + lane];
            const int bl = (int)(q >> 1), s = (q & 1) ? -1 : 1;
            const float2 v = value(bl);
            KbSpot sp;
            if (!vis_ok(v) || !kb_spot(g, wl, bl, K, kt, sp)) continue;
            const int rp = kSwap ? sp.up : sp.vp, cp = kSwap ? sp.vp : sp.up;
            const double* rk = kSwap ? sp.xk : sp.yk;
            const double* ck = kSwap ? sp.yk : sp.xk;
            const int rn = wrap_index(s * rp, n) - r0;
            if ((unsigned)rn < (unsigned)nr) count(rn, wrap_index(s * cp, n));
            if ((kHerm ? max(abs(cp), abs(rp)) : abs(cp)) >= far) {
                seen_far = 1;
                continue;
            }
            double cw[kX > 0 ? kX : 1];
            int cx[kX > 0 ? kX : 1];
            if constexpr (kX > 0) {
#pragma unroll
                for (int c = 0; c < kX; c++) {
                    cx[c] = -1;
                    if (c >= K) continue;
                    cw[c] = ck[c];
                    int x;
                    if (kb_cell(cp - mid + c, s, n, x)) cx[c] = x;
                }
            }
            unsigned hit = 0;  // rows j of the footprint that are here
            for (int j = 0; j < K; j++) {
                int y;
                if (kb_cell(rp - mid + j, s, n, y) && (unsigned)(y - r0) < (unsigned)nr) hit |= 1u << j;
            }
            for (; hit; hit &= hit - 1) {
                const int j = __ffs(hit) - 1;
                int y = 0;
                kb_cell(rp - mid + j, s, n, y);
                const double wr = rk[j];
                const int row = (y - r0) * n;
                auto put = [&](int x, double wc) {
                    const double w = wr * wc;
                    atomicAdd(&re[row + x], (double)v.x * w);
                    atomicAdd(&im[row + x], (double)s * (double)v.y * w);
                };
                if constexpr (kX > 0) {
#pragma unroll
                    for (int c = 0; c < kX; c++)
                        if (cx[c] >= 0) put(cx[c], cw[c]);
                } else {
                    for (int c = 0; c < K; c++) {
                        int x;
                        if (kb_cell(cp - mid + c, s, n, x)) put(x, ck[c]);
                    }
                }
            }
        }
        team_sync<false>();
    }
    if (!__any(seen_far)) return total;
    // the far footprints (few, if any), cell by cell
    auto in = [&](int p) { return p >= -n && p < n; };
    auto wrap = [&](int p) { return p < 0 ? p + n : (p == n ? 0 : p); };
    for (base = wave * 128; base < stride; base += 2 * NT) {
        cur = load(base);
        for (int e = 0; e < 4; e++) {
            const uint32_t cell = e < 2 ? cur.x : cur.y, r = cell >> 16;
            if (cell == kNoCell || !near((e & 1) && r ? n - r : r)) continue;
            const int bl = base + 2 * lane + (e >> 1), s = (e & 1) ? -1 : 1;
            const float2 v = value(bl);
            KbSpot sp;
            if (!vis_ok(v) || !kb_spot(g, wl, bl, K, kt, sp)) continue;
            const int rp = kSwap ? sp.up : sp.vp, cp = kSwap ? sp.vp : sp.up;
            if ((kHerm ? max(abs(cp), abs(rp)) : abs(cp)) < far) continue;
            for (int j = 0; j < K; j++) {
                const int py = s * (rp - mid + j), y = wrap(py) - r0;
                if (abs(py) > n || (!kHerm && py == n) || (unsigned)y >= (unsigned)nr) continue;
                for (int c = 0; c < K; c++) {
                    const int px = s * (cp - mid + c);
                    const bool own = in(px) && in(py), other = in(-px) && (!kHerm || in(-py));
                    if (!own && !other) continue;
                    const double w = (kHerm && own != other ? 0.5 : 1.0) *
                                     (kSwap ? sp.xk[j] * sp.yk[c] : sp.yk[j] * sp.xk[c]);
                    const double a = (double)v.x * w, b = (double)s * (double)v.y * w;
                    const bool plane = kHerm || own == other;
                    const int i = y * n + wrap(px);
                    atomicAdd(plane ? &re[i] : &edge[(own ? 0 : 2 * nr) + y], a);
                    atomicAdd(plane ? &im[i] : &edge[(own ? nr : 3 * nr) + y], plane || own ? b : -b);
                }
            }
        }
    }
    return total;
}

// Stage path: workgroup (slab, image) owns `rows` consecutive grid rows of the
// first `n_rows`; at the end the non-zero cells are added to the global grid (no
// other workgroup touches them).  n_rows = N, or N / 2 + 1 on an even side wider than
// the kernel: a cell of a footprint and the mirror cell of the conjugate's are
// then the conjugates of each other, so rows N - r are those of rows r, added by the
// same workgroup, except where the position is +-N (cells of an undersampled
// grid), which are summed apart (`edge` of kb_accumulate).  (A row at +-N is row 0,
// which is not mirrored.)
constexpr int kKbThreads = 512, kKbSlabRows = 8;  // (rows: the most)
template <int kX>
__global__ void __launch_bounds__(kKbThreads)
k_grid_kb_slabs(StageGrid g, int n_rows, int rows, int stride, const uint32_t* __restrict__ cells,
                int K, const double* __restrict__ kt) {
    extern __shared__ float4 kb_slabs_lds4[];
    const int n = g.n_pixels;
    double* re = (double*)kb_slabs_lds4;                     // [rows][n]
    double* im = re + (size_t)rows * n;                      // [rows][n]
    unsigned* cnt = (unsigned*)(im + (size_t)rows * n);      // [rows][n]
    uint32_t* queues = cnt + (size_t)rows * n;
    __shared__ double edge[4 * kKbSlabRows];                 // [4][nr]
    const bool mirror = n_rows < n;
    const int n_slab = (n_rows + rows - 1) / rows;
    const int r0 = (int)(blockIdx.x % (unsigned)n_slab) * rows, nr = min(rows, n_rows - r0);
    const int64_t img = blockIdx.x / (unsigned)n_slab;
    const int tid = threadIdx.x;
    for (int i = tid; i < rows * n; i += kKbThreads) {
        re[i] = im[i] = 0.0;
        cnt[i] = 0u;
    }
    if (tid < 4 * kKbSlabRows) edge[tid] = 0.0;
    __syncthreads();
    kb_accumulate<kKbThreads, kX, false, false>(
        g, wavelength_of(g.freq_hz[img % g.n_ch]), K, kt, cells + (img % g.n_ch) * stride, stride,
        r0, nr, re, im, edge, mirror, queues, [&](int bl) { return stage_value(g, img, bl); },
        [&](int r, int c) { atomicAdd(&cnt[r * n + c], 1u); });
    __syncthreads();
    float2* grid = g.grids + img * (int64_t)n * n;
    float* counts = g.counts + img * (int64_t)n * n;
    auto add = [&](int64_t at, double x, double y, unsigned k) {
        if (!(x == 0.0 && y == 0.0)) {
            const float2 o = grid[at];
            grid[at] = make_float2((float)((double)o.x + x), (float)((double)o.y + y));
        }
        if (k) counts[at] += (float)k;
    };
    for (int i = tid; i < nr * n; i += kKbThreads) {
        const double x = re[i], y = im[i];
        const unsigned k = cnt[i];
        const int lr = i / n, r = r0 + lr, c = i % n;
        const double* e = edge + lr;
        if (c) add((int64_t)r * n + c, x, y, k);
        else add((int64_t)r * n, x + e[0], y + e[nr], k);
        if (!mirror || r == 0 || 2 * r == n) continue;
        if (c) add((int64_t)(n - r) * n + (n - c), x, -y, k);
        else add((int64_t)(n - r) * n, x + e[2 * nr], e[3 * nr] - y, k);
    }
}

static size_t kb_slab_lds(int n, int rows) {
    return (size_t)20 * n * rows + kb_queue_bytes(kKbThreads);
}

// Rows to accumulate: see k_grid_kb_slabs.
static int kb_grid_rows(int n, int K) { return n % 2 == 0 && K < n ? n / 2 + 1 : n; }
// Rows per slab: up to kKbSlabRows (the wider, the fewer slabs compute a footprint's
// weights again), fewer while that leaves under four workgroups per CU or
// fills more than a third of a CU's LDS (16 x 256^2, K 7: 4 rows 147 us, 8 rows 161, 16 rows
// 321).
static int kb_slab_rows(int n, int K, int64_t n_img) {
    int rows = kKbSlabRows;
    while (rows > 1 && (3 * (int64_t)kb_slab_lds(n, rows) > g_lds_limit ||
                        n_img * ((kb_grid_rows(n, K) + rows - 1) / rows) < 4 * device_cu_count()))
        rows /= 2;
    return rows;
}

// Slabs pay their set-up (clearing, walking the channel's cells, the flush) per
// workgroup, global atomics 4 K^2 round trips per visibility.  Costs fitted to
// measurements (us): slabs 20 + 0.022 per workgroup (0.035 where one fills a CU's
// LDS) + 1.1e-5 per footprint cell (half with the mirror), atomics 2.3e-4 per
// footprint cell.  Measured, atomics -> slabs: 16 x 256^2, 32896 baselines, K 7
// 4914 -> 147; 1 x 180^2 803 -> 75; 2 x 225^2, K 15 5926 -> 231; 8256 baselines:
// 4 x 1024^2 349 -> 33, 2 x 4096^2 187 -> 177.
bool kb_grid_slabs(int n, int n_bl, int64_t n_img, int K) {
    if (n > kMaxPixels || n_img == 0) return false;
    const int rows = kb_slab_rows(n, K, n_img);
    if (!lds_fits(kb_slab_lds(n, rows))) return false;  // one row and the queues: N > 7475
    const int n_rows = kb_grid_rows(n, K);
    const double wgs = (double)n_img * ((n_rows + rows - 1) / rows);
    const double cells = (double)n_img * n_bl * K * K;
    const double per = 2 * (int64_t)kb_slab_lds(n, rows) > g_lds_limit ? 0.035 : 0.022;
    return 20.0 + per * wgs + (n_rows < n ? 5.5e-6 : 1.1e-5) * cells < 2.3e-4 * cells;
}

hipError_t launch_grid_kb(const float* vis, int n_ant, int n_ch, int n_t, const float* u_m,
                          const float* v_m, const int* flags, const double* freq_hz, double du,
                          double dv, double min_uv, int n_pixels, int pol, int kernel_size,
                          const double* table, uint32_t* cells, float* grids, float* counts,
                          hipStream_t stream) {
    const int n_bl = n_ant * (n_ant + 1) / 2;
    const int64_t n_img = (int64_t)n_ch * n_t;
    if (n_img == 0 || n_bl == 0) return hipSuccess;
    const StageGrid g{(const float2*)vis, u_m, v_m, flags, freq_hz, du, dv, min_uv,
                      n_bl, n_ch, n_pixels, pol, (float2*)grids, counts};
    if (!cells) {
        const int64_t n_rec = n_bl * n_img;
        hipLaunchKernelGGL(k_grid_kb, dim3(grid_for(n_rec, 256, 65536)), dim3(256), 0, stream, g,
                           n_rec, kernel_size, table);
        return hipGetLastError();
    }
    const int n_rows = kb_grid_rows(n_pixels, kernel_size);
    const int rows = kb_slab_rows(n_pixels, kernel_size, n_img);
    const size_t lds = kb_slab_lds(n_pixels, rows);
    const int64_t blocks = n_img * ((n_rows + rows - 1) / rows);
    if (!lds_fits(lds) || blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    const int stride = (int)stage_cell_stride(n_bl);
    hipLaunchKernelGGL(k_stage_cells, dim3(cell_blocks(stride), (unsigned)std::min(n_ch, 65535)),
                       dim3(256), 0, stream, g, stride, cells);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const auto k = kernel_size <= 8 ? k_grid_kb_slabs<8> : k_grid_kb_slabs<0>;
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(kKbThreads), lds, stream, g, n_rows, rows,
                       stride, cells, kernel_size, table);
    return hipGetLastError();
}

// ------------------------------------------ (b) gridding plans of a batched call
//
// One plan unit per (set, channel): the counting sort of the channel's 2 n_bl
// cells by grid row; `parts` workgroups per unit share its baselines.
//   count    the cell of every baseline of the part (FP64, bit-exact), kept
//            packed for the scatter, and the part's histogram by row;
//   scan     per unit: row starts, and each part's first slot in every row;
//   scatter  each part sorts its entries by row in LDS and writes them out
//            as contiguous runs (no FP64 work, no scattered 4-byte stores).
// Entry order inside a row is not fixed; the sums it feeds are FP32 sums in
// any order either way.  Histograms and slots cover the planned rows 0 .. N/2;
// the scan is bound by its chains of loads (16 parts of a row in flight: 48
// channels x 4096^2 25 us, all N rows with 8 in flight 38), the scatter by the
// part's row counts (22 us; 38 in strided chunks of all rows).

constexpr int kUnitThreads = 512;
// baselines per thread in a plan part (parts hold at most kPlanPartMax)
constexpr int kPlanPerThread = kPlanPartMax / kUnitThreads;
static_assert(kPlanPartMax % kUnitThreads == 0, "plan parts split evenly over the threads");

__device__ __forceinline__ void part_range(int n_bl, int parts, int part, int& b0, int& b1) {
    const int per = (n_bl + parts - 1) / parts;
    b0 = min(n_bl, part * per);
    b1 = min(n_bl, b0 + per);
}

// Exclusive scan of x over the workgroup (kUnitThreads threads); returns the
// thread's prefix and the total in *total.
__device__ __forceinline__ int unit_scan(int x, int* warp_tot, int* total) {
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    int y = x;
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(y, o, 64);
        if (lane >= o) y += t;
    }
    if (lane == 63) warp_tot[wid] = y;
    __syncthreads();
    int before = 0, tot = 0;
    for (int w = 0; w < kUnitThreads / 64; w++) {
        if (w < wid) before += warp_tot[w];
        tot += warp_tot[w];
    }
    *total = tot;
    return before + y - x;
}

__global__ void __launch_bounds__(kUnitThreads)
k_plan_count(const SetDesc* __restrict__ sets, const PlanUnit* __restrict__ units, int parts,
             int n_max, int* __restrict__ partial, uint32_t* __restrict__ cells) {
    extern __shared__ int unit_lds[];
    int* hist = unit_lds;  // [N/2 + 1]
    const int unit = blockIdx.x / parts, part = blockIdx.x % parts;
    const PlanUnit pu = units[unit];
    const SetDesc sd = sets[pu.set];
    const int n = sd.n_pixels, h1 = n / 2 + 1, n_bl = sd.g.n_bl;
    const CellUnit cu(sd.g.freq_hz[pu.ch], sd);
    for (int i = threadIdx.x; i < h1; i += kUnitThreads) hist[i] = 0;
    __syncthreads();
    int b0, b1;
    part_range(n_bl, parts, part, b0, b1);
    uint32_t* cl = cells + pu.cell_off;
    if (part == 0)  // the count sums of this channel's images start at zero
        for (int t = threadIdx.x; t < sd.n_img / sd.g.n_ch; t += kUnitThreads)
            sd.isums[(int64_t)t * sd.g.n_ch + pu.ch] = 0u;
    if (pu.ch == 0 && sd.g.corrections)  // one unit per set writes the phase coefficients
        for (int bl = b0 + (int)threadIdx.x; bl < b1; bl += kUnitThreads)
            sd.coef_out[bl] = phase_coefficient(sd.g.corrections, sd.w_m, sd.cable_m, (unsigned)bl);
    // at most kPlanPerThread baselines per thread: every load is issued first
    int fl[kPlanPerThread];
    float uu[kPlanPerThread], vv[kPlanPerThread];
#pragma unroll
    for (int k = 0; k < kPlanPerThread; k++) {
        const int bl = b0 + (int)threadIdx.x + k * kUnitThreads;
        fl[k] = 1;
        if (bl < b1) {
            fl[k] = sd.flags[bl];
            uu[k] = sd.u_m[bl];
            vv[k] = sd.v_m[bl];
        }
    }
#pragma unroll
    for (int k = 0; k < kPlanPerThread; k++) {
        const int bl = b0 + (int)threadIdx.x + k * kUnitThreads;
        if (bl >= b1) break;
        int up, vp;
        uint32_t packed = kNoCell;
        if (!fl[k] && plan_cell(uu[k], vv[k], cu, sd, up, vp)) {
            const int r = wrap_index(sd.uv_swap ? up : vp, n);
            packed = ((uint32_t)r << 16) | (uint32_t)wrap_index(sd.uv_swap ? vp : up, n);
            // only rows 0 .. N/2 are planned (the consumers rebuild the rest
            // from the Hermitian symmetry): the cell or its conjugate, or both
            // in rows 0 and N/2
            const int r2 = r == 0 ? 0 : n - r;
            if (r <= n / 2) atomicAdd(&hist[r], 1);
            if (r2 <= n / 2) atomicAdd(&hist[r2], 1);
        }
        cl[bl] = packed;
    }
    __syncthreads();
    int* out = partial + ((int64_t)unit * parts + part) * n_max;
    for (int i = threadIdx.x; i < h1; i += kUnitThreads) out[i] = hist[i];
}

__global__ void __launch_bounds__(kUnitThreads)
k_plan_scan(const SetDesc* __restrict__ sets, const PlanUnit* __restrict__ units, int parts,
            int n_max, int* __restrict__ partial) {
    extern __shared__ int unit_lds[];
    int* row_tot = unit_lds;  // [N/2 + 1] entries per row over all parts, then row starts
    __shared__ int warp_tot[kUnitThreads / 64];
    const int unit = blockIdx.x;
    const PlanUnit pu = units[unit];
    const SetDesc sd = sets[pu.set];
    const int n = sd.n_pixels, h1 = n / 2 + 1;
    int* rs = sd.row_start + (int64_t)pu.ch * (n + 1);
    int* base = partial + (int64_t)unit * parts * n_max;
    const int tid = threadIdx.x;
    // row totals: one thread per row, parts summed in order (coalesced reads)
    for (int i = tid; i < h1; i += kUnitThreads) {
        int t = 0;
#pragma unroll 16
        for (int p = 0; p < parts; p++) t += base[(int64_t)p * n_max + i];
        row_tot[i] = t;
    }
    __syncthreads();
    // exclusive scan of the row totals: contiguous chunks per thread
    const int chunk = (h1 + kUnitThreads - 1) / kUnitThreads;
    const int c0 = min(tid * chunk, h1), c1 = min(c0 + chunk, h1);
    int local = 0;
    for (int i = c0; i < c1; i++) local += row_tot[i];
    int total;
    int run = unit_scan(local, warp_tot, &total);
    for (int i = c0; i < c1; i++) {
        const int t = row_tot[i];
        row_tot[i] = run;
        run += t;
    }
    __syncthreads();
    // row starts, and each part's first slot in every row (one thread per row)
    for (int i = tid; i < h1; i += kUnitThreads) {
        int r = row_tot[i];
        rs[i] = r;
        for (int p0 = 0; p0 < parts; p0 += 16) {
            int h[16];  // independent loads in flight, then the running sums
#pragma unroll
            for (int k = 0; k < 16; k++)
                h[k] = p0 + k < parts ? base[(int64_t)(p0 + k) * n_max + i] : 0;
#pragma unroll
            for (int k = 0; k < 16; k++)
                if (p0 + k < parts) {
                    base[(int64_t)(p0 + k) * n_max + i] = r;
                    r += h[k];
                }
        }
    }
    for (int i = h1 + tid; i <= n; i += kUnitThreads) rs[i] = total;  // (not planned)
    // the non-empty rows 0 .. N/2 and their first entries (row_list_len)
    int* rl = sd.row_list + (int64_t)pu.ch * row_list_len(n);
    auto start = [&](int i) { return i < h1 ? row_tot[i] : total; };
    const int hc = (h1 + kUnitThreads - 1) / kUnitThreads;
    const int q0 = min(tid * hc, h1), q1 = min(q0 + hc, h1);
    int cnt = 0;
    for (int i = q0; i < q1; i++) cnt += start(i + 1) != start(i);
    __syncthreads();  // warp_tot is reused
    int n_rows;
    int at = unit_scan(cnt, warp_tot, &n_rows);
    for (int i = q0; i < q1; i++)
        if (start(i + 1) != start(i)) {
            rl[at] = i;
            rl[h1 + at] = start(i);
            at++;
        }
    for (int p = n_rows + tid; p <= h1; p += kUnitThreads) rl[h1 + p] = start(h1);
}

__global__ void __launch_bounds__(kUnitThreads)
k_plan_scatter(const SetDesc* __restrict__ sets, const PlanUnit* __restrict__ units, int parts,
               int n_max, const int* __restrict__ partial, const uint32_t* __restrict__ cells) {
    extern __shared__ int unit_lds[];
    __shared__ int warp_tot[kUnitThreads / 64];
    const int unit = blockIdx.x / parts, part = blockIdx.x % parts;
    const PlanUnit pu = units[unit];
    const SetDesc sd = sets[pu.set];
    const int n = sd.n_pixels, h1 = n / 2 + 1, n_bl = sd.g.n_bl;
    int* first = unit_lds;            // [h1] the part's first global slot per row
    int* lstart = first + n_max;      // [h1] the row's first local slot
    int* lfill = lstart + n_max;      // [h1]
    uint32_t* lent = (uint32_t*)(lfill + n_max);              // [2 kPlanPartMax]
    unsigned short* lrow = (unsigned short*)(lent + 2 * kPlanPartMax);  // [2 kPlanPartMax]
    const int* off = partial + ((int64_t)unit * parts + part) * n_max;
    const int* rs = sd.row_start + (int64_t)pu.ch * (n + 1);
    const int tid = threadIdx.x;
    // the part's count per row is the next part's first slot (or the row
    // end) minus its own; local starts are their exclusive scan
    for (int i = tid; i < h1; i += kUnitThreads) {
        const int o = off[i];
        const int e = part + 1 < parts ? off[n_max + i] : rs[i + 1];
        first[i] = o;
        lfill[i] = e - o;  // count, for now
    }
    __syncthreads();
    const int chunk = (h1 + kUnitThreads - 1) / kUnitThreads;
    const int c0 = min(tid * chunk, h1), c1 = min(c0 + chunk, h1);
    int local = 0;
    for (int i = c0; i < c1; i++) local += lfill[i];
    int n_local;
    int run = unit_scan(local, warp_tot, &n_local);
    for (int i = c0; i < c1; i++) {
        const int c = lfill[i];
        lstart[i] = run;
        lfill[i] = 0;
        run += c;
    }
    __syncthreads();
    int b0, b1;
    part_range(n_bl, parts, part, b0, b1);
    const uint32_t* cl = cells + pu.cell_off;
    uint32_t pk[kPlanPerThread];
#pragma unroll
    for (int k = 0; k < kPlanPerThread; k++) {
        const int bl = b0 + tid + k * kUnitThreads;
        pk[k] = bl < b1 ? cl[bl] : kNoCell;
    }
#pragma unroll
    for (int k = 0; k < kPlanPerThread; k++) {
        const int bl = b0 + tid + k * kUnitThreads;
        const uint32_t packed = pk[k];
        if (packed == kNoCell) continue;
        const int r = (int)(packed >> 16), u = (int)(packed & 0xffffu);
        if (r <= n / 2) {
            const int p = lstart[r] + atomicAdd(&lfill[r], 1);
            lent[p] = (uint32_t)u | ((uint32_t)bl << 14);
            lrow[p] = (unsigned short)r;
        }
        const int r2 = r == 0 ? 0 : n - r, u2 = u == 0 ? 0 : n - u;
        if (r2 <= n / 2) {
            const int q = lstart[r2] + atomicAdd(&lfill[r2], 1);
            lent[q] = (uint32_t)u2 | (1u << 13) | ((uint32_t)bl << 14);
            lrow[q] = (unsigned short)r2;
        }
    }
    __syncthreads();
    uint32_t* ent = sd.entries + (int64_t)pu.ch * 2 * n_bl;
    for (int i = tid; i < n_local; i += kUnitThreads) {
        const int r = lrow[i];
        ent[first[r] + (i - lstart[r])] = lent[i];
    }
}

hipError_t launch_plan_units(const SetDesc* sets, const PlanUnit* units, int n_units, int parts,
                             int n_max, int* partial, uint32_t* cells, hipStream_t stream) {
    if (n_units == 0) return hipSuccess;
    if (parts < 1 || n_max < 1 || n_max > kMaxPixels) return hipErrorInvalidValue;
    const int64_t blocks = (int64_t)n_units * parts;
    if (blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    const size_t lds_count = sizeof(int) * (size_t)n_max;
    const size_t lds_scatter = sizeof(int) * 3 * (size_t)n_max +
                               (sizeof(uint32_t) + sizeof(unsigned short)) * 2 * kPlanPartMax;
    if (!lds_fits(lds_scatter)) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(k_plan_count, dim3((unsigned)blocks), dim3(kUnitThreads), lds_count,
                       stream, sets, units, parts, n_max, partial, cells);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_plan_scan, dim3((unsigned)n_units), dim3(kUnitThreads), lds_count, stream,
                       sets, units, parts, n_max, partial);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_plan_scatter, dim3((unsigned)blocks), dim3(kUnitThreads), lds_scatter,
                       stream, sets, units, parts, n_max, (const int*)partial,
                       (const uint32_t*)cells);
    return hipGetLastError();
}

// Locates the tile row of entry e given the tile's row starts rs[0..nr].
__device__ __forceinline__ int row_of_entry(const int* rs, int nr, int e) {
    int r = 0;
    while (r + 1 < nr && rs[r + 1] <= e) r++;
    return r;
}

// Hermitian half plane for the DFT transform: rows v = 0 .. N/2 of each image
// of a chunk, gridded in LDS tiles of rb rows and written row-major
// to half[li][v][u] (rows of a chunk contiguous); rows without entries are
// written as zeros.  An entry in a row 0 < v < N/2 stands for its conjugate
// partner in row N - v too, so it counts twice in the count sum.
__global__ void __launch_bounds__(kTileThreads)
k_grid_half_rows(GatherArgs g, const int* __restrict__ row_start,
                 const uint32_t* __restrict__ entries, int n, int rb, int64_t img0,
                 float2* __restrict__ half, uint32_t* __restrict__ isums, int uniform) {
    extern __shared__ float4 ghr_lds4[];
    float4* tile4 = ghr_lds4;  // [rb][n] complex, as n/2 float4 per row
    float2* tile = (float2*)ghr_lds4;
    unsigned* cnt = (unsigned*)(tile + (size_t)rb * n);  // [rb][n] counts ("U" weighting)
    __shared__ int rs[kMaxTileRows + 1];
    __shared__ int red[kTileThreads / 64];
    const int h = n / 2;
    const int n_rb = (h + 1 + rb - 1) / rb;
    // XCD-aware order: each XCD gets a contiguous run of (image, tile) pairs,
    // so the tiles of one image share that XCD's L2 copy of its records.
    const unsigned bid = xcd_order(blockIdx.x, gridDim.x);
    const int tile_id = (int)(bid % n_rb);
    const int64_t li = bid / n_rb;
    const int64_t img = img0 + li;
    const int ch = (int)(img % g.n_ch);
    const int r0 = tile_id * rb;
    const int nr = min(rb, h + 1 - r0);
    const int* rsg = row_start + (int64_t)ch * (n + 1);
    if ((int)threadIdx.x <= nr) rs[threadIdx.x] = rsg[r0 + threadIdx.x];
    __syncthreads();
    float4* dst = (float4*)(half + (li * (h + 1) + r0) * (int64_t)n);
    const int q = nr * n / 2;
    if (rs[nr] == rs[0]) {  // no entries: zero rows (empty cells, NaN, under "U")
        const float z = uniform ? __builtin_nanf("") : 0.f;
        for (int i = threadIdx.x; i < q; i += blockDim.x) dst[i] = make_float4(z, z, z, z);
        return;
    }
    for (int i = threadIdx.x; i < q; i += blockDim.x) tile4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (uniform)
        for (int i = threadIdx.x; i < nr * n; i += blockDim.x) cnt[i] = 0u;
    __syncthreads();
    const uint32_t* ent = entries + (int64_t)ch * 2 * g.n_bl;
    const int n_ok = gather_range<4>(g, img, ch, ent, rs[0], rs[nr], (int)threadIdx.x,
                                     (int)blockDim.x, [&](int e, int u_idx, float2 v) {
        const int r = row_of_entry(rs, nr, e);
        lds_add(&tile[r * n + u_idx], v.x, v.y);
        if (uniform) atomicAdd(&cnt[r * n + u_idx], 1u);
        const int row = r0 + r;
        return (row == 0 || row == h) ? 1 : 2;
    });
    const int tot = block_sum_int(n_ok, red);
    if (threadIdx.x == 0 && tot) atomicAdd(&isums[img], (uint32_t)tot);
    __syncthreads();
    if (uniform) {  // grid / count per cell, 0 / 0 = NaN in empty cells
        for (int i = threadIdx.x; i < nr * n; i += blockDim.x) {
            const float k = (float)cnt[i];
            tile[i] = make_float2(tile[i].x / k, tile[i].y / k);
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < q; i += blockDim.x) dst[i] = tile4[i];
}

hipError_t launch_grid_half_rows(const GatherArgs& g, const int* row_start, const uint32_t* entries,
                                 int n, int64_t n_img, int64_t img0, float* half,
                                 uint32_t* isums, hipStream_t stream, bool uniform) {
    if (n_img == 0) return hipSuccess;
    if (n % 2) return hipErrorInvalidValue;
    // Two rows per workgroup: the gather of plan entries is latency bound, and
    // small tiles keep the most workgroups (and loads) in flight per CU; this
    // measured fastest against 4 to 16 rows on 768-channel 256-antenna sets.
    const int rb = 2;
    const int64_t n_rb = (n / 2 + 1 + rb - 1) / rb;
    const int64_t blocks = n_rb * n_img;
    const size_t lds = (sizeof(float2) + (uniform ? sizeof(unsigned) : 0)) * (size_t)rb * n;
    if (!lds_fits(lds) || blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(k_grid_half_rows, dim3((unsigned)blocks), dim3(kTileThreads), lds, stream, g,
                       row_start, entries, n, rb, img0, (float2*)half, isums, uniform ? 1 : 0);
    return hipGetLastError();
}

// Direct variant of k_grid_half_rows for dense sets with one timestep per
// channel (no plan; see k_grid_rows_direct_fft): one workgroup per image of
// the chunk holds rows v = 0 .. N/2 in LDS, walks every baseline in order and
// writes the half plane row-major to half[li][v][u], rows without entries as
// zeros.  The count sums start at zero (the direct set-up launch).
__global__ void __launch_bounds__(kDirectThreads)
k_grid_half_direct(SetDesc sd, int64_t img0, float2* __restrict__ half) {
    extern __shared__ float4 ghd_lds4[];
    const int n = sd.n_pixels, h = n / 2;
    float2* tile = (float2*)ghd_lds4;  // [h + 1][n]
    __shared__ int red[kDirectThreads / 64];
    const int64_t li = xcd_order(blockIdx.x, gridDim.x);
    const int64_t img = img0 + li;  // image within the set
    const int ch = (int)(img % sd.g.n_ch);
    const int q = (h + 1) * n / 2;  // float4 per image (N even)
    for (int i = threadIdx.x; i < q; i += kDirectThreads) ghd_lds4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();
    const int n_ok = direct_walk<2>(sd, img, ch, n, 0, h + 1, (int)threadIdx.x, kDirectThreads,
                                    [&](int r, int c) { return &tile[__mul24(r, n) + c]; });
    const int tot = block_sum_int(n_ok, red);
    if (threadIdx.x == 0 && tot) atomicAdd(&sd.isums[img], (uint32_t)tot);
    __syncthreads();
    float4* dst = (float4*)(half + li * (h + 1) * (int64_t)n);
    for (int i = threadIdx.x; i < q; i += kDirectThreads) dst[i] = ghd_lds4[i];
}

hipError_t launch_grid_half_direct(const SetDesc& sd, int64_t n_img, int64_t img0, float* half,
                                   hipStream_t stream) {
    if (n_img == 0) return hipSuccess;
    const int n = sd.n_pixels;
    if (n % 2 || sd.uv_swap) return hipErrorInvalidValue;
    const size_t lds = sizeof(float2) * (size_t)(n / 2 + 1) * n;
    if (!lds_fits(lds) || n_img > 0x7fffffff) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(k_grid_half_direct, dim3((unsigned)n_img), dim3(kDirectThreads), lds,
                       stream, sd, img0, (float2*)half);
    return hipGetLastError();
}

// grid /= count per cell, the "U" weighting of src/pacer_imager.cpp:421-428.
__global__ void k_uniform_weight(float2* __restrict__ grids, const float* __restrict__ counts,
                                 int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        float2 g = grids[i];
        const float c = counts[i];
        g.x = g.x / c;
        g.y = g.y / c;
        grids[i] = g;
    }
}

hipError_t launch_uniform_weight(float* grids, const float* counts, int64_t n_cells,
                                 hipStream_t stream) {
    if (n_cells == 0) return hipSuccess;
    hipLaunchKernelGGL(k_uniform_weight, dim3(grid_for(n_cells, 256, 65536)), dim3(256), 0, stream,
                       (float2*)grids, counts, n_cells);
    return hipGetLastError();
}

// ---------------------------------------------- (d) sums, shift+norm, averaging

// sums[img] = sum of values of one image, in double.  One block per image.
__global__ void __launch_bounds__(1024)
k_vector_sum(const float* __restrict__ values, int64_t image_size, double* __restrict__ sums) {
    __shared__ double part[16];
    const float* v = values + (int64_t)blockIdx.x * image_size;
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < image_size; i += blockDim.x) s += (double)v[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += part[w];
        sums[blockIdx.x] = t;
    }
}

hipError_t launch_vector_sum(const float* values, int64_t image_size, int n_images, double* sums,
                             hipStream_t stream) {
    if (n_images == 0) return hipSuccess;
    hipLaunchKernelGGL(k_vector_sum, dim3(n_images), dim3(1024), 0, stream, values, image_size, sums);
    return hipGetLastError();
}

// In-place fft_shift + scale.  Pixel p = (y, x) and its image q =
// (shift(y), shift(x)) form a 2-cycle (or p == q); the smaller index swaps.
__global__ void k_shift_norm(float2* __restrict__ img, int nx, int ny, int64_t n_total,
                             const double* __restrict__ sums, int n_sums) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t per = (int64_t)nx * ny;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_total; i += stride) {
        const int64_t im = i / per;
        const int64_t p = i % per;
        const int y = (int)(p / nx), x = (int)(p % nx);
        const int64_t q = (int64_t)shift_index(y, ny) * nx + shift_index(x, nx);
        if (q < p) continue;
        const float s = sums ? (float)(1.0 / sums[im % n_sums]) : 1.0f;
        float2* base = img + im * per;
        const float2 a = base[p];
        const float2 b = base[q];
        if (q == p) {
            base[p] = sums ? cscale(a, s) : a;
        } else {
            base[p] = sums ? cscale(b, s) : b;
            base[q] = sums ? cscale(a, s) : a;
        }
    }
}

hipError_t launch_shift_norm(float* images, int nx, int ny, int n_images, const double* sums,
                             int n_sums, hipStream_t stream) {
    const int64_t n = (int64_t)nx * ny * n_images;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_shift_norm, dim3(grid_for(n, 256, 65536)), dim3(256), 0, stream,
                       (float2*)images, nx, ny, n, sums, n_sums);
    return hipGetLastError();
}

// Mean over images per pixel, summed in image order in FP32
// (src/gpu/gpu_utils.cpp:143-150; real part only for src/utils.cpp:4-22).  One
// thread per pixel, kBatch images' loads ahead of their sums: images too small to
// fill the card with one load per thread are bound by latency (768 x 180^2 197 ->
// 33 us); large ones by HBM, where the plain loop is faster (24 x 1024^2 30
// against 35).
constexpr int64_t kSmallImage = 256 * 1024;
template <int kBatch>
__global__ void k_average(const float2* __restrict__ images, int64_t image_size, int n_images,
                          int real_only, float2* __restrict__ out) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < image_size; i += stride) {
        float2 t = images[i];
        int k = 1;
        for (; kBatch > 1 && k + kBatch <= n_images; k += kBatch) {
            float2 v[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; b++) v[b] = images[i + (int64_t)(k + b) * image_size];
#pragma unroll
            for (int b = 0; b < kBatch; b++) {
                t.x += v[b].x;
                t.y += v[b].y;
            }
        }
        for (; k < n_images; k++) {
            const float2 v = images[i + (int64_t)k * image_size];
            t.x += v.x;
            t.y += v.y;
        }
        const float n = (float)n_images;
        out[i] = real_only ? make_float2(t.x / n, 0.f) : make_float2(t.x / n, t.y / n);
    }
}

hipError_t launch_average(const float* images, int64_t image_size, int n_images, int real_only,
                          float* avg, hipStream_t stream) {
    if (image_size == 0) return hipSuccess;
    const bool small = image_size < kSmallImage;
    const int threads = small ? 64 : 256;
    hipLaunchKernelGGL(small ? k_average<16> : k_average<1>, dim3(grid_for(image_size, threads, 65536)),
                       dim3(threads), 0, stream, (const float2*)images, image_size, n_images,
                       real_only, (float2*)avg);
    return hipGetLastError();
}

// ------------------------------------- batched: gridding fused with row FFT

// Workgroup = (tile of RB rows, image).  Plan entries of the tile are
// gathered (pol, phase correction, NaN/MAX_VIS), accumulated with lds_add
// into the tile, each non-empty row is transformed in LDS and written to the
// row-pass buffer `inter` (image index relative to the chunk).  Empty rows are
// not written: the column pass reads the plan and treats them as zero.  The
// number of gridded cells per image goes to isums (integer atomics).
template <bool kMulti>
__global__ void __launch_bounds__(1024)
k_grid_rows_fft(SetDesc first, const SetDesc* __restrict__ sets, const int* __restrict__ img_set,
                FftPlan plan, int rb, int64_t gi0, float2* __restrict__ inter,
                const float2* __restrict__ tw) {
    extern __shared__ float4 grf_lds4[];
    const int n = plan.n;
    float2* tile = (float2*)grf_lds4;                 // [rb][n]
    float2* twl = tile + (size_t)rb * n;              // twiddle table copy [n]
    __shared__ int rs[kMaxTileRows + 1];
    __shared__ int red[1024 / 64];

    // Rows 0 .. N/2 only: the gridded plane is Hermitian, so row N - v is the
    // conjugate mirror of row v and the column pass rebuilds it.
    const int h = n / 2;
    const int n_rb = (h + 1 + rb - 1) / rb;
    // XCD-aware order: consecutive workgroup ids land on different XCDs, so
    // the ids are remapped to give each XCD a contiguous run of (image, tile)
    // pairs and keep an image's visibilities in one L2.
    const unsigned nwg = gridDim.x;
    unsigned bid = blockIdx.x;
    if ((nwg & 7u) == 0) bid = (bid & 7u) * (nwg >> 3) + (bid >> 3);
    const int tile_id = (int)(bid % n_rb);
    const int li = (int)(bid / n_rb);
    const int64_t gi = gi0 + li;
    const SetDesc sd = set_of<kMulti>(first, sets, img_set, gi);
    const GatherArgs& g = sd.g;
    const int img = (int)(gi - sd.img_base);  // image within its set
    const int ch = img % g.n_ch;
    const int r0 = tile_id * rb;
    const int nr = min(rb, h + 1 - r0);
    const int* rsg = sd.row_start + (int64_t)ch * (n + 1);
    const uint32_t* ent = sd.entries + (int64_t)ch * 2 * g.n_bl;
    if ((int)threadIdx.x <= nr) rs[threadIdx.x] = rsg[r0 + threadIdx.x];
    __syncthreads();
    if (rs[nr] == rs[0]) return;  // uniform: no entries in this tile
    // "U" weighting: a count per tile cell after the table
    unsigned* cnt = (unsigned*)(twl + n);
    const bool uniform = sd.uniform != 0;
    load_twiddles(twl, tw, n);
    for (int i = threadIdx.x; i < nr * n; i += blockDim.x) tile[i] = make_float2(0.f, 0.f);
    if (uniform)
        for (int i = threadIdx.x; i < nr * n; i += blockDim.x) cnt[i] = 0u;
    __syncthreads();
    const int n_ok = gather_range<4>(g, img, ch, ent, rs[0], rs[nr], (int)threadIdx.x,
                                     (int)blockDim.x, [&](int e, int u_idx, float2 v) {
        const int r = row_of_entry(rs, nr, e);
        lds_add(&tile[r * n + u_idx], v.x, v.y);
        if (uniform) atomicAdd(&cnt[r * n + u_idx], 1u);
        // an entry stands for its mirror too, except in the self-conjugate rows
        // (0, and N/2 for even N), which list both
        const int row = r0 + r;
        return (row == 0 || 2 * row == n) ? 1 : 2;
    });
    const int tot = block_sum_int(n_ok, red);
    if (threadIdx.x == 0 && tot) atomicAdd(&sd.isums[img], (uint32_t)tot);
    __syncthreads();
    if (uniform) {  // grid / count per cell (src/pacer_imager.cpp:421-428), 0 / 0 = NaN
        for (int i = threadIdx.x; i < nr * n; i += blockDim.x) {
            const float k = (float)cnt[i];
            tile[i] = make_float2(tile[i].x / k, tile[i].y / k);
        }
        __syncthreads();
    }
    fft_tile<1>(tile, nr, n, plan, twl);
    float2* dst = inter + ((int64_t)li * (h + 1) + r0) * n;
    for (int i = threadIdx.x; i < nr * n; i += blockDim.x) {
        const int r = i / n;
        if (rs[r + 1] != rs[r]) store_stream(&dst[i], tile[i]);  // (rows without entries: not read)
    }
}

// Second pass of the generic batched path, from the half-height row-major
// row-pass buffer inter[img][p][y], plan rows p = 0 .. N/2 (the plan is
// transposed: plan rows are grid columns u, transformed along v by the row
// pass).  As in the register path, the images are real, so one complex FFT
// over p of z = c_y + i c_{y+1} gives image rows y and y+1; plan rows N - p
// are the conjugates of rows p.  A workgroup owns `cb` (even) buffer columns
// = cb/2 pairs, staged through LDS with 16-byte loads, transformed by the
// teams, scaled by 1/sum and stored fftshifted with imaginary parts 0.
template <bool kMulti>
__global__ void __launch_bounds__(1024)
k_cols_half(SetDesc first, const SetDesc* __restrict__ sets, const int* __restrict__ img_set,
            FftPlan plan, int pairs, int64_t gi0, const float2* __restrict__ inter,
            const float2* __restrict__ tw) {
    extern __shared__ float4 ch_lds4[];
    const int n = plan.n, h = n / 2;
    const int ld = n + 1;                                   // padded LDS row
    float2* rows = (float2*)ch_lds4;                        // [pairs][ld]
    float2* twl = rows + (size_t)pairs * ld;                // twiddle table copy [n]
    unsigned char* nonempty = (unsigned char*)(twl + n);
    load_twiddles(twl, tw, n);

    // neighbouring blocks share lines of the buffer's rows: one XCD each
    const unsigned bid = xcd_order(blockIdx.x, gridDim.x);
    const int n_cb = (h + pairs - 1) / pairs;
    const int cbk = (int)(bid % n_cb);
    const int li = (int)(bid / n_cb);
    const int64_t gi = gi0 + li;
    const SetDesc sd = set_of<kMulti>(first, sets, img_set, gi);
    if (!sd.images) return;  // a set imaged for its average only (uniform per workgroup)
    const int img = (int)(gi - sd.img_base);
    const uint32_t count = sd.isums[img];
    if (cbk == 0 && threadIdx.x == 0 && sd.count_sums) sd.count_sums[img] = (double)count;
    const int* rsg = sd.row_start + (int64_t)(img % sd.g.n_ch) * (n + 1);
    const float empty = sd.uniform ? __builtin_nanf("") : 0.f;  // rows without entries
    for (int i = threadIdx.x; i <= h; i += blockDim.x)
        nonempty[i] = sd.all_rows || rsg[i + 1] != rsg[i];
    __syncthreads();

    const int c0 = cbk * 2 * pairs;
    pairs = min(pairs, h - cbk * pairs);  // (the last block's)
    const float2* src = inter + (int64_t)li * (h + 1) * n + c0;
    // four loads in flight per thread, then their LDS writes
    const int stage = (h + 1) * pairs, nt = (int)blockDim.x;
    for (int i0 = threadIdx.x; i0 < stage; i0 += 4 * nt) {
        float4 p[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = i0 + k * nt;
            const int v = i / pairs, t = i % pairs;
            p[k] = make_float4(empty, empty, empty, empty);
            if (i < stage && nonempty[v]) p[k] = *(const float4*)&src[(int64_t)v * n + 2 * t];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = i0 + k * nt;
            if (i >= stage) break;
            const int v = i / pairs, t = i % pairs;
            float2* zr = rows + (size_t)t * ld;
            zr[v] = make_float2(p[k].x - p[k].w, p[k].y + p[k].z);  // c_x[v] + i c_{x+1}[v]
            if (v > 0 && v < h) zr[n - v] = make_float2(p[k].x + p[k].w, p[k].z - p[k].y);  // row N - v
        }
    }
    __syncthreads();
    fft_tile<1>(rows, pairs, ld, plan, twl);
    const float s = (float)(1.0 / (double)count);
    float2* out = sd.images + (int64_t)img * n * n;
    // the plan is transposed: pair t holds Z_t[x] = img[y][x] + i img[y + 1][x]
    // for y = c0 + 2t, so it writes image rows shift(y) and shift(y + 1) (not
    // adjacent when N/2 is odd and y + 1 = N/2) whole, consecutive threads on
    // consecutive output column pairs (even, so 16-byte aligned as N is even)
    for (int i = threadIdx.x; i < h * pairs; i += blockDim.x) {
        const int t = i / h, ox = 2 * (i % h);
        const int x0 = ox < h ? ox + h : ox - h, x1 = ox + 1 < h ? ox + 1 + h : ox + 1 - h;
        const float2 z0 = rows[(size_t)t * ld + x0], z1 = rows[(size_t)t * ld + x1];
        const int y = c0 + 2 * t;
        const int oy0 = y < h ? y + h : y - h, oy1 = y + 1 < h ? y + 1 + h : y + 1 - h;
        store_stream((float4*)&out[(int64_t)oy0 * n + ox], make_float4(z0.x * s, 0.f, z1.x * s, 0.f));
        store_stream((float4*)&out[(int64_t)oy1 * n + ox], make_float4(z0.y * s, 0.f, z1.y * s, 0.f));
    }
}

// ------------------------------------------------------------ launchers

// Radices for n: 15s, then 10s (or 5s), 9s, and the 2s in even shares of at most 16,
// so that the passes are few; odd radices go first (the first pass writes
// with a lane stride of R, free of bank conflicts when R is odd).
bool make_fft_plan(int n, FftPlan& plan) {
    if (n < 2 || n > kMaxPixels) return false;
    int f[14] = {}, rem = n;
    for (int r : {2, 3, 5, 7, 11, 13})
        while (rem % r == 0) rem /= r, f[r]++;
    if (rem != 1) return false;
    int odd[kMaxFftPasses], even[kMaxFftPasses], n_odd = 0, n_even = 0;
    for (int r : {13, 11, 7})
        while (f[r] > 0) odd[n_odd++] = r, f[r]--;
    while (f[3] > 0 && f[5] > 0) odd[n_odd++] = 15, f[3]--, f[5]--;
    for (; f[5] > 0; f[5]--) {
        if (f[2] > 0) even[n_even++] = 10, f[2]--;
        else odd[n_odd++] = 5;
    }
    for (; f[3] > 1; f[3] -= 2) odd[n_odd++] = 9;
    if (f[3]) {
        if (f[2] > 1) even[n_even++] = 12, f[2] -= 2;
        else if (f[2]) even[n_even++] = 6, f[2]--;
        else odd[n_odd++] = 3;
    }
    for (int passes = (f[2] + 3) / 4; passes > 0; passes--) {
        const int e = (f[2] + passes - 1) / passes;
        even[n_even++] = 1 << e;
        f[2] -= e;
    }
    plan.n = n;
    plan.n_passes = 0;
    plan.cap = kPassValues;
    int span = 1;
    for (int i = 0; i < n_odd + n_even; i++) {
        const int r = i < n_odd ? odd[i] : even[i - n_odd];
        plan.radix[plan.n_passes] = r;
        plan.span[plan.n_passes++] = span;
        plan.cap = std::min(plan.cap, kPassValues / r * r);
        span *= r;
    }
    return true;
}

// Threads of a workgroup (256, 512 or 1024) that transforms `values` values of
// rows of length n at once (at least one row).
static int fft_threads(const FftPlan& plan, int64_t values) {
    int nt = 256;
    while (nt < 1024 && ((int64_t)nt * plan.cap < values || nt * plan.cap < plan.n)) nt *= 2;
    return nt;
}

hipError_t launch_grid_rows_fft(const SetDesc& first, const SetDesc* sets, const int* img_set,
                                int n_sets, const FftPlan& plan, int64_t gi0, int n_img,
                                float* inter, const float* tw, hipStream_t stream) {
    if (n_img == 0) return hipSuccess;
    const int n = plan.n;
    // rows per tile: as many as fit up to 4, and at least ~2048 workgroups in
    // the launch, so that a few images still spread over the whole chip.  The
    // gather of plan entries is latency bound: small tiles keep more
    // workgroups in flight (4 rows measured fastest against 2 to 16 at 180^2).
    const int64_t want = (int64_t)(n / 2 + 1) * n_img / 2048;
    int rb = (int)std::max<int64_t>(1, std::min<int64_t>({(int64_t)n, want, 4}));
    // uniform weighting keeps a count per tile cell beside the tile
    const bool uniform = first.uniform != 0;
    auto lds_of = [&](int r) {
        return sizeof(float2) * ((size_t)r * n + n) + (uniform ? sizeof(unsigned) * (size_t)r * n : 0);
    };
    while (rb > 1 && !lds_fits(lds_of(rb))) rb--;
    const int nt = fft_threads(plan, (int64_t)rb * n);
    const int n_rb = (n / 2 + 1 + rb - 1) / rb;
    const size_t lds = lds_of(rb);
    const int64_t blocks = (int64_t)n_rb * n_img;
    if (!lds_fits(lds) || blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    auto k = n_sets > 1 ? k_grid_rows_fft<true> : k_grid_rows_fft<false>;
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(nt), lds, stream, first, sets, img_set, plan,
                       rb, gi0, (float2*)inter, (const float2*)tw);
    return hipGetLastError();
}

// Direct row pass of the generic kernels (no plan), for dense sets with one
// timestep per channel, as k_grid_rows_direct does it for the register
// sides: one workgroup per image with the whole half plane (plan rows
// 0 .. N/2 of an even or odd side) in LDS, every baseline walked in order
// (direct_walk), then rows 0 .. the highest holding a cell transformed
// (fft_tile) and stored row-major as the generic second pass reads them, and
// the image's row starts written (the rows above empty).  Sides up to
// kDirectMaxSide, whose half plane leaves room for the table.  The count sums
// start at zero (the direct set-up launch).
constexpr int kDirectMaxSide = 186;
static size_t direct_fft_lds_bytes(int n) {
    return sizeof(float2) * ((size_t)(n / 2 + 1) * n + n);
}

template <bool kMulti>
__global__ void __launch_bounds__(kDirectThreads)
k_grid_rows_direct_fft(SetDesc first, const SetDesc* __restrict__ sets,
                       const int* __restrict__ img_set, FftPlan plan, int64_t gi0,
                       float2* __restrict__ inter, const float2* __restrict__ tw) {
    extern __shared__ float4 grd_lds4[];
    const int n = plan.n, h = n / 2;
    float2* tile = (float2*)grd_lds4;          // [h + 1][n]
    float2* twl = tile + (size_t)(h + 1) * n;  // twiddle table copy [n]
    __shared__ int red[kDirectThreads / 64];

    const int li = (int)xcd_order(blockIdx.x, gridDim.x);
    const int64_t gi = gi0 + li;
    const SetDesc sd = set_of<kMulti>(first, sets, img_set, gi);
    const int img = (int)(gi - sd.img_base);
    const int ch = img % sd.g.n_ch;
    for (int i = threadIdx.x; i < (h + 1) * n; i += kDirectThreads) tile[i] = make_float2(0.f, 0.f);
    load_twiddles(twl, tw, n);
    __syncthreads();
    int top = -1;
    const int n_ok = direct_walk<2>(
        sd, img, ch, n, 0, h + 1, (int)threadIdx.x, kDirectThreads,
        [&](int r, int c) { return &tile[__mul24(r, n) + c]; }, nullptr, &top);
    const int n_rows = block_max_int(top, red) + 1;
    const int tot = block_sum_int(n_ok, red);
    if (threadIdx.x == 0 && tot) atomicAdd(&sd.isums[img], (uint32_t)tot);
    __syncthreads();
    // rows 0 .. n_rows - 1 (the highest holding a cell); the row starts tell
    // the second pass that the others are empty
    fft_tile<1>(tile, n_rows, n, plan, twl);
    float2* dst = inter + (int64_t)li * (h + 1) * n;
    for (int i = threadIdx.x; i < n_rows * n; i += kDirectThreads) store_stream(&dst[i], tile[i]);
    int* rsg = sd.row_start + (int64_t)ch * (n + 1);
    for (int i = threadIdx.x; i <= n; i += kDirectThreads) rsg[i] = min(i, n_rows);
}

bool direct_half_plane_fits(int n) {
    return n % 2 == 0 && n <= kMaxPixels && lds_fits(sizeof(float2) * (size_t)(n / 2 + 1) * n);
}

bool direct_row_pass_fits(int n) {
    if (batch_reg_supported(n)) return batch_direct_supported(n);
    return n >= 2 && n <= kDirectMaxSide && lds_fits(direct_fft_lds_bytes(n));
}

hipError_t launch_grid_rows_direct_fft(const SetDesc& first, const SetDesc* sets,
                                       const int* img_set, int n_sets, const FftPlan& plan,
                                       int64_t gi0, int n_img, float* inter, const float* tw,
                                       hipStream_t stream) {
    if (n_img == 0) return hipSuccess;
    const size_t lds = direct_fft_lds_bytes(plan.n);
    if (!lds_fits(lds)) return hipErrorInvalidConfiguration;
    auto k = n_sets > 1 ? k_grid_rows_direct_fft<true> : k_grid_rows_direct_fft<false>;
    hipLaunchKernelGGL(k, dim3((unsigned)n_img), dim3(kDirectThreads), lds, stream, first, sets,
                       img_set, plan, gi0, (float2*)inter, (const float2*)tw);
    return hipGetLastError();
}

// Cells of a group's sets for the row pass below, as the plan's count pass packs
// them: SetDesc::entries holds kb_cell_stride(n_bl) words per channel.
__global__ void __launch_bounds__(256)
k_kb_cells(const SetDesc* __restrict__ sets) {
    const SetDesc sd = sets[blockIdx.z];
    const int n_bl = sd.g.n_bl, n = sd.n_pixels, stride = kb_cell_stride(n_bl);
    for (int ch = blockIdx.y; ch < sd.g.n_ch; ch += gridDim.y) {
        const CellUnit cu(sd.g.freq_hz[ch], sd);
#pragma unroll
        for (int k = 0; k < kCellsPer; k++) {
            const int bl = (int)(blockIdx.x * kCellsPer + k) * 256 + (int)threadIdx.x;
            if (bl >= stride) break;
            uint32_t packed = kNoCell;
            int up, vp;
            if (bl < n_bl && !sd.flags[bl] && plan_cell(sd.u_m[bl], sd.v_m[bl], cu, sd, up, vp))
                packed = ((uint32_t)wrap_index(up, n) << 16) | (uint32_t)wrap_index(vp, n);
            sd.entries[(int64_t)ch * stride + bl] = packed;
        }
    }
}

hipError_t launch_kb_cells(const SetDesc* sets, int n_sets, int max_bl, int max_ch,
                           hipStream_t stream) {
    if (n_sets == 0 || max_bl == 0 || max_ch == 0) return hipSuccess;
    for (int s0 = 0; s0 < n_sets; s0 += kMaxGridZ) {
        hipLaunchKernelGGL(k_kb_cells,
                           dim3(cell_blocks(kb_cell_stride(max_bl)), (unsigned)std::min(max_ch, 65535),
                                (unsigned)std::min(n_sets - s0, kMaxGridZ)),
                           dim3(256), 0, stream, sets + s0);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Row pass of convolutional gridding, any side: workgroup (slab, image) owns
// `rb` consecutive plan rows (grid columns u) of 0 .. N/2, accumulates their
// footprints in FP64 (kb_accumulate), transforms each row (the planes become
// the rows and their twiddles) and writes it, row-major or in the
// column-blocked layout of the register second pass.  The slabs nearest u = 0,
// the dense core, are launched first.  Bound by the LDS atomics: the LDS is busy
// 83 % of the time at 256^2 (20 clocks per wavefront instruction, a third of them
// bank conflicts).  Against a gather of plan entries with FP32 cells (a window of
// the plane at 256^2), whole calls: 256 x 256^2, K = 7 1336 -> 820 us, 64 x 180^2
// 1627 -> 313, 100 x 300^2, K = 9 2973 -> 578, 32 x 1024^2 418 -> 270, 4 x 4096^2
// 880 -> 568.
constexpr int kKbRowThreads = 1024;
template <int kX, bool kMulti>
__global__ void __launch_bounds__(kKbRowThreads)
k_grid_rows_kb(SetDesc first, const SetDesc* __restrict__ sets, const int* __restrict__ img_set,
               FftPlan plan, int rb, int64_t gi0, int n_img, float2* __restrict__ inter,
               const float2* __restrict__ tw, int blocked) {
    extern __shared__ float4 grk_lds4[];
    const int n = plan.n, h = n / 2, tid = threadIdx.x;
    double* re = (double*)grk_lds4;      // [rb][n]
    double* im = re + (size_t)rb * n;    // [rb][n]
    uint32_t* queues = (uint32_t*)(im + (size_t)rb * n);
    __shared__ int red[kKbRowThreads / 64];
    const int li = (int)(blockIdx.x % (unsigned)n_img);
    const int r0 = (int)(blockIdx.x / (unsigned)n_img) * rb, nr = min(rb, h + 1 - r0);
    const int64_t gi = gi0 + li;
    const SetDesc sd = set_of<kMulti>(first, sets, img_set, gi);
    const GatherArgs& g = sd.g;
    const int img = (int)(gi - sd.img_base), ch = img % g.n_ch;
    for (int i = tid; i < nr * n; i += kKbRowThreads) re[i] = im[i] = 0.0;
    __syncthreads();
    const StageGrid sg{nullptr, sd.u_m, sd.v_m, sd.flags, g.freq_hz, sd.du, sd.dv, sd.min_uv,
                       g.n_bl, g.n_ch, n, g.pol, nullptr, nullptr};
    const float2* rec = (const float2*)g.vis + 4 * ((int64_t)img * g.n_bl);
    const double nu = g.freq_hz[ch];
    const int p0 = g.pol == 1 ? 3 : (g.pol == 3 ? 1 : 0);
    const int p1 = g.pol == 3 ? 2 : 3;
    const int stride = kb_cell_stride(g.n_bl);
    int n_ok = 0;
    const int queued = kb_accumulate<kKbRowThreads, kX, true, true>(
        sg, wavelength_of(nu), sd.kb_size, sd.kb_table, sd.entries + (int64_t)ch * stride, stride,
        r0, nr, re, im, nullptr, false, queues,
        [&](int bl) {
            float2 v = select_pol2(rec[4 * (size_t)bl + p0],
                                   g.pol >= 2 ? rec[4 * (size_t)bl + p1] : make_float2(0.f, 0.f),
                                   g.pol);
            if (g.corrections) v = cmul(v, unit_phasor(g.phase_coef[bl] * (nu / kVelLight)));
            return v;
        },
        // a nearest cell stands for its mirror too, except in the
        // self-conjugate rows 0 and N/2, which hold both
        [&](int r, int) { n_ok += (r0 + r == 0 || 2 * (r0 + r) == n) ? 1 : 2; });
    const int tot = block_sum_int(n_ok, red);
    if (tid == 0 && tot) atomicAdd(&sd.isums[img], (uint32_t)tot);
    const bool any = __syncthreads_or(queued);
    // each cell's two sums become one FP32 complex value in its re slot
    for (int i = tid; i < nr * n; i += kKbRowThreads) {
        const float2 c = make_float2((float)re[i], (float)im[i]);
        *(float2*)&re[i] = c;
    }
    __syncthreads();
    const float2* rows = (float2*)re;
    if (any) {  // (uniform) else zeros
        float2* twl = (float2*)im;  // (rb >= 1 rows of n)
        load_twiddles(twl, tw, n);
        __syncthreads();
        fft_tile<1>((float2*)re, nr, n, plan, twl);
    }
    const int64_t h1 = h + 1;
    if (!blocked) {
        float2* dst = inter + ((int64_t)li * h1 + r0) * n;
        for (int i = tid; i < nr * n; i += kKbRowThreads) store_stream(&dst[i], rows[i]);
        return;
    }
    // element (v, x) at ((x / 32) (N/2+1) + v) 32 + x % 32 (n a power of two)
    float2* dst = inter + (int64_t)li * h1 * n + (int64_t)r0 * kInterBlockCols;
    for (int i = tid; i < nr * n; i += kKbRowThreads) {
        const int r = i / n, x = i - r * n;
        store_stream(&dst[(int64_t)(x / kInterBlockCols) * h1 * kInterBlockCols +
                          r * kInterBlockCols + x % kInterBlockCols],
                     rows[i]);
    }
}

hipError_t launch_grid_rows_kb(const SetDesc& first, const SetDesc* sets, const int* img_set,
                               int n_sets, const FftPlan& plan, int64_t gi0, int n_img,
                               float* inter, const float* tw, bool blocked, hipStream_t stream) {
    if (n_img == 0) return hipSuccess;
    if (first.kb_size < 1) return hipErrorInvalidValue;
    const int n = plan.n, h1 = n / 2 + 1;
    // as many rows as a CU's LDS holds (the taller the slab, the fewer slabs
    // compute a footprint's weights again), fewer while the images leave under
    // four workgroups per CU (rows above the array's reach have no work)
    const size_t queue = kb_queue_bytes(kKbRowThreads);
    int rb = (int)std::min<int64_t>(h1, (g_lds_limit - (int64_t)queue) / (16 * (int64_t)n));
    if (rb < 1) return hipErrorInvalidConfiguration;
    while (rb > 2 && (int64_t)n_img * ((h1 + rb - 1) / rb) < 4 * device_cu_count()) rb = (rb + 1) / 2;
    const size_t lds = (size_t)16 * n * rb + queue;
    const int64_t blocks = (int64_t)n_img * ((h1 + rb - 1) / rb);
    if (!lds_fits(lds) || blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    // (a group's sets share kb_size)
    auto pick = [&](auto kx) {
        constexpr int X = decltype(kx)::value;
        return n_sets > 1 ? k_grid_rows_kb<X, true> : k_grid_rows_kb<X, false>;
    };
    const auto k = first.kb_size <= 8 ? pick(std::integral_constant<int, 8>{})
                                      : pick(std::integral_constant<int, 0>{});
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(kKbRowThreads), lds, stream, first, sets,
                       img_set, plan, rb, gi0, n_img, (float2*)inter, (const float2*)tw,
                       blocked ? 1 : 0);
    return hipGetLastError();
}

// Second pass of the generic batched path for odd N = 2m + 1, from the
// row-major row-pass buffer inter[img][p][y], plan rows p = 0 .. m.  As for
// even N the images are real, so one complex FFT over p of z = c_y + i
// c_{y+1} gives image rows y and y + 1, with rows N - p (p = 1 .. m: an odd
// side has no self-conjugate middle row) the conjugates of rows p; column
// pairs are slots s = 0 .. m (y = 2s), and the last column N - 1 pairs with
// zero columns.  A workgroup owns `pairs` slots; 8-byte accesses (odd rows
// are not 16-byte aligned); the store applies the odd-side fftshift
// (shift_index: p <-> p + m + 1 for p < m, the middle element fixed,
// src/pacer_imager.cpp:30-35,110-128) element by element.
template <bool kMulti>
__global__ void __launch_bounds__(1024)
k_cols_half_odd(SetDesc first, const SetDesc* __restrict__ sets, const int* __restrict__ img_set,
                FftPlan plan, int pairs, int64_t gi0, const float2* __restrict__ inter,
                const float2* __restrict__ tw) {
    extern __shared__ float4 cho_lds4[];
    const int n = plan.n, h = n / 2;
    const int ld = n + 1;
    float2* rows = (float2*)cho_lds4;         // [pairs][ld]
    float2* twl = rows + (size_t)pairs * ld;  // twiddle table copy [n]
    unsigned char* nonempty = (unsigned char*)(twl + n);
    load_twiddles(twl, tw, n);

    const int n_slots = h + 1;
    const int n_cb = (n_slots + pairs - 1) / pairs;
    const unsigned bid = xcd_order(blockIdx.x, gridDim.x);
    const int cbk = (int)(bid % n_cb);
    const int li = (int)(bid / n_cb);
    const int64_t gi = gi0 + li;
    const SetDesc sd = set_of<kMulti>(first, sets, img_set, gi);
    if (!sd.images) return;  // uniform per workgroup
    const int img = (int)(gi - sd.img_base);
    const uint32_t count = sd.isums[img];
    if (cbk == 0 && threadIdx.x == 0 && sd.count_sums) sd.count_sums[img] = (double)count;
    const int* rsg = sd.row_start + (int64_t)(img % sd.g.n_ch) * (n + 1);
    const float empty = sd.uniform ? __builtin_nanf("") : 0.f;  // rows without entries
    for (int i = threadIdx.x; i <= h; i += blockDim.x)
        nonempty[i] = sd.all_rows || rsg[i + 1] != rsg[i];
    __syncthreads();

    const int s0 = cbk * pairs;
    const int np = min(pairs, n_slots - s0);  // slots of this workgroup (uniform)
    const float2* src = inter + (int64_t)li * (h + 1) * n;
    const int stage = (h + 1) * np;
    for (int i = threadIdx.x; i < stage; i += (int)blockDim.x) {
        const int v = i / np, t = i % np;
        const int y = 2 * (s0 + t);
        const bool has_b = y + 1 < n;  // the last column pairs with zeros
        float2 a = make_float2(empty, empty);
        float2 b = has_b ? make_float2(empty, empty) : make_float2(0.f, 0.f);
        if (nonempty[v]) {
            a = src[(int64_t)v * n + y];
            if (has_b) b = src[(int64_t)v * n + y + 1];
        }
        float2* zr = rows + (size_t)t * ld;
        zr[v] = make_float2(a.x - b.y, a.y + b.x);                   // c_y[v] + i c_{y+1}[v]
        if (v > 0) zr[n - v] = make_float2(a.x + b.y, b.x - a.y);    // row N - v
    }
    __syncthreads();
    fft_tile<1>(rows, np, ld, plan, twl);
    const float s = (float)(1.0 / (double)count);
    float2* out = sd.images + (int64_t)img * n * n;
    for (int i = threadIdx.x; i < np * n; i += (int)blockDim.x) {
        const int t = i / n, x = i % n;
        const int y = 2 * (s0 + t);
        const float2 z = rows[(size_t)t * ld + x];
        const int ox = shift_index(x, n);
        store_stream(&out[(int64_t)shift_index(y, n) * n + ox], make_float2(z.x * s, 0.f));
        if (y + 1 < n)
            store_stream(&out[(int64_t)shift_index(y + 1, n) * n + ox], make_float2(z.y * s, 0.f));
    }
}

// Pairs of buffer columns (image rows) per workgroup of the second pass: 8
// (128-byte runs of the buffer's rows) or, up to 256, 16, while the workgroup's threads hold them in
// registers and two workgroups, or one, fit a CU's LDS; fewer while the launch
// has under 512 workgroups (two per CU).
static int half_pairs(const FftPlan& plan, int n_slots, int64_t n_img) {
    const int n = plan.n;
    int pairs = std::min(n <= 256 ? 16 : 8, n_slots);
    auto lds_of = [&](int p) { return sizeof(float2) * ((size_t)p * (n + 1) + n) + n / 2 + 1; };
    while (pairs > 1 && ((int64_t)pairs * n > 1024 * plan.cap ||
                         (int64_t)lds_of(pairs) > g_lds_limit ||
                         (pairs > 4 && 2 * (int64_t)lds_of(pairs) > g_lds_limit) ||
                         (int64_t)((n_slots + pairs - 1) / pairs) * n_img < 512))
        pairs--;
    return pairs;
}

hipError_t launch_cols_half(const SetDesc& first, const SetDesc* sets, const int* img_set,
                            int n_sets, const FftPlan& plan, int64_t gi0, int n_img,
                            const float* inter, const float* tw, hipStream_t stream) {
    if (n_img == 0) return hipSuccess;
    const int n = plan.n;
    // odd N: the last column pairs with zeros
    const int n_slots = n % 2 ? n / 2 + 1 : n / 2;
    const int pairs = half_pairs(plan, n_slots, n_img);
    const size_t lds = sizeof(float2) * ((size_t)pairs * (n + 1) + n) + (size_t)(n / 2 + 1);
    const int64_t blocks = (int64_t)((n_slots + pairs - 1) / pairs) * n_img;
    if (!lds_fits(lds) || blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    const bool multi = n_sets > 1;
    auto k = n % 2 ? (multi ? k_cols_half_odd<true> : k_cols_half_odd<false>)
                   : (multi ? k_cols_half<true> : k_cols_half<false>);
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(fft_threads(plan, (int64_t)pairs * n)), lds,
                       stream, first, sets, img_set, plan, pairs, gi0, (const float2*)inter,
                       (const float2*)tw);
    return hipGetLastError();
}

__global__ void k_isums_to_double(const uint32_t* __restrict__ isums, double* __restrict__ sums,
                                  int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) sums[i] = (double)isums[i];
}

hipError_t launch_isums_to_double(const uint32_t* isums, double* sums, int n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_isums_to_double, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                       isums, sums, n);
    return hipGetLastError();
}

hipError_t set_kernel_attributes() {
    // Allow the dynamic LDS sizes used above.
    const int max_lds = (int)g_lds_limit;
    hipError_t e = hipSuccess;
    auto set = [&](const void* f) {
        hipError_t r = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
        if (r != hipSuccess && e == hipSuccess) e = r;
    };
    set((const void*)k_grid_half_direct);
    set((const void*)k_grid_rows_fft<false>);
    set((const void*)k_grid_rows_fft<true>);
    set((const void*)k_cols_half<false>);
    set((const void*)k_cols_half<true>);
    set((const void*)k_cols_half_odd<false>);
    set((const void*)k_cols_half_odd<true>);
    set((const void*)k_grid_rows_direct_fft<false>);
    set((const void*)k_grid_rows_direct_fft<true>);
    set((const void*)k_grid_slabs);
    set((const void*)k_grid_kb_slabs<8>);
    set((const void*)k_grid_kb_slabs<0>);
#define X(K) \
    set((const void*)k_grid_rows_kb<K, true>);        \
    set((const void*)k_grid_rows_kb<K, false>);
    X(8) X(0)
#undef X
    set((const void*)k_grid_half_rows);
    set((const void*)k_plan_count);
    set((const void*)k_plan_scatter);
    return e;
}

}  // namespace blink
