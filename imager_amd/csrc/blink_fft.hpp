// In-house LDS-staged mixed-radix FFT for gfx950, any N = 2^a 3^b 5^c 7^d 11^e
// 13^f.
//
// A workgroup transforms the rows of an LDS tile together (fft_tile).  Each pass
// is a radix-R Stockham autosort step (Govindaraju et al., "High Performance
// Discrete Fourier Transforms on Graphics Processors", SC'08): butterfly j
// reads x[j + r*N/R], multiplies by the twiddle w^(r*(j mod Ns)) of the
// current span Ns*R, does a radix-R DFT and writes
// y[(j/Ns)*Ns*R + (j mod Ns) + r*Ns].  The workgroup reads a whole pass into
// registers before it writes, so the rows stay where they are.
// Radices up to 16, composite odd ones among them (6, 9, 10, 12, 15), keep the
// passes few: each costs an LDS read and write of the tile and two barriers.
//
// Twiddles come from a table tw[m] = exp(+2 pi i m / N), m < N, built on the
// host in double and rounded to FP32 (accurate to 1/2 ulp); the forward
// direction uses the conjugate.
#pragma once

#include "blink_device.hpp"

namespace blink {

constexpr int kMaxFftPasses = 16;

// Values a thread of fft_tile keeps in registers during a pass: kPassValues / R
// butterflies of radix R.
constexpr int kPassValues = 20;

struct FftPlan {
    int n;                       // transform length
    int n_passes;
    int radix[kMaxFftPasses];    // radix of each pass
    int span[kMaxFftPasses];     // Ns before each pass (product of previous radices)
    int cap;                     // values per thread every pass can hold (fft_tile)
};

// Synchronisation of the lanes working on one row.
template <bool kBlockTeam>
__device__ __forceinline__ void team_sync() {
    if constexpr (kBlockTeam) {
        __syncthreads();
    } else {
        // One wavefront executes its LDS operations in order; the fences keep
        // the compiler from moving LDS accesses across this point.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// Radix-R DFTs with sign S: y[k] = sum_r x[r] exp(S 2 pi i r k / R).
template <int S>
__device__ __forceinline__ void dft2(float2* x) {
    const float2 a = x[0], b = x[1];
    x[0] = cadd(a, b);
    x[1] = csub(a, b);
}

template <int S>
__device__ __forceinline__ float2 rot_s(float2 a) {  // S * i * a
    return S > 0 ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

template <int S>
__device__ __forceinline__ void dft4(float2* x) {
    const float2 a = cadd(x[0], x[2]), b = csub(x[0], x[2]);
    const float2 c = cadd(x[1], x[3]), d = csub(x[1], x[3]);
    const float2 id = rot_s<S>(d);
    x[0] = cadd(a, c);
    x[2] = csub(a, c);
    x[1] = cadd(b, id);
    x[3] = csub(b, id);
}

template <int S>
__device__ __forceinline__ void dft3(float2* x) {
    constexpr float kC = -0.5f;
    constexpr float kS = 0.86602540378443864676f;  // sqrt(3)/2
    const float2 t = cadd(x[1], x[2]);
    const float2 d = csub(x[1], x[2]);
    const float2 m = make_float2(x[0].x + kC * t.x, x[0].y + kC * t.y);
    const float2 r = rot_s<S>(cscale(d, kS));
    x[0] = cadd(x[0], t);
    x[1] = cadd(m, r);
    x[2] = csub(m, r);
}

template <int S>
__device__ __forceinline__ void dft5(float2* x) {
    constexpr float c1 = 0.30901699437494742410f;   // cos(2 pi/5)
    constexpr float c2 = -0.80901699437494742410f;  // cos(4 pi/5)
    constexpr float s1 = 0.95105651629515357212f;   // sin(2 pi/5)
    constexpr float s2 = 0.58778525229247312917f;   // sin(4 pi/5)
    const float2 t1 = cadd(x[1], x[4]), t2 = cadd(x[2], x[3]);
    const float2 t3 = csub(x[1], x[4]), t4 = csub(x[2], x[3]);
    const float2 a1 = make_float2(x[0].x + c1 * t1.x + c2 * t2.x, x[0].y + c1 * t1.y + c2 * t2.y);
    const float2 a2 = make_float2(x[0].x + c2 * t1.x + c1 * t2.x, x[0].y + c2 * t1.y + c1 * t2.y);
    const float2 b1 = rot_s<S>(make_float2(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y));
    const float2 b2 = rot_s<S>(make_float2(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y));
    x[0] = cadd(x[0], cadd(t1, t2));
    x[1] = cadd(a1, b1);
    x[4] = csub(a1, b1);
    x[2] = cadd(a2, b2);
    x[3] = csub(a2, b2);
}

// exp(S 2 pi i k / 16), k < 8 (folds to constants once loops are unrolled).
template <int S>
__device__ __forceinline__ float2 root16(int k) {
    float c, sn;
    switch (k) {
        case 0: c = 1.0f; sn = 0.0f; break;
        case 1: c = 0.92387953251128675613f; sn = 0.38268343236508977173f; break;
        case 2: c = 0.70710678118654752440f; sn = 0.70710678118654752440f; break;
        case 3: c = 0.38268343236508977173f; sn = 0.92387953251128675613f; break;
        case 4: c = 0.0f; sn = 1.0f; break;
        case 5: c = -0.38268343236508977173f; sn = 0.92387953251128675613f; break;
        case 6: c = -0.70710678118654752440f; sn = 0.70710678118654752440f; break;
        default: c = -0.92387953251128675613f; sn = 0.38268343236508977173f; break;
    }
    return make_float2(c, S > 0 ? sn : -sn);
}

template <int S>
__device__ __forceinline__ void dft8(float2* x) {
    float2 e[4] = {x[0], x[2], x[4], x[6]};
    float2 o[4] = {x[1], x[3], x[5], x[7]};
    dft4<S>(e);
    dft4<S>(o);
    o[1] = cmul(o[1], root16<S>(2));
    o[2] = rot_s<S>(o[2]);
    o[3] = cmul(o[3], root16<S>(6));
#pragma unroll
    for (int k = 0; k < 4; k++) {
        x[k] = cadd(e[k], o[k]);
        x[k + 4] = csub(e[k], o[k]);
    }
}

template <int S>
__device__ __forceinline__ void dft16(float2* x) {
    float2 e[8], o[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        e[k] = x[2 * k];
        o[k] = x[2 * k + 1];
    }
    dft8<S>(e);
    dft8<S>(o);
#pragma unroll
    for (int k = 1; k < 8; k++) o[k] = (k == 4) ? rot_s<S>(o[k]) : cmul(o[k], root16<S>(k));
#pragma unroll
    for (int k = 0; k < 8; k++) {
        x[k] = cadd(e[k], o[k]);
        x[k + 8] = csub(e[k], o[k]);
    }
}

// exp(2 pi i m / N) for the constants of the odd radices.
template <int N>
struct Root;
template <> struct Root<7> {
    static constexpr float c[7] = {
        1.00000000000000000f, 0.62348980185873359f, -0.22252093395631434f, -0.90096886790241903f,
        -0.90096886790241915f, -0.22252093395631459f, 0.62348980185873337f};
    static constexpr float s[7] = {
        0.00000000000000000f, 0.78183148246802980f, 0.97492791218182362f, 0.43388373911755823f,
        -0.43388373911755801f, -0.97492791218182362f, -0.78183148246802991f};
};
template <> struct Root<9> {
    static constexpr float c[9] = {
        1.00000000000000000f, 0.76604444311897801f, 0.17364817766693041f, -0.49999999999999978f,
        -0.93969262078590832f, -0.93969262078590843f, -0.50000000000000044f, 0.17364817766692997f,
        0.76604444311897779f};
    static constexpr float s[9] = {
        0.00000000000000000f, 0.64278760968653925f, 0.98480775301220802f, 0.86602540378443871f,
        0.34202014332566888f, -0.34202014332566866f, -0.86602540378443837f, -0.98480775301220813f,
        -0.64278760968653958f};
};
template <> struct Root<11> {
    static constexpr float c[11] = {
        1.00000000000000000f, 0.84125353283118121f, 0.41541501300188644f, -0.14231483827328500f,
        -0.65486073394528499f, -0.95949297361449737f, -0.95949297361449748f, -0.65486073394528521f,
        -0.14231483827328523f, 0.41541501300188605f, 0.84125353283118121f};
    static constexpr float s[11] = {
        0.00000000000000000f, 0.54064081745559756f, 0.90963199535451833f, 0.98982144188093280f,
        0.75574957435425827f, 0.28173255684142967f, -0.28173255684142939f, -0.75574957435425816f,
        -0.98982144188093268f, -0.90963199535451855f, -0.54064081745559744f};
};
template <> struct Root<13> {
    static constexpr float c[13] = {
        1.00000000000000000f, 0.88545602565320991f, 0.56806474673115592f, 0.12053668025532301f,
        -0.35460488704253545f, -0.74851074817110119f, -0.97094181742605201f, -0.97094181742605212f,
        -0.74851074817110130f, -0.35460488704253590f, 0.12053668025532320f, 0.56806474673115481f,
        0.88545602565321002f};
    static constexpr float s[13] = {
        0.00000000000000000f, 0.46472317204376851f, 0.82298386589365635f, 0.99270887409805397f,
        0.93501624268541483f, 0.66312265824079519f, 0.23931566428755768f, -0.23931566428755743f,
        -0.66312265824079497f, -0.93501624268541472f, -0.99270887409805397f, -0.82298386589365702f,
        -0.46472317204376840f};
};

// Radix-R DFT for a prime R (7, 11, 13) with its real symmetry: the pairs
// x[m] +- x[R - m] meet the cosines and sines of 2 pi m k / R once for k and
// R - k.
template <int S, int R>
__device__ __forceinline__ void dft_prime(float2* x) {
    constexpr int H = R / 2;
    float2 p[H + 1], d[H + 1];
    float2 sum = x[0];
#pragma unroll
    for (int m = 1; m <= H; m++) {
        p[m] = cadd(x[m], x[R - m]);
        d[m] = rot_s<S>(csub(x[m], x[R - m]));  // S i (x[m] - x[R - m])
        sum = cadd(sum, p[m]);
    }
    float2 y[R];
    y[0] = sum;
#pragma unroll
    for (int k = 1; k <= H; k++) {
        float2 re = x[0], im = make_float2(0.f, 0.f);
#pragma unroll
        for (int m = 1; m <= H; m++) {
            const float c = Root<R>::c[(m * k) % R], sn = Root<R>::s[(m * k) % R];
            re = make_float2(re.x + c * p[m].x, re.y + c * p[m].y);
            im = make_float2(im.x + sn * d[m].x, im.y + sn * d[m].y);
        }
        y[k] = cadd(re, im);
        y[R - k] = csub(re, im);
    }
#pragma unroll
    for (int k = 0; k < R; k++) x[k] = y[k];
}

template <int S, int R>
__device__ __forceinline__ void dft_any(float2* x);

// Inverse of a modulo m.
__host__ __device__ constexpr int inverse_mod(int a, int m) {
    for (int i = 1; i < m; i++)
        if (a * i % m == 1) return i;
    return 1;
}

// Radix A B with coprime A, B by the prime-factor map (no twiddles): inputs
// B n1 + A n2, outputs at the k with k = k1 mod A, k = k2 mod B (Good, 1958).
template <int S, int A, int B>
__device__ __forceinline__ void dft_coprime(float2* x) {
    constexpr int N = A * B;
    float2 t[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; n2++) {
#pragma unroll
        for (int n1 = 0; n1 < A; n1++) t[n2][n1] = x[(B * n1 + A * n2) % N];
        dft_any<S, A>(t[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) {
        float2 u[B];
#pragma unroll
        for (int n2 = 0; n2 < B; n2++) u[n2] = t[n2][k1];
        dft_any<S, B>(u);
#pragma unroll
        for (int k2 = 0; k2 < B; k2++)
            x[(B * inverse_mod(B % A, A) * k1 + A * inverse_mod(A % B, B) * k2) % N] = u[k2];
    }
}

template <int S>
__device__ __forceinline__ void dft9(float2* x) {
    float2 t[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; n2++) {
#pragma unroll
        for (int n1 = 0; n1 < 3; n1++) t[n2][n1] = x[3 * n1 + n2];
        dft3<S>(t[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < 3; k1++) {
        float2 u[3];
#pragma unroll
        for (int n2 = 0; n2 < 3; n2++) {
            const float sn = S > 0 ? Root<9>::s[n2 * k1] : -Root<9>::s[n2 * k1];
            u[n2] = n2 * k1 ? cmul(t[n2][k1], make_float2(Root<9>::c[n2 * k1], sn)) : t[n2][k1];
        }
        dft3<S>(u);
#pragma unroll
        for (int k2 = 0; k2 < 3; k2++) x[k1 + 3 * k2] = u[k2];
    }
}

template <int S, int R>
__device__ __forceinline__ void dft_any(float2* x) {
    if constexpr (R == 2) dft2<S>(x);
    else if constexpr (R == 3) dft3<S>(x);
    else if constexpr (R == 4) dft4<S>(x);
    else if constexpr (R == 5) dft5<S>(x);
    else if constexpr (R == 6) dft_coprime<S, 2, 3>(x);
    else if constexpr (R == 8) dft8<S>(x);
    else if constexpr (R == 9) dft9<S>(x);
    else if constexpr (R == 10) dft_coprime<S, 2, 5>(x);
    else if constexpr (R == 12) dft_coprime<S, 4, 3>(x);
    else if constexpr (R == 15) dft_coprime<S, 3, 5>(x);
    else if constexpr (R == 16) dft16<S>(x);
    else dft_prime<S, R>(x);
}

// One Stockham pass of radix R over `rows` rows of the tile (row stride ld), in
// place: every butterfly of the workgroup is read and transformed in
// registers, then all of them are written.
template <int S, int R>
__device__ __forceinline__ void tile_pass(float2* __restrict__ tile, int rows, int ld, int n, int ns,
                                          const float2* __restrict__ tw) {
    constexpr int B = kPassValues / R;
    const int nb = n / R, total = rows * nb, nt = (int)blockDim.x;
    const int tstep = n / (ns * R);  // twiddle index step per (r * k)
    // quotients by one FP32 product: exact, as the dividends stay below 2^15
    // and lie half a unit from the multiples of the divisor
    const float inv_nb = 1.0f / (float)nb, inv_ns = 1.0f / (float)ns;
    float2 v[B][R];
    int at[B];
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int j = (int)threadIdx.x + b * nt;
        at[b] = -1;
        if (j >= total) continue;
        const int row = (int)(((float)j + 0.5f) * inv_nb), jj = j - row * nb;
        const int q = (int)(((float)jj + 0.5f) * inv_ns), k = jj - q * ns;
        const float2* src = tile + row * ld + jj;
#pragma unroll
        for (int r = 0; r < R; r++) v[b][r] = src[r * nb];
        if (ns > 1) {
#pragma unroll
            for (int r = 1; r < R; r++) {
                float2 w = tw[r * k * tstep];
                if (S < 0) w.y = -w.y;
                v[b][r] = cmul(v[b][r], w);
            }
        }
        dft_any<S, R>(v[b]);
        at[b] = row * ld + q * ns * R + k;
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; b++)
        if (at[b] >= 0)
#pragma unroll
            for (int r = 0; r < R; r++) tile[at[b] + r * ns] = v[b][r];
    __syncthreads();
}

// Transforms rows 0 .. rows - 1 of an LDS tile in place (row stride ld), all
// threads of the workgroup together; blockDim.x * plan.cap >= n.  Called and
// left with the tile synchronised.  All rows advance through a pass at once, so
// that a pass is one read, one write and two barriers whatever the number of
// rows, and no second buffer is needed.  (A team of lanes per row with its own
// scratch row, radices up to 16 without composites, left most of a workgroup
// waiting at sides above 300: second pass of 20 x 1500^2 427 us; the whole
// batched call there 601 -> 226 us, 16 x 4000^2 2964 -> 1336, 100 x 360^2 209 ->
// 139, 120 x 700^2 555 -> 274; stage calls at 1 x 4004^2 594 -> 328.)
template <int S>
__device__ __forceinline__ void fft_tile(float2* __restrict__ tile, int rows, int ld,
                                         const FftPlan& plan, const float2* __restrict__ tw) {
    const int n = plan.n, group = (int)blockDim.x * plan.cap / n;  // rows per pass
    for (int r0 = 0; r0 < rows; r0 += group) {
        float2* t = tile + r0 * ld;
        const int nr = min(group, rows - r0);
        for (int p = 0; p < plan.n_passes; p++) {
            // (opaque to the compiler, which would otherwise move the indexes
            // of every radix out of the loop, and spill them)
            int len = __builtin_amdgcn_readfirstlane(n);
            asm volatile("" : "+s"(len));
            const int ns = plan.span[p];
            switch (plan.radix[p]) {
#define BLINK_PASS(R) \
    case R: tile_pass<S, R>(t, nr, ld, len, ns, tw); break;
                BLINK_PASS(2) BLINK_PASS(3) BLINK_PASS(4) BLINK_PASS(5) BLINK_PASS(6)
                BLINK_PASS(7) BLINK_PASS(8) BLINK_PASS(9) BLINK_PASS(10) BLINK_PASS(11)
                BLINK_PASS(12) BLINK_PASS(13) BLINK_PASS(15)
                default: tile_pass<S, 16>(t, nr, ld, len, ns, tw); break;
#undef BLINK_PASS
            }
        }
    }
}

// Copies the twiddle table of a side to LDS.
__device__ __forceinline__ void load_twiddles(float2* __restrict__ twl, const float2* __restrict__ tw,
                                              int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) twl[i] = tw[i];
}

}  // namespace blink
