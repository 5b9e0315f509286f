// afft_kernels.hip -- gfx950 kernels of the FFT engine.
//
//   afft_stockham<Real, E, N, ...>  compile-time tiles of strided axes: N = 128 ... 1024 in Complex
//                                   Float, 256 in Complex Double
//   afft_chirp                      pointwise stages of multi-kernel chirp-z transforms
//   afft_gen_*                      FP64 twiddle / chirp generation, rounded to the element type
//
// The path is HBM-bound (about 0.3 log2 N flop per byte), so nothing here uses MFMA: the design
// goal is one HBM read and one HBM write per element per launch, with the passes of a transform
// exchanged through LDS.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "afft_device.hpp"
#include "afft_internal.hpp"
#include "afft_mixed.hpp"

namespace afft {

// ----------------------------------------------------------------------------------------------
// Column tiles of strided axes with compile-time radices Rs (CtStockham, the row kernels' passes) over
// the interleaved tile, twiddle bases loaded once from the table W_N^m.  Other lengths run the
// mixed-radix kernel (afft_mixed_kernel.hpp).
// TWG: the four-step twiddles on store come from the precomputed grid post_tab, loaded with the
// data so that they are in flight during the transform instead of in front of every store (the
// middle pass of the split six-step); otherwise from the two-level table post_hi / post_lo.

template <typename Real, int E, int N, bool TWG, int... Rs>
__global__ void __launch_bounds__(max_block_threads(sizeof(Real) == 8, E)) afft_stockham(const FftArgs a)
{
    using V = typename cplx_of<Real>::type;
    extern __shared__ __align__(16) unsigned char afft_smem[];
    V *lds = reinterpret_cast<V *>(afft_smem);

    constexpr int T = N / E;
    static_assert(T % 2 == 0, "elements i T apart share their centring sign");
    const int c = threadIdx.x % a.C, t = threadIdx.x / a.C; // neighbouring lanes, neighbouring columns
    CtStockham<V, N, E, Rs...> ct;
    ct.load(reinterpret_cast<const V *>(a.pw), t);
    const int64_t tile = a.xcd_remap ? xcd_tile(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x;
    const int64_t j = tile * a.C + c;
    const bool active = j < a.ntrans;

    int64_t j0, j1, j2;
    addr_split(a.div, a.ain, j, j0, j1, j2);
    const int64_t jl = a.post_level ? j1 : j0; // the four-step twiddle's index
    V reg[E];
    if (active) {
        const V *in = reinterpret_cast<const V *>(a.in);
        const int64_t base = addr_of(a.ain, j0, j1, j2);
        const bool nt = a.nt_in;
#pragma unroll
        for (int i = 0; i < E; ++i) {
            V v = c_load(in + base + (int64_t)(t + i * T) * a.ain.es, nt);
            reg[i] = a.conj_in ? c_conj(v) : v;
        }
        // apart from the loads, which stay one batch of independent instructions (T is even)
        if (a.sg_in.on) sign_run<E>(reg, a.sg_in, base + (int64_t)t * a.ain.es, false);
    } else {
#pragma unroll
        for (int i = 0; i < E; ++i) reg[i] = c_make<V>(0, 0);
    }
    V twv[TWG ? E : 1];
    if constexpr (TWG) {
        if (active) {
            const V *tab = reinterpret_cast<const V *>(a.post_tab) + jl;
#pragma unroll
            for (int i = 0; i < E; ++i) twv[i] = tab[(int64_t)(t + i * T) * a.post_ld];
        }
    }

    ct.run(reg, lds + c, a.C, t);

    if (active) {
        V *out = reinterpret_cast<V *>(a.out);
        const int64_t base = addr_of(a.aout, j0, j1, j2);
        const Real sc = (Real)a.scale;
        // apart from the stores, which stay one batch
        if (a.sg_out.on) sign_run<E>(reg, a.sg_out, base + (int64_t)t * a.aout.es, false);
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const int k = t + i * T;
            V v = reg[i];
            if constexpr (TWG) {
                v = c_mul(v, twv[TWG ? i : 0]);
            } else if (a.post_L) {
                // jl < n2 and k < n1, so jl * k < n1 * n2 = post_L: no reduction needed
                const int64_t e = jl * (int64_t)k;
                v = c_mul(v, power_lookup(reinterpret_cast<const V *>(a.post_hi),
                                          reinterpret_cast<const V *>(a.post_lo), e, a.post_shift));
            }
            if (a.conj_out) v = c_conj(v);
            c_store(out + base + (int64_t)k * a.aout.es, c_scale(v, sc), a.nt_out);
        }
    }
}

// ----------------------------------------------------------------------------------------------
// Pointwise stages of the multi-kernel Bluestein path.

template <typename Real>
__global__ void __launch_bounds__(256) afft_chirp(const ChirpArgs a)
{
    using V = typename cplx_of<Real>::type;
    const V *chirp = reinterpret_cast<const V *>(a.chirp);
    const int64_t per = a.mode == 2 ? a.n : a.M;
    const int64_t total = a.ntrans * per;
    for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = idx / per;
        const int64_t m = idx - j * per;
        if (a.mode == 0) {
            const V *x = reinterpret_cast<const V *>(a.in);
            V *aux = reinterpret_cast<V *>(a.out);
            V v = c_make<V>(0, 0);
            if (m < a.n) {
                const int64_t off = addr_base(a.a, j) + m * a.a.es;
                v = sign_apply(a.sg, off, c_load(x + off, (bool)a.nt_in));
                if (a.conj_in) v = c_conj(v);
                v = c_mul(v, chirp[m]);
            }
            aux[j * a.M + m] = v;
        } else if (a.mode == 1) {
            V *aux = reinterpret_cast<V *>(a.out);
            const V *filt = reinterpret_cast<const V *>(a.filt);
            aux[j * a.M + m] = c_conj(c_mul(aux[j * a.M + m], filt[m]));
        } else {
            const V *aux = reinterpret_cast<const V *>(a.in);
            V *y = reinterpret_cast<V *>(a.out);
            V v = c_mul(c_conj(aux[j * a.M + m]), chirp[m]);
            if (a.conj_out) v = c_conj(v);
            const int64_t off = addr_base(a.a, j) + m * a.a.es;
            c_store(y + off, sign_apply(a.sg, off, c_scale(v, (Real)a.scale)), (bool)a.nt_out);
        }
    }
}

// ----------------------------------------------------------------------------------------------
// Twiddle / chirp generation in FP64.

// exp(-2 pi i e / L), 0 <= e < L < 2^60: reduced to an eighth of a turn in integers, since the rounding of e / L itself
// would turn an angle near 2 pi by more than the result's rounding
__device__ __forceinline__ double2 unit_root(int64_t e, int64_t L)
{
    const int64_t o = 8 * e / L, f = o & 1 ? (o + 1) * L - 8 * e : 8 * e - o * L; // from the nearest quarter turn
    double s, c;
    sincospi((double)f / (4.0 * (double)L), &s, &c);
    if (f == L) s = c; // (the eighth itself: sinpi(1/4) comes out one unit low)
    if (o & 1) s = -s;
    switch ((o + 1) >> 1 & 3) {
    case 0: return make_double2(c, -s);
    case 1: return make_double2(-s, -c);
    case 2: return make_double2(-c, s);
    default: return make_double2(s, c);
    }
}

template <typename Real>
__global__ void afft_gen_pass_twiddles(typename cplx_of<Real>::type *out, const PassTable pt)
{
    using V = typename cplx_of<Real>::type;
    int Ns = 1;
    for (int p = 0; p < pt.npass; ++p) {
        const int R = pt.radix[p];
        const int L = Ns * R;
        for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < L; idx += gridDim.x * blockDim.x) {
            const int k = idx / R, r = idx % R;
            const int e = r * k; // < L, exact
            const double2 w = unit_root(e, L);
            out[pt.tw_off[p] + idx] = c_make<V>((Real)w.x, (Real)w.y);
        }
        Ns = L;
    }
}

struct MixTables { // of the passes after the first
    int npass;
    MixPass pass[kMixMaxPasses];
};

template <typename Real>
__global__ void afft_gen_mixed_twiddles(typename cplx_of<Real>::type *out, const MixTables t)
{
    using V = typename cplx_of<Real>::type;
    for (int p = 1; p < t.npass; ++p) {
        const int Ns = t.pass[p].Ns, R = t.pass[p].R, count = mixed_twiddle_elems(sizeof(Real) == 8, Ns, R);
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < R * Ns; i += gridDim.x * blockDim.x) {
            const int r = i / Ns + 1, k = i % Ns, at = mixed_twiddle_at(sizeof(Real) == 8, Ns, r, k);
            const double2 w = unit_root(r == R ? 0 : r * k, Ns * R); // (r = R: the spare halves)
            if (at < count) out[t.pass[p].toff + at] = c_make<V>((Real)w.x, (Real)w.y);
        }
    }
}

template <typename Real>
__global__ void afft_gen_power_table(typename cplx_of<Real>::type *out, int64_t L, int64_t step,
                                     int64_t count)
{
    using V = typename cplx_of<Real>::type;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count;
         i += (int64_t)gridDim.x * blockDim.x) {
        // exponent reduced exactly in integers; i*step < 2^62 for every table built here
        const int64_t e = (i * step) % L;
        const double2 w = unit_root(e, L);
        out[i] = c_make<V>((Real)w.x, (Real)w.y);
    }
}

template <typename Real>
__global__ void afft_gen_twiddle_grid(typename cplx_of<Real>::type *out, int64_t L, int64_t rows, int64_t cols)
{
    using V = typename cplx_of<Real>::type;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < rows * cols;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t q = i / cols, j = i - q * cols;
        const int64_t e = (q * j) % L;
        const double2 w = unit_root(e, L);
        out[i] = c_make<V>((Real)w.x, (Real)w.y);
    }
}

template <typename Real>
__global__ void afft_gen_chirp(typename cplx_of<Real>::type *out, int64_t n)
{
    using V = typename cplx_of<Real>::type;
    for (int64_t m = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; m < n;
         m += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e = (m * m) % (2 * n); // exp(-i pi m^2/n) has period 2n in m^2
        const double2 w = unit_root(e, 2 * n);
        out[m] = c_make<V>((Real)w.x, (Real)w.y);
    }
}

__global__ void afft_gen_bluestein_kernel(double2 *out, int64_t n, int64_t M)
{
    for (int64_t m = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; m < M;
         m += (int64_t)gridDim.x * blockDim.x) {
        int64_t src = -1;
        if (m < n) src = m;
        else if (M - m < n) src = M - m;
        double2 v = make_double2(0.0, 0.0);
        if (src >= 0) {
            const int64_t e = (src * src) % (2 * n);
            const double2 w = unit_root(e, 2 * n);
            v = make_double2(w.x, -w.y); // conj(chirp)
        }
        out[m] = v;
    }
}

template <typename Real>
__global__ void afft_convert_scale(typename cplx_of<Real>::type *out, const double2 *in,
                                   int64_t count, double scale)
{
    using V = typename cplx_of<Real>::type;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count;
         i += (int64_t)gridDim.x * blockDim.x) {
        const double2 v = in[i];
        out[i] = c_make<V>((Real)(v.x * scale), (Real)(v.y * scale));
    }
}

template <typename Real>
__global__ void afft_pointwise_mul(typename cplx_of<Real>::type *y, const typename cplx_of<Real>::type *x,
                                   const typename cplx_of<Real>::type *h, int64_t count, int64_t hcount,
                                   int conj_h, Real scale)
{
    using V = typename cplx_of<Real>::type;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count;
         i += (int64_t)gridDim.x * blockDim.x) {
        V hv = h[i % hcount];
        if (conj_h) hv = c_conj(hv);
        y[i] = c_scale(c_mul(x[i], hv), scale);
    }
}

// ----------------------------------------------------------------------------------------------
// Host launchers.

template <typename Kern, typename Args>
static hipError_t launch_one(Kern k, const Args &a, int block, int64_t grid, size_t lds, hipStream_t s)
{
    if (grid <= 0) return hipSuccess;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(block), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_stockham(int dtype, const FftArgs &a, int block, int64_t grid, size_t lds, hipStream_t s)
{
    if (dtype == 0) {
        // the twiddle-grid forms in Complex Float only: in FP64 its registers would cost the
        // strided tiles a wave per SIMD
        switch (a.pt.n) {
#define AFFT_TILE(N, ...)                                                                        \
    case N:                                                                                      \
        return a.post_tab ? launch_one(afft_stockham<float, 16, N, true, __VA_ARGS__>, a, block, grid, lds, s) \
                          : launch_one(afft_stockham<float, 16, N, false, __VA_ARGS__>, a, block, grid, lds, s);
            AFFT_TILE(128, 16, 8)
            AFFT_TILE(256, 16, 16)
            AFFT_TILE(512, 16, 16, 2)
            AFFT_TILE(1024, 16, 16, 4)
#undef AFFT_TILE
        default: return hipErrorInvalidValue;
        }
    }
    if (a.pt.n == 256) return launch_one(afft_stockham<double, 16, 256, false, 16, 16>, a, block, grid, lds, s);
    return hipErrorInvalidValue;
}

static int64_t gs_grid(int64_t count)
{
    int64_t g = (count + 255) / 256;
    if (g < 1) g = 1;
    if (g > 4096) g = 4096;
    return g;
}

hipError_t gen_pass_twiddles(int dtype, void *out, const PassTable &pt, hipStream_t s)
{
    const int64_t g = gs_grid(pt.n);
    if (dtype == 0)
        hipLaunchKernelGGL(afft_gen_pass_twiddles<float>, dim3(g), dim3(256), 0, s, (float2 *)out, pt);
    else
        hipLaunchKernelGGL(afft_gen_pass_twiddles<double>, dim3(g), dim3(256), 0, s, (double2 *)out, pt);
    return hipGetLastError();
}

hipError_t gen_mixed_twiddles(int dtype, void *out, const MixArgs &a, hipStream_t s)
{
    MixTables t;
    t.npass = a.npass;
    std::copy(a.pass, a.pass + a.npass, t.pass);
    const int64_t g = gs_grid(a.n);
    if (dtype == 0)
        hipLaunchKernelGGL(afft_gen_mixed_twiddles<float>, dim3(g), dim3(256), 0, s, (float2 *)out, t);
    else
        hipLaunchKernelGGL(afft_gen_mixed_twiddles<double>, dim3(g), dim3(256), 0, s, (double2 *)out, t);
    return hipGetLastError();
}

hipError_t gen_power_table(int dtype, void *out, int64_t L, int64_t step, int64_t count, hipStream_t s)
{
    const int64_t g = gs_grid(count);
    if (dtype == 0)
        hipLaunchKernelGGL(afft_gen_power_table<float>, dim3(g), dim3(256), 0, s, (float2 *)out, L, step, count);
    else
        hipLaunchKernelGGL(afft_gen_power_table<double>, dim3(g), dim3(256), 0, s, (double2 *)out, L, step, count);
    return hipGetLastError();
}

hipError_t gen_twiddle_grid(int dtype, void *out, int64_t L, int64_t rows, int64_t cols, hipStream_t s)
{
    const int64_t g = gs_grid(rows * cols);
    if (dtype == 0)
        hipLaunchKernelGGL(afft_gen_twiddle_grid<float>, dim3(g), dim3(256), 0, s, (float2 *)out, L, rows, cols);
    else
        hipLaunchKernelGGL(afft_gen_twiddle_grid<double>, dim3(g), dim3(256), 0, s, (double2 *)out, L, rows, cols);
    return hipGetLastError();
}

hipError_t gen_chirp(int dtype, void *out, int64_t n, hipStream_t s)
{
    const int64_t g = gs_grid(n);
    if (dtype == 0)
        hipLaunchKernelGGL(afft_gen_chirp<float>, dim3(g), dim3(256), 0, s, (float2 *)out, n);
    else
        hipLaunchKernelGGL(afft_gen_chirp<double>, dim3(g), dim3(256), 0, s, (double2 *)out, n);
    return hipGetLastError();
}

hipError_t gen_bluestein_kernel_f64(void *out, int64_t n, int64_t M, hipStream_t s)
{
    hipLaunchKernelGGL(afft_gen_bluestein_kernel, dim3(gs_grid(M)), dim3(256), 0, s, (double2 *)out, n, M);
    return hipGetLastError();
}

hipError_t convert_scale_from_f64(int dtype, void *out, const void *in, int64_t count, double scale,
                                  hipStream_t s)
{
    const int64_t g = gs_grid(count);
    if (dtype == 0)
        hipLaunchKernelGGL(afft_convert_scale<float>, dim3(g), dim3(256), 0, s, (float2 *)out,
                           (const double2 *)in, count, scale);
    else
        hipLaunchKernelGGL(afft_convert_scale<double>, dim3(g), dim3(256), 0, s, (double2 *)out,
                           (const double2 *)in, count, scale);
    return hipGetLastError();
}

hipError_t launch_chirp(int dtype, const ChirpArgs &a, hipStream_t s)
{
    const int64_t per = a.mode == 2 ? a.n : a.M;
    int64_t g = (a.ntrans * per + 255) / 256;
    if (g > 65536) g = 65536;
    if (g < 1) return hipSuccess;
    if (dtype == 0)
        hipLaunchKernelGGL(afft_chirp<float>, dim3((unsigned)g), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(afft_chirp<double>, dim3((unsigned)g), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t pointwise_mul(int dtype, void *y, const void *x, const void *h, int64_t count,
                         int64_t hcount, int conj_h, double scale, hipStream_t s)
{
    const int64_t g = gs_grid(count);
    if (dtype == 0)
        hipLaunchKernelGGL(afft_pointwise_mul<float>, dim3(g), dim3(256), 0, s, (float2 *)y,
                           (const float2 *)x, (const float2 *)h, count, hcount, conj_h, (float)scale);
    else
        hipLaunchKernelGGL(afft_pointwise_mul<double>, dim3(g), dim3(256), 0, s, (double2 *)y,
                           (const double2 *)x, (const double2 *)h, count, hcount, conj_h, scale);
    return hipGetLastError();
}

} // namespace afft
