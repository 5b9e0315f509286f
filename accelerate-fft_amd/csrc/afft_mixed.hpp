// afft_mixed.hpp -- descriptors of the mixed-radix kernel (afft_mixed_kernel.hpp): transforms of any length
// whose prime factors are at most 13 (31 where the length fits a workgroup), and chirp-z transforms of
// the others, for contiguous rows and for strided axes.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "afft_internal.hpp"

namespace afft {

constexpr int kMixMaxPasses = 8;
constexpr int kMixMaxRadix = 16;

// The kernel for lengths with a prime factor of 17 ... 31 (Complex Double: ... 23) holds one butterfly
// of it a thread: a prime p costs about p operations an element in one pass, a chirp-z transform
// 130 ... 200 in five (its E; the other radices as with 16 elements).  128 MiB of Complex Float rows of 31:
// 102 -> 60 us, of 289 138 -> 55 us, of 16337 563 -> 113 us; Complex Double rows of 4913 609 -> 92 us.
// Instances of their own, since a butterfly of 31 takes the registers of four waves a SIMD (the strided form
// spills 40 bytes a lane), one of 23 Complex Double those of two.
constexpr int kMixWide = 31;
constexpr int mixed_wide_radix(int dtype) { return dtype == 0 ? 31 : 23; }

// Butterflies of radix R a thread of the E = 16, E = 32 or kMixWide kernel owns in a pass: at most E
// elements, and few enough that their indexes and twiddles stay in registers.
__host__ __device__ constexpr int mixed_butterflies(int E, int R)
{
    return E == 32 ? (R <= 8 ? 4 : 2) : (R <= 8 ? 2 : 1);
}

// One pass: butterflies of radix R at stride Ns, nb = n / R of them per transform.
struct MixPass {
    int R, Ns, nb;
    int toff;          // elements in front of the pass's twiddles in MixArgs::tw
    uint32_t mnb, mns; // floor(2^32 / d) + 1 for d = nb and d = Ns (unused for d = 1)
    // LDS layouts, in elements: the pass reads block q of Ns elements rpad q elements on, its
    // butterflies' elements rstep apart, and writes its own blocks of Ns R elements wblock apart
    int rpad, rstep, wblock;
};

// Waves per SIMD the registers of a kernel must allow, and that the planner counts as resident.  Where
// more would spill the strided kernels keep what the compiler needs: forced to 7 (from 82 registers to
// 72, 15 spilled) the Complex Float tiles of 100 and 224 points took 53 us instead of 42 on 128 MiB.  (The
// Complex Float kMixWide kernels have 4 from their launch bound; counted as 4 the planner takes slower
// tiles for a few lengths and faster ones for none: 2^23 elements in rows of 58 65 -> 97 us, of 19 26 -> 31
// us.)
__host__ __device__ constexpr int mixed_waves(bool f64, int E, bool rows, bool chirpz)
{
    if (E == kMixWide) return f64 ? 2 : 3;
    if (E == 32) return f64 ? 2 : 4;
    if (f64) return rows && !chirpz ? 4 : 3;
    return chirpz ? 4 : rows ? 6 : 5;
}

// Where the table of a pass holds W_{Ns R}^{r k}, r = 1 ... R - 1, k < Ns, in elements from its start:
// neighbouring lanes have neighbouring k, and 16 bytes hold the Complex Float powers 2p + 1 and 2p + 2.
__host__ __device__ constexpr int mixed_twiddle_at(bool f64, int Ns, int r, int k)
{
    return f64 ? (r - 1) * Ns + k : 2 * ((r - 1) / 2 * Ns + k) + (r - 1) % 2;
}
__host__ __device__ constexpr int mixed_twiddle_elems(bool f64, int Ns, int R)
{
    return f64 ? (R - 1) * Ns : 2 * (R / 2) * Ns;
}

struct MixArgs {
    const void *in;
    void *out;
    const void *tw;    // the passes' twiddles (mixed_twiddle_at)
    int tw_elems;
    int64_t ntrans;
    Addr ain, aout;
    AddrDiv div;       // of a transform index by ain.cnt0 and ain.cnt1 (= aout's)
    int n;             // transform length (the padded length of a chirp-z transform)
    int len;           // length of the caller's rows: n, or the chirp-z length below n
    int npass;
    int C;             // transforms per workgroup (a power of two for strided tiles)
    int lc;            // log2 C of a strided tile
    int stage;         // rows: whole tiles go through LDS on load and store (short rows)
    int pitch;         // rows: LDS elements between transforms
    MixPass pass[kMixMaxPasses];
    int conj_in, conj_out;
    double scale;
    int xcd_remap;
    int nt_in, nt_out;
    SignSpec sg_in, sg_out;
    int odd_in, odd_out; // one step along the transform, in or out, is an odd step along its axis
    // four-step twiddle on store, as FftArgs
    int64_t post_L;
    int post_level, post_shift;
    const void *post_hi, *post_lo;
    // chirp-z: c[m], m < len, and the filter of n elements
    const void *chirp, *filt;
};

// The twiddles of one butterfly of a pass: W_{Ns R}^{r k}, r = 1 ... R - 1, read from the pass's table, B
// of them with the butterfly's elements (load) and the others B at a time (apply).  B = 0: the powers 1, 2, 3,
// 4, 8 and 12, and the others as one product of two of them; a prime radix beyond 16: the powers 1, 2,
// 4, 8 and 16, and the others as their products.
template <int R, typename V, int B> struct MixTwiddles {
    static constexpr bool f64 = sizeof(V) == 16;
    static constexpr int S = (int)sizeof(V);
    static constexpr int N = R > 16 ? 5 : B == 0 ? 6 : (B < R ? B : R);
    static_assert(B % 2 == 0, "whole loads");
    V w[N];
    __device__ __forceinline__ static uint32_t base(const MixPass &P, int k)
    {
        return (uint32_t)((P.toff + (f64 ? k : 2 * k)) * S);
    }
    __device__ __forceinline__ static void one(V &to, const BufView &tw, const MixPass &P, uint32_t off, int r)
    {
        to = buf_load<V>(tw, off, (uint32_t)(mixed_twiddle_at(f64, P.Ns, r, 0) * S));
    }
    // powers r and r + 1, r odd
    __device__ __forceinline__ static void two(V &a, V &b, const BufView &tw, const MixPass &P, uint32_t off, int r)
    {
        if constexpr (f64) {
            one(a, tw, P, off, r);
            if (r + 1 < R) one(b, tw, P, off, r + 1);
        } else {
            const float4 q = buf_load<float4>(tw, off, (uint32_t)((r - 1) / 2 * P.Ns * 16));
            a = c_make<V>(q.x, q.y);
            b = c_make<V>(q.z, q.w);
        }
    }
    // the powers from r0 on, as many as fit
    __device__ __forceinline__ void batch(const BufView &tw, const MixPass &P, uint32_t off, int r0)
    {
#pragma unroll
        for (int u = 0; u < N && r0 + u < R; u += 2) {
            if (u + 1 < N) two(w[u], w[u + 1], tw, P, off, r0 + u);
            else one(w[u], tw, P, off, r0 + u);
        }
    }
    __device__ __forceinline__ void load(const BufView &tw, const MixPass &P, int k)
    {
        const uint32_t off = base(P, k);
        if constexpr (R > 16) {
#pragma unroll
            for (int q = 0; q < 5; ++q) one(w[q], tw, P, off, 1 << q);
        } else if constexpr (B > 0) {
            batch(tw, P, off, 1);
        } else {
            if constexpr (R > 2) two(w[0], w[1], tw, P, off, 1);
            else one(w[0], tw, P, off, 1);
            if constexpr (R > 4) two(w[2], w[3], tw, P, off, 3);
            else if constexpr (R > 3) one(w[2], tw, P, off, 3);
            if constexpr (R > 8) one(w[4], tw, P, off, 8);
            if constexpr (R > 12) one(w[5], tw, P, off, 12);
        }
    }
    __device__ __forceinline__ void apply(V *v, const BufView &tw, const MixPass &P, int k)
    {
        if constexpr (R > 16) {
            power_twiddles<R>(v, w);
        } else if constexpr (B > 0) {
#pragma unroll
            for (int r0 = 1; r0 < R; r0 += N) {
                if (r0 > 1) {
                    __builtin_amdgcn_sched_barrier(0); // (registers)
                    batch(tw, P, base(P, k), r0);
                }
#pragma unroll
                for (int u = 0; u < N && r0 + u < R; ++u) v[r0 + u] = c_mul(v[r0 + u], w[u]);
            }
        } else {
#pragma unroll
            for (int r = 1; r < R; ++r) {
                const int g = r & 12, m = r & 3;
                if (g == 0) {
                    v[r] = c_mul(v[r], w[m - 1]);
                } else {
                    const V &q = w[g == 4 ? 3 : g == 8 ? 4 : 5];
                    v[r] = c_mul(v[r], m ? c_mul(q, w[m - 1]) : q);
                }
            }
        }
    }
};

// Host-side shape of a launch (afft_mixed_plan.cpp).
struct MixShape {
    int npass = 0;
    int radix[kMixMaxPasses];
    int C = 1, E = 16; // transforms per workgroup, elements a thread may hold
    int block = 0;
    size_t lds = 0;
    bool stage = false;
    bool stream_out = true; // the output's lines leave whole enough to bypass the caches
    int pad[kMixMaxPasses]; // rows: elements between the blocks each pass leaves in LDS
    int pitch = 0;          // rows: LDS elements of one transform
    double cost = 0; // rows: wavefront-level work per transform, to compare padded lengths by
};

// The cheapest radices of a transform of length n (every prime factor at most 13) whose passes fit
// `threads` threads of the E kernel; with `symmetric` there are at least two and the first and the
// last are equal.  False if there are none.
bool mixed_radices(int64_t n, bool symmetric, int E, int threads, MixShape &out, int most = kMixMaxRadix);
// The launch shape for ntrans transforms of length n: contiguous rows or a strided tile; cols
// (strided): columns per workgroup, 0 for the default; gathered: the rows start at arbitrary offsets;
// layout: choose the LDS padding too (a search for a length goes without).
// False if it does not fit a workgroup.
bool mixed_shape(int dtype, int64_t n, int64_t ntrans, bool strided, bool chirpz, size_t lds_bytes, int cus,
                 int cols, MixShape &out, bool gathered = false, bool layout = true);
int64_t bluestein_length(int64_t n);
// The padded length of a chirp-z transform of length n: the cheapest of at least 2n - 1 that fits `limit`
// elements and rounds no more than the lengths before it did; 0 if none.
int64_t mixed_chirpz_length(int dtype, int64_t n, int64_t limit, size_t lds_bytes);
// The shape of a tile of rows of length n for workgroups of `block` threads with 16 elements each, of at
// most `elems` elements (the items of ragged batches): as many rows as fit.  False if none does.
bool mixed_tile(int dtype, int64_t n, bool chirpz, int block, int elems, MixShape &out);

// padded length of a chirp-z transform of n points in such a tile, 0 if none fits
int64_t mixed_chirpz_tile(int dtype, int64_t n, int block, int elems);

void mixed_fill(int dtype, const MixShape &sh, int64_t n, MixArgs &a);
// The twiddle table of a's passes (tw_elems elements), in FP64 and rounded.
hipError_t gen_mixed_twiddles(int dtype, void *out, const MixArgs &a, hipStream_t s);

hipError_t launch_mixed(int dtype, const MixArgs &a, bool strided, int E, int block, int64_t grid, size_t lds,
                        hipStream_t s);

} // namespace afft
