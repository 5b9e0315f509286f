// afft_ragged.hip -- ragged batches: many 1D transforms of mixed lengths, stored back to back,
// in one launch or two (kernel afft_ragged<Real, BLOCK>).
//
// The host sorts the transforms into length classes and cuts the classes that fit one workgroup
// into work items of C transforms, ordered by decreasing cost; workgroup w runs item w, so the
// dispatcher balances them and a retiring workgroup's stores overlap the next one's loads.  There is
// no device-side state to reset between launches: the launch replays as a captured hipGraph.
// Longer classes run as plans of the batched engine over the rows of the class (gathered by offset).
//
// An item runs the passes of the mixed-radix kernel (afft_mixed) with its class's pass table read
// from constant memory, so one body serves every length: directly, for prime factors up to 13, or as
// the two transforms of a chirp-z one.  One body also keeps the instruction cache warm: with a
// compiled layout per length (22 of them) every class's first workgroup on a CU fetched its code
// from memory, and a batch of 3 MB in the two chirp-z classes took 27 us of device time; now 2.  Large
// batches are bound by memory (4096 x 4096: 144 -> 54 us, 5.0 TB/s), chirp-z ones by their arithmetic
// (20000 x 257: 109 -> 59 us), small ones by the launch.
#include <hip/hip_runtime.h>

#include "afft_device.hpp"
#include "afft_ragged.hpp"

namespace afft {

template <typename Real, int BLOCK, bool BLUE>
__device__ __forceinline__ void run_item(const RaggedArgs &a, const RaggedClass &K, int first, int count)
{
    using V = typename cplx_of<Real>::type;
    constexpr int S = (int)sizeof(V), EMAX = 16;
    extern __shared__ __align__(16) unsigned char afft_smem[];
    const int tid = threadIdx.x, bd = BLOCK;
    const int len = K.L, n = K.m.n;
    const V *__restrict__ in = reinterpret_cast<const V *>(a.in);
    V *__restrict__ out = reinterpret_cast<V *>(a.out);
    const int64_t *__restrict__ moffs = a.moffs + first;
    const Real sc = a.inverse ? (Real)(1.0 / (double)len) : (Real)1, sy = a.conj ? -sc : sc;
    const BufView vtw(reinterpret_cast<const V *>(K.m.tw), (uint32_t)(K.m.tw_elems * S));
    const BufView vchirp(reinterpret_cast<const V *>(K.m.chirp), (uint32_t)(len * S));
    const BufView vfilt(reinterpret_cast<const V *>(K.m.filt), (uint32_t)(n * S));
    const int npass = K.m.npass, pitch = K.m.pitch;

    if (npass == 0) { // length 1
        if (tid < count) {
            const V v = in[moffs[tid]];
            out[moffs[tid]] = c_make<V>(v.x * sc, (a.conj ? -v.y : v.y) * sy);
        }
        return;
    }

    auto chirp_mul = [&](auto &v, int b, int nb) __attribute__((always_inline)) {
        constexpr int R = (int)(sizeof(v) / S), B = S == 16 ? 4 : R;
#pragma unroll
        for (int r0 = 0; r0 < R; r0 += B) {
            V ch[B];
#pragma unroll
            for (int u = 0; u < B && r0 + u < R; ++u) {
                ch[u] = c_make<V>(0, 0);
                if ((r0 + u) * nb < len) ch[u] = buf_load<V>(vchirp, (uint32_t)((b + (r0 + u) * nb) * S), 0);
            }
#pragma unroll
            for (int u = 0; u < B && r0 + u < R; ++u) v[r0 + u] = c_mul(v[r0 + u], ch[u]);
            __builtin_amdgcn_sched_barrier(0); // (registers)
        }
    };

    const int nsteps = BLUE ? 2 * npass - 1 : npass;
    for (int s = 0; s < nsteps; ++s) {
        const MixPass P = K.m.pass[BLUE && s >= npass ? s - npass + 1 : s];
        const bool from_global = s == 0, to_global = s + 1 == nsteps;
        const bool turn = BLUE && s + 1 == npass; // the end of the first transform
        const int wblock = turn ? K.m.pass[0].wblock : P.wblock, wstep = (turn ? 1 : P.Ns) * S;

        auto body = [&](auto rc) __attribute__((always_inline)) {
            constexpr int R = decltype(rc)::value;
            constexpr int NK = mixed_butterflies(EMAX, R);
            V v[NK][R];
            MixTwiddles<R, V, S == 16 ? 6 : 16> w[NK];
            int cc[NK], cb[NK], cq[NK];
            bool ca[NK];
#pragma unroll
            for (int kk = 0; kk < NK; ++kk) {
                const int g = tid + kk * bd;
                cc[kk] = mix_div(g, P.nb, P.mnb);
                cb[kk] = g - cc[kk] * P.nb;
                ca[kk] = cc[kk] < count;
                cq[kk] = mix_div(cb[kk], P.Ns, P.mns);
                if (P.Ns > 1 && ca[kk]) w[kk].load(vtw, P, cb[kk] - cq[kk] * P.Ns);
            }
            if (from_global) {
#pragma unroll
                for (int kk = 0; kk < NK; ++kk) {
                    if (!ca[kk]) continue;
                    const V *src = in + moffs[cc[kk]] + cb[kk];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        if constexpr (BLUE) {
                            // padding is read from the row's last element (one batch of loads) and cleared
                            v[kk][r] = c_make<V>(0, 0);
                            if (r * P.nb >= len) continue;
                            v[kk][r] = src[(cb[kk] + r * P.nb < len ? cb[kk] + r * P.nb : len - 1) - cb[kk]];
                        } else {
                            v[kk][r] = src[r * P.nb];
                        }
                    }
                    if (a.conj) {
#pragma unroll
                        for (int r = 0; r < R; ++r) v[kk][r].y = -v[kk][r].y;
                    }
                    if constexpr (BLUE) {
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            if (cb[kk] + r * P.nb >= len) v[kk][r] = c_make<V>(0, 0);
                        chirp_mul(v[kk], cb[kk], P.nb);
                    }
                }
            } else {
#pragma unroll
                for (int kk = 0; kk < NK; ++kk) {
                    if (!ca[kk]) continue;
                    const unsigned char *src = afft_smem + (cc[kk] * pitch + cb[kk] + cq[kk] * P.rpad) * S;
#pragma unroll
                    for (int r = 0; r < R; ++r) v[kk][r] = *reinterpret_cast<const V *>(src + r * P.rstep * S);
                }
            }
            if (P.Ns > 1) {
#pragma unroll
                for (int kk = 0; kk < NK; ++kk) w[kk].apply(v[kk], vtw, P, cb[kk] - cq[kk] * P.Ns);
            }
#pragma unroll
            for (int kk = 0; kk < NK; ++kk) dft<R>::run(v[kk]);
            if constexpr (BLUE) {
                if (turn) {
#pragma unroll
                    for (int kk = 0; kk < NK; ++kk) {
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            v[kk][r] = c_conj(c_mul(v[kk][r], buf_load<V>(vfilt, (uint32_t)(cb[kk] * S), (uint32_t)(r * P.nb * S))));
                        dft<R>::run(v[kk]);
                        cq[kk] = cb[kk];
                    }
                }
            }
            if (!to_global) {
                if (!from_global) lds_sync(); // every butterfly of this pass has been read
#pragma unroll
                for (int kk = 0; kk < NK; ++kk) {
                    if (!ca[kk]) continue;
                    const int k = turn ? 0 : cb[kk] - cq[kk] * P.Ns;
                    unsigned char *dst = afft_smem + (cc[kk] * pitch + cq[kk] * wblock + k) * S;
#pragma unroll
                    for (int r = 0; r < R; ++r) *reinterpret_cast<V *>(dst + r * wstep) = v[kk][r];
                }
                lds_sync();
                return;
            }
#pragma unroll
            for (int kk = 0; kk < NK; ++kk) {
                if (!ca[kk]) continue;
                V *dst = out + moffs[cc[kk]] + cb[kk];
                if constexpr (BLUE) {
#pragma unroll
                    for (int r = 0; r < R; ++r) v[kk][r].y = -v[kk][r].y;
                    chirp_mul(v[kk], cb[kk], P.nb);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    v[kk][r].x *= sc;
                    v[kk][r].y *= sy;
                }
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (!BLUE || cb[kk] + r * P.nb < len) dst[r * P.nb] = v[kk][r];
            }
        };
        switch (P.R) { // (padded lengths of chirp-z transforms are products of 2, 3 and 5)
        case 2: body(IC<2>{}); break;
        case 3: body(IC<3>{}); break;
        case 4: body(IC<4>{}); break;
        case 5: body(IC<5>{}); break;
        case 6: body(IC<6>{}); break;
        case 7: if constexpr (!BLUE) body(IC<7>{}); break;
        case 8: body(IC<8>{}); break;
        case 9: body(IC<9>{}); break;
        case 10: body(IC<10>{}); break;
        case 11: if constexpr (!BLUE) body(IC<11>{}); break;
        case 12: body(IC<12>{}); break;
        case 13: if constexpr (!BLUE) body(IC<13>{}); break;
        case 14: if constexpr (!BLUE) body(IC<14>{}); break;
        case 15: body(IC<15>{}); break;
        case 16: body(IC<16>{}); break;
        default: break;
        }
    }
}

// (four waves a SIMD: the LDS of the longest classes allows no more)
template <typename Real, int BLOCK>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(sizeof(Real) == 8 ? 2 : 4, 8)))
afft_ragged(const RaggedArgs a)
{
    // items and class descriptors are read through scalar loads: one item to a workgroup
    const RaggedItem &it = *(const RaggedItem *)(const RaggedItem __attribute__((address_space(4))) *)(a.items + blockIdx.x);
    const int cls = __builtin_amdgcn_readfirstlane(it.cls);
    const RaggedClass &K = *(const RaggedClass *)(const RaggedClass __attribute__((address_space(4))) *)(a.classes + cls);
    if (K.m.chirp) run_item<Real, BLOCK, true>(a, K, it.first, it.count);
    else run_item<Real, BLOCK, false>(a, K, it.first, it.count);
}

hipError_t launch_ragged(int dtype, int bin, const RaggedArgs &a, int64_t grid, size_t lds, hipStream_t s)
{
    using Fn = void (*)(const RaggedArgs);
    static const Fn fns[2][2] = {{afft_ragged<float, kRaggedBlock[0][0]>, afft_ragged<float, kRaggedBlock[0][1]>},
                                 {afft_ragged<double, kRaggedBlock[1][0]>, afft_ragged<double, kRaggedBlock[1][1]>}};
    const Fn fn = fns[dtype][bin];
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(kRaggedBlock[dtype][bin]), lds, s, a);
    return hipGetLastError();
}

} // namespace afft
