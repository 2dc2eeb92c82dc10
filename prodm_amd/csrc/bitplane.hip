// bitplane.hip -- bitplane encoders/decoders and max-abs for gfx950.
//
// Layout: one lane per bitplane block (32 elements for u32 words, 64 for
// u64). A workgroup stages its blocks through LDS with coalesced global
// accesses (rows padded by one word so that each lane's block is read or
// written without bank conflicts), and each lane turns its block into plane
// words with an in-register bit-matrix transpose: after transpose32, word k
// holds bit k of every element, LSB = first element of the block
// (GroupedBPEncoder.hpp:345, NegaBinaryBPEncoder.hpp:246). Plane stores and
// loads are then one coalesced word per lane per plane.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "internal.hpp"

namespace prodm {

constexpr int kThreads = 256;

// wave-wide prefix sum (inclusive or not) and total (DPP reductions of the device library)
extern "C" __device__ uint32_t __ockl_wfscan_add_u32(uint32_t, bool);
extern "C" __device__ uint32_t __ockl_wfred_add_u32(uint32_t);

// ------------------------------------------------------------------------------
// fills
// ------------------------------------------------------------------------------
template <class U>
__global__ __launch_bounds__(kThreads) void k_fill(U *dst, uint64_t count, U value) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = value;
}

int launch_fill_u32(uint32_t *dst, uint64_t count, uint32_t value, hipStream_t s) {
    if (!count) return kOk;
    uint32_t grid = (uint32_t)std::min<uint64_t>(div_up(count, kThreads), 8192);
    hipLaunchKernelGGL(k_fill<uint32_t>, dim3(grid), dim3(kThreads), 0, s, dst, count, value);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
int launch_fill_u64(uint64_t *dst, uint64_t count, uint64_t value, hipStream_t s) {
    if (!count) return kOk;
    uint32_t grid = (uint32_t)std::min<uint64_t>(div_up(count, kThreads), 8192);
    hipLaunchKernelGGL(k_fill<uint64_t>, dim3(grid), dim3(kThreads), 0, s, dst, count, value);
    PRODM_CHECK_LAUNCH();
    return kOk;
}

// ------------------------------------------------------------------------------
// max-abs: NaN never compares greater (RefactorUtils.hpp:71-73)
// ------------------------------------------------------------------------------
template <class T>
__global__ __launch_bounds__(kThreads) void k_maxabs(const T *__restrict__ x, uint64_t n, KeyOf<T> *key) {
    using K = KeyOf<T>;
    K m = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        T v = x[i];
        if (v == v) { K k = abs_key(v); m = k > m ? k : m; }
    }
    for (int off = 32; off >= 1; off >>= 1) {
        K o = __shfl_xor(m, off, 64);
        m = o > m ? o : m;
    }
    if (lane_id() == 0 && m) atomicMax(key, m);
}

template <class T> int launch_maxabs(const T *x, uint64_t n, KeyOf<T> *key, hipStream_t s) {
    if (!n) return kOk;
    uint32_t grid = (uint32_t)std::min<uint64_t>(div_up(n, kThreads * 8ull), 4096);
    hipLaunchKernelGGL(k_maxabs<T>, dim3(grid), dim3(kThreads), 0, s, x, n, key);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_maxabs<float>(const float *, uint64_t, uint32_t *, hipStream_t);
template int launch_maxabs<double>(const double *, uint64_t, unsigned long long *, hipStream_t);

// The maximum for the host: every workgroup stores its own into out[its
// index] (pinned host memory, no initial value, no atomics on one address:
// 2350 workgroups' atomics had taken 24 us for 4.9 M floats, now 4 us).
template <class T>
__global__ __launch_bounds__(kThreads) void k_maxabs_blocks(const T *__restrict__ x, uint64_t n, KeyOf<T> *out) {
    using K = KeyOf<T>;
    constexpr int C = 16 / (int)sizeof(T);
    __shared__ K red[kThreads / 64];
    const uint64_t t0 = (uint64_t)blockIdx.x * kThreads + threadIdx.x, step = (uint64_t)gridDim.x * kThreads;
    K m = 0;
    auto take = [&](T v) __attribute__((always_inline)) {
        const K k = v == v ? (K)abs_key(v) : (K)0;
        m = k > m ? k : m;
    };
    uint64_t done = 0;
    if (((uintptr_t)x & 15) == 0) {  // 16-byte loads of the aligned part
        const uint64_t nv = n / C;
#pragma unroll 4
        for (uint64_t i = t0; i < nv; i += step) {
            T v[C];
            const float4 q = reinterpret_cast<const float4 *>(x)[i];
            __builtin_memcpy(v, &q, 16);
#pragma unroll
            for (int c = 0; c < C; c++) take(v[c]);
        }
        done = nv * C;
    }
#pragma unroll 4
    for (uint64_t i = done + t0; i < n; i += step) take(x[i]);
    for (int off = 32; off >= 1; off >>= 1) {
        const K o = __shfl_xor(m, off, 64);
        m = o > m ? o : m;
    }
    if (lane_id() == 0) red[threadIdx.x / 64] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; w++) m = red[w] > m ? red[w] : m;
        out[blockIdx.x] = m;
    }
}
template <class T> int launch_maxabs_blocks(const T *x, uint64_t n, KeyOf<T> *out, uint32_t blocks, hipStream_t s) {
    hipLaunchKernelGGL(k_maxabs_blocks<T>, dim3(blocks), dim3(kThreads), 0, s, x, n, out);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_maxabs_blocks<float>(const float *, uint64_t, uint32_t *, uint32_t, hipStream_t);
template int launch_maxabs_blocks<double>(const double *, uint64_t, unsigned long long *, uint32_t, hipStream_t);

template <class T> __device__ inline int level_exp(int32_t exp, const KeyOf<T> *key) {
    return key ? dev_frexp_exp(key_to_value<T>((uint64_t)*key)) : exp;
}

// ------------------------------------------------------------------------------
// bit-matrix transposes: A[r] bit c  ->  A[c] bit r
// ------------------------------------------------------------------------------
__device__ __forceinline__ void transpose32(uint32_t (&A)[32]) {
#pragma unroll
    for (int s = 0; s < 5; s++) {
        const int j = 16 >> s;
        const uint32_t m = s == 0 ? 0x0000FFFFu : s == 1 ? 0x00FF00FFu : s == 2 ? 0x0F0F0F0Fu : s == 3 ? 0x33333333u : 0x55555555u;
#pragma unroll
        for (int k = 0; k < 32; k++) {
            if ((k & j) == 0) {
                const uint32_t t = ((A[k] >> j) ^ A[k + j]) & m;
                A[k] ^= t << j;
                A[k + j] ^= t;
            }
        }
    }
}

template <int OFF, int N>
__device__ __forceinline__ void transpose32_at(uint32_t (&A)[N]) {
#pragma unroll
    for (int s = 0; s < 5; s++) {
        const int j = 16 >> s;
        const uint32_t m = s == 0 ? 0x0000FFFFu : s == 1 ? 0x00FF00FFu : s == 2 ? 0x0F0F0F0Fu : s == 3 ? 0x33333333u : 0x55555555u;
#pragma unroll
        for (int k = 0; k < 32; k++) {
            if ((k & j) == 0) {
                const uint32_t t = ((A[OFF + k] >> j) ^ A[OFF + k + j]) & m;
                A[OFF + k] ^= t << j;
                A[OFF + k + j] ^= t;
            }
        }
    }
}

// 64 x 64 as four in-place 32 x 32 blocks. Element-major layout: element e
// is (hi[e] << 32) | lo[e]. Word-major layout: word w (bit w of the 64
// elements, element 0 in bit 0) is (w < 32) ? lo[w] | lo[32 + w] << 32
// : hi[w - 32] | hi[w] << 32. The transform is its own inverse.
__device__ __forceinline__ void transpose64(uint32_t (&lo)[64], uint32_t (&hi)[64]) {
    transpose32_at<0>(lo);
    transpose32_at<32>(lo);
    transpose32_at<0>(hi);
    transpose32_at<32>(hi);
}
template <int W> __device__ __forceinline__ uint64_t word64_get(const uint32_t (&lo)[64], const uint32_t (&hi)[64]) {
    if constexpr (W < 32) return ((uint64_t)lo[32 + W] << 32) | lo[W];
    else return ((uint64_t)hi[W] << 32) | hi[W - 32];
}
template <int W> __device__ __forceinline__ void word64_set(uint32_t (&lo)[64], uint32_t (&hi)[64], uint64_t v) {
    if constexpr (W < 32) { lo[W] = (uint32_t)v; lo[32 + W] = (uint32_t)(v >> 32); }
    else { hi[W - 32] = (uint32_t)v; hi[W] = (uint32_t)(v >> 32); }
}
template <int I, int N, class F> __device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// ------------------------------------------------------------------------------
// block staging geometry
// ------------------------------------------------------------------------------
template <class T> struct BlkStage;
template <> struct BlkStage<float> {
    static constexpr int kTPB = 256;                // threads (= blocks) per workgroup
    static constexpr int kB = 32;                   // elements per block
    static constexpr int kPitch = kB + 1;           // LDS row pitch (words)
};
template <> struct BlkStage<double> {
    static constexpr int kTPB = 64;
    static constexpr int kB = 64;
    static constexpr int kPitch = kB + 1;
};

// coalesced load of the workgroup's TPB*B elements into LDS rows (0 past n)
template <class T, class XP = const T *>
__device__ inline void stage_in(XP __restrict__ x, uint64_t n, uint64_t e0, T *sx) {
    constexpr int TPB = BlkStage<T>::kTPB, B = BlkStage<T>::kB, PI = BlkStage<T>::kPitch;
    // all B loads in flight before the first LDS store
    T v[B];
#pragma unroll
    for (int i = 0; i < B; i++) {
        const uint64_t e = e0 + (uint32_t)(i * TPB) + threadIdx.x;
        v[i] = e < n ? x[e] : (T)0;
    }
#pragma unroll
    for (int i = 0; i < B; i++) {
        const uint32_t le = i * TPB + threadIdx.x;
        sx[(le / B) * PI + (le % B)] = v[i];
    }
}
template <class T>
__device__ inline void stage_out(T *__restrict__ out, uint64_t n, uint64_t e0, const T *sx) {
    constexpr int TPB = BlkStage<T>::kTPB, B = BlkStage<T>::kB, PI = BlkStage<T>::kPitch;
#pragma unroll 8
    for (int i = 0; i < B; i++) {
        const uint32_t le = i * TPB + threadIdx.x;
        const uint64_t e = e0 + le;
        if (e < n) out[e] = sx[(le / B) * PI + (le % B)];
    }
}

// ------------------------------------------------------------------------------
// wave rows: a wave's 64 lanes take 32 consecutive elements each
// ------------------------------------------------------------------------------
// f32: lane l holds block l of the wave (64 blocks of 32). f64: block i of the
// wave's 32 blocks of 64 is held by lanes i (elements 0..31, the low word of
// every plane word) and i + 32 (elements 32..63, the high word).
// Lanes read and write their elements through wave-private LDS rows of 128
// bytes (a whole cache line per row and global access; f64 in two rounds of
// 16 elements), so no barrier is involved. The row pitch of 36 words keeps
// the 16-byte LDS accesses of consecutive lanes on different banks.
constexpr int kRowElems = 32, kRowPitch = 36;
template <class T> struct WaveRows {
    static constexpr int kHalves = sizeof(T) / 4;             // lanes per block
    static constexpr int kBlocks = 64 / kHalves;              // blocks per wave
    static constexpr int kRound = 128 / (int)sizeof(T);       // elements of a row
    static constexpr int kRounds = kRowElems / kRound;
    // first element (in the wave's 2048) of lane row r in round h
    static __device__ __forceinline__ uint32_t first(uint32_t r, uint32_t h) {
        if constexpr (sizeof(T) == 4) return r * 32;
        else return (r & 31) * 64 + (r >> 5) * 32 + h * 16;
    }
};

// whether the wave's 2048 elements from e0 are all below n and 16-byte aligned
template <class T> __device__ __forceinline__ bool rows_whole(const T *x, uint64_t n, uint64_t e0) {
    return ((uintptr_t)x & 15) == 0 && e0 + 64 * kRowElems <= n;
}

// f(j, x_j) for the lane's 32 elements (0 past n) of the wave whose first
// element is e0, a round at a time (its conversions overlap the next loads)
template <class T, class Fn>
__device__ __forceinline__ void rows_in(const T *__restrict__ x, uint64_t n, uint64_t e0, uint32_t *rows, Fn &&f) {
    using R = WaveRows<T>;
    constexpr int E = R::kRound, C = 16 / (int)sizeof(T);  // elements of a row / of 16 bytes
    const uint32_t lane = lane_id();
    T *const tr = reinterpret_cast<T *>(rows);
    constexpr int kP = kRowPitch * 4 / (int)sizeof(T);     // row pitch in elements
    const bool whole = rows_whole(x, n, e0);
#pragma unroll
    for (int h = 0; h < R::kRounds; h++) {
        if (whole) {
            float4 q[8];
#pragma unroll
            for (int i = 0; i < 8; i++)
                q[i] = *reinterpret_cast<const float4 *>(x + e0 + R::first(8 * i + (lane >> 3), h) + (lane & 7) * C);
#pragma unroll
            for (int i = 0; i < 8; i++)
                *reinterpret_cast<float4 *>(rows + (8 * i + (lane >> 3)) * kRowPitch + (lane & 7) * 4) = q[i];
        } else {
            // the last wave of the data, or an input that starts off a 16-byte line
            T q[E];
#pragma unroll
            for (int i = 0; i < E; i++) {
                const uint32_t k = 64u * i + lane;
                const uint64_t e = e0 + R::first(k / E, h) + k % E;
                q[i] = e < n ? x[e] : (T)0;
            }
#pragma unroll
            for (int i = 0; i < E; i++) {
                const uint32_t k = 64u * i + lane;
                tr[(k / E) * kP + k % E] = q[i];
            }
        }
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < 8; i++) {
            T t[C];
            const float4 q = *reinterpret_cast<const float4 *>(rows + lane * kRowPitch + 4 * i);
            __builtin_memcpy(t, &q, 16);
#pragma unroll
            for (int c = 0; c < C; c++) f(h * E + i * C + c, t[c]);
        }
        wave_lds_sync();
    }
}
// the inverse: the lane's 32 elements to out (those below n)
template <class T>
__device__ __forceinline__ void rows_out(T *__restrict__ out, uint64_t n, uint64_t e0, uint32_t *rows,
                                         const T (&v)[kRowElems]) {
    using R = WaveRows<T>;
    constexpr int E = R::kRound, C = 16 / (int)sizeof(T);
    const uint32_t lane = lane_id();
    T *const tr = reinterpret_cast<T *>(rows);
    constexpr int kP = kRowPitch * 4 / (int)sizeof(T);
    const bool whole = rows_whole(out, n, e0);
#pragma unroll
    for (int h = 0; h < R::kRounds; h++) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            float4 t;
            __builtin_memcpy(&t, &v[h * E + i * C], 16);
            *reinterpret_cast<float4 *>(rows + lane * kRowPitch + 4 * i) = t;
        }
        wave_lds_sync();
        if (whole) {
#pragma unroll
            for (int i = 0; i < 8; i++)
                *reinterpret_cast<float4 *>(out + e0 + R::first(8 * i + (lane >> 3), h) + (lane & 7) * C) =
                    *reinterpret_cast<const float4 *>(rows + (8 * i + (lane >> 3)) * kRowPitch + (lane & 7) * 4);
        } else {
#pragma unroll
            for (int i = 0; i < E; i++) {
                const uint32_t k = 64u * i + lane, r = k / E, c = k % E;
                const uint64_t e = e0 + R::first(r, h) + c;
                if (e < n) out[e] = tr[r * kP + c];
            }
        }
        wave_lds_sync();
    }
}

// ------------------------------------------------------------------------------
// NegaBinary
// ------------------------------------------------------------------------------
// binary2negabinary of (T_fps) v (NegaBinaryBPEncoder.hpp:43,219-224)
template <class T> __device__ inline typename Traits<T>::Fixed to_negabinary(T v) {
    using F = typename Traits<T>::Fixed;
    using SF = typename Traits<T>::SFixed;
    SF q = 0;
    if (v == v && fabs(v) < (T)9.2233720368547758e18) q = (SF)(int64_t)v;
    return ((F)q + (F)Traits<T>::kNbMask) ^ (F)Traits<T>::kNbMask;
}

// workgroup bid encodes bitplane blocks [bid TPB, (bid + 1) TPB)
template <class T>
__device__ __forceinline__ void nb_encode_blocks(const T *__restrict__ x, uint32_t n, int32_t exp, const KeyOf<T> *key,
                                                 int nb, typename Traits<T>::Stream *__restrict__ planes,
                                                 uint64_t stride, uint32_t bid) {
    constexpr int TPB = BlkStage<T>::kTPB, B = BlkStage<T>::kB, PI = BlkStage<T>::kPitch;
    __shared__ T sx[TPB * PI];
    const uint64_t b0 = (uint64_t)bid * TPB;
    // global-space pointers: the grouped form reads them from memory
    using GS = PRODM_GLOBAL typename Traits<T>::Stream;
    GS *gplanes = (GS *)planes;
    stage_in<T, const PRODM_GLOBAL T *>((const PRODM_GLOBAL T *)x, n, b0 * B, sx);
    __syncthreads();
    const int shift = nb - (level_exp<T>(exp, key) + 2);  // exp += 2 (:21)
    const uint64_t b = b0 + threadIdx.x;
    const uint64_t nw = ((uint64_t)n + B - 1) / B;
    const T *row = sx + threadIdx.x * PI;
    if constexpr (sizeof(T) == 4) {
        uint32_t q[32];
#pragma unroll
        for (int j = 0; j < 32; j++) q[j] = to_negabinary<T>(dev_ldexp(row[j], shift));
        transpose32(q);
        if (b < nw) {
#pragma unroll
            for (int k = 0; k < 32; k++) {
                const int p = nb - 1 - k;  // plane p holds bit nb - 1 - p
                if (p >= 0) gplanes[(uint64_t)p * stride + b] = q[k];
            }
        }
    } else {
        uint32_t lo[64], hi[64];
#pragma unroll
        for (int j = 0; j < 64; j++) {
            const uint64_t q = to_negabinary<T>(dev_ldexp(row[j], shift));
            lo[j] = (uint32_t)q;
            hi[j] = (uint32_t)(q >> 32);
        }
        transpose64(lo, hi);
        if (b < nw) {
            static_for<0, 64>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const int p = nb - 1 - k;
                if (p >= 0) gplanes[(uint64_t)p * stride + b] = word64_get<k>(lo, hi);
            });
        }
    }
}

template <class T>
__global__ __launch_bounds__(BlkStage<T>::kTPB) void k_nb_encode(const T *__restrict__ x, uint32_t n, int32_t exp,
                                                              const KeyOf<T> *key, int nb,
                                                              typename Traits<T>::Stream *__restrict__ planes,
                                                              uint64_t stride) {
    nb_encode_blocks<T>(x, n, exp, key, nb, planes, stride, blockIdx.x);
}

// grouped form: one entry per level buffer of the batch (exponent from the
// level's max key, as the plan's refactor encodes)
template <class T> struct NbEntry {
    const T *x;
    const KeyOf<T> *key;
    typename Traits<T>::Stream *planes;
    uint64_t stride;
    uint32_t n, pad;
};
template <class T>
__global__ __launch_bounds__(BlkStage<T>::kTPB) void k_nb_encode_grouped(const NbEntry<T> *__restrict__ ps,
                                                                      const uint32_t *__restrict__ first,
                                                                      uint32_t nent, uint32_t total, int nb) {
    for (uint32_t vb = blockIdx.x; vb < total; vb += gridDim.x) {
        const uint32_t e = group_entry(first, nent, vb);
        const NbEntry<T> E = uniform_load(ps + e);
        const uint32_t f0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)first[e]);
        nb_encode_blocks<T>(E.x, E.n, 0, E.key, nb, E.planes, E.stride, vb - f0);
        __syncthreads();  // the staging rows are reused by the next workgroup's blocks
    }
}

template <class T>
int nb_batched_launch(const std::vector<EncodeRef> &levels, int nb, const GroupShape &shape, GroupLaunch &L) {
    constexpr int B = Traits<T>::kBlock, TPB = BlkStage<T>::kTPB;
    if (nb < 1 || nb > B) { set_error("batched negabinary encode: bad num_bitplanes"); return kErrArg; }
    L = GroupLaunch{};
    L.kind = kGrpNbEncode;
    L.elem = sizeof(T);
    L.nb = nb;
    L.block = TPB;
    L.shape = shape;
    std::vector<std::pair<uint32_t, NbEntry<T>>> v;
    for (const EncodeRef &r : levels) {
        if (!r.n) continue;
        const uint64_t nw = ((uint64_t)r.n + B - 1) / B;
        if (r.stride < nw || !r.x || !r.planes || !r.key) { set_error("batched negabinary encode: bad level"); return kErrArg; }
        NbEntry<T> E{};
        E.x = static_cast<const T *>(r.x);
        E.key = static_cast<const KeyOf<T> *>(r.key);
        E.planes = static_cast<typename Traits<T>::Stream *>(r.planes);
        E.stride = r.stride;
        E.n = r.n;
        v.push_back({div_up(nw, TPB), E});
    }
    std::stable_sort(v.begin(), v.end(), [](const auto &a, const auto &b) { return a.first > b.first; });
    L.first.push_back(0);
    for (auto &x : v) {
        const size_t o = L.params.size();
        L.params.resize(o + sizeof(NbEntry<T>));
        std::memcpy(L.params.data() + o, &x.second, sizeof(NbEntry<T>));
        L.first.push_back(L.first.back() + x.first);
        L.nent++;
    }
    L.total = L.first.back();
    return kOk;
}
template int nb_batched_launch<float>(const std::vector<EncodeRef> &, int, const GroupShape &, GroupLaunch &);
template int nb_batched_launch<double>(const std::vector<EncodeRef> &, int, const GroupShape &, GroupLaunch &);

struct ZeroEntry {
    uint32_t *p;
    uint32_t words, pad;
};
__global__ __launch_bounds__(kThreads) void k_zero_grouped(const ZeroEntry *__restrict__ ps,
                                                          const uint32_t *__restrict__ first, uint32_t nent,
                                                          uint32_t total) {
    for (uint32_t vb = blockIdx.x; vb < total; vb += gridDim.x) {
        const uint32_t e = group_entry(first, nent, vb);
        const ZeroEntry E = uniform_load(ps + e);
        const uint32_t f0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)first[e]);
        const uint32_t i = (vb - f0) * kThreads + threadIdx.x;
        if (i < E.words) E.p[i] = 0u;
    }
}

int zero_batched_launch(const std::vector<std::pair<void *, uint32_t>> &buffers, GroupLaunch &L) {
    L = GroupLaunch{};
    L.kind = kGrpZero;
    L.block = kThreads;
    L.first.push_back(0);
    for (const auto &b : buffers) {
        if (!b.second) continue;
        if (!b.first) { set_error("batched zero: null buffer"); return kErrArg; }
        ZeroEntry E{static_cast<uint32_t *>(b.first), b.second, 0};
        const size_t o = L.params.size();
        L.params.resize(o + sizeof(E));
        std::memcpy(L.params.data() + o, &E, sizeof(E));
        L.first.push_back(L.first.back() + div_up(b.second, kThreads));
        L.nent++;
    }
    L.total = L.first.back();
    return kOk;
}

int bitplane_group_run(const GroupLaunch &L, hipStream_t s) {
    if (L.kind != kGrpNbEncode && L.kind != kGrpZero) { set_error("grouped launch: not a bitplane kind"); return kErrArg; }
    if (!L.d_params || !L.d_first) { set_error("grouped launch: tables not uploaded"); return kErrState; }
    const uint32_t grid = L.grid();
    if (!grid || !L.nent) return kOk;
    if (L.kind == kGrpZero)
        hipLaunchKernelGGL(k_zero_grouped, dim3(grid), dim3(L.block), 0, s, static_cast<const ZeroEntry *>(L.d_params),
                           L.d_first, L.nent, L.total);
    else if (L.elem == 8)
        hipLaunchKernelGGL(k_nb_encode_grouped<double>, dim3(grid), dim3(L.block), 0, s,
                           static_cast<const NbEntry<double> *>(L.d_params), L.d_first, L.nent, L.total, L.nb);
    else
        hipLaunchKernelGGL(k_nb_encode_grouped<float>, dim3(grid), dim3(L.block), 0, s,
                           static_cast<const NbEntry<float> *>(L.d_params), L.d_first, L.nent, L.total, L.nb);
    PRODM_CHECK_LAUNCH();
    return kOk;
}

template <class T>
int launch_nb_encode(const T *x, uint32_t n, int32_t exp, const KeyOf<T> *key, int nb,
                     typename Traits<T>::Stream *planes, uint64_t stride, hipStream_t s) {
    constexpr int B = Traits<T>::kBlock;
    if (n == 0 || nb < 1 || nb > B) { set_error("negabinary encode: bad n or num_bitplanes"); return kErrArg; }
    const uint64_t nw = ((uint64_t)n + B - 1) / B;
    if (stride < nw) { set_error("negabinary encode: plane stride below the words per plane"); return kErrArg; }
    const uint32_t grid = div_up(nw, BlkStage<T>::kTPB);
    hipLaunchKernelGGL(k_nb_encode<T>, dim3(grid), dim3(BlkStage<T>::kTPB), 0, s, x, n, exp, key, nb, planes, stride);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_nb_encode<float>(const float *, uint32_t, int32_t, const uint32_t *, int, uint32_t *, uint64_t,
                                     hipStream_t);
template int launch_nb_encode<double>(const double *, uint32_t, int32_t, const unsigned long long *, int, uint64_t *,
                                      uint64_t, hipStream_t);

// workgroup bid decodes its blocks from planes [start, start + k), plane(i)
// giving the words of plane start + i
template <class T, class PlaneFn>
__device__ __forceinline__ void nb_decode_blocks(PlaneFn &&plane, uint32_t n, int32_t exp, const KeyOf<T> *key,
                                                 int start, int k, T *__restrict__ out, uint32_t bid) {
    using S = typename Traits<T>::Stream;
    using SF = typename Traits<T>::SFixed;
    constexpr int TPB = BlkStage<T>::kTPB, B = BlkStage<T>::kB, PI = BlkStage<T>::kPitch;
    __shared__ T sx[TPB * PI];
    const uint64_t b0 = (uint64_t)bid * TPB;
    const uint64_t b = b0 + threadIdx.x;
    const uint64_t nw = ((uint64_t)n + B - 1) / B;
    const int e2 = level_exp<T>(exp, key) + 2;
    const int end = start + k;
    T *row = sx + threadIdx.x * PI;
    // acc bit (k - 1 - i) comes from plane start + i
    if constexpr (sizeof(T) == 4) {
        uint32_t a[32];
#pragma unroll
        for (int r = 0; r < 32; r++) {
            const int i = k - 1 - r;
            a[r] = (i >= 0 && b < nw) ? plane(i)[b] : 0u;
        }
        transpose32(a);
#pragma unroll
        for (int j = 0; j < 32; j++) {
            const SF val = (SF)((a[j] ^ (uint32_t)Traits<T>::kNbMask) - (uint32_t)Traits<T>::kNbMask);
            const T y = dev_ldexp((T)val, e2 - end);
            row[j] = (end & 1) ? -y : y;  // odd ending plane flips the sign (:153,172-189)
        }
    } else {
        uint32_t lo[64], hi[64];
        static_for<0, 64>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            const int i = k - 1 - r;
            const uint64_t w = (i >= 0 && b < nw) ? plane(i)[b] : 0ull;
            word64_set<r>(lo, hi, w);
        });
        transpose64(lo, hi);
#pragma unroll
        for (int j = 0; j < 64; j++) {
            const uint64_t acc = ((uint64_t)hi[j] << 32) | lo[j];
            const SF val = (SF)((acc ^ (uint64_t)Traits<T>::kNbMask) - (uint64_t)Traits<T>::kNbMask);
            const T y = dev_ldexp((T)val, e2 - end);
            row[j] = (end & 1) ? -y : y;
        }
    }
    __syncthreads();
    stage_out<T>(out, n, b0 * B, sx);
}

template <class T>
__global__ __launch_bounds__(BlkStage<T>::kTPB) void k_nb_decode(PlanePtrs pl, uint32_t n, int32_t exp,
                                                              const KeyOf<T> *key, int start, int k,
                                                              T *__restrict__ out) {
    using S = typename Traits<T>::Stream;
    nb_decode_blocks<T>([&](int i) __attribute__((always_inline)) { return static_cast<const S *>(pl.p[i]); }, n, exp,
                        key, start, k, out, blockIdx.x);
}

template <class T>
int launch_nb_decode(const PlanePtrs &planes, uint32_t n, int32_t exp, const KeyOf<T> *key, int start, int k, T *out,
                     hipStream_t s) {
    constexpr int B = Traits<T>::kBlock;
    if (n == 0) return kOk;
    if (k < 0 || start < 0 || start + k > B) { set_error("negabinary decode: bad plane range"); return kErrArg; }
    if (k == 0) {
        // k == 0: the reference returns zeros (:135-138)
        if constexpr (sizeof(T) == 4) return launch_fill_u32(reinterpret_cast<uint32_t *>(out), n, 0u, s);
        else return launch_fill_u64(reinterpret_cast<uint64_t *>(out), n, 0ull, s);
    }
    const uint64_t nw = ((uint64_t)n + B - 1) / B;
    const uint32_t grid = div_up(nw, BlkStage<T>::kTPB);
    hipLaunchKernelGGL(k_nb_decode<T>, dim3(grid), dim3(BlkStage<T>::kTPB), 0, s, planes, n, exp, key, start, k, out);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_nb_decode<float>(const PlanePtrs &, uint32_t, int32_t, const uint32_t *, int, int, float *,
                                     hipStream_t);
template int launch_nb_decode<double>(const PlanePtrs &, uint32_t, int32_t, const unsigned long long *, int, int,
                                      double *, hipStream_t);

// ---- small levels of a plan together ---------------------------------------------
// A plan's small levels take one launch per kernel (LevelSet by value) instead
// of one each: a launch costs some 3 us of host time and 3 to 6 us on the GPU
// whatever its size, and a 33^3 refactor + retrieve was 40 of them.
template <class T>
__global__ __launch_bounds__(BlkStage<T>::kTPB) void k_nb_encode_set(LevelSet<NbLevel<T>> L, int nb) {
    const uint32_t i = set_entry(L, blockIdx.x);
    const NbLevel<T> &E = L.e[i];
    nb_encode_blocks<T>(E.x, E.n, 0, E.key, nb, E.planes, E.stride, blockIdx.x - L.first[i]);
}
template <class T>
__global__ __launch_bounds__(BlkStage<T>::kTPB) void k_nb_decode_set(LevelSet<NbLevel<T>> L) {
    const uint32_t i = set_entry(L, blockIdx.x);
    const NbLevel<T> &E = L.e[i];
    const typename Traits<T>::Stream *planes = E.planes;
    const uint64_t stride = E.stride;
    nb_decode_blocks<T>([&](int p) __attribute__((always_inline)) { return planes + (uint64_t)p * stride; }, E.n, 0,
                        E.key, 0, E.k, E.x, blockIdx.x - L.first[i]);
}
template <class T> static uint32_t nb_workgroups(uint32_t n) {
    return div_up(((uint64_t)n + Traits<T>::kBlock - 1) / Traits<T>::kBlock, BlkStage<T>::kTPB);
}
template <class T> int launch_nb_encode_set(LevelSet<NbLevel<T>> L, int nb, hipStream_t s) {
    if (!L.n) return kOk;
    for (uint32_t i = 0; i < L.n; i++)
        if (L.e[i].n == 0 || nb < 1 || nb > Traits<T>::kBlock) {
            set_error("negabinary encode: bad n or num_bitplanes");
            return kErrArg;
        }
    set_sizes(L, [](const NbLevel<T> &e) { return nb_workgroups<T>(e.n); });
    hipLaunchKernelGGL(k_nb_encode_set<T>, dim3(L.first[L.n]), dim3(BlkStage<T>::kTPB), 0, s, L, nb);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template <class T> int launch_nb_decode_set(LevelSet<NbLevel<T>> L, hipStream_t s) {
    if (!L.n) return kOk;
    for (uint32_t i = 0; i < L.n; i++)
        if (L.e[i].k < 0 || L.e[i].k > Traits<T>::kBlock) { set_error("negabinary decode: bad plane range"); return kErrArg; }
    set_sizes(L, [](const NbLevel<T> &e) { return nb_workgroups<T>(e.n); });
    if (!L.first[L.n]) return kOk;
    hipLaunchKernelGGL(k_nb_decode_set<T>, dim3(L.first[L.n]), dim3(BlkStage<T>::kTPB), 0, s, L);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_nb_encode_set<float>(LevelSet<NbLevel<float>>, int, hipStream_t);
template int launch_nb_encode_set<double>(LevelSet<NbLevel<double>>, int, hipStream_t);
template int launch_nb_decode_set<float>(LevelSet<NbLevel<float>>, hipStream_t);
template int launch_nb_decode_set<double>(LevelSet<NbLevel<double>>, hipStream_t);

// ------------------------------------------------------------------------------
// GroupedBP
// ------------------------------------------------------------------------------
// magnitude of (int64_t) ldexp(x, nb - exp), sign folded (GroupedBPEncoder.hpp:40-44);
// |v| >= 2^63 is undefined in C++: compat reproduces the x86 result 2^63,
// otherwise the truncated magnitude is used (hazard B1).
template <class T>
__device__ inline typename Traits<T>::Fixed gb_mag(T x, int shift, int compat) {
    using F = typename Traits<T>::Fixed;
    const T v = dev_ldexp(x, shift);
    if constexpr (sizeof(T) == 4) {  // one conversion where the magnitude fits the word
        const float a = fabsf(v);
        if (a < 4294967296.0f) return (F)a;
    }
    if (v != v) return 0;
    const T av = fabs(v);
    if (av < (T)9.2233720368547758e18) {
        const int64_t q = (int64_t)v;
        const uint64_t m = (x < 0) ? (uint64_t)0 - (uint64_t)q : (uint64_t)q;
        return (F)m;
    }
    if (compat) return (F)0x8000000000000000ull;
    if (av < (T)1.8446744073709552e19) return (F)(uint64_t)av;
    return (F)~0ull;
}

// recording plane of a block from the OR of its magnitudes
template <class F> __device__ inline int rb_of(F orv, int nb) {
    const F mask = (nb >= (int)(8 * sizeof(F))) ? ~(F)0 : (((F)1 << nb) - 1);
    orv &= mask;
    if (!orv) return nb;
    const int msb = (int)(8 * sizeof(F)) - 1 - (sizeof(F) == 4 ? __clz((uint32_t)orv) : __clzll((uint64_t)orv));
    return nb - 1 - msb;
}

// Encode and decode run in workgroups of 4 waves (f32: 256 blocks, f64: 128),
// each wave on its own rows, bound by the memory's rate and the compacted
// stores. 1025 x 1025 x 257 f64, 64 planes, finest level (1.9 GB): rb 0.78 ->
// 0.37 ms, words 1.70 -> 0.76 ms, decode of 24 planes 1.68 -> 0.71 ms against
// workgroups of one wave per 64 blocks (33 KB of LDS, 4 waves per CU, two
// barriers per plane); the whole refactor + retrieve 13.06 -> 7.11 ms.
// A row of the workspace holds, per workgroup, the words of every plane p,
// #(rb <= p) + #(rb == p); the scan turns rows into offsets in place.
constexpr int kGbWaves = 4, kGbTPB = 64 * kGbWaves;
template <class T> constexpr uint32_t gb_wg_blocks() { return kGbWaves * WaveRows<T>::kBlocks; }

// h[r] counts a workgroup's blocks by recording plane: the words of planes
// pstart .. pstart + k - 1 into row[0 .. k), by the first wave (k <= 64)
__device__ __forceinline__ void gb_row(const uint32_t *h, int pstart, int k, uint32_t *__restrict__ row) {
    const int lane = (int)lane_id();
    const uint32_t below = __ockl_wfscan_add_u32(h[lane], true);  // #(rb <= lane)
    if (lane >= pstart && lane < pstart + k) row[lane - pstart] = below + h[lane];
}

// Pass 1: rb per block and the words row of each workgroup. The recording
// plane is the top bit of the OR of the block's magnitudes; they are monotone
// in |x| while the largest stays below 2^nb, so the largest |x| alone gives
// it and a block needs no lane of its own: 8 (f32) or 32 (f64) lanes share
// it through 16-byte loads and the pass reads at the memory's rate. Blocks
// with a larger value (an exponent below the level's, infinities) take the OR.
template <class T>
__device__ __forceinline__ void gb_rb_blocks(const T *__restrict__ x, uint32_t n, int32_t exp, const KeyOf<T> *key,
                                             int nb, int compat, uint8_t *__restrict__ rb,
                                             uint32_t *__restrict__ rowsum, uint32_t bid) {
    using F = typename Traits<T>::Fixed;
    using K = KeyOf<T>;
    constexpr int B = Traits<T>::kBlock, C = 16 / (int)sizeof(T);
    constexpr int G = B / C;                               // lanes per block
    constexpr int kLoads = 64 * kRowElems / (64 * C);      // 16-byte loads per lane
    constexpr K kInf = sizeof(T) == 4 ? (K)0x7f800000u : (K)0x7ff0000000000000ull;
    __shared__ uint32_t h[128];
    if (threadIdx.x < 128) h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t lane = lane_id(), wv = threadIdx.x / 64;
    const uint64_t b0 = (uint64_t)bid * gb_wg_blocks<T>() + (uint64_t)wv * WaveRows<T>::kBlocks;
    const uint64_t e0 = b0 * B;
    const uint64_t nblk = ((uint64_t)n - 1) / B + 1;
    const int shift = nb - level_exp<T>(exp, key);
    auto mag_key = [](T v) __attribute__((always_inline)) -> K {
        const K q = (K)abs_key(v);
        return q > kInf ? (K)0 : q;  // NaN has magnitude 0
    };
    K m[kLoads];
    if (rows_whole(x, n, e0)) {
        float4 q[kLoads];
#pragma unroll
        for (int i = 0; i < kLoads; i++) q[i] = *reinterpret_cast<const float4 *>(x + e0 + (64u * i + lane) * C);
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            T t[C];
            __builtin_memcpy(t, &q[i], 16);
            m[i] = 0;
#pragma unroll
            for (int c = 0; c < C; c++) { const K a = mag_key(t[c]); m[i] = a > m[i] ? a : m[i]; }
        }
    } else {
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            m[i] = 0;
#pragma unroll
            for (int c = 0; c < C; c++) {
                const uint64_t e = e0 + (64u * i + lane) * C + c;
                const K a = e < n ? mag_key(x[e]) : (K)0;
                m[i] = a > m[i] ? a : m[i];
            }
        }
    }
    // load i's lane group g holds block i * (64 / G) + g; lane g G + i of
    // the group's lanes keeps block i's maximum
    K mine = 0;
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        K a = m[i];
#pragma unroll
        for (int o = 1; o < G; o <<= 1) {
            const K t = __shfl_xor(a, o, 64);
            a = t > a ? t : a;
        }
        if ((lane % G) == (uint32_t)i % G) mine = a;
    }
    static_assert(kLoads <= G, "a lane of the group per load");
    const uint32_t bl = (lane % G) * (64 / G) + lane / G;  // this lane's block in the wave
    const uint64_t b = b0 + bl;
    if (lane % G < (uint32_t)kLoads && b < nblk) {
        F orv = 0;
        const T top = key_to_value<T>((uint64_t)mine);
        if (dev_ldexp(top, shift) < dev_ldexp((T)1, nb)) {
            orv = gb_mag<T>(top, shift, compat);
        } else {
            const uint64_t end = min((uint64_t)n, b * B + B);
            for (uint64_t e = b * B; e < end; e++) orv |= gb_mag<T>(x[e], shift, compat);
        }
        const int r = rb_of<F>(orv, nb);
        rb[b] = (uint8_t)r;
        atomicAdd(&h[r], 1u);
    }
    __syncthreads();
    if (wv == 0) gb_row(h, 0, nb, rowsum + (uint64_t)bid * nb);
}

template <class T>
__global__ __launch_bounds__(kGbTPB) void k_gb_rb(const T *__restrict__ x, uint32_t n, int32_t exp,
                                                  const KeyOf<T> *key, int nb, int compat, uint8_t *__restrict__ rb,
                                                  uint32_t *__restrict__ rowsum) {
    gb_rb_blocks<T>(x, n, exp, key, nb, compat, rb, rowsum, blockIdx.x);
}

// Offsets: rows of k words are scanned down the workgroups, a lane per plane
// (k <= 64), kGbScanRows rows per workgroup with every row load in flight.
// k_gb_sums takes the column sums of each such group, k_gb_offsets adds those
// of the groups before its own. (One workgroup per plane that summed the
// histogram bins of every row took 1,600 us for 57,700 rows x 64 planes; the
// two launches take 13 us for that level, now 28,850 rows.) A level of at
// most kGbDirectRows workgroups takes no scan launch: gb_wave_base adds the rows
// of the workgroups before its own, which costs less than the two launches
// (129^3 GroupedBP refactor + retrieve 413 -> 361 us; encode and a decode of two
// planes of floats: 367 rows 25 -> 21 and 22 -> 15 us, 733 rows 29 -> 27 and
// 24 -> 20, 977 rows 31 and 24 either way).
constexpr int kGbScanRows = 256, kGbScanPer = kGbScanRows / kGbWaves;
constexpr int kGbDirectRows = 768;
__device__ __forceinline__ void gb_scan_load(const uint32_t *__restrict__ rows, uint32_t nrow, int k, uint32_t r0,
                                             uint32_t (&v)[kGbScanPer], uint32_t &sum) {
    const uint32_t lane = lane_id();
    const auto r = buf_rsrc(rows, true);
    // masked by offset (rows take at most 2^27 bytes, so a masked lane's stays
    // out of range): a select between addresses becomes a branch per load, and
    // each is waited for by itself (367 rows: k_gb_sums 17 us, now 3)
    const uint32_t at = (int)lane < k ? (r0 * (uint32_t)k + lane) * 4 : kOffNone;
#pragma unroll
    for (int i = 0; i < kGbScanPer; i++) {
        const uint32_t in = at + i * (uint32_t)k * 4;
        v[i] = buf_load<uint32_t>(r, r0 + i < nrow ? in : kOffNone);
    }
    sum = 0;
#pragma unroll
    for (int i = 0; i < kGbScanPer; i++) sum += v[i];
}
__global__ __launch_bounds__(kGbTPB) void k_gb_sums(const uint32_t *__restrict__ rows, uint32_t nrow, int k,
                                                    uint32_t *__restrict__ sums) {
    __shared__ uint32_t part[kGbWaves][64];
    const uint32_t lane = lane_id(), wv = threadIdx.x / 64;
    uint32_t v[kGbScanPer], s;
    gb_scan_load(rows, nrow, k, blockIdx.x * kGbScanRows + wv * kGbScanPer, v, s);
    part[wv][lane] = s;
    __syncthreads();
    if (wv == 0 && (int)lane < k)
        sums[(uint64_t)blockIdx.x * k + lane] = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
}
__global__ __launch_bounds__(kGbTPB) void k_gb_offsets(uint32_t *__restrict__ rows, uint32_t nrow, int k,
                                                       const uint32_t *__restrict__ sums,
                                                       uint32_t *__restrict__ totals) {
    __shared__ uint32_t part[kGbWaves][64], below[kGbWaves][64];
    const uint32_t lane = lane_id(), wv = threadIdx.x / 64;
    const uint32_t r0 = blockIdx.x * kGbScanRows + wv * kGbScanPer;
    uint32_t v[kGbScanPer], s;
    gb_scan_load(rows, nrow, k, r0, v, s);
    // the scan groups before this one, a quarter per wave
    uint32_t b = 0;
    if ((int)lane < k) {
#pragma unroll 8
        for (uint32_t c = wv; c < blockIdx.x; c += kGbWaves) b += sums[(uint64_t)c * k + lane];
    }
    part[wv][lane] = s;
    below[wv][lane] = b;
    __syncthreads();
    uint32_t o = (below[0][lane] + below[1][lane]) + (below[2][lane] + below[3][lane]);
    for (uint32_t w = 0; w < wv; w++) o += part[w][lane];
    if ((int)lane >= k) return;
#pragma unroll
    for (int i = 0; i < kGbScanPer; i++) {
        if (r0 + i < nrow) rows[(uint64_t)(r0 + i) * k + lane] = o;
        o += v[i];
    }
    if (totals && blockIdx.x == gridDim.x - 1 && wv == kGbWaves - 1) totals[lane] = o;  // the whole plane's words
}
static int gb_scan(uint32_t *rows, uint32_t nrow, int k, uint32_t *sums, uint32_t *totals, hipStream_t s) {
    const uint32_t grid = div_up(nrow, kGbScanRows);
    if (nrow <= (uint32_t)kGbDirectRows) return kOk;  // gb_wave_base sums the rows itself
    hipLaunchKernelGGL(k_gb_sums, dim3(grid), dim3(kGbTPB), 0, s, rows, nrow, k, sums);
    PRODM_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_gb_offsets, dim3(grid), dim3(kGbTPB), 0, s, rows, nrow, k, sums, totals);
    PRODM_CHECK_LAUNCH();
    return kOk;
}

// Positions of a wave's blocks in the planes. Lane p of the result holds where
// the wave's first word of plane pstart + p goes: the workgroup's offset plus
// the words of the waves before it, from the recording planes of the
// workgroup's blocks (one barrier). rows: offsets per workgroup, or with at
// most kGbDirectRows workgroups their words, which are summed here; totals
// (then, if any) takes the words of every plane. r: the lane's block's rb, 255
// past the data. Both lanes of an f64 block hold the same r.
struct GbWaveLds {
    uint32_t hw[kGbWaves][64], below[kGbWaves][64];
};
template <class T>
__device__ __forceinline__ uint32_t gb_wave_base(int r, const uint32_t *__restrict__ rows, int pstart, int k,
                                                 uint32_t *__restrict__ totals, GbWaveLds &lds, uint32_t bid,
                                                 uint32_t nwg) {
    const uint32_t lane = lane_id(), wv = threadIdx.x / 64;
    const bool on = (int)lane < k, direct = nwg <= (uint32_t)kGbDirectRows;
    lds.hw[wv][lane] = 0;
    if (r < 64 && lane < (uint32_t)WaveRows<T>::kBlocks) atomicAdd(&lds.hw[wv][r], 1u);
    uint32_t b = 0;
    if (direct && on) {
#pragma unroll 8
        for (uint32_t c = wv; c < bid; c += kGbWaves) b += rows[(uint64_t)c * k + lane];
    }
    lds.below[wv][lane] = b;
    __syncthreads();
    uint32_t hb = 0;
    for (uint32_t w = 0; w < wv; w++) hb += lds.hw[w][lane];
    const uint32_t words = __ockl_wfscan_add_u32(hb, true) + hb;  // lane p: plane p
    // window lane i <- plane pstart + i
    const uint32_t shifted = __shfl(words, (int)((lane + (uint32_t)pstart) & 63u), 64);
    uint32_t own = on && (!direct || totals) ? rows[(uint64_t)bid * k + lane] : 0u;
    if (direct) {
        const uint32_t o = (lds.below[0][lane] + lds.below[1][lane]) + (lds.below[2][lane] + lds.below[3][lane]);
        if (totals && on && wv == 0 && bid == nwg - 1) totals[lane] = o + own;
        own = o;
    }
    return on ? own + shifted : 0u;
}
// word index of this lane's block in plane window index i, from the wave's
// ballots of (rb <= p) and (rb == p)
template <class T>
__device__ __forceinline__ uint32_t gb_pos(uint32_t base, int i, uint64_t le, uint64_t eq) {
    if constexpr (sizeof(T) == 4) {
        return readlane_u32(base, i) + lanes_below(le) + lanes_below(eq);
    } else {
        const uint32_t bm = (1u << (lane_id() & 31u)) - 1u;
        return readlane_u32(base, i) + __popc((uint32_t)le & bm) + __popc((uint32_t)eq & bm);
    }
}

// Pass 2: plane words, compacted per plane. The positions need no barrier
// inside the plane loop (gb_wave_base).
template <class T>
__device__ __forceinline__ void gb_write_blocks(const T *__restrict__ x, uint32_t n, int32_t exp, const KeyOf<T> *key,
                                                int nb, int compat, const uint8_t *__restrict__ rb,
                                                const uint32_t *__restrict__ off,
                                                typename Traits<T>::Stream *__restrict__ planes, uint64_t stride,
                                                uint32_t *__restrict__ totals, uint32_t bid, uint32_t nwg) {
    using R = WaveRows<T>;
    constexpr int B = Traits<T>::kBlock, W = 8 * (int)sizeof(T);
    __shared__ __align__(16) uint32_t rows[kGbWaves][64 * kRowPitch];
    __shared__ GbWaveLds wl;
    const uint32_t lane = lane_id(), wv = threadIdx.x / 64;
    const uint64_t b0 = (uint64_t)bid * gb_wg_blocks<T>() + (uint64_t)wv * R::kBlocks;
    const uint32_t bl = lane % R::kBlocks, half = lane / R::kBlocks;
    const uint64_t b = b0 + bl, nblk = ((uint64_t)n - 1) / B + 1;
    const int r = b < nblk ? rb[b] : 255;
    // before the elements: its loop over rows would hold registers beside them
    const uint32_t base = gb_wave_base<T>(r, off, 0, nb, totals, wl, bid, nwg);
    const int shift = nb - level_exp<T>(exp, key);
    uint32_t w[W], sg = 0;
    rows_in<T>(x, n, b0 * B, rows[wv], [&](int j, T v) __attribute__((always_inline)) {
        const uint64_t q = gb_mag<T>(v, shift, compat);
        w[j] = (uint32_t)q;
        if constexpr (sizeof(T) == 8) w[32 + j] = (uint32_t)(q >> 32);
        sg |= (uint32_t)(v < 0) << j;
    });
    transpose32_at<0>(w);
    if constexpr (sizeof(T) == 8) transpose32_at<32>(w);
    static_for<0, W>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        const int p = nb - 1 - k;  // plane p holds bit nb - 1 - p
        if (p >= 0) {
            const uint64_t le = ballot64(r <= p), eq = ballot64(r == p);
            uint32_t pos = gb_pos<T>(base, p, le, eq);
            uint32_t *dst = reinterpret_cast<uint32_t *>(planes + (uint64_t)p * stride) + half;
            if (r == p) { dst[(uint64_t)pos * R::kHalves] = sg; pos++; }
            if (r <= p) dst[(uint64_t)pos * R::kHalves] = w[k];
        }
    });
}

template <class T>
__global__ __launch_bounds__(kGbTPB) void k_gb_write(const T *__restrict__ x, uint32_t n, int32_t exp,
                                                     const KeyOf<T> *key, int nb, int compat,
                                                     const uint8_t *__restrict__ rb, const uint32_t *__restrict__ off,
                                                     typename Traits<T>::Stream *__restrict__ planes, uint64_t stride,
                                                     uint32_t *__restrict__ totals) {
    gb_write_blocks<T>(x, n, exp, key, nb, compat, rb, off, planes, stride, totals, blockIdx.x, gridDim.x);
}

// workgroups of the formula the workspace sizes were first given out with;
// the buffers below need less
template <class T> static uint32_t gb_ws_rows(uint32_t n) {
    const uint32_t nblk = (n - 1) / Traits<T>::kBlock + 1;
    return div_up(nblk, BlkStage<T>::kTPB);
}
template <class T> static uint32_t gb_nwg(uint32_t n) {
    const uint32_t nblk = (n - 1) / Traits<T>::kBlock + 1;
    return div_up(nblk, gb_wg_blocks<T>());
}

template <class T> size_t gb_workspace_bytes(uint32_t n, int nb) {
    const uint32_t nwg = gb_ws_rows<T>(n);
    return (size_t)nwg * (nb + 1) * 4 + (size_t)nwg * nb * 4 + 256;
}
template size_t gb_workspace_bytes<float>(uint32_t, int);
template size_t gb_workspace_bytes<double>(uint32_t, int);
// rows and the scan's column sums, in words
template <class T> static size_t gb_scan_words(uint32_t n, int k) {
    const uint32_t nwg = gb_nwg<T>(n);
    return ((size_t)nwg + div_up(nwg, kGbScanRows)) * k;
}

template <class T>
int launch_gb_encode(const T *x, uint32_t n, int32_t exp, const KeyOf<T> *key, int nb, int compat, uint8_t *rb,
                     typename Traits<T>::Stream *planes, uint64_t stride, uint32_t *words_per_plane, void *ws,
                     size_t ws_bytes, hipStream_t s) {
    constexpr int B = Traits<T>::kBlock;
    if (n == 0 || nb < 1 || nb > B) { set_error("grouped encode: bad n or num_bitplanes"); return kErrArg; }
    const uint32_t nblk = (n - 1) / B + 1;
    if (stride < 2ull * nblk) { set_error("grouped encode: plane stride below 2 * nblocks"); return kErrArg; }
    if (ws_bytes < gb_workspace_bytes<T>(n, nb) || ws_bytes < gb_scan_words<T>(n, nb) * 4) {
        set_error("grouped encode: workspace too small");
        return kErrArg;
    }
    const uint32_t nwg = gb_nwg<T>(n);
    uint32_t *rows = static_cast<uint32_t *>(ws), *sums = rows + (size_t)nwg * nb;
    hipLaunchKernelGGL(k_gb_rb<T>, dim3(nwg), dim3(kGbTPB), 0, s, x, n, exp, key, nb, compat, rb, rows);
    PRODM_CHECK_LAUNCH();
    if (int rc = gb_scan(rows, nwg, nb, sums, words_per_plane, s)) return rc;
    hipLaunchKernelGGL(k_gb_write<T>, dim3(nwg), dim3(kGbTPB), 0, s, x, n, exp, key, nb, compat, rb, rows, planes,
                       stride, words_per_plane);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_gb_encode<float>(const float *, uint32_t, int32_t, const uint32_t *, int, int, uint8_t *,
                                     uint32_t *, uint64_t, uint32_t *, void *, size_t, hipStream_t);
template int launch_gb_encode<double>(const double *, uint32_t, int32_t, const unsigned long long *, int, int,
                                      uint8_t *, uint64_t *, uint64_t, uint32_t *, void *, size_t, hipStream_t);

// ---- GroupedBP progressive decode ----------------------------------------------
// words rows of planes [start, start + k) from the recording planes
template <class T>
__device__ __forceinline__ void gb_rbrows_blocks(const uint8_t *__restrict__ rb, uint32_t nblk, int start, int k,
                                                 uint32_t *__restrict__ rows, uint32_t bid) {
    __shared__ uint32_t h[64];
    if (threadIdx.x < 64) h[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t b = (uint64_t)bid * gb_wg_blocks<T>() + threadIdx.x;
    if (threadIdx.x < gb_wg_blocks<T>() && b < nblk) {
        const int r = rb[b];
        if (r < 64) atomicAdd(&h[r], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 64) gb_row(h, start, k, rows + (uint64_t)bid * k);
}

template <class T>
__global__ __launch_bounds__(kGbTPB) void k_gb_rbrows(const uint8_t *__restrict__ rb, uint32_t nblk, int start, int k,
                                                      uint32_t *__restrict__ rows) {
    gb_rbrows_blocks<T>(rb, nblk, start, k, rows, blockIdx.x);
}

// 32-bit word at any byte offset (stream 0's words follow its header)
__device__ __forceinline__ uint32_t load_bytes32(const uint8_t *p) {
    return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}

// Lanes hold 32 elements of a block as in the encode. The words of all k
// planes are loaded without branches: a lane without a word in a plane (rb
// above it) takes the offset past the buffer's range and reads 0. A plane
// holds at most 2 words per block, 2^30 bytes at 2^32 elements.
template <class T, class PlaneFn>
__device__ __forceinline__ void gb_decode_blocks(PlaneFn &&plane, uint32_t n, int32_t exp, const KeyOf<T> *key,
                                                 int start, int k, const uint8_t *__restrict__ rb,
                                                 typename Traits<T>::Stream *__restrict__ signs,
                                                 const uint32_t *__restrict__ off, T *__restrict__ out, uint64_t hdr0,
                                                 uint32_t bid, uint32_t nwg) {
    using R = WaveRows<T>;
    constexpr int B = Traits<T>::kBlock, W = 8 * (int)sizeof(T);
    __shared__ __align__(16) uint32_t rows[kGbWaves][64 * kRowPitch];
    __shared__ GbWaveLds wl;
    const uint32_t lane = lane_id(), wv = threadIdx.x / 64;
    const uint64_t b0 = (uint64_t)bid * gb_wg_blocks<T>() + (uint64_t)wv * R::kBlocks;
    const uint32_t bl = lane % R::kBlocks, half = lane / R::kBlocks;
    const uint64_t b = b0 + bl, nblk = ((uint64_t)n - 1) / B + 1;
    const bool valid = b < nblk;
    const int e0 = level_exp<T>(exp, key);
    const int end = start + k;
    const int r = valid ? rb[b] : 255;
    uint32_t *const sgw = reinterpret_cast<uint32_t *>(signs) + b * R::kHalves + half;
    uint32_t sg = valid ? *sgw : 0u;
    const uint32_t base = gb_wave_base<T>(r, off, start, k, nullptr, wl, bid, nwg);
    // acc bit (end - 1 - p) comes from plane p; planes below rb are zero
    const uint8_t *sgat = nullptr;
    uint32_t w[W];
    static_for<0, W>([&](auto qc) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value;
        const int p = end - 1 - q, i = p - start;
        w[q] = 0;
        if (i >= 0) {
            const uint64_t le = ballot64(r <= p), eq = ballot64(r == p);
            const uint32_t pos = gb_pos<T>(base, i, le, eq), at = (pos * R::kHalves + half) * 4;
            const uint8_t *sb = plane(i) + (i == 0 ? hdr0 : 0);
            if (eq && r == p) sgat = sb + at;
            const uint32_t word = at + (r == p ? 4 * R::kHalves : 0);
            if (i == 0 && (hdr0 & 3)) {
                if (r <= p) w[q] = load_bytes32(sb + word);
            } else {
                w[q] = buf_load<uint32_t>(buf_rsrc(sb, true), r <= p ? word : kOffNone);
            }
        }
    });
    const bool fresh = r >= start && r < end;  // recorded in this window: its sign word precedes plane r's
    if (fresh) sg = r == start && (hdr0 & 3) ? load_bytes32(sgat) : *reinterpret_cast<const uint32_t *>(sgat);
    if (fresh) *sgw = sg;
    transpose32_at<0>(w);
    if constexpr (sizeof(T) == 8) transpose32_at<32>(w);
    T v[kRowElems];
#pragma unroll
    for (int j = 0; j < kRowElems; j++) {
        T y;
        if constexpr (sizeof(T) == 4) y = dev_ldexp((T)w[j], e0 - end);
        else y = dev_ldexp((T)(((uint64_t)w[32 + j] << 32) | w[j]), e0 - end);
        if ((sg >> j) & 1u) y = -y;
        v[j] = (r >= end) ? (T)0 : y;
    }
    rows_out<T>(out, n, b0 * B, rows[wv], v);
}

template <class T>
__global__ __launch_bounds__(kGbTPB) void k_gb_decode(PlanePtrs pl, uint32_t n, int32_t exp, const KeyOf<T> *key,
                                                      int start, int k, const uint8_t *__restrict__ rb,
                                                      typename Traits<T>::Stream *__restrict__ signs,
                                                      const uint32_t *__restrict__ off, T *__restrict__ out,
                                                      uint64_t hdr0) {
    gb_decode_blocks<T>([&](int i) __attribute__((always_inline)) { return static_cast<const uint8_t *>(pl.p[i]); }, n,
                        exp, key, start, k, rb, signs, off, out, hdr0, blockIdx.x, gridDim.x);
}

template <class T>
int launch_gb_decode(const PlanePtrs &streams, uint32_t n, int32_t exp, const KeyOf<T> *key, int start, int k,
                     const uint8_t *rb, typename Traits<T>::Stream *signs, T *out, void *ws, size_t ws_bytes,
                     uint64_t hdr0, hipStream_t s) {
    constexpr int B = Traits<T>::kBlock;
    if (n == 0) return kOk;
    if (k < 0 || start < 0 || start + k > B) { set_error("grouped decode: bad plane range"); return kErrArg; }
    if (k == 0) {
        if constexpr (sizeof(T) == 4) return launch_fill_u32(reinterpret_cast<uint32_t *>(out), n, 0u, s);
        else return launch_fill_u64(reinterpret_cast<uint64_t *>(out), n, 0ull, s);
    }
    const uint32_t nblk = (n - 1) / B + 1;
    const uint32_t nwg = gb_nwg<T>(n);
    if (ws_bytes < gb_decode_workspace_bytes<T>(n, start, k) || ws_bytes < gb_scan_words<T>(n, k) * 4) {
        set_error("grouped decode: workspace too small");
        return kErrArg;
    }
    uint32_t *rows = static_cast<uint32_t *>(ws), *sums = rows + (size_t)nwg * k;
    if (nwg > 1) {  // a single workgroup has no offset
        hipLaunchKernelGGL(k_gb_rbrows<T>, dim3(nwg), dim3(kGbTPB), 0, s, rb, nblk, start, k, rows);
        PRODM_CHECK_LAUNCH();
    }
    if (int rc = gb_scan(rows, nwg, k, sums, nullptr, s)) return rc;
    hipLaunchKernelGGL(k_gb_decode<T>, dim3(nwg), dim3(kGbTPB), 0, s, streams, n, exp, key, start, k, rb, signs, rows,
                       out, hdr0);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_gb_decode<float>(const PlanePtrs &, uint32_t, int32_t, const uint32_t *, int, int, const uint8_t *,
                                     uint32_t *, float *, void *, size_t, uint64_t, hipStream_t);
template int launch_gb_decode<double>(const PlanePtrs &, uint32_t, int32_t, const unsigned long long *, int, int,
                                      const uint8_t *, uint64_t *, double *, void *, size_t, uint64_t, hipStream_t);

template <class T> size_t gb_decode_workspace_bytes(uint32_t n, int start, int k) {
    const uint32_t nwg = gb_ws_rows<T>(n);
    return (size_t)nwg * (start + 2 * k) * 4 + 64 * 4 + 256;
}
template size_t gb_decode_workspace_bytes<float>(uint32_t, int, int);
template size_t gb_decode_workspace_bytes<double>(uint32_t, int, int);

// ---- small levels of a plan together (at most kGbDirectRows workgroups each) -------
template <class T> __global__ __launch_bounds__(kGbTPB) void k_gb_rb_set(LevelSet<GbLevel<T>> L, int nb) {
    const uint32_t i = set_entry(L, blockIdx.x);
    const GbLevel<T> &E = L.e[i];
    gb_rb_blocks<T>(E.x, E.n, 0, E.key, nb, 0, E.rb, E.rows, blockIdx.x - L.first[i]);
}
template <class T> __global__ __launch_bounds__(kGbTPB) void k_gb_write_set(LevelSet<GbLevel<T>> L, int nb) {
    const uint32_t i = set_entry(L, blockIdx.x);
    const GbLevel<T> &E = L.e[i];
    gb_write_blocks<T>(E.x, E.n, 0, E.key, nb, 0, E.rb, E.rows, E.planes, E.stride, E.words, blockIdx.x - L.first[i],
                       L.first[i + 1] - L.first[i]);
}
template <class T> __global__ __launch_bounds__(kGbTPB) void k_gb_rbrows_set(LevelSet<GbLevel<T>> L) {
    const uint32_t i = set_entry(L, blockIdx.x);
    const GbLevel<T> &E = L.e[i];
    gb_rbrows_blocks<T>(E.rb, (E.n - 1) / Traits<T>::kBlock + 1, 0, E.k, E.rows, blockIdx.x - L.first[i]);
}
template <class T> __global__ __launch_bounds__(kGbTPB) void k_gb_decode_set(LevelSet<GbLevel<T>> L) {
    const uint32_t i = set_entry(L, blockIdx.x);
    const GbLevel<T> &E = L.e[i];
    const typename Traits<T>::Stream *planes = E.planes;
    const uint64_t stride = E.stride;
    gb_decode_blocks<T>(
        [&](int p) __attribute__((always_inline)) { return reinterpret_cast<const uint8_t *>(planes + (uint64_t)p * stride); },
        E.n, 0, E.key, 0, E.k, E.rb, E.signs, E.rows, E.x, 0, blockIdx.x - L.first[i], L.first[i + 1] - L.first[i]);
}
template <class T> size_t gb_set_row_words(uint32_t n, int nb) {
    const uint32_t nwg = gb_nwg<T>(n);
    return nwg <= (uint32_t)kGbDirectRows ? (size_t)nwg * nb : 0;
}
template size_t gb_set_row_words<float>(uint32_t, int);
template size_t gb_set_row_words<double>(uint32_t, int);
template <class T> int launch_gb_encode_set(LevelSet<GbLevel<T>> L, int nb, hipStream_t s) {
    if (!L.n) return kOk;
    for (uint32_t i = 0; i < L.n; i++)
        if (L.e[i].n == 0 || nb < 1 || nb > Traits<T>::kBlock || !gb_set_row_words<T>(L.e[i].n, nb)) {
            set_error("grouped encode: bad n or num_bitplanes");
            return kErrArg;
        }
    set_sizes(L, [](const GbLevel<T> &e) { return gb_nwg<T>(e.n); });
    hipLaunchKernelGGL(k_gb_rb_set<T>, dim3(L.first[L.n]), dim3(kGbTPB), 0, s, L, nb);
    PRODM_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_gb_write_set<T>, dim3(L.first[L.n]), dim3(kGbTPB), 0, s, L, nb);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template <class T> int launch_gb_decode_set(LevelSet<GbLevel<T>> L, hipStream_t s) {
    if (!L.n) return kOk;
    for (uint32_t i = 0; i < L.n; i++)
        if (L.e[i].k < 0 || L.e[i].k > Traits<T>::kBlock || (L.e[i].n && !gb_set_row_words<T>(L.e[i].n, 1))) {
            set_error("grouped decode: bad plane range or level size");
            return kErrArg;
        }
    set_sizes(L, [](const GbLevel<T> &e) { return e.n ? gb_nwg<T>(e.n) : 0; });
    if (!L.first[L.n]) return kOk;
    hipLaunchKernelGGL(k_gb_rbrows_set<T>, dim3(L.first[L.n]), dim3(kGbTPB), 0, s, L);
    PRODM_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_gb_decode_set<T>, dim3(L.first[L.n]), dim3(kGbTPB), 0, s, L);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_gb_encode_set<float>(LevelSet<GbLevel<float>>, int, hipStream_t);
template int launch_gb_encode_set<double>(LevelSet<GbLevel<double>>, int, hipStream_t);
template int launch_gb_decode_set<float>(LevelSet<GbLevel<float>>, hipStream_t);
template int launch_gb_decode_set<double>(LevelSet<GbLevel<double>>, hipStream_t);

// ------------------------------------------------------------------------------
// PerBit
// ------------------------------------------------------------------------------
// Stream p carries bit nb - 1 - p of every element's magnitude, element by
// element, and right after an element's first 1 bit (over planes 0..nb-1)
// its sign; bits fill 64-bit words LSB first (PerBitBPEncoder.hpp:9-39,
// 96-143). Encode runs in three passes over runs of 64 lanes x B
// consecutive elements (one wave): count (first-1 flags per plane), scan
// (bit offset of every wave's run in every stream) and write (each lane
// expands its plane word with its sign bits; the wave assembles its run
// in LDS and stores whole words).

// T_fp of the reference, sign ? -(int64_t) v : (int64_t) v with
// v = ldexp(x, nb - exp) (PerBitBPEncoder.hpp:101-104). The conversion of
// |v| >= 2^63 or NaN is undefined in C++: compat gives the x86 result
// (INT64_MIN, which is its own negation), otherwise the truncated
// magnitude is used, as for GroupedBP (hazard B1).
template <class T>
__device__ inline typename Traits<T>::Fixed pb_mag(T x, int shift, int compat) {
    using F = typename Traits<T>::Fixed;
    if (!compat) return gb_mag<T>(x, shift, 0);
    const T v = dev_ldexp(x, shift);
    if constexpr (sizeof(T) == 4) {  // trunc(|v|): the low word of either sign's conversion
        const float a = fabsf(v);
        if (a < 4294967296.0f) return (F)a;
    }
    const int64_t q = fabs(v) < (T)9.2233720368547758e18 ? (int64_t)v : INT64_MIN;
    return (F)(x < 0 ? (uint64_t)0 - (uint64_t)q : (uint64_t)q);
}

// Every lane takes 32 consecutive elements (f32 and f64), a wave 2048, a
// workgroup of 4 waves 8192; a lane's run in a stream is at most 64 bits.
constexpr int kPbTPB = 256, kPbB = 32;

// The lane's 32 elements straight from global memory (16-byte loads when
// the row is whole and aligned) as plane words kept in registers: w[k] bit
// j = bit k of element j's magnitude (k < 32 for f32, < 64 for f64); sg
// bit j = element j < 0.
template <class T> struct PbLane {
    static constexpr int kWords = 8 * sizeof(T);
    uint32_t w[kWords];
    uint32_t sg;
    __device__ __forceinline__ void load(const T *__restrict__ x, uint64_t e, uint32_t n, int shift, int compat, bool vec) {
        T v[kPbB];
        if (vec && e + kPbB <= n) {
            if constexpr (sizeof(T) == 4) {
                const float4 *q = reinterpret_cast<const float4 *>(x + e);
#pragma unroll
                for (int i = 0; i < kPbB / 4; i++) {
                    const float4 t = q[i];
                    v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
                }
            } else {
                const double2 *q = reinterpret_cast<const double2 *>(x + e);
#pragma unroll
                for (int i = 0; i < kPbB / 2; i++) {
                    const double2 t = q[i];
                    v[2 * i] = t.x; v[2 * i + 1] = t.y;
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < kPbB; j++) v[j] = e + j < n ? x[e + j] : (T)0;
        }
        sg = 0;
#pragma unroll
        for (int j = 0; j < kPbB; j++) {
            const uint64_t q = pb_mag<T>(v[j], shift, compat);
            w[j] = (uint32_t)q;
            if constexpr (sizeof(T) == 8) w[32 + j] = (uint32_t)(q >> 32);
            sg |= (uint32_t)(v[j] < 0) << j;
        }
        transpose32_at<0>(w);
        if constexpr (sizeof(T) == 8) transpose32_at<32>(w);
    }
};
// f(p, D, F) for the planes p = 0..nb-1 in order: D = the plane word (bit
// nb - 1 - p of the lane's elements), F = the elements whose first 1 bit is
// in plane p. Unrolled, so that the words stay in registers.
template <class T, class Fn> __device__ __forceinline__ void pb_for_planes(const PbLane<T> &P, int nb, Fn &&f) {
    constexpr int W = PbLane<T>::kWords;
    uint32_t H = 0;
    static_for<0, W>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = W - 1 - decltype(kc)::value;
        const int p = nb - 1 - k;
        if (p >= 0) {
            const uint32_t D = P.w[k];
            const uint32_t F = D & ~H;
            H |= D;
            f(p, D, F);
        }
    });
}

// The first-1 counts of planes 2i and 2i + 1 packed in one word (low and
// high 16 bits: a lane counts at most 32 per plane, a wave at most 2048), so
// that one wave-wide scan or sum serves two planes. f(i, packed count) for
// the pairs i in plane order; planes p < 0 (nb below the word count) count 0.
template <class T, class Fn> __device__ __forceinline__ void pb_for_plane_pairs(const PbLane<T> &P, int nb, Fn &&f) {
    constexpr int W = PbLane<T>::kWords;
    uint32_t H = 0, acc = 0;
    static_for<0, W>([&](auto kc) __attribute__((always_inline)) {
        constexpr int i = decltype(kc)::value;
        constexpr int k = W - 1 - i;
        const bool on = nb - 1 - k >= 0;
        const uint32_t D = on ? P.w[k] : 0u;
        const uint32_t c = (uint32_t)__popc(D & ~H);
        H |= D;
        if constexpr (i % 2 == 0) acc = c;
        else f(i / 2, acc | (c << 16));
    });
}

// Runs are cut per wave (64 lanes x 32 consecutive elements).
template <class T> static uint32_t pb_nwg(uint32_t n) { return div_up(n, (uint64_t)kPbTPB * kPbB); }
template <class T> static uint32_t pb_nwaves(uint32_t n) { return pb_nwg<T>(n) * (kPbTPB / 64); }

// valid elements of wave gw
template <class T> __device__ inline uint32_t pb_wave_valid(uint32_t n, uint32_t gw) {
    constexpr uint64_t E = 64ull * kPbB;
    const uint64_t e = (uint64_t)gw * E;
    return e < n ? (uint32_t)min(E, (uint64_t)n - e) : 0u;
}

// Pass 1: bits[p][gw] = bits of wave gw's run in plane p: its valid
// elements plus those whose first 1 bit is in plane p.
template <class T>
__global__ __launch_bounds__(kPbTPB) void k_pb_count(const T *__restrict__ x, uint32_t n, int32_t exp,
                                                  const KeyOf<T> *key, int nb, int compat,
                                                  uint32_t *__restrict__ bits, uint32_t nwv) {
    constexpr int NW = kPbTPB / 64;
    const int lane = (int)lane_id();
    const uint32_t gw = blockIdx.x * NW + threadIdx.x / 64;
    PbLane<T> P;
    P.load(x, ((uint64_t)blockIdx.x * kPbTPB + threadIdx.x) * kPbB, n, nb - level_exp<T>(exp, key), compat,
           ((uintptr_t)x & 15) == 0);
    uint32_t mine = 0;  // lane p: plane p's first-1 flags of the wave
    constexpr int W = PbLane<T>::kWords;
    pb_for_plane_pairs(P, nb, [&](int i, uint32_t pc) {
        const uint32_t s = __ockl_wfred_add_u32(pc);
        // pair i holds the planes with word indices W - 1 - 2i, W - 2 - 2i
        const int pa = nb - W + 2 * i, pb = pa + 1;
        if (lane == pa) mine = s & 0xFFFFu;
        if (lane == pb) mine = s >> 16;
    });
    if (lane < nb) bits[(uint64_t)lane * nwv + gw] = pb_wave_valid<T>(n, gw) + mine;
}

// Pass 2: exclusive bit offsets off[p][gw] of the wave runs and the stream
// sizes in bytes (whole words). Blocks of kPbScanBlk waves per plane: their
// sums, then every block's waves with the sum of the blocks below.
constexpr int kPbScanT = 1024, kPbScanPer = 4, kPbScanBlk = kPbScanT * kPbScanPer;

// sum over the workgroup (all threads call it); result on thread 0
__device__ inline uint64_t pb_block_sum(uint64_t v, uint64_t *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane_id() == 0) red[threadIdx.x / 64] = v;
    __syncthreads();
    uint64_t t = 0;
    if (threadIdx.x == 0)
        for (uint32_t i = 0; i < blockDim.x / 64; i++) t += red[i];
    return t;
}

__global__ __launch_bounds__(kPbScanT) void k_pb_scan_sum(const uint32_t *__restrict__ bits, uint32_t nwv,
                                                         uint64_t *__restrict__ sums) {
    __shared__ uint64_t red[kPbScanT / 64];
    const int p = blockIdx.y;
    const uint32_t *row = bits + (uint64_t)p * nwv;
    uint32_t v = 0;
#pragma unroll
    for (int i = 0; i < kPbScanPer; i++) {
        const uint32_t w = blockIdx.x * kPbScanBlk + i * kPbScanT + threadIdx.x;
        if (w < nwv) v += row[w];
    }
    const uint64_t t = pb_block_sum(v, red);
    if (threadIdx.x == 0) sums[(uint64_t)p * gridDim.x + blockIdx.x] = t;
}

__global__ __launch_bounds__(kPbScanT) void k_pb_scan_off(const uint32_t *__restrict__ bits, uint32_t nwv,
                                                         const uint64_t *__restrict__ sums,
                                                         uint64_t *__restrict__ off, uint32_t *__restrict__ sizes) {
    __shared__ uint64_t red[kPbScanT / 64];
    __shared__ uint32_t wtot[kPbScanT / 64];
    __shared__ uint64_t base_s;
    const int p = blockIdx.y;
    const uint32_t blk = blockIdx.x, lane = lane_id(), wv = threadIdx.x / 64;
    const uint32_t *row = bits + (uint64_t)p * nwv;
    uint64_t *orow = off + (uint64_t)p * nwv;
    // bits below this block
    const uint64_t b = pb_block_sum(threadIdx.x < blk ? sums[(uint64_t)p * gridDim.x + threadIdx.x] : 0, red);
    if (threadIdx.x == 0) base_s = b;
    // this thread's waves [w0, w0 + kPbScanPer)
    const uint32_t w0 = blk * kPbScanBlk + threadIdx.x * kPbScanPer;
    uint32_t v[kPbScanPer], local = 0;
#pragma unroll
    for (int i = 0; i < kPbScanPer; i++) {
        v[i] = w0 + i < nwv ? row[w0 + i] : 0;
        local += v[i];
    }
    const uint32_t pre = __ockl_wfscan_add_u32(local, false);
    if (lane == 63) wtot[wv] = pre + local;
    __syncthreads();
    uint64_t o = base_s + pre;
    for (uint32_t i = 0; i < wv; i++) o += wtot[i];
#pragma unroll
    for (int i = 0; i < kPbScanPer; i++) {
        if (w0 + i < nwv) {
            orow[w0 + i] = o;
            o += v[i];
            if (w0 + i == nwv - 1) sizes[p] = (uint32_t)(((o + 63) >> 6) * 8);  // the stream's end
        }
    }
}

// Pass 3: the streams. Lane t of wave gw starts its run in plane p at bit
// off[p][gw] + min(t B, valid) + (first-1 flags of the lanes below). The
// wave assembles its run in its own LDS words (in wave order, no
// barriers) and stores them.
template <class T>
__global__ __launch_bounds__(kPbTPB) void k_pb_write(const T *__restrict__ x, uint32_t n, int32_t exp,
                                                  const KeyOf<T> *key, int nb, int compat,
                                                  const uint64_t *__restrict__ off, uint32_t nwv,
                                                  uint64_t *__restrict__ streams, uint64_t stride,
                                                  uint64_t *__restrict__ side) {
    constexpr int B = kPbB, NW = kPbTPB / 64;
    constexpr int kRunWords = (2 * 64 * B + 63) / 64 + 2;  // a wave's run plus its start offset
    __shared__ unsigned long long run[NW][kRunWords];
    const int lane = (int)lane_id();
    const uint32_t wv = threadIdx.x / 64, gw = blockIdx.x * NW + wv;
    unsigned long long *buf = run[wv];
    for (int i = lane; i < kRunWords; i += 64) buf[i] = 0;
    const uint64_t my_off = lane < nb ? off[(uint64_t)lane * nwv + gw] : 0;  // lane p: plane p's offset
    const uint32_t nv = pb_wave_valid<T>(n, gw);
    const uint32_t below = min((uint32_t)lane * B, nv);  // valid elements of the lanes below
    PbLane<T> P;
    P.load(x, ((uint64_t)blockIdx.x * kPbTPB + threadIdx.x) * B, n, nb - level_exp<T>(exp, key), compat,
           ((uintptr_t)x & 15) == 0);
    const uint32_t S = P.sg, S1 = S << 1;  // sign bits of the lane's elements
    // first-1 flags of the lanes below and of the wave: for f32 two planes
    // per scan, computed before the plane loop (16 words); f64's 64 planes
    // would hold 32 of them, so it scans per plane
    constexpr int W = PbLane<T>::kWords;
    constexpr bool kPairs = sizeof(T) == 4;
    uint32_t pre2[kPairs ? W / 2 : 1], tot2[kPairs ? W / 2 : 1];
    if constexpr (kPairs)
        pb_for_plane_pairs(P, nb, [&](int i, uint32_t pc) __attribute__((always_inline)) {
            pre2[i] = __ockl_wfscan_add_u32(pc, false);
            tot2[i] = readlane_u32(pre2[i] + pc, 63);
        });
    pb_for_planes(P, nb, [&](int p, uint32_t D, uint32_t F) __attribute__((always_inline)) {
        const uint64_t o = ((uint64_t)readlane_u32((uint32_t)(my_off >> 32), p) << 32) |
                           readlane_u32((uint32_t)my_off, p);
        uint32_t pre, flags;
        if constexpr (kPairs) {
            // p = nb - W + i for the plane order index i, in pair i / 2
            const int i = p - nb + W;
            const uint32_t sh16 = (i & 1) ? 16u : 0u;
            pre = (pre2[i >> 1] >> sh16) & 0xFFFFu;
            flags = (tot2[i >> 1] >> sh16) & 0xFFFFu;  // the wave's total
        } else {
            const uint32_t c = (uint32_t)__popc(F);
            pre = __ockl_wfscan_add_u32(c, false);
            flags = readlane_u32(pre + c, 63);
        }
        const uint32_t q = (uint32_t)(o & 63) + below + pre;
        // insert each flagged element's sign after its bit, highest first:
        // adding the bits above an element to themselves moves them up by
        // one (the low word's carry is the high word's new bit 0). c = the bit
        // above the element; element 31, whose c is in the high word, first. The
        // loop runs as often as the lane with the most flags needs and is what
        // bounds the kernel: with 64-bit masks and shifts 2^27 - 2^24 fp32
        // elements took 431 us, the whole encode 580 -> 513
        uint32_t lo = D, hi = (S & F) >> 31;
        uint32_t ff = F << 1;
        while (ff) {
            const uint32_t c = 0x80000000u >> __clz(ff);
            ff ^= c;
            const uint64_t up = (uint64_t)lo + (lo & (0u - c));
            hi = hi + hi + (uint32_t)(up >> 32);
            lo = (uint32_t)up | (S1 & c);
        }
        const uint64_t r = ((uint64_t)hi << 32) | lo;
        const uint32_t wi = q >> 6, sh = q & 63;
        const uint64_t w0 = r << sh, w1 = (r >> 1) >> (63 - sh);
        atomicOr(&buf[wi], w0);  // unconditional: OR-ing zero is harmless and needs no branch
        atomicOr(&buf[wi + 1], w1);
        // whole words of this run are stored; a first word shared with the
        // run below (head) and a last word not wholly this run's (tail) go to
        // side[p][gw] for k_pb_fixup
        const uint64_t end = o + nv + flags;
        const uint32_t nwords = (uint32_t)(((o & 63) + nv + flags + 63) >> 6);
        uint64_t *st = streams + (uint64_t)p * stride + (o >> 6);
        uint64_t *sd = side + 2 * ((uint64_t)p * nwv + gw);
        for (uint32_t w = lane; w < nwords; w += 64) {
            const uint64_t v = buf[w];
            buf[w] = 0;
            const bool head = w == 0 && (o & 63);
            const bool tail = !head && w == nwords - 1 && (end & 63);
            // one store to the selected word (no branches)
            *(head ? sd : tail ? sd + 1 : st + w) = v;
        }
    });
}

// Pass 4: the words at run boundaries. Only the last non-empty run can be
// shorter than a word (the others hold 2048 elements), so a word is shared
// by at most two runs: run g's head word is its head ORed with run g - 1's
// tail; the last run's tail word is its own.
__global__ __launch_bounds__(256) void k_pb_fixup(const uint32_t *__restrict__ bits, const uint64_t *__restrict__ off,
                                                  const uint64_t *__restrict__ side, uint32_t nwv, uint32_t glast,
                                                  uint64_t *__restrict__ streams, uint64_t stride) {
    const uint32_t g = blockIdx.x * 256 + threadIdx.x;
    const int p = blockIdx.y;
    if (g > glast) return;
    const uint64_t i = (uint64_t)p * nwv + g;
    const uint64_t o = off[i], end = o + bits[i];
    uint64_t *st = streams + (uint64_t)p * stride;
    if (o & 63) st[o >> 6] = side[2 * i] | side[2 * (i - 1) + 1];
    const bool one_word = (o & 63) && ((o & 63) + bits[i] <= 64);  // the head word is also the last
    if (g == glast && (end & 63) && !one_word) st[(end - 1) >> 6] = side[2 * i + 1];
}

uint64_t pb_stream_words(uint32_t n) { return (2ull * n + 63) / 64; }

template <class T> size_t pb_workspace_bytes(uint32_t n, int nb) {
    const uint64_t nwv = pb_nwaves<T>(n), nblk = div_up(nwv, kPbScanBlk);
    return nwv * nb * (8 + 16 + 4) + nblk * nb * 8 + 256;
}
template size_t pb_workspace_bytes<float>(uint32_t, int);
template size_t pb_workspace_bytes<double>(uint32_t, int);

template <class T>
int launch_pb_encode(const T *x, uint32_t n, int32_t exp, const KeyOf<T> *key, int nb, int compat,
                     uint64_t *streams, uint64_t stride, uint32_t *sizes, void *ws, size_t ws_bytes, hipStream_t s) {
    if (n == 0 || nb < 1 || nb > (int)(8 * sizeof(T))) { set_error("perbit encode: bad n or num_bitplanes"); return kErrArg; }
    if (stride < pb_stream_words(n)) { set_error("perbit encode: stream stride below ceil(2 n / 64) words"); return kErrArg; }
    if (ws_bytes < pb_workspace_bytes<T>(n, nb)) { set_error("perbit encode: workspace too small"); return kErrArg; }
    const uint32_t nwg = pb_nwg<T>(n), nwv = pb_nwaves<T>(n);
    const uint32_t nblk = div_up(nwv, kPbScanBlk);
    if (nblk > kPbScanT) { set_error("perbit encode: too many elements"); return kErrArg; }
    uint64_t *off = static_cast<uint64_t *>(ws);
    uint64_t *side = off + (size_t)nwv * nb;
    uint64_t *sums = side + 2 * (size_t)nwv * nb;
    uint32_t *bits = reinterpret_cast<uint32_t *>(sums + (size_t)nblk * nb);
    hipLaunchKernelGGL(k_pb_count<T>, dim3(nwg), dim3(kPbTPB), 0, s, x, n, exp, key, nb, compat, bits, nwv);
    PRODM_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_pb_scan_sum, dim3(nblk, nb), dim3(kPbScanT), 0, s, bits, nwv, sums);
    PRODM_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_pb_scan_off, dim3(nblk, nb), dim3(kPbScanT), 0, s, bits, nwv, sums, off, sizes);
    PRODM_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_pb_write<T>, dim3(nwg), dim3(kPbTPB), 0, s, x, n, exp, key, nb, compat, off, nwv,
                       streams, stride, side);
    PRODM_CHECK_LAUNCH();
    const uint32_t glast = (n - 1) / (64u * kPbB);  // the last wave with elements
    hipLaunchKernelGGL(k_pb_fixup, dim3(div_up(glast + 1, 256), nb), dim3(256), 0, s, bits, off, side, nwv, glast,
                       streams, stride);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int launch_pb_encode<float>(const float *, uint32_t, int32_t, const uint32_t *, int, int, uint64_t *,
                                     uint64_t, uint32_t *, void *, size_t, hipStream_t);
template int launch_pb_encode<double>(const double *, uint32_t, int32_t, const unsigned long long *, int, int,
                                      uint64_t *, uint64_t, uint32_t *, void *, size_t, hipStream_t);

}  // namespace prodm
