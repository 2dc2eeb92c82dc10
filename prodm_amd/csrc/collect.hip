// collect.hip -- SquaredErrorCollector (SquaredErrorCollector.hpp:23-65) and the
// encoders' level errors on gfx950.
//
// The reference adds, per element, the squared truncation error of every
// bitplane prefix (computed in T) into a double table, sequentially. A
// parallel FP64 sum cannot reproduce that order, so each table entry is
// defined as the EXACTLY ROUNDED sum of the same terms: order independent,
// and identical between these kernels and the CPU restatement.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "internal.hpp"

namespace prodm {

template <class T> __device__ inline typename Traits<T>::Bits to_bits(T v) {
    typename Traits<T>::Bits b;
    __builtin_memcpy(&b, &v, sizeof(b));
    return b;
}
template <class T> __device__ inline T from_bits(typename Traits<T>::Bits b) {
    T v;
    __builtin_memcpy(&v, &b, sizeof(v));
    return v;
}

// ---- exact host summation and rounding ---------------------------------------------
namespace {
struct Big {
    std::vector<uint64_t> w;  // little endian
    explicit Big(size_t limbs) : w(limbs, 0) {}
    void add_shifted(uint64_t v, int shift) {  // v << shift, shift >= 0
        if (!v) return;
        const size_t li = (size_t)shift / 64;
        const int off = shift % 64;
        uint64_t parts[2] = {v << off, off ? (v >> (64 - off)) : 0};
        uint64_t carry = 0;
        for (size_t j = li; j < w.size(); j++) {
            const uint64_t add = (j - li < 2) ? parts[j - li] : 0;
            if (j - li >= 2 && !carry) break;
            const uint64_t s1 = w[j] + add;
            const uint64_t c1 = s1 < add;
            const uint64_t s2 = s1 + carry;
            const uint64_t c2 = s2 < carry;
            w[j] = s2;
            carry = c1 | c2;
        }
    }
    void sub_shifted(uint64_t v, int shift) {  // the total stays >= 0
        if (!v) return;
        const size_t li = (size_t)shift / 64;
        const int off = shift % 64;
        const uint64_t parts[2] = {v << off, off ? (v >> (64 - off)) : 0};
        uint64_t borrow = 0;
        for (size_t j = li; j < w.size(); j++) {
            if (j - li >= 2 && !borrow) break;
            const uint64_t sub = (j - li < 2) ? parts[j - li] : 0;
            const uint64_t s1 = w[j] - sub, s2 = s1 - borrow;
            borrow = (w[j] < sub) | (s1 < borrow);
            w[j] = s2;
        }
    }
    void add128(__int128 v, int shift, bool negatives) {  // the value, or nothing if its sign is not asked for
        if ((v < 0) != negatives) return;
        const unsigned __int128 m = negatives ? (unsigned __int128)(-v) : (unsigned __int128)v;
        const uint64_t lo = (uint64_t)m, hi = (uint64_t)(m >> 64);
        if (negatives) { sub_shifted(lo, shift); sub_shifted(hi, shift + 64); }
        else { add_shifted(lo, shift); add_shifted(hi, shift + 64); }
    }
    int bit(long i) const { return i < 0 ? 0 : (int)((w[(size_t)i / 64] >> (i % 64)) & 1u); }
    // value * 2^scale rounded to nearest even
    double to_double(int scale) const {
        long top = -1;
        for (long i = (long)w.size() - 1; i >= 0; i--)
            if (w[i]) { top = i * 64 + 63 - __builtin_clzll(w[i]); break; }
        if (top < 0) return 0.0;
        if (top <= 52) return std::ldexp((double)w[0], scale);
        const long lsb = top - 52;
        uint64_t mant = 0;
        for (long b = top; b >= lsb; b--) mant = (mant << 1) | (uint64_t)bit(b);
        const int rb = bit(lsb - 1);
        int sticky = 0;
        for (long b = lsb - 2; b >= 0 && !sticky; b--) sticky = bit(b);
        if (rb && (sticky || (mant & 1u))) mant++;
        return std::ldexp((double)mant, (int)(scale + lsb));
    }
};
}  // namespace


// ---- exact sums in FP64 (float data) --------------------------------------------
// Error-free extraction onto fixed grids, the idea of Demmel and Nguyen's binned
// summation, with every grid's sum kept as an integer.
// A term below 2^T and a multiple of 2^Q is added to up to three accumulators
// of decreasing grid 2^u. An accumulator starts at 1.5 2^(u + 52), so that it
// stays in one binade, whose numbers are the multiples of 2^u: adding a term
// rounds it to the grid, the rounding error is exact and goes to the next one,
// and the last grid is 2^Q itself. The sum in units of 2^u is the difference of
// the bit patterns, an integer. 32 terms per accumulator, then the integers go to
// LDS (a slot per lane pair), to one partial sum per workgroup, and to 96-bit
// totals that the host adds and rounds once. A term costs 3 operations per
// accumulator but the last, which costs 1; the tables' lower entries need
// three, most two (carrying integers over the words of the same window took
// some 50 operations, a wave reduction of them per 16 terms, and a host sum
// over every workgroup's partials: 257^3 finest level, both tables 2.94 ms, now
// 0.43 ms).
namespace {

constexpr int kExThreads = 256, kExEPT = 32, kExChunk = kExThreads * kExEPT;
constexpr int kExMaxChunks = 8;  // 2^16 terms below 2^(u + 45) per workgroup: sums stay in 63 bits
constexpr int kExSlots = 32;     // LDS words per accumulator
constexpr int kExBins = 35;      // nb + 1 entries and two for the tiny elements

struct Grid3 {
    int n;     // accumulators used
    int u[3];  // exponents of their grids; the last is [2]
};
// grids of terms of at most 2^T, multiples of 2^Q
__host__ __device__ inline Grid3 grid3(int T, int Q) {
    Grid3 g;
    // 32 terms of at most 2^T in the first, remainders of at most 2^(T - 46),
    // 2^(T - 92) in the others, each sum below half of the bias's binade
    g.n = T - Q <= 45 ? 1 : T - Q <= 91 ? 2 : 3;
    g.u[0] = T - 45;
    g.u[1] = T - 91;
    g.u[2] = Q;
    return g;
}
// the tiny elements' grids: no Q, what the third does not hold is refused
__host__ __device__ inline Grid3 grid3_open(int T) {
    Grid3 g{3, {T - 45, T - 91, T - 137}};
    return g;
}
__device__ __forceinline__ double grid_bias(int u) { return ldexp(1.5, u + 52); }

struct Acc3 {
    double a[3], b[3];
    __device__ __forceinline__ void start(const Grid3 &g) {
#pragma unroll
        for (int i = 0; i < 3; i++) a[i] = b[i] = grid_bias(g.u[i]);
    }
    template <int N> __device__ __forceinline__ void add(double t) {
        if constexpr (N >= 2) { const double n = a[0] + t; t -= n - a[0]; a[0] = n; }
        if constexpr (N >= 3) { const double n = a[1] + t; t -= n - a[1]; a[1] = n; }
        a[2] += t;
    }
    // adds t if the three grids hold it
    __device__ __forceinline__ bool add_open(double t) {
        const double n0 = a[0] + t, t1 = t - (n0 - a[0]);
        const double n1 = a[1] + t1, t2 = t1 - (n1 - a[1]);
        const double n2 = a[2] + t2;
        if (t2 - (n2 - a[2]) != 0.0) return false;
        a[0] = n0; a[1] = n1; a[2] = n2;
        return true;
    }
    __device__ __forceinline__ void flush(unsigned long long *slot) const {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            // unconditional: behind a test, the second and third chains of the
            // sums would sink to their uses, with all terms held until then
            const uint64_t d = to_bits(a[i]) - to_bits(b[i]);
            atomicAdd(slot + i * kExSlots + (threadIdx.x % kExSlots), (unsigned long long)d);
        }
    }
};

// Terms outside the grids go to 128-bit sums of their exponents: buckets
// [first, first + n) of double exponents for each entry.
struct Under {
    unsigned long long *sum;
    uint32_t *flag;  // set once any is used
    int first, n;
    __device__ __forceinline__ void add(int bin, int be, unsigned long long v) const {
        unsigned long long *bk = sum + ((size_t)bin * n + (be - first)) * 2;
        const unsigned long long old = atomicAdd(bk, v);
        if (old + v < old) atomicAdd(bk + 1, 1ull);
        *flag = 1u;
    }
};
// exponent and mantissa of a term. One that is infinite or NaN has no sum and
// is left out (M = 0), or (over) counts as its float's bits read as a number:
// infinity is 2^128.
__device__ __forceinline__ unsigned long long term_bits(double t, bool over, int &be) {
    const uint64_t tb = to_bits(t);
    be = (int)((tb >> 52) & 0x7ff);
    unsigned long long M = (tb & ((1ull << 52) - 1)) | (be ? (1ull << 52) : 0);
    if (be == 0x7ff) {
        be = 1023 + 128;
        if (!over) M = 0;
    }
    be = be ? be : 1;
    return M;
}
__device__ __forceinline__ void add_under(double t, int bin, const Under &U, bool over) {
    int be;
    const unsigned long long M = term_bits(t, over, be);
    if (M) U.add(bin, be, M);
}
// The terms of the wave's elements named by `past` (element 0 of the lane's in
// bit 31; term(x, k) for entries 0 .. nb) through windows of 64 exponents in
// LDS, kPastEntries entries at a time, whose used words go to the buckets in one
// addition each: every element's own additions there meet on a few addresses
// (3 M floats, a third of them past the bound: 6.5 ms, now 0.29). At most 2^11
// additions below 2^53 per word.
constexpr int kPastEntries = 4;
template <class Term>
__device__ __forceinline__ void add_past(uint32_t past, const float *x, int nb, bool over, const Under &U,
                                         unsigned long long (*win)[64], Term &&term) {
    if (!__any(past != 0)) return;
    const int lane = (int)lane_id();
    auto each = [&](auto &&fn) __attribute__((always_inline)) {
        for (uint32_t left = past; left;) {
            const int i = __clz(left);
            left ^= 0x80000000u >> i;
            fn(x[(uint64_t)i * kExThreads + threadIdx.x]);
        }
    };
    // entry 0 has the largest terms, those of the others are at most some times that
    int base = 0;
    each([&](float v) __attribute__((always_inline)) {
        int be;
        if (term_bits(term(v, 0), over, be)) base = max(base, be);
    });
    for (int o = 32; o >= 1; o >>= 1) base = max(base, __shfl_xor(base, o, 64));
    base -= 59;
    for (int k0 = 0; k0 <= nb; k0 += kPastEntries) {
        for (int j = 0; j < kPastEntries; j++) win[j][lane] = 0;
        wave_lds_sync();
        each([&](float v) __attribute__((always_inline)) {
            for (int j = 0; j < kPastEntries && k0 + j <= nb; j++) {
                int be;
                const unsigned long long M = term_bits(term(v, k0 + j), over, be);
                if (!M) continue;
                if (be >= base && be < base + 64) atomicAdd(&win[j][be - base], M);
                else U.add(k0 + j, be, M);
            }
        });
        wave_lds_sync();
        for (int j = 0; j < kPastEntries; j++)
            if (win[j][lane]) U.add(k0 + j, base + lane, win[j][lane]);
        wave_lds_sync();
    }
}

// the workgroup's sums of every accumulator (kExBins * 3 of kExSlots words)
__device__ __forceinline__ void store_partials(const unsigned long long *acc, int bins, uint64_t *__restrict__ partial) {
    for (int s = threadIdx.x; s < bins * 3; s += kExThreads) {
        uint64_t v = 0;
#pragma unroll
        for (int i = 0; i < kExSlots; i++) v += acc[s * kExSlots + ((i + threadIdx.x) % kExSlots)];
        partial[(uint64_t)s * gridDim.x + blockIdx.x] = v;
    }
}
// total of accumulator blockIdx.x over the workgroups: out[2 s] low and
// out[2 s + 1] high parts in units of 1 and 2^32
__global__ __launch_bounds__(kExThreads) void k_exact_totals(const uint64_t *__restrict__ partial, uint32_t nwg,
                                                             uint64_t *__restrict__ out) {
    __shared__ uint64_t red[2][kExThreads / 64];
    uint64_t lo = 0, hi = 0;
    for (uint32_t i = threadIdx.x; i < nwg; i += kExThreads) {
        const int64_t v = (int64_t)partial[(uint64_t)blockIdx.x * nwg + i];
        lo += (uint32_t)v;
        hi += (uint64_t)(v >> 32);
    }
    for (int o = 32; o >= 1; o >>= 1) { lo += __shfl_xor(lo, o, 64); hi += __shfl_xor(hi, o, 64); }
    if (lane_id() == 0) { red[0][threadIdx.x / 64] = lo; red[1][threadIdx.x / 64] = hi; }
    __syncthreads();
    if (threadIdx.x < 2) {
        uint64_t v = 0;
        for (int w = 0; w < kExThreads / 64; w++) v += red[threadIdx.x][w];
        out[2 * blockIdx.x + threadIdx.x] = v;
    }
}

// workspace: [totals: bins * 3 * 2 words][flag][partials][exponent buckets]
struct ExLayout {
    uint32_t nwg;
    int bins, first, buckets;
    size_t flag, partial, under, total;
};
ExLayout ex_layout(uint64_t n, int nb, int first, int buckets) {
    ExLayout L;
    L.first = first;
    L.buckets = buckets;
    const uint64_t chunks = std::max<uint64_t>(1, (n + kExChunk - 1) / kExChunk);
    // one chunk per workgroup up to 4 workgroups per CU, then up to kExMaxChunks
    const uint64_t per = std::min<uint64_t>(kExMaxChunks, std::max<uint64_t>(1, chunks / 1024));
    L.nwg = (uint32_t)((chunks + per - 1) / per);
    L.bins = nb + 3;
    L.flag = (size_t)L.bins * 3 * 16;
    L.partial = L.flag + 16;
    L.under = L.partial + (size_t)L.bins * 3 * 8 * L.nwg;
    L.total = L.under + (size_t)L.bins * buckets * 16;
    return L;
}

// Sums the totals of the kernel's accumulators: out[k] = main k + the tiny
// sums that tiny(k) names (bit 0: entry nb + 1, bit 1: entry nb + 2), times
// 2^scale. grid(i): the grids of entry i.
template <class GridOf, class TinyOf>
int exact_finish(const ExLayout &L, int nb, GridOf grid, TinyOf tiny, int scale, double *out, void *ws, hipStream_t s) {
    char *base = static_cast<char *>(ws);
    hipLaunchKernelGGL(k_exact_totals, dim3(L.bins * 3), dim3(kExThreads), 0, s,
                       reinterpret_cast<const uint64_t *>(base + L.partial), L.nwg, reinterpret_cast<uint64_t *>(base));
    PRODM_CHECK_LAUNCH();
    std::vector<uint64_t> tot((L.flag + 16) / 8), under;
    PRODM_HIP(hipMemcpyAsync(tot.data(), base, tot.size() * 8, hipMemcpyDeviceToHost, s));
    PRODM_HIP(hipStreamSynchronize(s));
    if (tot[L.flag / 8]) {
        under.resize((L.total - L.under) / 8);
        PRODM_HIP(hipMemcpyAsync(under.data(), base + L.under, under.size() * 8, hipMemcpyDeviceToHost, s));
        PRODM_HIP(hipStreamSynchronize(s));
    }
    constexpr int kEmin = -1074;
    for (int k = 0; k <= nb; k++) {
        Big b((2048 + 128 + 64 * 4 + 64) / 64 + 2);
        const int from[3] = {k, tiny(k) & 1 ? nb + 1 : -1, tiny(k) & 2 ? nb + 2 : -1};
        for (int neg = 0; neg < 2; neg++)
            for (int i : from) {
                if (i < 0) continue;
                const Grid3 g = grid(i);
                for (int a = 0; a < 3; a++) {
                    const uint64_t *t = tot.data() + ((size_t)i * 3 + a) * 2;
                    b.add128(((__int128)(int64_t)t[1] << 32) + (__int128)t[0], g.u[a] - kEmin, neg);
                }
                if (!neg && !under.empty())
                    for (int e = 0; e < L.buckets; e++) {
                        const uint64_t *u = under.data() + ((size_t)i * L.buckets + e) * 2;
                        b.add_shifted(u[0], L.first + e - 1);
                        b.add_shifted(u[1], L.first + e - 1 + 64);
                    }
            }
        out[k] = std::ldexp(b.to_double(kEmin), scale);
    }
    return kOk;
}

// The thread's elements of chunk c (0 past n): i-th at i * kExThreads + its
// index. A buffer descriptor ends with the data, so no address is per lane
// and all loads are in flight together.
__device__ __forceinline__ void load_chunk(const float *x, uint64_t n, uint64_t c, float (&v)[kExEPT]) {
    const uint64_t e0 = c * kExChunk;
    const uint32_t bytes = (uint32_t)min((uint64_t)kExChunk, n - e0) * 4u;
    const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(x + e0), 0, bytes, 0x00020000);
#pragma unroll
    for (int i = 0; i < kExEPT; i++)
        v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)threadIdx.x * 4, i * kExThreads * 4, 0));
}

// adds term(i), i < kExEPT, in N accumulators and flushes them
template <int N, class Fn>
__device__ __forceinline__ void sum_terms(const Grid3 &g, unsigned long long *slot, Fn &&term) {
    Acc3 A;
    A.start(g);
#pragma unroll
    for (int i = 0; i < kExEPT; i++) {
        A.add<N>(term(i));
        // the scheduler would form all terms before the serial sums (256
        // VGPRs, one wave per SIMD)
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    A.flush(slot);
}
template <class Fn> __device__ __forceinline__ void sum_bin(const Grid3 &g, unsigned long long *slot, Fn &&term) {
    if (g.n == 1) sum_terms<1>(g, slot, term);
    else if (g.n == 2) sum_terms<2>(g, slot, term);
    else sum_terms<3>(g, slot, term);
}

}  // namespace

// term of bin k for element x, restating the reference loop (:326-356):
// bins s_idx, s_idx-1, ... get the squared residual after clearing mantissa
// bits 0..b (b = b0, b0+1, ..., prec-1); the remaining bins get x^2.
template <class T>
__device__ inline T sq_term(T x, int de, int le, int nb, int k) {
    using Bits = typename Traits<T>::Bits;
    constexpr int P = Traits<T>::kPrec;
    const int exp_diff = le - de + P - nb;
    const int s_idx = exp_diff > 0 ? nb : nb + exp_diff;
    const int b0 = exp_diff > 0 ? exp_diff : 0;
    if (s_idx <= 0 || k > s_idx) return (T)0;
    if (b0 < P && k >= s_idx - (P - 1 - b0)) {
        const int b = b0 + (s_idx - k);
        const Bits mask = ~(((Bits)2 << b) - 1);  // clears bits 0..b
        const T xb = from_bits<T>(to_bits<T>(x) & mask);
        const T d = x - xb;
        return d * d;
    }
    return x * x;
}

// SquaredErrorCollector, float. An element of exponent de has the term
// (x - x cleared of mantissa bits 0 .. b)^2 in entry k, b = le + 23 - de - k
// (x^2 from b = 23 on, 0 below b = 0). With le - nb < de <= le its terms are at
// most 2^(2 (le - k)) and multiples of 2^(2 (le - nb - 23)). Smaller elements
// have the term x^2 in every entry and are summed once; ones past the bound go
// term by term to the buckets.
// Squares are float. One past the largest float counts as 2^128, as in the CPU
// restatement (infinity's bits read as a number), so that no term is above 2^128
// and 2^128 is on the grid of any step up to it. Only entries with le - k > 64
// reach it and take the minimum. Elements past the bound, infinite or NaN have
// such terms too: theirs count where a 128-bit window from 2^q reaches 2^128
// (le > nb + 23), and are left out elsewhere.
constexpr double kSqOver = 0x1p128;
__host__ __device__ inline Grid3 sq_grid(int k, int le, int nb) {
    if (k > nb) return grid3_open(2 * (le - nb));
    const int q = 2 * (le - nb - 23), t = 2 * (le - k);
    return grid3(t < 128 ? t : 128, q < -149 ? -149 : q > 128 ? 128 : q);
}
__global__ __launch_bounds__(kExThreads) void k_collect_squared_f32(const float *__restrict__ x, uint64_t n, int nb,
                                                                    int le, uint64_t *__restrict__ partial, Under U) {
    __shared__ unsigned long long acc[kExBins * 3 * kExSlots];
    __shared__ unsigned long long win[kExThreads / 64][kPastEntries][64];
    for (int i = threadIdx.x; i < (nb + 3) * 3 * kExSlots; i += kExThreads) acc[i] = 0;
    __syncthreads();
    for (uint64_t c = blockIdx.x; c * kExChunk < n; c += gridDim.x) {
        float v[kExEPT];
        int cut[kExEPT];  // mantissa bits cleared in entry 0
        load_chunk(x, n, c, v);
        uint32_t rest = 0;  // elements not summed by the loops over entries, element 0 in bit 31
#pragma unroll
        for (int i = 0; i < kExEPT; i++) {
            const int de = dev_frexp_exp(v[i]);
            const float a = fabsf(v[i]);
            cut[i] = le + 24 - de;
            const bool main = de > le - nb && de <= le && a >= 1.17549435e-38f && a < __builtin_inff();
            rest = 2 * rest + (!main && !(a < 1.17549435e-38f));  // a subnormal element's squares are 0
            v[i] = main ? v[i] : 0.0f;
            // formed here: left to the loop below, the selects and what they
            // read would both stay live (256 VGPRs instead of 111)
            asm volatile("" : "+v"(v[i]), "+v"(cut[i]));
        }
        uint32_t past = 0;
        if (__any(rest != 0)) {
            Acc3 tiny;
            tiny.start(sq_grid(nb + 1, le, nb));
            while (rest) {
                const int i = __clz(rest);  // element 0 is bit 31
                rest ^= 0x80000000u >> i;
                const float t = x[c * kExChunk + (uint64_t)i * kExThreads + threadIdx.x];
                const int de = dev_frexp_exp(t);
                if (de <= le - nb && fabsf(t) < __builtin_inff()) {
                    const float tt = t * t;
                    const double td = fmin((double)tt, kSqOver);
                    if (!tiny.add_open(td)) add_under(td, nb + 1, U, false);
                } else {
                    past |= 0x80000000u >> i;
                }
            }
            tiny.flush(acc + (nb + 1) * 3 * kExSlots);
        }
        for (int k = 0; k <= nb; k++) {
            auto term = [&](int i) __attribute__((always_inline)) -> double {
                const int b = cut[i] - k;
                const uint32_t keep = 0xffffffffu << (b > 23 ? 31 : max(b, 0));
                const float d = v[i] - from_bits<float>(to_bits(v[i]) & keep);
                const float t = d * d;
                return (double)t;
            };
            const Grid3 g = sq_grid(k, le, nb);
            unsigned long long *const slot = acc + k * 3 * kExSlots;
            if (le - k > 64)
                sum_bin(g, slot, [&](int i) __attribute__((always_inline)) -> double { return fmin(term(i), kSqOver); });
            else
                sum_bin(g, slot, term);
        }
        // last, when the elements' registers are free
        add_past(past, x + c * kExChunk, nb, le > nb + 23, U, win[threadIdx.x / 64],
                 [&](float t, int k) __attribute__((always_inline)) -> double {
                     return (double)sq_term<float>(t, dev_frexp_exp(t), le, nb, k);
                 });
    }
    __syncthreads();
    store_partials(acc, nb + 3, partial);
}

// float squares: exponents of 2^-149 to 2^128 as doubles
ExLayout sq_layout(uint64_t n, int nb) { return ex_layout(n, nb, 1023 - 149, 149 + 128 + 1); }
size_t sq_workspace_bytes_f32(uint64_t n, int nb) { return sq_layout(n, nb).total; }
static int squared_errors_f32(const float *x, uint64_t n, int nb, float maxerr, double *out, void *ws, hipStream_t s) {
    int le = 0;
    std::frexp(maxerr, &le);
    const ExLayout L = sq_layout(n, nb);
    char *base = static_cast<char *>(ws);
    uint32_t *flag = reinterpret_cast<uint32_t *>(base + L.flag);
    if (int rc = launch_fill_u32(flag, 4, 0u, s)) return rc;
    if (int rc = launch_fill_u64(reinterpret_cast<uint64_t *>(base + L.under), (L.total - L.under) / 8, 0ull, s)) return rc;
    hipLaunchKernelGGL(k_collect_squared_f32, dim3(L.nwg), dim3(kExThreads), 0, s, x, n, nb, le,
                       reinterpret_cast<uint64_t *>(base + L.partial),
                       Under{reinterpret_cast<unsigned long long *>(base + L.under), flag, L.first, L.buckets});
    PRODM_CHECK_LAUNCH();
    return exact_finish(L, nb, [&](int i) { return sq_grid(i, le, nb); }, [](int) { return 1; }, 0, out, ws, s);
}

// ---- SquaredErrorCollector, double -------------------------------------------------
// Terms are doubles over a window of up to 232 bits, accumulated as integers
// in units of Q = max(q^2, min_sub), q = 2^(le - nb - 52), in per-thread
// multi-limb registers, reduced across the wave and workgroup with carries,
// and summed exactly on the host. The rare squares of elements far below
// the level maximum that are not multiples of Q go to a per-(entry, exponent)
// histogram of mantissa sums.
constexpr int kSqLimbs = 4;  // 2^256 > 2^(2 * 64 + 104) * 2^12 terms per workgroup
constexpr int kSqExpBuckets = 2048, kSqEmin = -1074;
constexpr int kSqThreads = 256;
constexpr int kSqEPT = 16;  // elements per thread
__global__ __launch_bounds__(kSqThreads) void k_collect_squared_f64(const double *__restrict__ x, uint64_t n, int nb, int le,
                                                                int log2q, uint64_t *__restrict__ partial,
                                                                unsigned long long *__restrict__ under) {
    using T = double;
    using Bits = typename Traits<T>::Bits;
    constexpr int LM = kSqLimbs, MB = 52;
    __shared__ uint64_t wacc[kSqThreads / 64][65][LM];
    const uint32_t lane = lane_id(), wv = threadIdx.x / 64;
    const uint64_t base = (uint64_t)blockIdx.x * kSqThreads * kSqEPT;
    T v[kSqEPT];
    int de[kSqEPT];
#pragma unroll
    for (int i = 0; i < kSqEPT; i++) {
        const uint64_t e = base + (uint64_t)i * kSqThreads + threadIdx.x;
        v[i] = e < n ? x[e] : (T)0;
        de[i] = dev_frexp_exp(v[i]);
    }
    for (int k = 0; k <= nb; k++) {
        uint64_t a[LM];
#pragma unroll
        for (int j = 0; j < LM; j++) a[j] = 0;
#pragma unroll
        for (int i = 0; i < kSqEPT; i++) {
            if (v[i] == (T)0) continue;
            const T t = sq_term<T>(v[i], de[i], le, nb, k);
            if (t == (T)0) continue;
            const Bits tb = to_bits<T>(t);
            const int be = (int)((tb >> MB) & ((1u << 11) - 1));
            const uint64_t M = (uint64_t)(tb & (((Bits)1 << MB) - 1)) | (be ? ((uint64_t)1 << MB) : 0);
            const int E = (be ? be : 1) - 1 + kSqEmin;  // t = M * 2^E
            const int s = E - log2q;
            if (s < 0) {
                atomicAdd(&under[(size_t)k * kSqExpBuckets + (be ? be : 1)], (unsigned long long)M);
                continue;
            }
            const int li = s >> 6, off = s & 63;
            const uint64_t plo = M << off;
            const uint64_t phi = off ? (M >> (64 - off)) : 0;
            uint64_t carry = 0;
#pragma unroll
            for (int j = 0; j < LM; j++) {
                const uint64_t add = (j == li ? plo : 0) + (j == li + 1 ? phi : 0);
                const uint64_t s1 = a[j] + add;
                const uint64_t c1 = s1 < add;
                const uint64_t s2 = s1 + carry;
                const uint64_t c2 = s2 < carry;
                a[j] = s2;
                carry = c1 | c2;
            }
        }
        // wave reduction with carries
        for (int o = 32; o >= 1; o >>= 1) {
            uint64_t b[LM];
#pragma unroll
            for (int j = 0; j < LM; j++) b[j] = __shfl_xor(a[j], o, 64);
            uint64_t carry = 0;
#pragma unroll
            for (int j = 0; j < LM; j++) {
                const uint64_t s1 = a[j] + b[j];
                const uint64_t c1 = s1 < b[j];
                const uint64_t s2 = s1 + carry;
                const uint64_t c2 = s2 < carry;
                a[j] = s2;
                carry = c1 | c2;
            }
        }
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < LM; j++) wacc[wv][k][j] = a[j];
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k <= nb; k += kSqThreads) {
        uint64_t a[LM];
#pragma unroll
        for (int j = 0; j < LM; j++) a[j] = 0;
        for (int w = 0; w < kSqThreads / 64; w++) {
            uint64_t carry = 0;
#pragma unroll
            for (int j = 0; j < LM; j++) {
                const uint64_t bj = wacc[w][k][j];
                const uint64_t s1 = a[j] + bj;
                const uint64_t c1 = s1 < bj;
                const uint64_t s2 = s1 + carry;
                const uint64_t c2 = s2 < carry;
                a[j] = s2;
                carry = c1 | c2;
            }
        }
#pragma unroll
        for (int j = 0; j < LM; j++) partial[((uint64_t)blockIdx.x * (nb + 1) + k) * LM + j] = a[j];
    }
}


// workspace: [partials][underflow histogram]
static uint32_t sq_nwg(uint64_t n) { return (uint32_t)std::max<uint64_t>(1, (n + kSqThreads * kSqEPT - 1) / (kSqThreads * kSqEPT)); }
static size_t sq_partial_bytes(uint64_t n, int nb) { return (size_t)sq_nwg(n) * (nb + 1) * kSqLimbs * 8; }
static size_t sq_under_bytes(int nb) { return (size_t)(nb + 1) * kSqExpBuckets * 8; }
static int squared_errors_f64(const double *x, uint64_t n, int nb, double maxerr, double *out, void *ws,
                              hipStream_t s) {
    int le = 0;
    std::frexp(maxerr, &le);
    const int log2q = (int)std::max<long>(2L * ((long)le - nb - 52), kSqEmin);
    const uint32_t nwg = sq_nwg(n);
    const size_t pb = sq_partial_bytes(n, nb), ub = sq_under_bytes(nb);
    uint64_t *partial = static_cast<uint64_t *>(ws);
    unsigned long long *under = reinterpret_cast<unsigned long long *>(static_cast<char *>(ws) + pb);
    if (int rc = launch_fill_u64(reinterpret_cast<uint64_t *>(under), ub / 8, 0ull, s)) return rc;
    if (n == 0) {
        if (int rc = launch_fill_u64(partial, pb / 8, 0ull, s)) return rc;
    } else {
        hipLaunchKernelGGL(k_collect_squared_f64, dim3(nwg), dim3(kSqThreads), 0, s, x, n, nb, le, log2q, partial, under);
        PRODM_CHECK_LAUNCH();
    }
    std::vector<uint64_t> host((pb + ub) / 8);
    PRODM_HIP(hipMemcpyAsync(host.data(), ws, pb + ub, hipMemcpyDeviceToHost, s));
    PRODM_HIP(hipStreamSynchronize(s));
    const uint64_t *hp = host.data(), *hu = host.data() + pb / 8;
    // common scale: 2^emin; window terms sit at 2^log2q = 2^emin * 2^(log2q - emin)
    const int wshift = log2q - kSqEmin;
    const size_t limbs = (size_t)(wshift + 64 * kSqLimbs + 64 + 64 + 2 * 1100) / 64 + 2;
    for (int k = 0; k <= nb; k++) {
        Big b(limbs);
        for (uint64_t g = 0; g < nwg; g++)
            for (int j = 0; j < kSqLimbs; j++) b.add_shifted(hp[(g * (nb + 1) + k) * kSqLimbs + j], wshift + 64 * j);
        for (int e = 1; e < kSqExpBuckets; e++) b.add_shifted(hu[(size_t)k * kSqExpBuckets + e], e - 1);
        out[k] = b.to_double(kSqEmin);
    }
    return kOk;
}

template <class T> size_t sq_workspace_bytes(uint64_t n, int nb) {
    return sizeof(T) == 4 ? sq_workspace_bytes_f32(n, nb) : 64 + sq_partial_bytes(n, nb) + sq_under_bytes(nb);
}
template size_t sq_workspace_bytes<float>(uint64_t, int);
template size_t sq_workspace_bytes<double>(uint64_t, int);
template <> int squared_errors<float>(const float *x, uint64_t n, int nb, float maxerr, double *out, void *ws, hipStream_t s) {
    return squared_errors_f32(x, n, nb, maxerr, out, ws, s);
}
template <> int squared_errors<double>(const double *x, uint64_t n, int nb, double maxerr, double *out, void *ws, hipStream_t s) {
    return squared_errors_f64(x, n, nb, maxerr, out, ws, s);
}

// ---- encoder-fused level errors ------------------------------------------------------
// NegaBinaryBPEncoder::encode(..., level_errors) (NegaBinaryBPEncoder.hpp:65-125,
// collect_level_errors :231-239) and GroupedBPEncoder::encode(..., level_errors)
// (GroupedBPEncoder.hpp:76-145, :324-335), for fp32 data (the reference's
// collectors take float / uint32). Per element, in the shifted units
// s = x 2^(nb - e) (e + 2 for NegaBinary), bin nb - k holds the squared
// value of the digits below the top nb - k planes plus the fraction m, bin
// nb the fraction alone and bin 0 s^2; bins 0 and nb square in float as the
// reference does. Each entry is the exactly rounded sum over elements, then
// scaled by 2^(2 (e - nb)).
//
// Exactness: an element with 1 <= |s| < 2^min(nb, kFeTop) has terms of at most
// 2^(2 (nb - k) + 2) in entry k that are multiples of 2^-46 (the fraction's step
// is at least 2^-23). One with |s| < 1 has no digit: its term is s^2 in every
// entry, as a double, or squared in float where the reference squares in
// float; both are summed once. Larger ones (an exponent below the data's) go
// term by term to the buckets.
namespace {
__device__ __forceinline__ uint32_t fe_mask(int k) { return k >= 31 ? 0x7fffffffu : ((1u << k) - 1u); }

template <int ENC>
__device__ __forceinline__ double fe_term(float s, float m, uint32_t bits, int nb, int bin) {
    if (ENC == 0) {  // NegaBinary: bits = negabinary digits of (int32) s
        if (bin == nb) { const float mm = m * m; return (double)mm; }
        if (bin == 0) { const float ss = s * s; return (double)ss; }
        const int32_t v = (int32_t)(((bits & fe_mask(nb - bin)) ^ 0xaaaaaaaau) - 0xaaaaaaaau);
        const double d = (double)v + (double)m;
        return d * d;
    }
    // GroupedBP: s = |shifted|, bits = (uint32) s, m = s - bits (float)
    const double md = (double)m;
    if (bin == nb) return md * md;
    if (bin == 0) { const float ss = s * s; return (double)ss; }
    const double d = (double)(bits & fe_mask(nb - bin)) + md;
    return d * d;
}


// an element's shifted value (its magnitude for GroupedBP), fraction and digits
template <int ENC>
__device__ __forceinline__ void fe_split(float x, int shift, float &s, float &m, uint32_t &bits) {
    const float sh = ldexpf(x, shift);
    const float a = fabsf(sh);
    if (ENC == 0) {
        // (int32) shifted as in the reference (in range: |x| < 2^e)
        const int32_t q = (sh == sh && a < 2147483648.0f) ? (int32_t)sh : (int32_t)0x80000000;
        bits = ((uint32_t)q + 0xaaaaaaaau) ^ 0xaaaaaaaau;
        s = sh;
        m = sh - (float)q;
    } else {
        const uint32_t fp = (a == a && a < 4294967296.0f) ? (uint32_t)a : 0u;
        bits = fp;
        s = a;
        m = a - (float)fp;
    }
}

constexpr int kFeQ = -46;
// digits end at 2^31 (int32) and 2^32 (uint32)
template <int ENC> constexpr int kFeTop = ENC == 0 ? 31 : 32;
ExLayout fe_layout(uint64_t n, int nb) { return ex_layout(n, nb, 1, 2046); }
__host__ __device__ inline Grid3 fe_grid(int k, int nb) {
    return k > nb ? grid3_open(0) : grid3(2 * (nb - k) + 2, kFeQ);
}

template <int ENC>
__global__ __launch_bounds__(kExThreads) void k_fused_errors(const float *__restrict__ x, uint64_t n, int shift,
                                                             int nb, uint64_t *__restrict__ partial, Under U) {
    __shared__ unsigned long long acc[kExBins * 3 * kExSlots];
    __shared__ unsigned long long win[kExThreads / 64][kPastEntries][64];
    for (int i = threadIdx.x; i < (nb + 3) * 3 * kExSlots; i += kExThreads) acc[i] = 0;
    __syncthreads();
    const float top = ldexpf(1.0f, min(nb, kFeTop<ENC>));
    for (uint64_t c = blockIdx.x; c * kExChunk < n; c += gridDim.x) {
        float m[kExEPT];
        uint32_t bits[kExEPT];
        load_chunk(x, n, c, m);
        uint32_t rest = 0;  // elements not summed by the loops over entries, element 0 in bit 31
#pragma unroll
        for (int i = 0; i < kExEPT; i++) {
            float s;
            fe_split<ENC>(m[i], shift, s, m[i], bits[i]);
            const float a = fabsf(s);
            const bool main = a >= 1.0f && a < top;
            rest = 2 * rest + (!main && s != 0.0f);
            m[i] = main ? m[i] : 0.0f;
            bits[i] = main ? bits[i] : 0u;
            asm volatile("" : "+v"(m[i]), "+v"(bits[i]));  // as above
        }
        uint32_t past = 0;
        if (__any(rest != 0)) {
            Acc3 tinyd, tinyf;
            tinyd.start(fe_grid(nb + 1, nb));
            tinyf.start(fe_grid(nb + 2, nb));
            while (rest) {
                const int i = __clz(rest);  // element 0 is bit 31
                rest ^= 0x80000000u >> i;
                float s, mm;
                uint32_t bb;
                fe_split<ENC>(x[c * kExChunk + (uint64_t)i * kExThreads + threadIdx.x], shift, s, mm, bb);
                if (fabsf(s) < 1.0f) {
                    const double d = (double)s * (double)s;
                    const float ff = s * s;
                    if (!tinyd.add_open(d)) add_under(d, nb + 1, U, false);
                    if (!tinyf.add_open((double)ff)) add_under((double)ff, nb + 2, U, false);
                } else {
                    past |= 0x80000000u >> i;
                }
            }
            tinyd.flush(acc + (nb + 1) * 3 * kExSlots);
            tinyf.flush(acc + (nb + 2) * 3 * kExSlots);
        }
        // entries 0 and nb: s = digits + fraction again, exactly
        sum_bin(fe_grid(0, nb), acc, [&](int i) __attribute__((always_inline)) -> double {
            const float q = ENC == 0 ? (float)(int32_t)((bits[i] ^ 0xaaaaaaaau) - 0xaaaaaaaau) : (float)bits[i];
            return fe_term<ENC>(q + m[i], m[i], bits[i], nb, 0);
        });
        sum_bin(fe_grid(nb, nb), acc + nb * 3 * kExSlots,
                [&](int i) __attribute__((always_inline)) -> double { return fe_term<ENC>(0.0f, m[i], bits[i], nb, nb); });
        for (int k = 1; k < nb; k++) {
            const uint32_t mask = fe_mask(nb - k);
            sum_bin(fe_grid(k, nb), acc + k * 3 * kExSlots, [&](int i) __attribute__((always_inline)) -> double {
                const uint32_t low = bits[i] & mask;
                const double v = ENC == 0 ? (double)(int32_t)((low ^ 0xaaaaaaaau) - 0xaaaaaaaau) : (double)low;
                const double d = v + (double)m[i];
                return d * d;
            });
        }
        add_past(past, x + c * kExChunk, nb, false, U, win[threadIdx.x / 64],
                 [&](float t, int k) __attribute__((always_inline)) -> double {
                     float s, mm;
                     uint32_t bb;
                     fe_split<ENC>(t, shift, s, mm, bb);
                     return fe_term<ENC>(s, mm, bb, nb, k);
                 });
    }
    __syncthreads();
    store_partials(acc, nb + 3, partial);
}
}  // namespace

size_t fused_errors_workspace_bytes(uint64_t n, int nb) { return fe_layout(n, nb).total; }

int fused_level_errors(int enc, const float *x, uint64_t n, int32_t exp, int nb, double *out, void *ws,
                       size_t ws_bytes, hipStream_t s) {
    if (nb < 1 || nb > 32 || !out || (enc != 0 && enc != 1)) { set_error("level errors: bad arguments"); return kErrArg; }
    if (n > 0 && !x) { set_error("level errors: null input"); return kErrArg; }
    const ExLayout L = fe_layout(n, nb);
    if (ws_bytes < L.total || !ws) { set_error("level errors: workspace too small"); return kErrArg; }
    const int e = enc == 0 ? exp + 2 : exp;  // NegaBinaryBPEncoder.hpp:68
    char *base = static_cast<char *>(ws);
    uint64_t *partial = reinterpret_cast<uint64_t *>(base + L.partial);
    uint32_t *flag = reinterpret_cast<uint32_t *>(base + L.flag);
    const Under under{reinterpret_cast<unsigned long long *>(base + L.under), flag, L.first, L.buckets};
    if (int rc = launch_fill_u32(flag, 4, 0u, s)) return rc;
    if (int rc = launch_fill_u64(reinterpret_cast<uint64_t *>(base + L.under), (L.total - L.under) / 8, 0ull, s)) return rc;
    if (enc == 0)
        hipLaunchKernelGGL(k_fused_errors<0>, dim3(L.nwg), dim3(kExThreads), 0, s, x, n, nb - e, nb, partial, under);
    else
        hipLaunchKernelGGL(k_fused_errors<1>, dim3(L.nwg), dim3(kExThreads), 0, s, x, n, nb - e, nb, partial, under);
    PRODM_CHECK_LAUNCH();
    // entries whose terms of tiny elements are squared in float take the second sum
    return exact_finish(L, nb, [&](int i) { return fe_grid(i, nb); },
                        [&](int k) { return k == 0 || (enc == 0 && k == nb) ? 2 : 1; }, 2 * (e - nb), out, ws, s);
}

}  // namespace prodm
