// perbit_host.cpp -- progressive decode of PerBit streams
// (PerBitBPEncoder.hpp:290-382), host code.
//
// An element takes one bit of a stream, or two where its first 1 bit is
// (the bit, then its sign), and the streams carry no index of where each
// element's bits begin: the position of element e in stream i depends on
// the bits of every element before it. Each stream is therefore parsed from
// its start, on the host, 64 elements at a time: of the next 64 bits, those
// of elements whose sign is known are data; the first other 1 bit is followed
// by a sign, which is taken out, and the search goes on behind it. Only the
// elements that get their sign cost a step of their own. Plane i of a group
// needs the signs known after plane i - 1 of the same group and nothing else,
// so long levels are parsed by a pipeline of threads, some planes each.
// (1.87 M float elements x 32 planes on an 8-CPU host: 45 ms in one thread, 14 ms
// in eight; a 129^3 hierarchical refactor + retrieve beside an MI355X 143 to 149
// ms bit by bit, now 7.4 to 9.2 by the host.)
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "prodm_mdr.h"

namespace prodm {
void set_error(const std::string &msg);
}

// Per-level sign state, keyed by `level` (the reference keys it by call
// order, PerBitBPEncoder.hpp:304-309; the explicit key also serves levels
// first decoded with zero planes).
struct prodm_perbit_state {
    struct Level {
        uint32_t n = 0;
        std::vector<uint64_t> sign, flag;  // per element: sign recorded, sign known
    };
    std::map<int, Level> levels;
};

namespace {

int fail(const char *fmt, ...) {
    char buf[256];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    prodm::set_error(buf);
    return -1;
}

// LSB-first bit reader over 64-bit words (PerBitBPEncoder.hpp:41-67),
// bounded by the stream's size when one is given
struct BitReader {
    const uint64_t *w = nullptr;
    uint64_t nwords = ~0ull, next = 0, buf = 0;
    int left = 0;
    bool overrun = false;
    uint64_t load() {
        if (next >= nwords) {
            overrun = true;
            return 0;
        }
        uint64_t v;
        std::memcpy(&v, reinterpret_cast<const char *>(w) + 8 * next, 8);  // any alignment
        next++;
        return v;
    }
    uint64_t get() {
        if (!left) {
            buf = load();
            left = 64;
        }
        const uint64_t b = buf & 1u;
        buf >>= 1;
        left--;
        return b;
    }
    // m bits (1..64), reading no word past the last of them
    uint64_t get(int m) {
        uint64_t v = buf;
        if (left < m) {
            const uint64_t x = load();
            if (left) v |= x << left;
            else v = x;
            const int used = m - left;
            buf = used == 64 ? 0 : x >> used;
            left = 64 - used;
        } else {
            buf = m == 64 ? 0 : buf >> m;
            left -= m;
        }
        return m == 64 ? v : v & ((1ull << m) - 1);
    }
};

// one plane of a group of m elements: its bits; F, S: signs known / signs
uint64_t group_plane(BitReader &r, int m, uint64_t &F, uint64_t &S) {
    uint64_t d = r.get(m);
    uint64_t c = d & ~F;
    if (!c) return d;
    const uint64_t open = ~F;
    do {
        const int j = __builtin_ctzll(c);
        const uint64_t upto = (2ull << j) - 1, next = r.get();
        uint64_t sg = next;  // the last element's sign is past the m bits
        if (j != m - 1) {
            sg = (d >> (j + 1)) & 1u;
            d = (d & upto) | ((d >> 1) & ~upto) | (next << (m - 1));
        }
        S |= sg << j;
        F |= 1ull << j;
        c = d & open & ~upto;
    } while (c);
    return d;
}

// two 32 x 32 bit transposes, of the words' low and of their high halves
void transpose2x32(uint64_t *A) {
    static const uint64_t masks[5] = {0x0000FFFF0000FFFFull, 0x00FF00FF00FF00FFull, 0x0F0F0F0F0F0F0F0Full,
                                      0x3333333333333333ull, 0x5555555555555555ull};
    for (int s = 0, j = 16; j; s++, j >>= 1)
        for (int k0 = 0; k0 < 32; k0 += 2 * j)
            for (int k = k0; k < k0 + j; k++) {
                const uint64_t t = ((A[k] >> j) ^ A[k + j]) & masks[s];
                A[k] ^= t << j;
                A[k + j] ^= t;
            }
}

// values of a group from its k plane words D[i] (plane i is bit k - 1 - i),
// times 2^e, with their signs
template <class T> void group_values(const uint64_t *D, int k, int m, uint64_t S, int e, T *out) {
    using F = typename std::conditional<std::is_same<T, double>::value, uint64_t, uint32_t>::type;
    constexpr int kParts = sizeof(F) / 4;
    uint64_t A[kParts][32];
    for (int p = 0; p < kParts; p++) {
        for (int b = 0; b < 32; b++) {
            const int i = k - 1 - (32 * p + b);
            A[p][b] = i >= 0 ? D[i] : 0;
        }
        transpose2x32(A[p]);
    }
    // one multiplication by a power of two rounds as ldexp does; powers
    // outside the normal range take ldexp itself
    const bool normal = sizeof(T) == 4 ? e >= -126 && e <= 127 : e >= -1022 && e <= 1023;
    const T scale = normal ? std::ldexp((T)1, e) : (T)0;
    for (int j = 0; j < m; j++) {
        const int h = 32 * (j >> 5), r = j & 31;
        F fp = (F)(uint32_t)(A[0][r] >> h);
        if (kParts == 2) fp |= (F)((uint64_t)(uint32_t)(A[kParts - 1][r] >> h) << 32);
        const T y = normal ? (T)fp * scale : std::ldexp((T)fp, e);
        F bits;
        std::memcpy(&bits, &y, sizeof(T));
        bits |= (F)((S >> j) & 1u) << (8 * sizeof(F) - 1);  // y >= 0
        std::memcpy(&out[j], &bits, sizeof(T));
    }
}

constexpr uint32_t kChunk = 64;          // groups a stage passes on at a time
constexpr uint32_t kWindow = 1u << 14;   // groups decoded together (bounds the plane words held)
constexpr int kMaxStages = 8;

// Groups [g0, g1) of a level: the stages' threads parse their planes chunk by
// chunk behind each other, then all turn finished chunks into values.
template <class T>
void decode_groups(std::vector<BitReader> &rd, uint64_t *flag, uint64_t *sign, uint32_t n, uint32_t g0, uint32_t g1,
                   const std::vector<int> &cut, int e, std::vector<uint64_t> &words, T *out) {
    const int k = (int)rd.size(), stages = (int)cut.size() - 1;  // stage st: planes [cut[st], cut[st + 1])
    const uint32_t chunks = (g1 - g0 + kChunk - 1) / kChunk;
    std::atomic<uint32_t> done[kMaxStages], next{0};
    for (auto &d : done) d.store(0, std::memory_order_relaxed);
    auto len = [&](uint32_t g) { return (int)std::min<uint64_t>(64, (uint64_t)n - 64ull * g); };
    auto wait = [](const std::atomic<uint32_t> &d, uint32_t c) {
        while (d.load(std::memory_order_acquire) <= c) std::this_thread::yield();
    };
    auto parse = [&](int st) {
        const int i0 = cut[st], i1 = cut[st + 1];
        for (uint32_t c = 0; c < chunks; c++) {
            if (st) wait(done[st - 1], c);
            const uint32_t ge = std::min(g1, g0 + (c + 1) * kChunk);
            for (uint32_t g = g0 + c * kChunk; g < ge; g++) {
                uint64_t F = flag[g], S = sign[g];
                for (int i = i0; i < i1; i++) words[(size_t)(g - g0) * k + i] = group_plane(rd[i], len(g), F, S);
                flag[g] = F;
                sign[g] = S;
            }
            done[st].store(c + 1, std::memory_order_release);
        }
    };
    auto finish = [&] {
        for (uint32_t c; (c = next.fetch_add(1, std::memory_order_relaxed)) < chunks;) {
            wait(done[stages - 1], c);
            const uint32_t ge = std::min(g1, g0 + (c + 1) * kChunk);
            for (uint32_t g = g0 + c * kChunk; g < ge; g++)
                group_values<T>(words.data() + (size_t)(g - g0) * k, k, len(g), sign[g], e, out + 64ull * g);
        }
    };
    std::vector<std::thread> pool;
    int own = 0;  // stages [own, stages) run on this thread
    pool.reserve(stages);
    for (; own < stages - 1; own++) {
        const int st = own;
        try {
            pool.emplace_back([&, st] { parse(st); finish(); });
        } catch (const std::exception &) {  // no thread to be had: the rest runs here
            break;
        }
    }
    for (int st = own; st < stages; st++) parse(st);
    finish();
    for (auto &t : pool) t.join();
}

template <class T>
int perbit_decode(prodm_perbit_state *s, int level, const uint64_t *const *streams, const uint32_t *sizes, uint32_t n,
                  int32_t exp, int start, int k, T *out) {
    if (!s || (n && !out)) return fail("perbit decode: null state or output");
    if (k == 0) {  // (:296-299)
        for (uint32_t e = 0; e < n; e++) out[e] = 0;
        return 0;
    }
    if (k < 0 || start < 0 || start + k > (int)(8 * sizeof(T))) return fail("perbit decode: bad plane range");
    if (!streams) return fail("perbit decode: null stream array");
    for (int i = 0; i < k; i++)
        if (!streams[i] && n) return fail("perbit decode: null stream %d", i);
    prodm_perbit_state::Level &L = s->levels[level];
    const uint32_t groups = (uint32_t)(((uint64_t)n + 63) / 64);
    if (L.n == 0) {
        L.sign.assign(groups, 0);
        L.flag.assign(groups, 0);
        L.n = n;
    } else if (L.n != n) {
        return fail("perbit decode: level %d has %u elements, not %u", level, L.n, n);
    }
    std::vector<BitReader> rd(k);
    for (int i = 0; i < k; i++) {
        rd[i].w = streams[i];
        if (sizes) rd[i].nwords = sizes[i] / 8;
    }
    // threads where they have more to parse than they cost to start (some 20 us
    // each, again for every window): 128 groups of 32 planes, at the line, take
    // 189 us in one thread and 184 in two; 256 groups 416 and 237 (in four),
    // 512 groups 1038 and 461 (in eight)
    const uint64_t work = (uint64_t)groups * k;
    const int cpus = (int)std::max(1u, std::thread::hardware_concurrency());
    const int stages = work < 4096 ? 1 : std::min({kMaxStages, cpus, k, (int)std::min<uint64_t>(work / 2048, 64)});
    // planes per stage by what they cost: some 4 ns a group, 11 ns a sign (a
    // stream's bits beyond one per element)
    std::vector<double> upto(k + 1, 0.0);
    for (int i = 0; i < k; i++) {
        const double signs = sizes ? std::max(0.0, 8.0 * sizes[i] - n) : 0.0;
        upto[i + 1] = upto[i] + 4.0 * groups + 11.0 * signs;
    }
    std::vector<int> cut(1, 0);
    for (int st = 1; st < stages; st++) {
        const double at = upto[k] * st / stages;
        const int i = (int)(std::lower_bound(upto.begin(), upto.end(), at) - upto.begin());
        const int near = i > 0 && at - upto[i - 1] < upto[i] - at ? i - 1 : i;
        if (near > cut.back() && near < k) cut.push_back(near);
    }
    cut.push_back(k);
    std::vector<uint64_t> words((size_t)k * std::min(groups, kWindow));
    for (uint32_t g = 0; g < groups; g += kWindow)
        decode_groups<T>(rd, L.flag.data(), L.sign.data(), n, g, std::min(groups, g + kWindow), cut, exp - (start + k), words, out);
    for (int i = 0; i < k; i++)
        if (rd[i].overrun) return fail("perbit decode: stream %d is shorter than its content", i);
    return 0;
}

// no exception leaves a C entry point (the decode allocates)
template <class Fn> int guarded(Fn &&fn) {
    try {
        return fn();
    } catch (const std::exception &e) {
        return fail("perbit decode: %s", e.what());
    }
}

}  // namespace

extern "C" {

int prodm_perbit_state_create(prodm_perbit_state **out) {
    if (!out) return fail("perbit state: null output");
    *out = new prodm_perbit_state();
    return 0;
}
int prodm_perbit_state_destroy(prodm_perbit_state *s) {
    delete s;
    return 0;
}
int prodm_perbit_decode_f32(prodm_perbit_state *s, int level, const uint64_t *const *h_streams,
                            const uint32_t *h_sizes, uint32_t n, int32_t exp, int start, int k, float *h_out) {
    return guarded([&] { return perbit_decode<float>(s, level, h_streams, h_sizes, n, exp, start, k, h_out); });
}
int prodm_perbit_decode_f64(prodm_perbit_state *s, int level, const uint64_t *const *h_streams,
                            const uint32_t *h_sizes, uint32_t n, int32_t exp, int start, int k, double *h_out) {
    return guarded([&] { return perbit_decode<double>(s, level, h_streams, h_sizes, n, exp, start, k, h_out); });
}

}  // extern "C"
