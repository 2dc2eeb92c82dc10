// adjoint.hip -- transpose of the MGARD orthogonal recompose (FP64).
//
// One recompose level maps (u_c', W) to u = P (u_c' - S R W) + E W, with P
// the multilinear prolongation (injection at coarse nodes), R = P^T M the
// load operator (M: fine mass matrix, 3/h-scaled [1/2, 2, 1/2] per dim, ends
// 1), S = M_c^-1 the coarse solve and E the embedding of the coefficients.
// Its transpose, given g = dJ/du on the fine grid:
//   h   = P^T g                     (coarse; the next coarser level's g)
//   t   = S h                       (coarse line solves, S symmetric)
//   r   = M P t                     (fine)
//   dJ/dW = g - r                   at the coefficient nodes
// applied from the finest level to the coarsest, where dJ/du_0 = h.
// The result is laid out like a decompose output (coarse nodes first along
// each dim inside every level box). ProDM has no adjoint; this serves
// QoI-guided retrieval (sensitivities of a QoI to each level's coefficients).
#include "internal.hpp"

#include <type_traits>

namespace prodm {

namespace {

// dJ/dW = g - M P t at the coefficient nodes of the level box, written at the
// decompose layout position (rpos per dim) of the output array.
//
// M P is a stencil of the coarse values along each dim: at fine node 2 j
// [1/4, 5/2, 1/4] on t_{j-1..j+1} (centre 5/4 at the two ends), at 2 j + 1
// [3/2, 3/2] on t_j, t_{j+1}: the transpose of the load stencil. A workgroup
// takes 8 x 8 x 64 fine nodes: their coarse neighbourhood (6 x 6 x 34) goes to
// LDS, is expanded along dim 2 there (36 rows of 64), then along dims 1 and 0
// in the registers of a thread's two columns of 8 nodes. Bound by reading g
// once and writing the result once; as separate prolongation, mass (per dim)
// and store passes over FP64 fine grids it took 430 + 126 + 160 us of a 257^3
// f32 backward, now 36 + 28 us.
constexpr int kA0 = 8, kA1 = 8, kA2 = 64;
constexpr int kT0 = kA0 / 2 + 2, kT1 = kA1 / 2 + 2, kT2 = kA2 / 2 + 2;
struct AdjBox {
    uint32_t n[3], c[3];
};
template <class G, class T>
__global__ __launch_bounds__(256) void k_adj_coef(const double *__restrict__ t, uint32_t tp, AdjBox box,
                                                  const G *__restrict__ g, uint64_t gs0, uint64_t gs1,
                                                  T *__restrict__ out, uint64_t os0, uint64_t os1) {
    __shared__ double C[kT0 * kT1 * kT2], E[kT0 * kT1 * kA2];
    const uint32_t n0 = box.n[0], n1 = box.n[1], n2 = box.n[2], c0 = box.c[0], c1 = box.c[1], c2 = box.c[2];
    const uint32_t t2n = (n2 + kA2 - 1) / kA2, t1n = (n1 + kA1 - 1) / kA1, t0n = (n0 + kA0 - 1) / kA0;
    const uint32_t bt = xcd_remap(blockIdx.x, t0n * t1n * t2n);
    const uint32_t s2 = (bt % t2n) * kA2, s1 = ((bt / t2n) % t1n) * kA1, s0 = (bt / (t2n * t1n)) * kA0;
    const uint32_t lane = threadIdx.x % kA2, wv = threadIdx.x / kA2;
    const uint32_t i2 = s2 + lane;
    constexpr int kCols = kA1 / 4;  // columns of kA0 nodes per thread
    // every load of the thread in flight before the first LDS write
    G gv[kCols][kA0];
#pragma unroll
    for (int q = 0; q < kCols; q++) {
        const uint32_t i1 = s1 + wv + 4 * q;
#pragma unroll
        for (int k = 0; k < kA0; k++) {
            const bool in = s0 + k < n0 && i1 < n1 && i2 < n2;
            gv[q][k] = g[in ? (uint64_t)(s0 + k) * gs0 + (uint64_t)i1 * gs1 + i2 : 0];
        }
    }
    constexpr int kStage = (kT0 * kT1 * kT2 + 255) / 256;
    double sv[kStage];
#pragma unroll
    for (int k = 0; k < kStage; k++) {
        const uint32_t idx = threadIdx.x + 256u * k;
        // coarse node s / 2 - 1 + a of each dim; outside the grid 0
        const uint32_t j2 = s2 / 2 + idx % kT2 - 1, j1 = s1 / 2 + (idx / kT2) % kT1 - 1, j0 = s0 / 2 + idx / (kT2 * kT1) - 1;
        const bool in = idx < kT0 * kT1 * kT2 && j0 < c0 && j1 < c1 && j2 < c2;  // -1 wraps past c
        const double v = t[in ? ((uint64_t)j0 * c1 + j1) * tp + j2 : 0];
        sv[k] = in ? v : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kStage; k++)
        if (threadIdx.x + 256u * k < kT0 * kT1 * kT2) C[threadIdx.x + 256u * k] = sv[k];
    __syncthreads();
    // weight of the centre at fine node 2 j; an extent-1 dim keeps its value
    auto centre = [](uint32_t j, uint32_t c) __attribute__((always_inline)) -> double {
        return c == 1 ? 1.0 : (j == 0 || j == c - 1) ? 1.25 : 2.5;
    };
    const bool odd2 = lane & 1;
    const double w2 = centre(i2 >> 1, c2);
#pragma unroll
    for (int r = 0; r < kT0 * kT1 / 4; r++) {
        const uint32_t row = wv + 4 * r;
        const double *p = C + row * kT2 + (lane >> 1);
        const double a = p[0], b = p[1], d = p[2];
        E[row * kA2 + lane] = odd2 ? 1.5 * (b + d) : fma(w2, b, 0.25 * (a + d));
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kCols; q++) {
        const uint32_t l1 = wv + 4 * q, i1 = s1 + l1;
        const bool odd1 = l1 & 1;
        const double w1 = centre(i1 >> 1, c1);
        double F[kT0];
#pragma unroll
        for (int a0 = 0; a0 < kT0; a0++) {
            const double *p = E + (a0 * kT1 + (l1 >> 1)) * kA2 + lane;
            const double a = p[0], b = p[kA2], d = p[2 * kA2];
            F[a0] = odd1 ? 1.5 * (b + d) : fma(w1, b, 0.25 * (a + d));
        }
        const bool in12 = i1 < n1 && i2 < n2, coarse12 = !odd1 && !odd2;
        T *const o12 = out + (uint64_t)rpos(i1, c1) * os1 + rpos(i2, c2);
#pragma unroll
        for (int k = 0; k < kA0; k++) {
            const uint32_t i0 = s0 + k;
            const double r = (k & 1) ? 1.5 * (F[k / 2 + 1] + F[k / 2 + 2])
                                     : fma(centre(i0 >> 1, c0), F[k / 2 + 1], 0.25 * (F[k / 2] + F[k / 2 + 2]));
            if (in12 && i0 < n0 && !(coarse12 && !(k & 1)))
                o12[(uint64_t)rpos(i0, c0) * os0] = (T)((double)gv[q][k] - r);
        }
    }
}

// a box copy with conversion (the coarsest grid's adjoint into the output)
template <class G, class T>
__global__ __launch_bounds__(256) void k_adj_copy(const G *__restrict__ h, uint64_t hs0, uint64_t hs1, uint32_t n2,
                                                     T *__restrict__ out, uint64_t os0, uint64_t os1) {
    const uint32_t i2 = blockIdx.x * 256 + threadIdx.x;
    if (i2 >= n2) return;
    const uint32_t i1 = blockIdx.y, i0 = blockIdx.z;
    out[(uint64_t)i0 * os0 + (uint64_t)i1 * os1 + i2] = (T)h[(uint64_t)i0 * hs0 + (uint64_t)i1 * hs1 + i2];
}

dim3 grid_of(const uint32_t *n) { return dim3(div_up(n[2], 256), n[1], n[0]); }

// g: the dense copy of a box that meets its output or has planes of 2 GiB (the
// size query sees neither)
struct AdjLayout {
    size_t g, h0, h1, mgard, total;
};
AdjLayout adj_layout(const LevelGeom &g) {
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const uint64_t pL = g.points[g.L], p1 = g.L >= 1 ? g.points[g.L - 1] : 1;
    AdjLayout a{};
    a.g = 0;
    a.h0 = al(a.g + pL * 8);
    a.h1 = al(a.h0 + p1 * 8);
    a.mgard = al(a.h1 + p1 * 8);
    a.total = a.mgard + mgard_workspace_bytes(g, 8);
    return a;
}

}  // namespace

size_t adjoint_workspace_bytes(const LevelGeom &g) { return adj_layout(g).total; }

template <class T>
int mgard_recompose_adjoint(const T *g_in, const uint64_t *in_strides, const LevelGeom &g, T *out,
                            const uint64_t *out_strides, void *ws, size_t ws_bytes, hipStream_t s) {
    const AdjLayout A = adj_layout(g);
    if (ws_bytes < A.total) { set_error("adjoint: workspace too small"); return kErrArg; }
    char *base = static_cast<char *>(ws);
    double *hb[2] = {reinterpret_cast<double *>(base + A.h0), reinterpret_cast<double *>(base + A.h1)};
    void *mws = base + A.mgard;
    const size_t mws_bytes = A.total - A.mgard;
    // the sweep reads g in place, after the output's first stores: a box whose
    // memory meets the output's is first copied to a dense FP64 grid, and so
    // is one whose plane spans 2 GiB or more of its array (31-bit offsets)
    const uint32_t *n = g.ld[g.L];
    auto bytes = [&](const uint64_t *st) {
        return ((uint64_t)(n[0] - 1) * st[0] + (uint64_t)(n[1] - 1) * st[1] + n[2]) * sizeof(T);
    };
    const uintptr_t gi = reinterpret_cast<uintptr_t>(g_in), oi = reinterpret_cast<uintptr_t>(out);
    bool dense = gi < oi + bytes(out_strides) && oi < gi + bytes(in_strides);
    const double *cur = nullptr;
    uint64_t cs[2] = {(uint64_t)n[1] * n[2], n[2]};
    auto copy_in = [&]() -> int {
        double *gd = reinterpret_cast<double *>(base + A.g);
        hipLaunchKernelGGL((k_adj_copy<T, double>), grid_of(n), dim3(256), 0, s, g_in, in_strides[0], in_strides[1],
                           n[2], gd, cs[0], cs[1]);
        PRODM_CHECK_LAUNCH();
        cur = gd;
        return kOk;
    };
    if (g.L == 0 && !dense) {
        hipLaunchKernelGGL((k_adj_copy<T, T>), grid_of(n), dim3(256), 0, s, g_in, in_strides[0], in_strides[1], n[2], out,
                           out_strides[0], out_strides[1]);
        PRODM_CHECK_LAUNCH();
        return kOk;
    }
    // one level: h = P^T g and t = S h (the transposed load and the coarse
    // solves), then dJ/dW = g - M P t at the coefficient nodes
    auto level = [&](auto *cur, const uint64_t *cs, int l, double *h) -> int {
        const uint32_t *nl = g.ld[l], *c = g.ld[l - 1];
        if (int rc = mgard_adjoint_coarse(cur, cs, g, l, h, mws, mws_bytes, s)) return rc;
        uint32_t tp = 0;
        const double *t = mgard_adjoint_solution(g, l, mws, &tp);
        AdjBox box;
        for (int d = 0; d < 3; d++) { box.n[d] = nl[d]; box.c[d] = c[d]; }
        const uint32_t tiles = div_up(nl[2], kA2) * div_up(nl[1], kA1) * div_up(nl[0], kA0);
        using G = std::remove_const_t<std::remove_pointer_t<decltype(cur)>>;
        hipLaunchKernelGGL((k_adj_coef<G, T>), dim3(tiles), dim3(256), 0, s, t, tp, box, cur, cs[0], cs[1], out,
                           out_strides[0], out_strides[1]);
        PRODM_CHECK_LAUNCH();
        return kOk;
    };
    if (g.L > 0 && (uint64_t)n[1] * n[2] * sizeof(double) >= 0x7FFFFFFFull) {
        set_error("a fine plane of this level spans 2 GiB or more; the sweeps address planes with 31-bit offsets");
        return kErrUnsupported;
    }
    dense = dense || ((uint64_t)(n[1] - 1) * in_strides[1] + n[2]) * sizeof(T) >= 0x7FFFFFFFull;
    if (dense)
        if (int rc = copy_in()) return rc;
    for (int l = g.L, which = 0; l >= 1; l--, which ^= 1) {
        const int rc = cur ? level(cur, cs, l, hb[which]) : level(g_in, in_strides, l, hb[which]);
        if (rc) return rc;
        cur = hb[which];
        cs[0] = (uint64_t)g.ld[l - 1][1] * g.ld[l - 1][2];
        cs[1] = g.ld[l - 1][2];
    }
    hipLaunchKernelGGL((k_adj_copy<double, T>), grid_of(g.ld[0]), dim3(256), 0, s, cur, cs[0], cs[1], g.ld[0][2], out,
                       out_strides[0], out_strides[1]);
    PRODM_CHECK_LAUNCH();
    return kOk;
}
template int mgard_recompose_adjoint<float>(const float *, const uint64_t *, const LevelGeom &, float *,
                                            const uint64_t *, void *, size_t, hipStream_t);
template int mgard_recompose_adjoint<double>(const double *, const uint64_t *, const LevelGeom &, double *,
                                             const uint64_t *, void *, size_t, hipStream_t);

}  // namespace prodm
