// AdamW steps with bf16 moments for gfx950: the BF16-moment AdamW of TritonAdamW and the
// hybrid's AdamW groups (muon_sr/triton_adamw.py:9-72), and the bf16-moment branch of the
// 8-bit optimizer (muon_sr/triton_adamw_8bit.py:90-99), many tensors per launch.
//
// A launch's 8-element groups are cut into tiles that never cross a tensor; a work-group
// finds its tile's tensor once (a uniform search in the kernel-argument table).  14 bytes move
// per element, so HBM bounds the step once the arithmetic is short enough: three Philox
// streams, a correctly rounded square root and up to two correctly rounded quotients per
// element.  The wave takes one of two uniform branches:
//  * fast: every value in the ranges where sqrt_rn_x2p32, div_rn and div_upd (common.hpp) equal
//    the IEEE operations (the usual case);
//  * exact: the reference arithmetic with IEEE square root and division (non-finite gradients,
//    extreme moments, a denominator that could leave the range).
// Both give the same bits where both apply.  Measured on 128256 x 4096 (525 M elements, 7.35 GB):
// 1735 us with IEEE square root and divisions throughout, 1260 us now (5.84 TB/s; a copy kernel
// reaches 6.27).  The 73 tensors of an 8-layer d = 384 model: 536 us as 73 launches, 100 us as two
// (host time; the kernels take 52).
#include <cmath>
#include <algorithm>
#include <vector>

#include "common.hpp"
#include "vecio.hpp"
#include "../../include/muon_sr_amd.h"

namespace msr {

// A tile is 128 threads x 2 groups (2048 elements).  Measured on 128256 x 4096 with philox8 noise,
// and on half of it with the reference's: 1260 and 981 us; 256 x 1 1280 and 1044, 256 x 2 1276 and
// 1004, 512 x 1 1281 and 1175.  Tiles in dispatch order: runs of 64 per XCD measured equal.
#ifndef MSR_A16_THREADS
#define MSR_A16_THREADS 128
#endif
#ifndef MSR_A16_U
#define MSR_A16_U 2
#endif
constexpr int A16_THREADS = MSR_A16_THREADS, A16_U = MSR_A16_U, A16_TILE = A16_THREADS * A16_U;   // groups of 8
constexpr int A16_MAXT = 56;            // tensors per launch (4 KiB of kernel arguments)
constexpr uint32_t A16_VEC = 1, A16_FAST = 2;

enum : int { A16_ADAMW = 0, A16_ADAM8 = 1 };   // triton_adamw.py:9-72 | triton_adamw_8bit.py:90-99

struct A16Item {
    uint16_t *p;
    const uint16_t *g;
    uint16_t *m, *v;
    int64_t n;
    uint32_t seed, flags;
    float step;          // lr / bc                  | lr sqrt(BC2) / BC1
    float den, rden;     // sqrt(bias corr.) 2^32, RN of its reciprocal | sqrt(BC2) eps, unused
    uint32_t mmin;       // bits of the smallest nonzero |m'| of the fast branch, minus 1 (`ok` in a16_group)
};

struct A16Args {
    int count;
    float b1, b2, omb1, omb2, eps, decay;
    float strength;           // gradient centralization
    const uint16_t *inject;   // NOISE_INJECT (one tensor): uint16 [3][n]
    int32_t tstart[A16_MAXT + 1];
    int32_t cols[A16_MAXT];   // gradient centralization: elements of a row
    A16Item it[A16_MAXT];
};
static_assert(sizeof(A16Args) <= 4096, "kernel arguments");

// Wave-uniform constants, held in VGPRs (an SGPR operand takes the slow issue rate).
struct A16Consts {
    float b1, b2, omb1, omb2, eps, decay, step, den, rden;
    uint32_t mmin;
    bool fast;
};
__device__ __forceinline__ A16Consts a16_consts(const A16Args &a, const A16Item &it) {
    A16Consts c;
    c.b1 = vgpr(a.b1); c.b2 = vgpr(a.b2); c.omb1 = vgpr(a.omb1); c.omb2 = vgpr(a.omb2);
    c.eps = vgpr(a.eps); c.decay = vgpr(a.decay);
    c.step = vgpr(it.step); c.den = vgpr(it.den); c.rden = vgpr(it.rden);
    c.mmin = it.mmin;
    c.fast = (it.flags & A16_FAST) != 0;
    return c;
}

// One group of 8 elements: p, m, v updated in place in their packed words.  active: the lane's
// values count for the choice of the branch.
template <int MODE, int FORM>
__device__ __forceinline__ void a16_group(const A16Consts &c, const Noise (&ns)[3], int64_t o0, int valid,
                                          uint32_t (&wp)[4], const uint32_t (&wg)[4], uint32_t (&wm)[4],
                                          uint32_t (&wv)[4], bool active = true) {
    float p[8], g[8], m[8], v[8];
    unpack8(wp, p); unpack8(wg, g); unpack8(wm, m); unpack8(wv, v);
    // new moments; extremes of 2 bits(|m'|) and bits(v') (unsigned: NaN, infinities and negative v'
    // are the largest)
    uint32_t tmin = 0xffffffffu, tmax = 0u, vmax = 0u;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        m[j] = c.b1 * m[j] + c.omb1 * g[j];
        v[j] = c.b2 * v[j] + (c.omb2 * g[j]) * g[j];
        const uint32_t t = __float_as_uint(m[j]) << 1;
        tmin = min(tmin, t - 2u);               // +-0 gives 0xfffffffe
        tmax = max(tmax, t);
        vmax = max(vmax, __float_as_uint(v[j]));
    }
    // fast ranges: v' in [0, 2^24], m' = 0 or 2^-90 <= |step m'| with |m'| < 2^40 (step <= 2^20 is the
    // launcher's check), so that the root, both quotients and the denominator (in [eps, 2^31]) are in
    // the ranges of the correctly rounded sequences
    const bool ok = c.fast && vmax <= 0x4b800000u && tmax < (0x53800000u << 1) && (tmin >> 1) >= c.mmin;
    uint32_t r[8];
    uint32_t om[8], ov[8], op[8];
    const bool exact = __builtin_amdgcn_ballot_w64(active && !ok) != 0;
    if (!exact) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float s = sqrt_rn_x2p32(v[j]);
            if constexpr (FORM == A16_ADAMW) {
                const float d = div_rn(s, c.den, c.rden) + c.eps;
                p[j] = p[j] * c.decay - div_upd(c.step * m[j], d);
            } else {
                const float d = __builtin_fmaf(s, 0x1p-32f, c.den);
                p[j] = (p[j] - div_upd(c.step * m[j], d)) * c.decay;
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if constexpr (FORM == A16_ADAMW) {
                const float d = sqrtf(v[j]) / (c.den * 0x1p-32f) + c.eps;
                const float pj = p[j] * c.decay;
                p[j] = pj - (c.step * m[j]) / d;
            } else {
                const bool fin = fabsf(g[j]) < __builtin_huge_valf();
                m[j] = fin ? m[j] : 0.0f;
                v[j] = fin ? v[j] : 0.0f;
                const float upd = (p[j] - (c.step * m[j]) / (sqrtf(v[j]) + c.den)) * c.decay;
                p[j] = upd;
            }
        }
    }
    // FORM ADAMW: streams m: SEED, v: SEED + 1, p: SEED + 2; ADAM8: p: SEED, m: SEED + 1, v: SEED + 2
    constexpr int KP = FORM == A16_ADAMW ? 2 : 0, KM = FORM == A16_ADAMW ? 0 : 1, KV = FORM == A16_ADAMW ? 1 : 2;
    auto round = [&](const float (&x)[8], const Noise &n, uint32_t (&o)[8]) __attribute__((always_inline)) {
        noise8<MODE>(n, o0, valid, r);
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = __float_as_uint(x[j]) + r[j];
    };
    auto pack = [&](const uint32_t (&o)[8], uint32_t (&w)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = __builtin_amdgcn_perm(o[2 * j + 1], o[2 * j], 0x07060302u);
    };
    round(m, ns[KM], om);
    pack(om, wm);
    round(v, ns[KV], ov);
    pack(ov, wv);
    round(p, ns[KP], op);
    if (FORM == A16_ADAM8 && exact) {   // a non-finite gradient leaves the parameter as it is
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool fin = fabsf(g[j]) < __builtin_huge_valf();
            const uint32_t pin = (j & 1) ? (wp[j >> 1] & 0xffff0000u) : (wp[j >> 1] << 16);
            op[j] = fin ? op[j] : pin;
        }
    }
    pack(op, wp);
}

template <int MODE, int FORM, bool VEC>
__device__ __forceinline__ void a16_tile(const A16Args &a, const A16Item &it, int64_t g0) {
    Noise ns[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        ns[k].key = seed_key(it.seed, k);
        ns[k].inject = MODE == NOISE_INJECT ? a.inject + (int64_t)k * it.n : nullptr;
    }
    const A16Consts c = a16_consts(a, it);
    uint32_t wp[A16_U][4], wg[A16_U][4], wm[A16_U][4], wv[A16_U][4];
    int valid[A16_U];
#pragma unroll
    for (int u = 0; u < A16_U; ++u) {
        const int64_t o0 = (g0 + u * A16_THREADS + threadIdx.x) * 8;
        valid[u] = clamp_valid(it.n, o0);
        load_bf16x8<VEC>(it.p, o0, valid[u], wp[u]);
        load_bf16x8<VEC>(it.g, o0, valid[u], wg[u]);
        load_bf16x8<VEC>(it.m, o0, valid[u], wm[u]);
        load_bf16x8<VEC>(it.v, o0, valid[u], wv[u]);
    }
#pragma unroll
    for (int u = 0; u < A16_U; ++u) {
        const int64_t o0 = (g0 + u * A16_THREADS + threadIdx.x) * 8;
        a16_group<MODE, FORM>(c, ns, o0, valid[u], wp[u], wg[u], wm[u], wv[u]);
        store_bf16x8<VEC>(it.m, o0, valid[u], wm[u]);
        store_bf16x8<VEC>(it.v, o0, valid[u], wv[u]);
        store_bf16x8<VEC>(it.p, o0, valid[u], wp[u]);
    }
}

template <int MODE, int FORM>
__global__ __launch_bounds__(A16_THREADS) void adamw16_kernel(A16Args a) {
    const int32_t total = a.tstart[a.count];
    for (int64_t tile = blockIdx.x; tile < total; tile += gridDim.x) {
        int lo = 0, hi = a.count - 1;   // last t with tstart[t] <= tile (uniform)
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (a.tstart[mid] <= tile) lo = mid; else hi = mid - 1;
        }
        const A16Item &it = a.it[lo];
        const int64_t g0 = (tile - a.tstart[lo]) * A16_TILE;
        if (it.flags & A16_VEC) a16_tile<MODE, FORM, true>(a, it, g0);
        else a16_tile<MODE, FORM, false>(a, it, g0);
    }
}

// ---------------------------------------------------------------------------
// AdamW with gradient centralization (muon_sr/triton_adamw.py:179-187): the row's mean is taken
// from gradients that stay in registers, so the centred gradient is never written or read
// and every operand moves once (14 bytes per element; centralize.hip and the step above move
// 20).  A work-group of 256 threads takes a row of more than 1024 elements, or 256 / TPR
// narrower ones, TPR the power of two that holds a row's 8-element groups.  The mean is
// summed in centralize.hip's order (its 256 threads, then its tree; threads without elements add
// exact zeros), so results are the same bits.  Rows of up to 4096 elements (two groups per
// thread in flight): four groups took 172 VGPRs, and wider rows are centred first.  Measured on
// 128256 x 4096: 1253 us (5.87 TB/s, HBM-bound), where centring first and the step above take 1723.
// ---------------------------------------------------------------------------

constexpr int CEN_THREADS = 256;

__host__ __device__ inline int a16_tpr(int cols) {   // threads of a row
    int t = 8;
    while (t < 256 && t < cols / 8) t *= 2;
    return t;
}

// G (1 or 2): groups of a thread, all in flight at once.  row0: first row of the work-group.
template <int MODE, int G>
__device__ __forceinline__ void a16_rows(const A16Args &a, const A16Item &it, int cols, int64_t row0, float *red) {
    const int tpr = a16_tpr(cols), groups = cols >> 3;
    const int lr = threadIdx.x & (tpr - 1);
    const int64_t base0 = row0 * cols, base = base0 + (int64_t)(threadIdx.x / tpr) * cols;
    // Lanes without elements load and store nothing and have no say in the choice of the branch.  One
    // group: they compute on whatever their registers hold.  Two: their loads are out of the buffer
    // resource's range and give 0.  Against loads of the tensor's first group in their place, which its
    // owner stores meanwhile (us before, now): 128256 x 4096 1260, 1258 (with the form of one group
    // 1284); 400000 x 1000 1040, 1043; 400000 x 520 686, 695; 128256 x 2048 596, 620 on one box and
    // 588, 588 on another.
    bool in[G];
    int64_t at[G];
    uint32_t wp[G][4], wg[G][4], wm[G][4], wv[G][4];
    auto load = [&](const uint16_t *t, int u, uint32_t (&w)[4]) __attribute__((always_inline)) {
        if constexpr (G == 1) {
            asm volatile("" : "=v"(w[0]), "=v"(w[1]), "=v"(w[2]), "=v"(w[3]));
            if (in[u]) load_bf16x8<true>(t, at[u], 8, w);
        } else {
            const u32x4_t x = ldu_nt4(t + base0, in[u] ? (uint32_t)((at[u] - base0) * 2) : LDU_NONE);
            w[0] = x.x; w[1] = x.y; w[2] = x.z; w[3] = x.w;
        }
    };
#pragma unroll
    for (int u = 0; u < G; ++u) {
        in[u] = base < it.n && lr + u * tpr < groups;
        at[u] = base + (int64_t)(lr + u * tpr) * 8;
        load(it.g, u, wg[u]);
        load(it.p, u, wp[u]);
        load(it.m, u, wm[u]);
        load(it.v, u, wv[u]);
    }
    float s = 0.0f;
#pragma unroll
    for (int u = 0; u < G; ++u) {
        if (in[u]) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                s = s + bf16_lo(wg[u][k]);
                s = s + bf16_hi(wg[u][k]);
            }
        }
    }
    // the tree of centralize.hip's block_sum: halves of 128 and 64 through LDS, the rest in the wave
    const int lane = threadIdx.x & 63;
    if (tpr > 64) {
        red[threadIdx.x] = s;
        __syncthreads();
        const float *r = red + (threadIdx.x & ~(tpr - 1)) + lane;
        s = tpr == 256 ? (r[0] + r[128]) + (r[64] + r[192]) : r[0] + r[64];
    }
    const int width = tpr < 64 ? tpr : 64;
    for (int w = width >> 1; w > 0; w >>= 1) s = s + __shfl_down(s, w, 64);
    s = __shfl(s, lane & ~(width - 1), 64);
    const float mean = (0.0f + s) / (float)cols * a.strength;
    Noise ns[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        ns[k].key = seed_key(it.seed, k);
        ns[k].inject = nullptr;
    }
    const A16Consts c = a16_consts(a, it);
#pragma unroll
    for (int u = 0; u < G; ++u) {
#pragma unroll
        for (int k = 0; k < 4; ++k) wg[u][k] = rne_bf16x2(bf16_lo(wg[u][k]) - mean, bf16_hi(wg[u][k]) - mean);
        a16_group<MODE, A16_ADAMW>(c, ns, at[u], 8, wp[u], wg[u], wm[u], wv[u], G > 1 || in[u]);
        if (in[u]) {
            store_bf16x8<true>(it.m, at[u], 8, wm[u]);
            store_bf16x8<true>(it.v, at[u], 8, wv[u]);
            store_bf16x8<true>(it.p, at[u], 8, wp[u]);
        }
    }
}

// Two groups: 4 waves per SIMD (128256 x 4096, on one box: 1272 us; left to the compiler, 5 waves and 1311).
template <int MODE, int G>
__global__ __launch_bounds__(CEN_THREADS) __attribute__((amdgpu_waves_per_eu(G == 2 ? 4 : 1, G == 2 ? 4 : 8)))
void adamw16_central_kernel(A16Args a) {
    __shared__ float red[CEN_THREADS];
    const int32_t total = a.tstart[a.count];
    for (int64_t tile = blockIdx.x; tile < total; tile += gridDim.x) {
        int lo = 0, hi = a.count - 1;   // last t with tstart[t] <= tile (uniform)
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (a.tstart[mid] <= tile) lo = mid; else hi = mid - 1;
        }
        const int cols = a.cols[lo];
        a16_rows<MODE, G>(a, a.it[lo], cols, (tile - a.tstart[lo]) * (CEN_THREADS / a16_tpr(cols)), red);
        __syncthreads();   // the next tile writes red again
    }
}

// The fp32 constants of one tensor, in the reference's expression order, and whether its
// hyperparameters allow the fast branch.
static A16Item a16_item(int form, const msr_adamw_item &x, float lr, float eps) {
    A16Item it;
    it.p = x.p; it.g = x.g; it.m = x.m; it.v = x.v; it.n = x.n; it.seed = x.seed;
    float eps_c;
    if (form == A16_ADAMW) {
        it.step = lr / x.bc1;                              // muon_sr/triton_adamw.py:33
        it.den = x.bc2 * 0x1p32f;                          // exact
        it.rden = 1.0f / it.den;
        eps_c = eps;
    } else {
        const float sqrt_bc2 = sqrtf(x.bc2);
        it.step = (lr * sqrt_bc2) / x.bc1;                 // muon_sr/triton_adamw_8bit.py:95
        it.den = sqrt_bc2 * eps;
        it.rden = 0.0f;
        eps_c = it.den;
    }
    const float as = fabsf(it.step);
    // eps in [2^-60, 2^30] and, for AdamW, sqrt(bias correction) in [2^-16, 1]: the denominator is
    // then in [2^-60, 2^31]
    const bool fast = eps_c >= 0x1p-60f && eps_c <= 0x1p30f && as <= 0x1p20f &&
                      (form != A16_ADAMW || (x.bc2 >= 0x1p-16f && x.bc2 <= 1.0f));
    // |step m'| >= 2^-90 for |m'| >= 2^-90 / |step| (rounded up a little)
    const float lim = as > 0.0f ? (0x1p-90f / as) * 1.00001f : 0.0f;
    it.mmin = lim > 0.0f ? __builtin_bit_cast(uint32_t, lim) - 1u : 0u;
    it.flags = (fast && lim < 0x1p100f ? A16_FAST : 0u) |
               (aligned(x.p, 16) && aligned(x.g, 16) && aligned(x.m, 16) && aligned(x.v, 16) ? A16_VEC : 0u);
    return it;
}

// One launch over its items (at most A16_MAXT, none empty).  central: the items' gradients are
// centred by `strength` over rows of item.cols elements.
int adamw16_launch(int form, const msr_adamw_item *items, int32_t count, float lr, float b1, float b2, float eps, float wd,
                   int32_t mode, const uint16_t *inject, hipStream_t s, bool central, float strength) {
    A16Args a;
    a.strength = strength;
    a.count = count;
    a.b1 = b1; a.b2 = b2; a.omb1 = 1.0f - b1; a.omb2 = 1.0f - b2; a.eps = eps; a.decay = 1.0f - lr * wd;
    a.inject = inject;
    int64_t tiles = 0;
    for (int32_t i = 0; i < count; ++i) {
        a.tstart[i] = (int32_t)tiles;
        a.it[i] = a16_item(form, items[i], lr, eps);
        if (central) {
            const int64_t rows = items[i].n / items[i].cols, per = CEN_THREADS / a16_tpr(items[i].cols);
            a.cols[i] = items[i].cols;
            tiles += (rows + per - 1) / per;
        } else {
            tiles += ((items[i].n + 7) / 8 + A16_TILE - 1) / A16_TILE;
        }
    }
    if (tiles >= (int64_t(1) << 31)) { set_error("adamw: more than 2^31 tiles in a launch"); return MSR_ERR_ARG; }
    a.tstart[count] = (int32_t)tiles;
    const dim3 grid((unsigned)std::min<int64_t>(tiles, 1 << 20)), block(central ? CEN_THREADS : A16_THREADS);
    if (central) {   // items of one class: rows of up to 2048 elements, or more
        const bool two = items[0].cols > 8 * CEN_THREADS;
#define CEN_LAUNCH(MODE, G) hipLaunchKernelGGL((adamw16_central_kernel<MODE, G>), grid, block, 0, s, a)
        if (mode == NOISE_TRITON) { if (two) CEN_LAUNCH(NOISE_TRITON, 2); else CEN_LAUNCH(NOISE_TRITON, 1); }
        else { if (two) CEN_LAUNCH(NOISE_PHILOX8, 2); else CEN_LAUNCH(NOISE_PHILOX8, 1); }
#undef CEN_LAUNCH
        return check_launch("adamw16_central_kernel");
    }
    if (form == A16_ADAMW) { MSR_DISPATCH_NOISE(mode, M, hipLaunchKernelGGL((adamw16_kernel<M, A16_ADAMW>), grid, block, 0, s, a)); }
    else { MSR_DISPATCH_NOISE(mode, M, hipLaunchKernelGGL((adamw16_kernel<M, A16_ADAM8>), grid, block, 0, s, a)); }
    return check_launch("adamw16_kernel");
}

void item_ranges(const msr_adamw_item &x, int32_t id, ItemRange *r) {
    const size_t b = 2 * (size_t)x.n;
    const void *q[4] = {x.p, x.m, x.v, x.g};
    for (int k = 0; k < 4; ++k) r[k] = {(uintptr_t)q[k], (uintptr_t)q[k] + b, id, k < 3};
}

static bool items_conflict(const msr_adamw_item *items, int32_t count) {
    ItemRange r[4 * A16_MAXT];
    for (int32_t i = 0; i < count; ++i) item_ranges(items[i], i, r + 4 * i);
    return ranges_conflict(r, 4 * count);
}

// Every item's own operands distinct (or the same buffer, updated in place).
int check_item(const msr_adamw_item &x, const char *name, int32_t i) {
    if (x.n < 0 || (x.n > 0 && (!x.p || !x.g || !x.m || !x.v))) {
        set_error("%s: bad arguments in item %d", name, (int)i);
        return MSR_ERR_ARG;
    }
    const void *ops[4] = {x.p, x.g, x.m, x.v};
    for (int k = 0; k < 4; ++k)
        for (int l = k + 1; l < 4; ++l)
            if (partial_overlap(ops[k], 2 * (size_t)x.n, ops[l], 2 * (size_t)x.n)) {
                set_error("%s: operands %d and %d of item %d overlap", name, k, l, (int)i);
                return MSR_ERR_OVERLAP;
            }
    return MSR_OK;
}

}  // namespace msr

using namespace msr;

extern "C" {

int msr_adamw_bf16_step(uint16_t *p, const uint16_t *g, uint16_t *ema, uint16_t *ema_sq, int64_t n, float lr,
                        float beta1, float beta2, float eps, float weight_decay, float bias_correction,
                        float bias_correction_sqrt, uint32_t seed, int32_t noise_mode, const uint16_t *inject,
                        msr_stream_t stream) {
    if (noise_mode < 0 || noise_mode > 2) { set_error("noise_mode %d is not 0, 1 or 2", (int)noise_mode); return MSR_ERR_ARG; }
    if (noise_mode == NOISE_INJECT && !inject) { set_error("noise_mode INJECT needs an inject buffer"); return MSR_ERR_ARG; }
    const msr_adamw_item it{p, g, ema, ema_sq, n, bias_correction, bias_correction_sqrt, seed, 0};
    const int rc = check_item(it, "msr_adamw_bf16_step", 0);
    if (rc || n == 0) return rc;
    return adamw16_launch(A16_ADAMW, &it, 1, lr, beta1, beta2, eps, weight_decay, noise_mode, inject, (hipStream_t)stream);
}

int msr_adamw_multi(const msr_adamw_item *items, int32_t count, int32_t form, float strength, float lr, float beta1,
                    float beta2, float eps, float weight_decay, int32_t noise_mode, msr_stream_t stream) {
    const bool central = form == MSR_ADAMW_CENTRALIZED;
    if (count < 0 || (count > 0 && !items) || (form != MSR_ADAMW && form != MSR_ADAMW_8BIT16 && !central)) {
        set_error("msr_adamw_multi: bad arguments");
        return MSR_ERR_ARG;
    }
    if (noise_mode != NOISE_TRITON && noise_mode != NOISE_PHILOX8) {
        set_error("msr_adamw_multi: noise_mode must be TRITON or PHILOX8 (got %d)", (int)noise_mode);
        return MSR_ERR_ARG;
    }
    for (int32_t i = 0; i < count; ++i) {
        const msr_adamw_item &x = items[i];
        const int rc = check_item(x, "msr_adamw_multi", i);
        if (rc) return rc;
        if (central && x.n > 0 &&
            (x.cols < 8 || x.cols > MSR_ADAMW_CENTRAL_MAX_COLS || x.cols % 8 || x.n % x.cols || !aligned(x.p, 16) ||
             !aligned(x.g, 16) || !aligned(x.m, 16) || !aligned(x.v, 16))) {
            set_error("msr_adamw_multi: centralization needs 16-byte aligned tensors and rows of a multiple of 8 elements, "
                      "at most %d (item %d: %lld in rows of %d)", MSR_ADAMW_CENTRAL_MAX_COLS, (int)i, (long long)x.n, (int)x.cols);
            return MSR_ERR_ARG;
        }
    }
    for (int32_t i = 0; i < count;) {
        msr_adamw_item run[A16_MAXT];
        int32_t n = 0;
        for (; i < count && n < A16_MAXT; ++i)
            if (items[i].n > 0) run[n++] = items[i];
        int32_t cut = n;   // central: first the items of narrow rows, then the wide ones
        const bool apart = n > 1 && items_conflict(run, n);
        if (central && !apart)
            cut = (int32_t)(std::stable_partition(run, run + n, [](const msr_adamw_item &x) { return x.cols <= 8 * CEN_THREADS; }) - run);
        for (int32_t j = 0; j < n;) {
            const int32_t k = apart ? 1 : (j < cut ? cut : n) - j;
            const int rc = adamw16_launch(central ? MSR_ADAMW : form, run + j, k, lr, beta1, beta2, eps, weight_decay,
                                          noise_mode, nullptr, (hipStream_t)stream, central, strength);
            if (rc) return rc;
            j += k;
        }
    }
    return MSR_OK;
}

}  // extern "C"
