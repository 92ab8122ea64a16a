// Matrix products in 64 x 64 and 128 x 128 tiles, for products too small to fill the
// chip with 256 x 256 ones (ns_gemm.hip): Newton-Schulz of few or small matrices, and
// weight gradients of modest layers.
//
// What bounds them is not the matrix cores but how many CUs have a tile and how long
// one tile takes from its first load to its last store.  So the tile is small, K streams
// through a ring of LDS stages filled by direct global->LDS loads several slabs ahead
// (counted vmcnt waits, one barrier per slab), and a work-group does one tile.
// Symmetric products compute their upper tiles and store each off-diagonal one twice
// (transposed through the epilogue's LDS staging), so every operand of the iteration is
// a full row-major matrix and the K loop has a single range.
//
// Every output element is the same chain of 32x32x16 MFMAs over ascending k as in the
// 256 x 256 kernel, with the same epilogue arithmetic, so results are the same bits
// whichever tile a call takes (zero padding adds exact zeros).
#include <algorithm>
#include <type_traits>

#include "gemm.hpp"
#include "tile_gemm.hpp"
#include "../../include/muon_sr_amd.h"

namespace msr {

constexpr int TBK = 64;            // k per slab
constexpr int TG_THREADS = 256;    // 4 waves, 2 x 2, each T/2 x T/2 of the tile

constexpr int PR_A = TILE_A, PR_B = TILE_B, PR_X = TILE_X, PR_W = TILE_W;
constexpr int OUT_WS = TILE_WS, OUT_D = TILE_D, OUT_DT = TILE_DT, OUT_PD = TILE_PD, OUT_PT = TILE_PT;

struct NoTab {};

// PROD: A = alpha X X^T | B' = alpha A A + beta A + diag I | X' = alpha (B' X + r X) |
// the weight gradient's SR accumulation.  OUT (X'): workspace matrix, caller's output as is
// or transposed (bounded stores), or the Muon apply on the parameters in either layout.
// MODE: noise mode of the apply or accumulation.  T: tile; S: LDS stages.
// Two work-groups per CU, but for the 128 KiB ring, of which the LDS holds one.
template <int T, int S, int PROD, int OUT, int MODE, typename TAB>
__global__ __launch_bounds__(TG_THREADS, T * S == 512 ? 1 : 2) void tile_gemm_kernel(TileArgs a, TAB tab) {
    constexpr int W = T / 2, F = W / 32;            // a wave's sub-tile and its 32-wide blocks per side
    constexpr int SLAB = T * TBK * 2;               // bytes of one operand's slab
    constexpr int NL = SLAB / 4096;                 // direct-to-LDS loads per wave, operand and slab
    constexpr int LPS = 2 * NL;                     // ... per wave and slab
    constexpr bool PK = PROD == PR_W, QK = PROD == PR_W || PROD == PR_X;   // K-major operands
    constexpr bool SYM = PROD == PR_A || PROD == PR_B;
    static_assert(S == 2 || S == 4, "an even ring: a slab's fragments go to the register set of its stage's parity");
    static_assert((S - 1) * LPS < 64, "vmcnt is 6 bits");
    // one variable per stage, so that the compiler knows that the fragment reads of one
    // stage do not alias the loads into another (it would wait for those loads otherwise)
    __shared__ __attribute__((aligned(1024))) char st0[2 * SLAB], st1[2 * SLAB];
    __shared__ __attribute__((aligned(1024))) char st2[S > 2 ? 2 * SLAB : 16], st3[S > 3 ? 2 * SLAB : 16];
    auto stage = [&](auto ST) __attribute__((always_inline)) -> char * {
        constexpr int s = decltype(ST)::value;
        if constexpr (s == 0) return st0;
        else if constexpr (s == 1) return st1;
        else if constexpr (s == 2) return st2;
        else return st3;
    };

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int r32 = lane & 31, khalf = lane >> 5;

    // Work-group -> (matrix, tile).  Consecutive work-groups go to the 8 XCDs in turn: each
    // XCD takes a contiguous eighth of the launch's tiles, so that tiles sharing operand rows
    // share its L2.
    const int per = a.total / NXCD;
    const int b = blockIdx.x;
    const int v = b < per * NXCD ? (b % NXCD) * per + b / NXCD : b;
    const int64_t bz = v / a.tiles;
    const int t = v % a.tiles;
    int ti, tj;
    if constexpr (SYM) {   // upper triangle, column by column
        tj = (int)((__builtin_amdgcn_sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
        while (tj * (tj + 1) / 2 > t) --tj;
        while ((tj + 1) * (tj + 2) / 2 <= t) ++tj;
        ti = t - tj * (tj + 1) / 2;
    } else {               // 4 tile-rows at a time, column by column
        const int pg = 4 * a.tiles_n, g = t / pg, first = 4 * g, rows = min(4, a.tiles_m - first), r = t - g * pg;
        ti = first + r % rows;
        tj = r / rows;
    }
    const int m0 = ti * T, n0 = tj * T;

    const uint16_t *Pb = a.P + bz * a.sP, *Qb = a.Q + bz * a.sQ;
    const uint32_t ldbP = (uint32_t)(a.ldp * 2), ldbQ = (uint32_t)(a.ldq * 2);
    const __amdgpu_buffer_rsrc_t rP = __builtin_amdgcn_make_buffer_rsrc((void *)Pb, (short)0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rQ = __builtin_amdgcn_make_buffer_rsrc((void *)Qb, (short)0, 0x7fffffff, 0x00020000);

    // Global -> LDS: load i (0..NL-1) of wave w moves 64 lanes x 16 B into block 4 i + w (1 KiB)
    // of the slab (lane l to byte 16 l).
    //  * row-major slab (T rows x 128 B): block = 8 rows; row r holds logical chunk c at
    //    c ^ ((r >> 1) & 7), so a fragment read's 16 rows cover all 64 banks;
    //  * K-major slab (64 rows of k x 2 T B): T = 128: block = 4 rows, chunk c of row k at
    //    c ^ 4 (k & 3); T = 64: block = 8 rows, chunk c at c ^ 4 ((k >> 1) & 1) (rows k and
    //    k + 1 fall in different halves of the banks by themselves).
    const int lrow = lane >> 3, lchunk = (lane & 7) ^ (4 * (wave & 1) + (lane >> 4));
    const int kr = T == 128 ? 4 * wave + (lane >> 4) : 8 * wave + (lane >> 3);
    const int kc = T == 128 ? (lane & 15) ^ (4 * (lane >> 4)) : (lane & 7) ^ (4 * ((lane >> 4) & 1));
    constexpr int KSTEP = T == 128 ? 16 : 32;       // k rows per load index of a K-major slab
    const uint32_t vP = PK ? (uint32_t)(((int64_t)kr * a.ldp + m0 + 8 * kc) * 2)
                           : (uint32_t)(((int64_t)(m0 + wave * 8 + lrow) * a.ldp + lchunk * 8) * 2);
    const uint32_t vQ = QK ? (uint32_t)(((int64_t)kr * a.ldq + n0 + 8 * kc) * 2)
                           : (uint32_t)(((int64_t)(n0 + wave * 8 + lrow) * a.ldq + lchunk * 8) * 2);
    // load j of the slab at k0 (even: P block j / 2, odd: Q block j / 2)
    auto issue1 = [&](auto ST, int k0, int j) __attribute__((always_inline)) {
        const int i = j >> 1, dst = (4 * i + wave) * 1024;
        if (j & 1) {
            const uint32_t oQ = QK ? (uint32_t)(k0 + KSTEP * i) * ldbQ : (uint32_t)(32 * i) * ldbQ + (uint32_t)k0 * 2u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rQ, (lds_void_t *)(stage(ST) + SLAB + dst), 16, vQ, oQ, 0, 0);
        } else {
            const uint32_t oP = PK ? (uint32_t)(k0 + KSTEP * i) * ldbP : (uint32_t)(32 * i) * ldbP + (uint32_t)k0 * 2u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rP, (lds_void_t *)(stage(ST) + dst), 16, vP, oP, 0, 0);
        }
    };
    auto issue = [&](auto ST, int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < LPS; ++j) issue1(ST, k0, j);
    };

    // Fragment reads.  Row-major: chunk (2 ks + khalf) ^ ((row >> 1) & 7) of row.  K-major: two
    // transposing reads of 4 k each; in a read, lane i of a 16-lane group fetches row k = i / 4,
    // columns 4 (i % 4) .. +3 of its group's 16 and returns element i % 4 of 4 lanes' rows.
    const int sw = (r32 >> 1) & 7;
    const int G = lane >> 4, gi = lane & 15;
    const uint32_t rowP = (uint32_t)((wm * W + r32) * 128), rowQ = (uint32_t)((wn * W + r32) * 128);
    const uint32_t krow = (uint32_t)((8 * (G >> 1) + (gi >> 2)) * (2 * T) + (gi & 1) * 8);
    const int kc0 = 2 * (G & 1) + ((gi >> 1) & 1), kx = T == 128 ? 4 * (gi >> 2) : 4 * (gi >> 3);
    auto trfrag = [](const char *p) __attribute__((always_inline)) {
        const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t *)(p));
        const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t *)(p + 4 * (2 * T)));
        return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    auto frag = [&](auto KM, const char *base, uint32_t row, int wcol, int ks, int f) __attribute__((always_inline)) {
        if constexpr (decltype(KM)::value)
            return trfrag(base + ks * 16 * (2 * T) + krow + (uint32_t)((((wcol + 32 * f) / 8 + kc0) ^ kx) * 16));
        else
            return *reinterpret_cast<const bf16x8_t *>(base + row + f * 4096 + (((2 * ks) ^ khalf ^ sw) * 16));
    };

    f32x16_t acc[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // X' = B' X + r X: bf16(r) of the wave's rows; the term enters as MFMAs with a one-hot
    // operand right after the substep that holds k = m (as in the 256 x 256 kernel)
    uint32_t rb16[F];
    const int wm0 = m0 + wm * W, wn0 = n0 + wn * W;
    if constexpr (PROD == PR_X) {
#pragma unroll
        for (int mi = 0; mi < F; ++mi) {
            const float rf = a.rvec[bz * a.sv + wm0 + 32 * mi + r32];
            rb16[mi] = rne_bf16x2(rf, 0.0f) & 0xffffu;
        }
    }

    const int KT = a.K / TBK;
    // A slab's 4 substeps go in groups of H; while the matrix cores multiply one group, the next
    // one is read into the other register set.  T = 64: a whole slab at a time (one MFMA per
    // substep would not cover a read's latency); T = 128: half a slab (two sets of whole slabs
    // would not leave registers for two work-groups per CU).
    constexpr int H = T == 64 ? 4 : 2, NG = 4 / H;
    bf16x8_t fp[2][H][F], fq[2][H][F];
    constexpr int NF = 2 * F * H, NM = H * F * F;   // fragments and MFMAs of a group
    static_assert(NF % NM == 0 && LPS % NM == 0, "a group's reads and a slab's loads spread over its MFMAs");
    auto read1 = [&](auto ST, auto GR, int j) __attribute__((always_inline)) {   // fragment j of group GR of stage ST's slab
        constexpr int g = decltype(GR)::value, pr = NG == 1 ? decltype(ST)::value & 1 : g;
        const char *const base = stage(ST);
        const int h = j / (2 * F), f = (j >> 1) % F;
        if (j & 1) fq[pr][h][f] = frag(std::integral_constant<bool, QK>{}, base + SLAB, rowQ, wn * W, g * H + h, f);
        else fp[pr][h][f] = frag(std::integral_constant<bool, PK>{}, base, rowP, wm * W, g * H + h, f);
    };
    auto read = [&](auto ST, auto GR) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NF; ++j) read1(ST, GR, j);
    };
    // dg: the slab holds the diagonal of (some of) this wave's rows (X' only): in substep ks the
    // diagonal crosses the wave's 32-row block ks / 2 (T = 128), or, for the waves with wm = ks / 2,
    // its one block (T = 64); lane l's fragment (row r32, k = 8 khalf + e) holds it at
    // e = r32 - 16 (ks & 1) - 8 khalf.
    // before(x): what is issued ahead of the group's MFMA x
    auto mult = [&](auto ST, auto GR, bool dg, auto before) __attribute__((always_inline)) {
        constexpr int g = decltype(GR)::value, pr = NG == 1 ? decltype(ST)::value & 1 : g;
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const int ks = g * H + h;
#pragma unroll
            for (int mi = 0; mi < F; ++mi)
#pragma unroll
                for (int ni = 0; ni < F; ++ni) {
                    before((h * F + mi) * F + ni);
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fq[pr][h][ni], fp[pr][h][mi], acc[mi][ni], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            if constexpr (PROD == PR_X) {
                if (dg && (T == 128 || wm == (ks >> 1))) {   // uniform per wave
                    const int mi = T == 128 ? ks >> 1 : 0;
                    int row = r32;   // an opaque copy: the operand is formed here, not kept over the loop
                    asm volatile("" : "+v"(row));
                    const int e = row - 16 * (ks & 1) - 8 * khalf;
                    const uint32_t x = (unsigned)e < 8u ? rb16[mi] << (16 * (e & 1)) : 0u;
                    const int w = e >> 1;
                    const u32x4_t words = {w == 0 ? x : 0u, w == 1 ? x : 0u, w == 2 ? x : 0u, w == 3 ? x : 0u};
                    const bf16x8_t rf = __builtin_bit_cast(bf16x8_t, words);
#pragma unroll
                    for (int ni = 0; ni < F; ++ni)
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fq[pr][h][ni], rf, acc[mi][ni], 0, 0, 0);
                }
            }
        }
    };
    using T_ = std::true_type;
    using F_ = std::false_type;
    using I0_ = std::integral_constant<int, 0>;
    using I1_ = std::integral_constant<int, 1>;
    using I2_ = std::integral_constant<int, 2>;
    using I3_ = std::integral_constant<int, 3>;
    // Slab k, whose first group has been read: its MFMAs, the reads of its other groups, then,
    // after the barrier that frees its stage, slab k + S into that stage (ISSUE) and the first
    // group of slab k + 1 (NEXT).  AFTER: slabs later than k + 1 in flight at the barrier.
    auto body = [&](auto ST, int k, auto ISSUE, auto AFTER, auto NEXT) __attribute__((always_inline)) {
        constexpr int s = decltype(ST)::value;
        using SN = std::integral_constant<int, (s + 1) % S>;
        const bool dg = PROD == PR_X && k * TBK == (T == 128 ? wm0 : m0);
        if constexpr (NG > 1)
            mult(ST, I0_{}, dg, [&](int x) __attribute__((always_inline)) { read1(ST, I1_{}, x); });
        using GL = std::integral_constant<int, NG - 1>;
        if constexpr (decltype(NEXT)::value) {
            wait_vm<decltype(AFTER)::value * LPS>();                           // own loads of slab k + 1
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");    // everyone's; slab k is read
            // reads and loads go out between the MFMAs: one after the other they would stall the
            // wave (one wave per SIMD) on the full LDS and texture queues
            mult(ST, GL{}, dg, [&](int x) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < NF / NM; ++j) read1(SN{}, I0_{}, x * (NF / NM) + j);
                if constexpr (decltype(ISSUE)::value) {
#pragma unroll
                    for (int j = 0; j < LPS / NM; ++j) issue1(ST, (k + S) * TBK, x * (LPS / NM) + j);
                }
            });
        } else {
            mult(ST, GL{}, dg, [](int) __attribute__((always_inline)) {});
        }
    };
    // Every loop and tail below has a fixed sequence of loads and counted waits: with a
    // conditional load the compiler would have to wait for everything before the fragment reads.
    issue(I0_{}, 0);                          // a K of fewer than S slabs loads its last one again
    issue(I1_{}, min(1, KT - 1) * TBK);
    if constexpr (S > 2) {
        issue(I2_{}, min(2, KT - 1) * TBK);
        issue(I3_{}, min(3, KT - 1) * TBK);
    }
    using AF = std::integral_constant<int, S - 2>;
    // N slabs from k that load another one each, then the last S
    auto tail = [&](auto N, int k) __attribute__((always_inline)) {
        constexpr int n = decltype(N)::value;
        if constexpr (n > 0) body(I0_{}, k, T_{}, AF{}, T_{});
        if constexpr (n > 1) body(I1_{}, k + 1, T_{}, AF{}, T_{});
        if constexpr (n > 2) body(std::integral_constant<int, 2 % S>{}, k + 2, T_{}, AF{}, T_{});
        body(std::integral_constant<int, n % S>{}, k + n, F_{}, AF{}, T_{});
        if constexpr (S > 2) {
            body(std::integral_constant<int, (n + 1) % S>{}, k + n + 1, F_{}, std::integral_constant<int, (S > 2 ? S - 3 : 0)>{}, T_{});
            body(std::integral_constant<int, (n + 2) % S>{}, k + n + 2, F_{}, I0_{}, T_{});
        }
        body(std::integral_constant<int, (n + S - 1) % S>{}, k + n + S - 1, F_{}, I0_{}, F_{});
    };
    if (KT < S) {
        wait_vm<0>();
        asm volatile("s_barrier" ::: "memory");
        read(I0_{}, I0_{});
        if (KT == 1) {
            body(I0_{}, 0, F_{}, I0_{}, F_{});
        } else if constexpr (S > 2) {
            body(I0_{}, 0, F_{}, I0_{}, T_{});
            if (KT == 2) {
                body(I1_{}, 1, F_{}, I0_{}, F_{});
            } else {
                body(I1_{}, 1, F_{}, I0_{}, T_{});
                body(I2_{}, 2, F_{}, I0_{}, F_{});
            }
        }
    } else {
        wait_vm<(S - 1) * LPS>();
        asm volatile("s_barrier" ::: "memory");
        read(I0_{}, I0_{});
        int k = 0;
#pragma clang loop unroll(disable)
        for (; k + 2 * S <= KT; k += S) {
            body(I0_{}, k, T_{}, AF{}, T_{});
            body(I1_{}, k + 1, T_{}, AF{}, T_{});
            if constexpr (S > 2) {
                body(I2_{}, k + 2, T_{}, AF{}, T_{});
                body(I3_{}, k + 3, T_{}, AF{}, T_{});
            }
        }
        const int n = KT - k - S;   // 0 .. S - 1
        if (n == 0) tail(I0_{}, k);
        else if (n == 1) tail(I1_{}, k);
        else if constexpr (S > 2) {
            if (n == 2) tail(I2_{}, k);
            else tail(I3_{}, k);
        }
    }

    // ---------------- epilogue ----------------
    // Each wave stages its sub-tile through a private LDS region, one 32-row block at a time
    // (LDS accesses of one wave execute in order: no barrier after this one).  Lane l holds
    // D[m = l % 32][n = 8 r + 4 (l / 32) + q] of each 32 x 32 block.
    wait_vm<0>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    constexpr int EP = W + 8;                        // staging row pitch (elements; 16-byte rows)
    static_assert(4 * 32 * EP * 2 <= 2 * SLAB, "the staging fits one stage");
    char *const wst = st0 + wave * (32 * EP * 2);
    auto est = [&](int row) __attribute__((always_inline)) { return reinterpret_cast<uint16_t *>(wst + row * (EP * 2)); };
    constexpr int WC = W / 8, RPP = 64 / WC, NP = 32 / RPP;   // 16-byte chunks per row, rows per access, accesses per block
    constexpr int TP = W / 16;                                 // transposed accesses per block (16 output rows each)
    const int crow = lane / WC, cchk = lane % WC;
    const int tq = lane & 3, tn = lane >> 2;
    const float alpha = a.alpha_b ? a.alpha_b[bz] : a.alpha;
    const bool dtile = SYM && m0 == n0;
    auto block = [&](auto MI) __attribute__((always_inline)) {
        constexpr int mi = decltype(MI)::value;
        const int bm0 = wm0 + 32 * mi;
        if constexpr (PROD == PR_B) {   // this block of A into the staging
            const uint16_t *Cb = a.C + bz * a.sC + (int64_t)(bm0 + crow) * a.ldc + wn0 + 8 * cchk;
            u32x4_t c[NP];
#pragma unroll
            for (int i = 0; i < NP; ++i) c[i] = *reinterpret_cast<const u32x4_t *>(Cb + (int64_t)(RPP * i) * a.ldc);
#pragma unroll
            for (int i = 0; i < NP; ++i) *reinterpret_cast<u32x4_t *>(est(crow + RPP * i) + 8 * cchk) = c[i];
        }
        float rho = 0.0f;
        if constexpr (PROD == PR_B) {
            if (dtile) rho = a.rvec[bz * a.sv + bm0 + r32];
        }
        float res = 0.0f;
        bool has = false;
#pragma unroll
        for (int ni = 0; ni < F; ++ni) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = bm0 + r32, n = wn0 + ni * 32 + 8 * r + 4 * khalf;
                uint2 *sp = reinterpret_cast<uint2 *>(est(r32) + ni * 32 + 8 * r + 4 * khalf);
                float x[4], cv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    x[q] = acc[mi][ni][4 * r + q];
                    if constexpr (PROD != PR_W) x[q] = alpha * x[q];
                }
                if constexpr (PROD == PR_B) {
                    const uint2 cw = *sp;
                    cv[0] = bf16_lo(cw.x);
                    cv[1] = bf16_hi(cw.x);
                    cv[2] = bf16_lo(cw.y);
                    cv[3] = bf16_hi(cw.y);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        x[q] = x[q] + a.beta * cv[q];
                        if (dtile && m == n + q) x[q] = x[q] + (a.diag + rho * (a.beta + 2.0f * alpha * cv[q]));
                    }
                }
                const uint2 w = make_uint2(rne_bf16x2(x[0], x[1]), rne_bf16x2(x[2], x[3]));
                *sp = w;
                if constexpr (SYM) {
                    const float rq[4] = {bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y)};
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const bool on = dtile && m == n + q;
                        res = on ? x[q] - rq[q] : res;
                        has = has || on;
                    }
                }
            }
        }
        if constexpr (SYM) {
            if (has) a.resid[bz * a.sv + bm0 + r32] = res;
        }
        // block rows bm0 + crow + RPP i, columns wn0 + 8 cchk
        if constexpr (PROD == PR_W) {
            uint16_t *Db = a.D + bz * a.sD;
            uint4 c[NP];
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int64_t o0 = (int64_t)(bm0 + crow + RPP * i) * a.ldd + wn0 + 8 * cchk;
                c[i] = a.zero_init ? make_uint4(0u, 0u, 0u, 0u) : *reinterpret_cast<const uint4 *>(Db + o0);
            }
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int64_t o0 = (int64_t)(bm0 + crow + RPP * i) * a.ldd + wn0 + 8 * cchk;
                const uint4 w = *reinterpret_cast<const uint4 *>(est(crow + RPP * i) + 8 * cchk);
                const uint32_t gw[4] = {w.x, w.y, w.z, w.w}, cw[4] = {c[i].x, c[i].y, c[i].z, c[i].w};
                uint32_t rn[8], o[4];
                noise8<MODE>(a.ns, o0, 8, rn);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    o[j] = pack2(sr_bf16(bf16_lo(cw[j]) + bf16_lo(gw[j]), rn[2 * j]),
                                 sr_bf16(bf16_hi(cw[j]) + bf16_hi(gw[j]), rn[2 * j + 1]));
                *reinterpret_cast<uint4 *>(Db + o0) = make_uint4(o[0], o[1], o[2], o[3]);
            }
        } else if constexpr (OUT == OUT_WS) {
            uint16_t *Db = a.D + bz * a.sD + (int64_t)(bm0 + crow) * a.ldd + wn0 + 8 * cchk;
#pragma unroll
            for (int i = 0; i < NP; ++i)
                *reinterpret_cast<uint4 *>(Db + (int64_t)(RPP * i) * a.ldd) = *reinterpret_cast<const uint4 *>(est(crow + RPP * i) + 8 * cchk);
        } else if constexpr (OUT == OUT_D || OUT == OUT_PD) {
            const int n = wn0 + 8 * cchk, valid = min(8, a.Nv - n);
            const bool vec = a.d_vec != 0;
            if constexpr (OUT == OUT_PD) {
                uint16_t *Pp = tab.p[bz];
                Noise ns;
                ns.key = seed_key(tab.seed[bz], 0);
                ns.inject = tab.inject ? tab.inject + bz * tab.numel : nullptr;
                u32x4_t pw[NP];
#pragma unroll
                for (int i = 0; i < NP; ++i) {
                    const int m = bm0 + crow + RPP * i;
                    pw[i] = m < a.Mv && valid > 0 ? apply_load(Pp, (int64_t)m * a.ldd + n, valid, vec) : u32x4_t{0u, 0u, 0u, 0u};
                }
#pragma unroll
                for (int i = 0; i < NP; ++i) {
                    const int m = bm0 + crow + RPP * i;
                    if (m >= a.Mv || valid <= 0) continue;
                    const uint4 w = *reinterpret_cast<const uint4 *>(est(crow + RPP * i) + 8 * cchk);
                    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
                    apply_chunk<MODE>(tab, Pp, ns, (int64_t)m * a.ldd + n, valid, vec, u, pw[i]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < NP; ++i) {
                    const int m = bm0 + crow + RPP * i;
                    if (m >= a.Mv || valid <= 0) continue;
                    const uint4 w = *reinterpret_cast<const uint4 *>(est(crow + RPP * i) + 8 * cchk);
                    uint16_t *dp = a.D + bz * a.sD + (int64_t)m * a.ldd + n;
                    if (vec && valid == 8) {
                        *reinterpret_cast<uint4 *>(dp) = w;
                    } else {
                        const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            if (j < valid) dp[j] = (uint16_t)(u[j >> 1] >> (16 * (j & 1)));
                    }
                }
            }
        }
        // transposed: output row n = wn0 + tn + 16 i, the 8 consecutive m from bm0 + 8 tq
        if constexpr (SYM || OUT == OUT_DT || OUT == OUT_PT) {
            if (SYM && dtile) return;
            const int m = bm0 + 8 * tq, valid = SYM ? 8 : min(8, a.Mv - m);
            const bool vec = SYM || a.dt_vec != 0;
            Noise ns;
            uint16_t *Pp = nullptr;
            u32x4_t pw[TP];
            if constexpr (OUT == OUT_PT) {
                Pp = tab.p[bz];
                ns.key = seed_key(tab.seed[bz], 0);
                ns.inject = tab.inject ? tab.inject + bz * tab.numel : nullptr;
#pragma unroll
                for (int i = 0; i < TP; ++i) {
                    const int n = wn0 + tn + 16 * i;
                    pw[i] = n < a.Nv && valid > 0 ? apply_load(Pp, (int64_t)n * a.lddt + m, valid, vec) : u32x4_t{0u, 0u, 0u, 0u};
                }
            }
#pragma unroll
            for (int i = 0; i < TP; ++i) {
                const int nl = tn + 16 * i, n = wn0 + nl;
                uint32_t u[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    u[j] = (uint32_t)est(8 * tq + 2 * j)[nl] | ((uint32_t)est(8 * tq + 2 * j + 1)[nl] << 16);
                if constexpr (SYM) {
                    *reinterpret_cast<uint4 *>(a.D + bz * a.sD + (int64_t)n * a.ldd + m) = make_uint4(u[0], u[1], u[2], u[3]);
                } else {
                    if (n >= a.Nv || valid <= 0) continue;
                    if constexpr (OUT == OUT_PT) {
                        apply_chunk<MODE>(tab, Pp, ns, (int64_t)n * a.lddt + m, valid, vec, u, pw[i]);
                    } else {
                        uint16_t *tp = a.DT + bz * a.sDT + (int64_t)n * a.lddt + m;
                        if (vec && valid == 8) {
                            *reinterpret_cast<uint4 *>(tp) = make_uint4(u[0], u[1], u[2], u[3]);
                        } else {
#pragma unroll
                            for (int j = 0; j < 8; ++j)
                                if (j < valid) tp[j] = (uint16_t)(u[j >> 1] >> (16 * (j & 1)));
                        }
                    }
                }
            }
        }
    };
    block(I0_{});
    if constexpr (F > 1) block(I1_{});
}

template <int T, int S>
static int launch_tiles(int prod, int out, int mode, TileArgs &a, int64_t batch, const ApplyTab *tab, hipStream_t s) {
    const int64_t tm = a.M / T, tn = a.N / T, tiles = prod == PR_A || prod == PR_B ? tm * (tm + 1) / 2 : tm * tn;
    if (a.M % T || a.N % T || a.K % TBK || tiles * batch >= (int64_t(1) << 30)) {
        set_error("tile_gemm: a %d x %d x %d product of %lld matrices does not fit %d-wide tiles", a.M, a.N, a.K,
                  (long long)batch, T);
        return MSR_ERR_ARG;
    }
    a.tiles_m = (int)tm; a.tiles_n = (int)tn; a.tiles = (int)tiles; a.total = (int)(tiles * batch);
    const dim3 grid((unsigned)a.total), block(TG_THREADS);
#define TG_LAUNCH(PROD, OUT, MODE, TAB, tab) hipLaunchKernelGGL((tile_gemm_kernel<T, S, PROD, OUT, MODE, TAB>), grid, block, 0, s, a, tab)
    if (prod == PR_A) TG_LAUNCH(PR_A, OUT_WS, 0, NoTab, NoTab{});
    else if (prod == PR_B) TG_LAUNCH(PR_B, OUT_WS, 0, NoTab, NoTab{});
    else if (prod == PR_W) { MSR_DISPATCH_NOISE(mode, M, TG_LAUNCH(PR_W, OUT_D, M, NoTab, NoTab{})); }
    else if (out == OUT_WS) TG_LAUNCH(PR_X, OUT_WS, 0, NoTab, NoTab{});
    else if (out == OUT_D) TG_LAUNCH(PR_X, OUT_D, 0, NoTab, NoTab{});
    else if (out == OUT_DT) TG_LAUNCH(PR_X, OUT_DT, 0, NoTab, NoTab{});
    else if (out == OUT_PD) { MSR_DISPATCH_NOISE(mode, M, TG_LAUNCH(PR_X, OUT_PD, M, ApplyTab, *tab)); }
    else { MSR_DISPATCH_NOISE(mode, M, TG_LAUNCH(PR_X, OUT_PT, M, ApplyTab, *tab)); }
#undef TG_LAUNCH
    return check_launch("tile_gemm_kernel");
}

// Estimated time (us) of a product in `tiles` tiles of T (ring of S stages) over `slabs` K slabs:
// rounds of the work-groups that run at once (LDS and registers allow 512 of 64/4, 768 of 64/2, 256
// of 128/4 and 512 of 128/2), each the slabs plus a tile's start and end.  Fitted to kernel times
// of A, B' and X' at 20 Newton-Schulz shapes (1-64 matrices of 256-2048 x 256-5632).  Some of the
// times, us (64/4, 64/2, 128/4, 128/2), and what the estimates pick:
//   40 tiles of 64 (12 of 128),  4 slabs   4.1   4.4   6.9   6.6   64/4, the fastest
//   168 (48),                   24 slabs   6.8   8.8  13.4  13.7   64/4, the fastest
//   528 (136),                  88 slabs  59.3  44.8  38.2  57.3   64/2, 17 % over 128/4
//   576 (144),                  12 slabs  12.0   9.9  10.5  10.5   64/2, the fastest
//   1024 (256),                 32 slabs  30.9  30.6  20.6  24.3   128/4, the fastest
//   1152 (288),                  6 slabs  12.0  11.0  14.0   9.8   64/2, 12 % over 128/2
//   8192 (2048),                16 slabs   121   105    90    72   128/2, the fastest
// The two misses are 64/2, whose term is one line in `slabs` and a plain share of a round: 0.6 us
// more for it mends the second and makes 40 other shapes 1.1 % slower (geometric mean).
// 256-wide tiles (ns_gemm.hip): one work-group per CU.
static double tile_cost(int T, int S, int64_t tiles, int64_t slabs) {
    const double f = (double)tiles / TILE_CUS, k = (double)slabs;
    // whole rounds of n work-groups, and a last one that is shorter when it leaves CUs less shared
    auto rounds = [&](int64_t n, double least) {
        const int64_t rest = tiles % n;
        return (double)(tiles / n) + (rest ? least + (1.0 - least) * (double)rest / (double)n : 0.0);
    };
    if (T == 256) return 9.0 + 1.3 * k * (double)((tiles + TILE_CUS - 1) / TILE_CUS);
    if (T == 64 && S == 4) return f <= 1.0 ? 3.4 + k * (0.13 + 0.13 * f) : 3.4 + rounds(512, 0.4) * (0.42 * k + 1.0);
    if (T == 64) return 3.4 + std::max(0.5, f / 3.0) * (0.57 * k + 1.2);
    if (S == 4) return 5.2 + (f <= 1.0 ? k * (0.33 + 0.17 * f) : rounds(TILE_CUS, 0.66) * (0.5 * k + 1.0));
    return 5.0 + rounds(512, 0.45) * (0.98 * k + 1.2);
}

struct TileCfg {
    int T, S;
};
constexpr TileCfg TILE_CFGS[4] = {{64, 4}, {64, 2}, {128, 4}, {128, 2}};

// Tiles of an M x N product in T-wide tiles (upper ones only if symmetric).
static int64_t tiles_of(int T, bool sym, int64_t M, int64_t N) {
    const int64_t tm = M / T, tn = N / T;
    return sym ? tm * (tm + 1) / 2 : tm * tn;
}

// The cheapest of the four for a product whose extents are multiples of 64.
static TileCfg best_cfg(bool sym, int64_t M, int64_t N, int64_t K, int64_t batch, double *cost) {
    TileCfg best = TILE_CFGS[0];
    double least = -1.0;
    for (const TileCfg &c : TILE_CFGS) {
        if (M % c.T || N % c.T) continue;
        const double t = tile_cost(c.T, c.S, tiles_of(c.T, sym, M, N) * batch, K / TBK);
        if (least < 0.0 || t < least) { least = t; best = c; }
    }
    *cost = least;
    return best;
}

int launch_tile_gemm(int prod, int out, int mode, const TileArgs &a0, int64_t batch, const ApplyTab *tab, hipStream_t s) {
    TileArgs a = a0;
    if (batch == 0) return MSR_OK;
    double cost;
    const TileCfg c = best_cfg(prod == PR_A || prod == PR_B, a.M, a.N, a.K, batch, &cost);
    if (c.T == 64) return c.S == 4 ? launch_tiles<64, 4>(prod, out, mode, a, batch, tab, s) : launch_tiles<64, 2>(prod, out, mode, a, batch, tab, s);
    return c.S == 4 ? launch_tiles<128, 4>(prod, out, mode, a, batch, tab, s) : launch_tiles<128, 2>(prod, out, mode, a, batch, tab, s);
}

static int64_t up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// Padding of a Newton-Schulz call (m <= n): the smallest estimate of one iteration's three
// products, each in its best tile, with what the padding costs; 256 means the 256-wide kernel.
// Measured times in us (all products 256 / 128 / 64 wide):
//   4 of 256 x 256   165 / 104 / 65      1 of 2048 x 2048   710 / 286 / 371
//   8 of 384 x 1536  351 / 170 / 121     2 of 2048 x 5632  1308 / 910 / 1333
//   1 of 1024 x 1024 364 / 185 / 118     4 of 2048 x 2048   795 / 845 / 1126
//   12 of 768 x 3072 1259 / 541 / 640    1 of 4096 x 4096  1371 / 1576 / 2520
int ns_tile_choice(int64_t batch, int64_t m, int64_t n) {
    int best = 256;
    double least = 0.0;
    for (int T : {256, 128, 64}) {
        const int64_t mp = up(m, T), np = up(n, T);
        double c;
        if (T == 256) {
            const int64_t sym = tiles_of(256, true, mp, mp) * batch;
            c = tile_cost(256, 2, sym, np / TBK) + tile_cost(256, 2, sym, mp / TBK) +
                tile_cost(256, 2, tiles_of(256, false, mp, np) * batch, mp / TBK);
        } else {
            if (tiles_of(64, false, mp, np) * batch >= (int64_t(1) << 28) || mp * np >= (int64_t(1) << 29)) continue;
            double ca, cb, cx;
            best_cfg(true, mp, mp, np, batch, &ca);
            best_cfg(true, mp, mp, mp, batch, &cb);
            best_cfg(false, mp, np, mp, batch, &cx);
            c = ca + cb + cx;
        }
        if (T == 256 || c < least) { best = T; least = c; }
    }
    return best;
}

// Whether a weight gradient M x N over K tokens (M, N multiples of 256) takes these tiles rather
// than the 256-wide ones.  Measured times in us (256 / 128 / 64): 2048 x 2048 of 4096 tokens
// 78 / 35 / 66, 1024 x 4096 of 8192 139 / 62 / 129, 768 x 768 of 8192 140 / 47 / 27, 5632 x 2048
// of 4096 85 / 92 / 155, 4096 x 4096 of 2048 60 / 66 / 94, 256 x 256 of 128 12 / 7.5 / 7.6.
bool wgrad_takes_tiles(int64_t M, int64_t N, int64_t K) {
    double c;
    best_cfg(false, M, N, K, 1, &c);
    return c < tile_cost(256, 2, (M / 256) * (N / 256), K / TBK);
}

}  // namespace msr

using namespace msr;

extern "C" int msr_tile_gemm(int32_t product, int32_t tile, int32_t stages, const uint16_t *p, const uint16_t *q,
                             uint16_t *d, int64_t batch, int64_t m, int64_t n, int64_t k, float alpha, float beta,
                             float diag, const float *rvec, float *resid, uint32_t seed, int32_t noise_mode,
                             msr_stream_t stream) {
    const bool sym = product == TILE_A || product == TILE_B;
    const int64_t lim = 1 << 14;   // operands below 2 GiB
    if (product < TILE_A || product > TILE_W || !p || !d || (!sym && !q) || batch < 1 || batch > 1024 || m < 1 || m > lim ||
        n < 1 || n > lim || k < 1 || k > lim || (sym && m != n) || ((product == TILE_B || product == TILE_X) && (k != m || !rvec)) ||
        (sym && !resid) || (product == TILE_W && batch != 1) || (noise_mode != NOISE_TRITON && noise_mode != NOISE_PHILOX8)) {
        set_error("msr_tile_gemm: bad arguments");
        return MSR_ERR_ARG;
    }
    if (!aligned(p, 16) || !aligned(q, 16) || !aligned(d, 16)) { set_error("msr_tile_gemm: operands must be 16-byte aligned"); return MSR_ERR_ALIGN; }
    const size_t np = 2 * (size_t)batch * m * k, nq = sym ? 0 : 2 * (size_t)batch * k * n, nd = 2 * (size_t)batch * m * n;
    auto touch = [&](const void *x, size_t nx) { return x && (uintptr_t)x < (uintptr_t)d + nd && (uintptr_t)d < (uintptr_t)x + nx; };
    if (touch(p, np) || touch(q, nq)) { set_error("msr_tile_gemm: d overlaps an operand"); return MSR_ERR_OVERLAP; }
    TileArgs a = {};
    const bool w = product == TILE_W;
    a.P = p; a.ldp = w ? m : k; a.sP = m * k;
    a.Q = sym ? p : q; a.ldq = sym ? k : n; a.sQ = sym ? m * k : k * n;
    a.C = product == TILE_B ? p : nullptr; a.ldc = k; a.sC = m * k;
    a.D = d; a.ldd = n; a.sD = m * n;
    a.M = (int)m; a.N = (int)n; a.K = (int)k;
    a.alpha = alpha; a.beta = beta; a.diag = diag;
    a.rvec = rvec; a.resid = resid; a.sv = m;
    a.ns.key = seed_key(seed, 0);
    const hipStream_t s = (hipStream_t)stream;
    if (tile == 64 && stages == 4) return launch_tiles<64, 4>(product, TILE_WS, noise_mode, a, batch, nullptr, s);
    if (tile == 64 && stages == 2) return launch_tiles<64, 2>(product, TILE_WS, noise_mode, a, batch, nullptr, s);
    if (tile == 128 && stages == 4) return launch_tiles<128, 4>(product, TILE_WS, noise_mode, a, batch, nullptr, s);
    if (tile == 128 && stages == 2) return launch_tiles<128, 2>(product, TILE_WS, noise_mode, a, batch, nullptr, s);
    set_error("msr_tile_gemm: no kernel of tile %d with %d stages", (int)tile, (int)stages);
    return MSR_ERR_ARG;
}
