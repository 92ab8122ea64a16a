// Launch interface of the 64 x 64 / 128 x 128 tile products (tile_gemm.hip).
#pragma once

#include "gemm.hpp"

namespace msr {

// D = alpha P Q^T (+ beta C + diag I) of `batch` matrices; extents are multiples of 64,
// and each operand matrix spans less than 2 GiB.
struct TileArgs {
    const uint16_t *P; int64_t ldp, sP;
    const uint16_t *Q; int64_t ldq, sQ;
    const uint16_t *C; int64_t ldc, sC;
    uint16_t *D; int64_t ldd, sD;
    uint16_t *DT; int64_t lddt, sDT;
    int M, N, K;
    int Mv, Nv;              // bounded stores: m < Mv, n < Nv
    float alpha, beta, diag;
    const float *alpha_b;    // per-matrix alpha (replaces alpha when not null)
    float *resid;            // PR_A, PR_B: fp32 rounding residuals of the diagonal, [batch][sv]
    const float *rvec;       // PR_B: A's residuals; PR_X: B''s residuals, [batch][sv]
    int64_t sv;
    int d_vec, dt_vec;       // D / DT (or parameter) rows allow 16-byte accesses
    int zero_init;           // PR_W: the accumulator reads as zero
    Noise ns;                // PR_W: noise of element offset m * ldd + n
    int tiles_m, tiles_n, tiles, total;   // set by the launch
};

constexpr int64_t TILE_CUS = 256;   // work-groups that run at once, one per CU

enum TileProd : int { TILE_A = 0, TILE_B = 1, TILE_X = 2, TILE_W = 3 };
enum TileOut : int { TILE_WS = 0, TILE_D = 1, TILE_DT = 2, TILE_PD = 3, TILE_PT = 4 };

// mode: noise mode of TILE_PD / TILE_PT (with `tab`, at most APPLY_MAX matrices) and TILE_W.
// The tile (64 or 128 wide, where the extents allow it) is the one with the least estimated time.
int launch_tile_gemm(int prod, int out, int mode, const TileArgs &a, int64_t batch, const ApplyTab *tab, hipStream_t s);

// What a Newton-Schulz call of `batch` m x n matrices (m <= n) pads to: 64 or 128 (these tiles),
// or 256 (ns_gemm.hip's kernel); and whether a weight gradient M x N over K tokens takes these tiles.
int ns_tile_choice(int64_t batch, int64_t m, int64_t n);
bool wgrad_takes_tiles(int64_t M, int64_t N, int64_t K);

}  // namespace msr
