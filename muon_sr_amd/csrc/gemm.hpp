// Pieces shared by the two matrix-product kernels (ns_gemm.hip: 256 x 256 tiles;
// tile_gemm.hip: 64 x 64 and 128 x 128 tiles): fragment types, the fused Muon
// apply, counted waits and the Newton-Schulz epilogues.
#pragma once

#include "common.hpp"
#include "vecio.hpp"

namespace msr {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int NXCD = 8;

// Wait until at most N vector memory operations of this wave are outstanding
// (s_waitcnt: vmcnt in bits 3:0 and 15:14; expcnt and lgkmcnt at their maxima).
// Vector memory operations complete in issue order, so every operation issued
// before the last N has completed.
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Muon apply fused into the store of the last Newton-Schulz product
// (msr_muon_ns_apply): matrix b of a launch updates params p[b] with seed[b].
constexpr int APPLY_MAX = 128;   // matrices per launch (kernel-argument table)
struct ApplyTab {
    uint16_t *p[APPLY_MAX];
    uint32_t seed[APPLY_MAX];
    const uint16_t *inject;      // uint16 [count][numel] of this launch (NOISE_INJECT), or null
    int64_t numel;
    float lr, decay, scale;      // decay = 1 - lr * wd
};

// p[off + j] <- SR(p*(1 - lr*wd) - lr*(f32(u_j)*scale)) for the j < valid bf16 values u
// (packed in u[4]) of one 8-element chunk: the arithmetic and noise of
// muon_apply_kernel (muon_sr/triton_muon_sr.py:53-80); off is the element index in p.
// vec: the chunk is 16-byte aligned and off a multiple of 8.
// The parameter chunk of apply_chunk (loaded ahead so that the loads of a thread's
// chunks overlap).
__device__ __forceinline__ u32x4_t apply_load(const uint16_t *P, int64_t off, int valid, bool vec) {
    if (vec && valid == 8) return ld_nt4(P + off);
    uint32_t wp[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if (j < valid) wp[j >> 1] |= (uint32_t)P[off + j] << (16 * (j & 1));
    return u32x4_t{wp[0], wp[1], wp[2], wp[3]};
}

template <int MODE>
__device__ __forceinline__ void apply_chunk(const ApplyTab &ap, uint16_t *P, const Noise &ns, int64_t off, int valid,
                                            bool vec, const uint32_t u[4], u32x4_t pw) {
    const uint32_t wp[4] = {pw.x, pw.y, pw.z, pw.w};
    uint32_t r[8];
    if (vec && valid == 8) {
        noise8<MODE>(ns, off, 8, r);
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = j < valid ? noise1<MODE>(ns, off + j) : 0u;
    }
    uint32_t op[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float uf = (j & 1) ? bf16_hi(u[j >> 1]) : bf16_lo(u[j >> 1]);
        const float pf = (j & 1) ? bf16_hi(wp[j >> 1]) : bf16_lo(wp[j >> 1]);
        const float t1 = uf * ap.scale;                                   // :70
        float pj = pf * ap.decay;                                         // :72
        pj = pj - ap.lr * t1;                                             // :73
        op[j] = sr_bf16(pj, r[j]);                                        // :75-80
    }
    if (vec && valid == 8) {
        st_nt4(P + off, u32x4_t{pack2(op[0], op[1]), pack2(op[2], op[3]), pack2(op[4], op[5]), pack2(op[6], op[7])});
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j < valid) P[off + j] = (uint16_t)op[j];
    }
}

// Epilogues of the Newton-Schulz products.  The iteration keeps A, B' and X
// in bf16 between products; the diagonals of A and B' are the largest
// entries of those matrices (B' carries a = 3.4445 on it), so their bf16
// rounding is the largest rounding error of the iteration.  These epilogues
// carry the rounding residual of every diagonal element in fp32 to the next
// product:
//   EPI_A  A = alpha X X^T:  rho[m] = A_mm - bf16(A_mm)                 (resid)
//   EPI_B  B' = alpha (A A) + beta A + diag I with the diagonal corrected
//          for rho to first order, B'_mm += rho[m] (beta + 2 alpha A_mm)
//          (d/dA_mm of beta A_mm + alpha (A A)_mm with A_mm dominant):
//          r[m] = B'_mm - bf16(B'_mm)                                   (resid)
//   EPI_X  X' = alpha (B' X + bf16(r[m]) X), the second term as MFMAs of the diagonal
//          block (see mmdiag)
// EPI_NONE is the plain alpha P Q^T + beta C + diag I of the diagnostic GEMMs.
enum : int { EPI_NONE = 0, EPI_A = 1, EPI_B = 2, EPI_X = 3 };

}  // namespace msr
