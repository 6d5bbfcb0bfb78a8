// What the dense-layer kernels share (gemm.hip, gemm_rows.hip): the epilogue's
// operands and arithmetic, the FLOP tally.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>

#include "split_bf16.h"

namespace pet_gemm {

using pet_split::f4;
using pet_split::u2;
using pet_split::u4;

// The hardware's exp and reciprocal, with one Newton step on the reciprocal
// (its own ulp of error has a mean that a model's activations add up), except
// where that is 0 (x below -88): the step would make NaN of it.
__device__ __forceinline__ float sig_fast(float x) {
  const float d = 1.0f + __expf(-x), r = __builtin_amdgcn_rcpf(d), n = fmaf(fmaf(-d, r, 1.0f), r, r);
  return r == 0.f ? r : n;
}

struct Epi {
  const float* row_scale = nullptr;  // [M]
  const float* bias = nullptr;       // [N]
  const float* cin = nullptr;        // [M, N] (ld ldcin), scaled by beta
  int64_t ldcin = 0;
  float beta = 0.f;
  float* pre = nullptr;              // [M, N] (ld ldpre): v before the activation
  int64_t ldpre = 0;
  int act = 0;                       // 0 none, 1 SiLU, 2 SwiGLU (C has N/2 columns),
                                     // 3 / 4 the backward of SiLU / SwiGLU (below)
  // Block pairs in place of C (the row kernels only): the output row i as
  // fp16 pairs in pair_act_kernel's layout (kgo k groups of 8 a row, each
  // group's hi then lo 16 bytes), scaled per (row, column tile) -- the tile's
  // output columns are one K block of the product that reads them -- with the
  // block's inverse scale at pinv[block ldinv + i].
  u4* pout = nullptr;
  float* pinv = nullptr;
  int64_t ldinv = 0;
  int kgo = 0;
};

// FLOPs (2 M N K) of the products this library's dense kernels have launched,
// by the instructions that run them: 0 the fp32 fused kernel (fp32 matrix
// cores), 1 split-fp32 as three bf16 parts (six bf16 products), 2 fp16 pairs
// (three fp16 products), 3 the three-part kernels (five fp16 products). A
// measurement aid, process-wide (pet_gemm_flop_tally).
extern std::atomic<uint64_t> g_flops[4];  // gemm.hip
inline void tally(int cls, int64_t M, int64_t N, int64_t K) {
  g_flops[cls].fetch_add(uint64_t(2) * uint64_t(M) * uint64_t(N) * uint64_t(K), std::memory_order_relaxed);
}

// The K loop's barrier: no memory fence, since any fence, even one on LDS
// alone, makes the compiler wait for every global-to-LDS load in flight (the
// prefetches too). The loop's own vmcnt wait before it covers the step's
// loads; an explicit lgkmcnt(0) wait (vmcnt and expcnt left at their maxima)
// makes every LDS read a wave issued in the step before complete before it
// passes, so no wave's global_load_lds can overwrite a stage another is still
// reading, whatever order the compiler gives the products; the empty asm
// keeps the compiler from moving memory accesses across it.
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}


// 16 bytes a lane from global memory into LDS, a wave's 64 lanes filling
// dst .. dst + 1 KB in lane order (dst wave-uniform). A device function: the
// builtin, called in a lambda of a kernel, stops the host side from emitting
// the kernel.
__device__ __forceinline__ void ring_load(const u4* src, u4* dst) {
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}

// s_waitcnt on the vector-memory counter alone (gfx9 encoding: vmcnt in bits
// 3:0 and 15:14; expcnt 7 and lgkmcnt 15 wait for nothing).
template <int n>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}

}  // namespace pet_gemm

// gemm_rows.hip: C = epilogue(A B^T) from three-part weights (pet_gemm_pair_weights)
int pet_gemm_nt_p3(int M, int N, int K, const float* A, int64_t lda, const void* Bp, float* C, int64_t ldc,
                   const pet_gemm::Epi& e, hipStream_t st);
// ... and on the row kernels, P parts of weights a value; as: how A comes
enum { kRowsOnline = 0, kRowsExact = 1, kRowsPairs = 2 };
int pet_gemm_nt_rows(int M, int N, int K, const void* A, int64_t lda, int as, int kb, const void* Bp, int P, float* C,
                     int64_t ldc, const pet_gemm::Epi& e, hipStream_t st, int cfg);
