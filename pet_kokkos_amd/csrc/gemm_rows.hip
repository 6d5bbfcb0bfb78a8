// The dense layers' row-streaming product on gfx950: C = epi(A B^T), A [M, K]
// activations, B [N, K] weights split once into P fp16 parts a value (2: hi and
// lo; 3: hi, mid and lo, the weight exactly), the sums in fp32 on the
// 16x16x32 f16 matrix instruction (three products a value for two parts, five
// for three).
//
// What bounds it, and the split that follows. Both operands are staged a K step
// of 32 at a time in an LDS ring by loads straight into LDS (A's rows as fp32,
// split in registers by the wave that reads them; a load of 16 rows of a
// fragment into registers meets 16 cache lines a quarter wave, 20 to 25% slower),
// one barrier a step, conflict-free swizzles. A wave of 16 TM x 64 results reads
// 2 TM + 4 P fragments for 4 TM (2 P - 1) instructions: large tiles are bound by the
// matrix unit and its clock (1.65 to 1.88 PFLOP/s with random data), small ones
// by LDS and the chain of a step, so the tile is as large as still fills the
// chip (the dispatch at the end). The weights are the instruction's first
// operand, so a lane's results belong to its own row c (scales are undone in the
// lane), and the columns of four tiles are interleaved (col_of) so that a lane
// holds sixteen consecutive columns.
//
// A is split with a power-of-two scale a row. Three forms (AS):
//   kOnline: the scale follows the row as it streams: it puts the largest |x|
//     so far of the row's first step in [2^11, 2^12), and a later value past
//     2^15 lowers it (rare: eight times the first 32 values' largest; the
//     accumulators are then rescaled by the exact power of two). A value keeps
//     22 significand bits down to 2^-14 of the row's largest (under the row's own
//     scale, kExact, to 2^-17), and below an error of at most 2^-36 of it (2^-39).
//   kExact: the row's largest |x| is found first, in a pass over the wave's rows
//     (whose second reading comes from cache): the bits of the pair rows
//     (pair_act_kernel) read in form kPairs.
//   kPairs: A already as fp16 pairs with a scale per (row, K block): a step's
//     sum, made from zero at its block's own scale, is brought to the row's
//     smallest scale in fp32 as it is added, so that a block far below the row's
//     largest keeps all of its bits.
// In one kernel a row's results depend on that row alone, and repeat bit for bit.
// The tile kernel's shapes and the strip share one order of sums; the kernel that
// splits K over its waves (three parts, K from 256, few rows) has its own.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "../../include/pet_model.h"
#include "attn_common.h"
#include "gemm_common.h"
#include "split_bf16.h"

namespace pet_gemm {

using pet_attn::max_g;
using pet_split::mfma_h;

enum { kOnline = kRowsOnline, kExact = kRowsExact, kPairs = kRowsPairs };  // A
enum { kVec = 0, kAny = 1, kBlocks = 2 };  // the output: fp32 of a width a multiple of 4, of any width, block pairs

namespace {

// The largest |x| of eight floats in two registers of four.
__device__ __forceinline__ float amax8(const u4& x, const u4& y) {
  float m;
  asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(m) : "v"(x[0]), "v"(x[1]), "v"(x[2]));
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(x[3]), "v"(y[0]));
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(y[1]), "v"(y[2]));
  asm("v_max3_f32 %0, |%1|, |%1|, %0" : "+v"(m) : "v"(y[3]));
  return m;
}

// Eight floats (x then y) times s, a power of two, as fp16 to nearest, in
// place: the hi parts in x, the lo parts (of the remainders, exact) in y.
__device__ __forceinline__ void split8x(u4& x, u4& y, float s) {
#pragma clang fp contract(off)
  const u4 in[2] = {x, y};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float a = __uint_as_float(in[j >> 1][2 * (j & 1)]), b = __uint_as_float(in[j >> 1][2 * (j & 1) + 1]);
    const pet_split::h2v h = {(_Float16)fmaf(a, s, 0.f), (_Float16)fmaf(b, s, 0.f)};
    const pet_split::h2v lo = {(_Float16)fmaf(a, s, -float(h[0])), (_Float16)fmaf(b, s, -float(h[1]))};
    x[j] = __builtin_bit_cast(unsigned, h);
    y[j] = __builtin_bit_cast(unsigned, lo);
  }
}

// A row's running scale sa (kOnline) once |x| up to m, this lane's share of the
// row, comes past the limit lim it holds: the new scale and limit, and the
// factor onto them of sums made under the old (0 at the first).
__device__ __forceinline__ float outgrow(float m, float& sa, float& lim) {
  const float rm = max_g(m);
  float f = 1.f;
  if (rm > lim) {  // (an infinity: any scale, special_rows makes the row's results)
    const int k = min(12 - __builtin_amdgcn_frexp_expf(rm), 126);
    f = __builtin_amdgcn_ldexpf(lim, k - 15);
    sa = __builtin_amdgcn_ldexpf(1.f, k), lim = fminf(__builtin_amdgcn_ldexpf(1.f, 15 - k), pet_split::kFltMax);
  }
  return f;
}

// Rows of A that hold an infinity or a NaN. Split into parts an infinity makes
// NaN of its row (inf - inf), every column alike; such a row's results are made
// again after its K loop, on the matrix cores, from its infinities and NaNs
// alone (no finite value has a say) and the weights' signs: infinite times the
// weight's sign, NaN against a zero weight or where both signs meet, as fp32
// gives. A weight's first part carries its sign, unless the weight itself is
// infinite: then the last (pair3). The check is one ballot a tile; kept in the K
// loop, where the rows' scales are, it cost 1 to 2% of the model's layers.
__device__ __forceinline__ unsigned special_half(unsigned x) {
  const unsigned m = x & 0x7fffffffu;
  return m < 0x7f800000u ? 0u : (x >> 16 & 0x8000u) | (m > 0x7f800000u ? 0x7e00u : 0x7c00u);
}
// acc: the row's tiles; row(c, s): this lane's 8 floats of step s; weight(c, b, s,
// hi, lo): its parts of tile b.
template <int TN, class R, class W>
__device__ __forceinline__ void special_rows(f4 (&acc)[TN], int steps, int c, R&& row, W&& weight) {
  const bool bad = acc[0][0] != acc[0][0];
  if (__builtin_amdgcn_ballot_w64(bad) == 0) return;
  // the lane's row and column of a tile, c, past the compiler's sight: the
  // addresses are made here and not held in registers by the callers' loops
  asm volatile("" : "+v"(c));
#pragma unroll
  for (int b = 0; b < TN; ++b) {
    f4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = 0; s < steps; ++s) {
      const u4* p = row(c, s);
      const u4 x = p[0], y = p[1];
      const u4 v = {special_half(x[0]) | special_half(x[1]) << 16, special_half(x[2]) | special_half(x[3]) << 16,
                    special_half(y[0]) | special_half(y[1]) << 16, special_half(y[2]) | special_half(y[3]) << 16};
      u4 h, lo;
      weight(c, b, s, h, lo);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned lh = h[j] & 0x7fffu ? h[j] : lo[j], hh = h[j] & 0x7fff0000u ? h[j] : lo[j];
        h[j] = (lh & 0xffffu) | (hh & 0xffff0000u);
      }
      t = mfma_h(h, v, t);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[b][e] = bad ? t[e] : acc[b][e];
  }
}

// A step of 32 is summed from zero and added to the running sum; with three-part
// weights the rows of odd steps are negated and their sums subtracted. The
// matrix instruction rounds its sums, and each product as it aligns it, toward
// minus infinity: summed in place, an error of 1.6e-7 (K 128) to 3.2e-7 (K 512) of
// a result with a mean of -1.6e-8 to -3.3e-8 that a model sums over its atoms
// (random operands on MI355X; the fp32 matrix core 2.6e-7 to 5.1e-7, mean 0). So it
// is 0.9e-7 to 1.3e-7, and the steps of either sign cancel the mean. Two-part
// weights come with their odd steps negated where the mean adds up (their
// inverse scales are negative then): the energies of 64 structures on a 512-wide
// model are 5.4e-6 eV an atom (rms) from float64, 9.3e-6 with steps of one sign.
__device__ __forceinline__ void add_step(f4& acc, const f4& t, float sg) {
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = fmaf(t[e], sg, acc[e]);
}

// The tile column of LDS row r: fragment row 4 q + e of tile 4 b + s (r = 64 b +
// 16 s + 4 q + e) is column 64 b + 16 q + 4 s + e, so that a lane's results of
// four tiles are sixteen consecutive columns.
__device__ __forceinline__ int col_of(int r) { return (r & ~63) | ((r & 12) << 2) | ((r & 48) >> 2) | (r & 3); }

// The slot of chunk q (of 4 P; A's rows as P = 2) in LDS row r: with rows of
// 128 bytes an XOR by bits 1 and 3 of r, with 192 (P = 3) a rotation by two for
// r with bit 3. Measured on MI355X over every XOR by bits of r and every such
// rotation: a 16-byte read of 16 rows by four k groups at the conflict-free
// rate of consecutive lanes, 5.8 cycles (8.5 with an odd pitch or bits 2 and 3
// in the XOR, 16 with neither).
template <int P>
__device__ __forceinline__ int swizzle(int q, int r) {
  if constexpr (P == 2) return q ^ (((r >> 1) & 1) | ((r >> 1) & 4));
  const int x = q + ((r >> 2) & 2);
  return x < 12 ? x : x - 12;
}
template <int P>
__device__ __forceinline__ int unswizzle(int x, int r) {
  if constexpr (P == 2) return swizzle<2>(x, r);
  const int q = x - ((r >> 2) & 2);
  return q < 0 ? q + 12 : q;
}

// A workgroup's tile: WR x WC waves of 16 TM rows by 16 TN columns, and its LDS.
template <int TM, int TN, int WR, int WC, int P>
struct RowsTile {
  static constexpr int BM = 16 * TM * WR, BN = 16 * TN * WC, CH = 4 * P;
  static constexpr int STAGE = BM * 8 + BN * CH;  // 16-byte chunks
  static constexpr int ST = STAGE <= 1280 ? 3 : 2;
  static constexpr size_t bytes = size_t(ST) * STAGE * 16 + BM * 4;
};
constexpr int rows_waves(int TM, int TN) { return TM * TN >= 16 ? 2 : TM * TN >= 8 ? 3 : 4; }

// A 4 x 4 transpose over each quad of lanes: x[r] of lane i becomes x[i] of
// lane r.
__device__ __forceinline__ void quad_transpose(float (&x)[4]) {
  const bool b0 = threadIdx.x & 1, b1 = threadIdx.x & 2;
  auto dpp = [](float v, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  using x1 = std::integral_constant<int, 0xb1>;  // quad_perm 1, 0, 3, 2
  using x2 = std::integral_constant<int, 0x4e>;  // quad_perm 2, 3, 0, 1
  // (every exchange before its select: all lanes take part)
  const float t0 = dpp(x[0], x1{}), t1 = dpp(x[1], x1{}), t2 = dpp(x[2], x1{}), t3 = dpp(x[3], x1{});
  const float y0 = b0 ? t1 : x[0], y1 = b0 ? x[1] : t0, y2 = b0 ? t3 : x[2], y3 = b0 ? x[3] : t2;
  const float u0 = dpp(y0, x2{}), u1 = dpp(y1, x2{}), u2 = dpp(y2, x2{}), u3 = dpp(y3, x2{});
  x[0] = b1 ? u2 : y0, x[1] = b1 ? u3 : y1, x[2] = b1 ? y2 : u0, x[3] = b1 ? y3 : u1;
}

// Lane i of this lane's quad's x.
template <int i>
__device__ __forceinline__ int quad_lane(int x) {
  return __builtin_amdgcn_update_dpp(0, x, 0x55 * i, 0xf, 0xf, true);
}

// n consecutive columns of an epilogue operand. Every address is a float's: the
// 4-byte alignment of the vectors costs nothing on gfx950 (an access of 16 bytes
// at any of them is one instruction). Element by element, outputs that are not
// 16-byte aligned took 1.3 to 2.7 times as long (100000 x 128 x 128 on MI355X: 72 us
// against 30), and in 256 x 256 tiles, their accumulators in scratch, 12 times
// (62291 x 512 x 1024 from pairs: 2240 against 181). ANY (the width no multiple of
// 4): the last chunk's `left` columns one by one.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
template <bool ANY, int n>
__device__ __forceinline__ void get_cols(const float* p, float (&x)[n], int left) {
  if (!ANY || left >= n) {
#pragma unroll
    for (int e = 0; e < n; e += 4) {
      const f4u q = *reinterpret_cast<const f4u*>(p + e);
      x[e] = q[0], x[e + 1] = q[1], x[e + 2] = q[2], x[e + 3] = q[3];
    }
  } else {
#pragma unroll
    for (int e = 0; e < n; ++e) x[e] = p[min(e, left - 1)];
  }
}
template <bool ANY, int n>
__device__ __forceinline__ void put_cols(float* p, const float (&x)[n], int left) {
  if (!ANY || left >= n) {
    if constexpr (n == 2) *reinterpret_cast<f2u*>(p) = f2u{x[0], x[1]};
#pragma unroll
    for (int e = 0; e + 4 <= n; e += 4) *reinterpret_cast<f4u*>(p + e) = f4u{x[e], x[e + 1], x[e + 2], x[e + 3]};
  } else {
#pragma unroll
    for (int e = 0; e < n; ++e)
      if (e < left) p[e] = x[e];
  }
}

}  // namespace

// The epilogue of a wave's TM x TN tiles: acc times the row's inverse scale ia
// and the columns' inv_b (a row past 2^64 apart from that factor of its scale,
// which follows inv_b: sums of 2^30 and more times a scale up to 2^116 can pass the
// range of a float where the result does not; FAR: three-part weights, whose
// products ran in fp32, and block pairs out, whose kernel spills 69 registers
// with it and 101 without), then epi_elem's arithmetic in its order. A lane holds
// sixteen consecutive columns of its row c; a 4 x 4 transpose of those 16-byte
// chunks over each quad of lanes makes an instruction's quad cover 64 bytes of
// one row (r of the four), so a quarter of a wave meets 4 rows' lines, not 16:
// stores of 16 bytes to 16 rows bounded the products of short K with an
// activation (26670 x 512 x 128 with SiLU and its kept input on MI355X: 35 us
// without the transpose, 31 with it).
template <int TM, int TN, int OUT, bool FAR>
__device__ __forceinline__ void rows_epilogue(const f4 (&acc)[TM][TN], const float (&ia)[TM], const float* inv_b,
                                              int m0, int n0, int c, int g, int M, int N, float* C, int64_t ldc,
                                              const Epi& epi) {
  static_assert(TN % 4 == 0, "64 columns at a time");
  constexpr bool ANY = OUT == kAny;
  const int r0 = m0 + (c & 12), j0 = n0 + 16 * g + 4 * (c & 3);  // this lane's first row and column
  auto run = [&](auto act) {
    constexpr int ACT = decltype(act)::value, NG = TN / 4;
    constexpr int Z = ACT == 4 ? 8 : 4, R = ACT == 2 ? 2 : ACT == 4 ? 8 : 4;  // values read and written a chunk
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      const bool far = FAR && ia[a] > 0x1p64f, afar = __builtin_amdgcn_ballot_w64(far) != 0;
      const float ia1 = far ? ia[a] * 0x1p-64f : ia[a];
      float res[OUT == kBlocks ? NG : 1][4][R], mx[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < NG; ++b) {
        // (a lane past the last column reads the last ones and writes nothing)
        const int j = min(j0 + 64 * b, ANY ? N - 1 : N - 4), left = N - j;
        const bool in = OUT == kBlocks || j0 + 64 * b < N;
        constexpr int ZC = ACT == 4 ? 2 : 1;  // cin's and the bias's columns a column
        // the chunk's operands, four rows' together
        float z[4][Z], ib[4], bb[Z];
        const bool hz = ACT >= 3 || epi.cin != nullptr;
        if (hz)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            get_cols<ANY>(epi.cin + int64_t(min(r0 + 16 * a + r, M - 1)) * epi.ldcin + ZC * j, z[r], ZC * left);
          }
        get_cols<ANY>(inv_b + j, ib, left);
        if (epi.bias) get_cols<ANY>(epi.bias + ZC * j, bb, ZC * left);
        float v[4][4];  // [element][row]
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int s = 0; s < 4; ++s) v[e][s] = acc[a][4 * b + s][e] * ia1;
          quad_transpose(v[e]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = r0 + 16 * a + r;
          const bool live = in && i < M;
          float u[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) u[e] = v[e][r] * fabsf(ib[e]);  // (the sign: add_step)
          if (afar) {
            const int f = far;
            const float p = (r == 0 ? quad_lane<0>(f) : r == 1 ? quad_lane<1>(f) : r == 2 ? quad_lane<2>(f) : quad_lane<3>(f)) ? 0x1p64f : 1.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) u[e] *= p;
          }
          float (&o)[R] = res[OUT == kBlocks ? b : 0][r];
          if constexpr (ACT == 3) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float x = z[r][e] + (epi.bias ? bb[e] : 0.f), sg = sig_fast(x);
              o[e] = u[e] * (sg * (1.0f + x * (1.0f - sg)));
            }
          } else if constexpr (ACT == 4) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float y = z[r][2 * e] + (epi.bias ? bb[2 * e] : 0.f);
              const float sg = sig_fast(z[r][2 * e + 1] + (epi.bias ? bb[2 * e + 1] : 0.f));
              o[2 * e] = u[e] * sg, o[2 * e + 1] = u[e] * y * sg * (1.0f - sg);
            }
          } else {
            if (epi.row_scale) {
              const float rs = epi.row_scale[min(i, M - 1)];
#pragma unroll
              for (int e = 0; e < 4; ++e) u[e] *= rs;
            }
            if (epi.bias)
#pragma unroll
              for (int e = 0; e < 4; ++e) u[e] += bb[e];
            if (epi.cin)
#pragma unroll
              for (int e = 0; e < 4; ++e) u[e] += epi.beta * z[r][e];
            if (epi.pre && live) put_cols<ANY>(epi.pre + int64_t(i) * epi.ldpre + j, u, left);
            if constexpr (ACT == 2) {
              o[0] = u[0] * sig_fast(u[1]), o[1] = u[2] * sig_fast(u[3]);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) o[e] = epi.act == 1 ? u[e] * sig_fast(u[e]) : u[e];
            }
          }
          if constexpr (OUT != kBlocks) {
            if (live) put_cols<ANY>(C + int64_t(i) * ldc + (ACT == 2 ? j / 2 : ZC * j), o, ACT == 2 ? left / 2 : ZC * left);
          } else {
#pragma unroll
            for (int e = 0; e < R; ++e) mx[r] = fmaxf(mx[r], fabsf(o[e]));
          }
        }
        if constexpr (OUT != kBlocks) asm volatile("" ::: "memory");  // (the next chunk's operands are not held as well)
      }
      if constexpr (OUT == kBlocks) {
        // each row's 128 columns of the product scaled by their own power of
        // two, as fp16 pairs: groups of 8 outputs hi then lo, 16 bytes each
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int m = __float_as_int(mx[r]);  // |values|: the bit patterns order as the values
          m = max(m, __builtin_amdgcn_update_dpp(0, m, 0xb1, 0xf, 0xf, true));
          m = max(m, __builtin_amdgcn_update_dpp(0, m, 0x4e, 0xf, 0xf, true));
          const float sc = pet_split::block_scale(max_g(__int_as_float(m)));
          const int i = r0 + 16 * a + r;
          if (i < M) {
            unsigned* rowp = reinterpret_cast<unsigned*>(epi.pout + int64_t(i) * epi.kgo * 2);
#pragma unroll
            for (int b = 0; b < NG; ++b) {
              const int jo = (ACT == 2 ? 1 : ACT == 4 ? 4 : 2) * (j0 + 64 * b) / 2;  // the first output
              unsigned h[R / 2], lw[R / 2];
#pragma unroll
              for (int e = 0; e < R / 2; ++e)
                pet_split::pair2(res[b][r][2 * e] * sc, res[b][r][2 * e + 1] * sc, h[e], lw[e]);
              unsigned* q = rowp + (jo / 8) * 8 + (jo % 8) / 2;
              if constexpr (R == 2) q[0] = h[0], q[4] = lw[0];
              if constexpr (R == 4) *reinterpret_cast<u2*>(q) = u2{h[0], h[1]}, *reinterpret_cast<u2*>(q + 4) = u2{lw[0], lw[1]};
              if constexpr (R == 8) {
                *reinterpret_cast<u4*>(q) = u4{h[0], h[1], h[2], h[3]};
                *reinterpret_cast<u4*>(q + 4) = u4{lw[0], lw[1], lw[2], lw[3]};
              }
            }
            if (g == 0 && (c & 3) == 0) epi.pinv[int64_t(n0 / 128) * epi.ldinv + i] = 1.f / sc;
          }
        }
        asm volatile("" ::: "memory");
      }
    }
  };
  if (epi.act == 2) run(std::integral_constant<int, 2>{});
  else if (epi.act == 3) run(std::integral_constant<int, 3>{});
  else if (epi.act == 4) run(std::integral_constant<int, 4>{});
  else run(std::integral_constant<int, 0>{});
}

// The tile kernel. From pairs it takes the place of a kernel with 128 x 128 tiles
// of eight waves that read 12 operand fragments for 24 instructions a step and met
// LDS bank conflicts (MI355X, 62291 rows: 512 x 2048 424 -> 337 us, 512 x 1024 237 -> 176,
// 2048 x 512 424 -> 408); from fp32 rows, of one that split them on their way into LDS
// (26670 x 128 x 1024: 58.5 -> 48.6).
template <int TM, int TN, int WR, int WC, int P, int AS, int OUT>
__global__ void __launch_bounds__(64 * WR * WC) __attribute__((amdgpu_waves_per_eu(rows_waves(TM, TN))))
gemm_rows_kernel(int M, int N, int K, const void* A, int64_t lda, const u4* B, float* C, int64_t ldc, Epi epi, int kbs,
                 int win) {
  using Sh = RowsTile<TM, TN, WR, WC, P>;
  constexpr int BM = Sh::BM, BN = Sh::BN, CH = Sh::CH, ST = Sh::ST, NW = WR * WC;
  constexpr int TG = TN < 4 / TM ? TN : TM >= 4 ? 1 : 4 / TM;  // tiles whose products interleave
  constexpr int NG = TN / TG;
  static_assert(TN % 4 == 0 && (P == 2 || P == 3) && TN % TG == 0 && (NG == 1 || NG % 2 == 0), "64 columns, whole groups");
  constexpr int LA = BM / 8 / NW, NIB = BN * CH / 64, LB = (NIB + NW - 1) / NW;  // a wave's loads a stage
  static_assert(LA * 8 * NW == BM, "whole loads");
  extern __shared__ u4 lds[];  // ST stages: BM rows of A's 8 chunks of 16 bytes, BN rows of B's CH; then BM floats
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, c = l & 15, g = l >> 4;
  const int KG = K / 8, steps = K / 32;
  // XCD x takes a contiguous run of tiles, windows of `win` row blocks swept
  // column tile by column tile (the weights' strips and the rows in flight
  // share its L2)
  const int NT = (N + BN - 1) / BN, RBk = (M + BM - 1) / BM;
  const int t = pet_attn::xcd_item(blockIdx.x, gridDim.x);
  const int wi = t / (win * NT), wr_ = min(win, RBk - wi * win), within = t - wi * win * NT;
  const int mt = (wi * win + within % wr_) * BM, nt = (within / wr_) * BN;  // the tile's corner
  const int ar = 16 * TM * (w / WC), bc = 16 * TN * (w % WC);              // the wave's rows and columns in it
  const int m0 = mt + ar, n0 = nt + bc;

  // ---- this lane's source of each of the wave's stage loads. A: LDS chunk e,
  // slot e % 8 of row e / 8; B: slot e % CH of row e / CH (column col_of(row))
  const char* pa[LA];
  const int64_t arow = 4 * (AS == kPairs ? int64_t(K) : lda);
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int e = 64 * (w * LA + q) + l, r = e >> 3;
    pa[q] = static_cast<const char*>(A) + min(mt + r, M - 1) * arow + 16 * swizzle<2>(e & 7, r);
  }
  const u4* pb[LB];
#pragma unroll
  for (int q = 0; q < LB; ++q) {
    const int e = min(64 * (w + NW * q) + l, BN * CH - 1), r = e / CH;
    pb[q] = B + int64_t(min(nt + col_of(r), N - 1)) * KG * P + unswizzle<P>(e - r * CH, r);
  }
  auto issue = [&](int s, int stage) {  // (past the last step: its chunks again, unused)
    const int k = min(s, steps - 1);
    u4* dst = lds + stage * Sh::STAGE;
#pragma unroll
    for (int q = 0; q < LA; ++q) ring_load(reinterpret_cast<const u4*>(pa[q] + 128 * int64_t(k)), dst + 64 * (w * LA + q));
#pragma unroll
    for (int q = 0; q < LB; ++q)
      if (NIB % NW == 0 || w + NW * q < NIB) ring_load(pb[q] + k * CH, dst + BM * 8 + 64 * (w + NW * q));
  };

  f4 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};
  // the sign of odd steps' sums (add_step): the rows are split with it (three
  // parts), or the weights were
  const float* inv_b = reinterpret_cast<const float*>(B + int64_t(N) * KG * P);
  unsigned alt = 0x80000000u;
  if constexpr (P == 2) alt &= __builtin_amdgcn_readfirstlane(__float_as_uint(inv_b[min(nt, N - 1)]));
  // the row's scale and the largest |x| it takes (kOnline), 1 / scale at the end
  float sa[TM], lim[TM], sg = 1.f;
  // kPairs: the row's largest inverse scale (as its exponent field, a byte a row:
  // registers), the current block's factor onto it (a power of two, at most 1:
  // the fp16 operands themselves would lose bits to it, or with a factor below
  // 2^-24 the whole block)
  unsigned imax = 0;
  float inext[TM], fac[TM];
  const float* inv_a = nullptr;
  float* smax = reinterpret_cast<float*>(lds + ST * Sh::STAGE);
  if constexpr (AS == kExact) {
    // the tile's rows' largest |x|: eight lanes a row, as the stage loads read them
    float m[LA];
#pragma unroll
    for (int q = 0; q < LA; ++q) m[q] = 0.f;
    for (int s = 0; s < steps; ++s)
#pragma unroll
      for (int q = 0; q < LA; ++q) {
        const float4 x = *reinterpret_cast<const float4*>(pa[q] + 128 * int64_t(s));
        asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m[q]) : "v"(x.x), "v"(x.y));
        asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m[q]) : "v"(x.z), "v"(x.w));
      }
#pragma unroll
    for (int q = 0; q < LA; ++q) {
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) m[q] = fmaxf(m[q], __shfl_xor(m[q], o));
      if ((l & 7) == 0) smax[8 * (w * LA + q) + (l >> 3)] = m[q];
    }
  } else if constexpr (AS == kOnline) {
#pragma unroll
    for (int a = 0; a < TM; ++a) sa[a] = 1.f, lim[a] = 0.f;
  } else {
    inv_a = reinterpret_cast<const float*>(static_cast<const char*>(A) + 4 * int64_t(M) * K);
    const int nblk = steps / kbs;
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      const int row = min(m0 + 16 * a + c, M - 1);
      float m = 0.f;
      for (int b = g; b < nblk; b += 4) m = fmaxf(m, inv_a[int64_t(b) * M + row]);
      imax |= (__float_as_uint(max_g(m)) >> 23) << (8 * a);
      inext[a] = inv_a[row];
      fac[a] = 1.f;
    }
  }
#pragma unroll
  for (int s = 0; s < ST - 1; ++s) issue(s, s);

  f4 ts[NG > 1 ? 2 : 1][TM][TG];  // a group's step
  // kExact: the running sum turned with the steps' sign (turn: t - acc, the sign of
  // the last step at the end) in a K loop of its own: with the sign a multiplier,
  // as in the other forms, the 256 x 256 tiles spill in the loop (62291 x 1024 x 512
  // 290 us against 259)
  auto add_group = [&](auto set, int bg, auto turn) {
    constexpr int X = decltype(set)::value;
#pragma unroll
    for (int j = 0; j < TG; ++j)
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        f4& s = acc[a][TG * bg + j];
        if constexpr (AS == kExact) s = turn ? ts[X][a][j] - s : ts[X][a][j] + s;
        else add_step(s, ts[X][a][j], AS == kPairs ? fac[a] : sg);
      }
  };
  using last_ = std::integral_constant<int, (NG > 1 ? 1 : 0)>;  // the last group's set
  int stage = 0;          // step s's
  int left = 0, blk = 0;  // kPairs: steps left in the K block, the next block
  // this lane's slots in a stage row (row & 15 = c): A's two chunks, B's parts
  const int sa0 = swizzle<2>(2 * g, c), sa1 = swizzle<2>(2 * g + 1, c);
  int sb[P];
#pragma unroll
  for (int p = 0; p < P; ++p) sb[p] = swizzle<P>(g * P + p, c);
  auto k_loop = [&](auto turn) {
    for (int s = 0; s < steps; ++s) {
      // the step's stage in LDS for this wave's loads (those of the stages after
      // it may still fly), then for every wave's; no wave still reads the stage
      // of step s - 1, which the next loads fill
      wait_vm<(ST - 2) * (LA + (NIB % NW == 0 ? LB : LB - 1))>();
      ring_barrier();
      issue(s + ST - 1, stage == 0 ? ST - 1 : stage - 1);
      const u4* at = lds + stage * Sh::STAGE + ar * 8;
      const u4* bt = lds + stage * Sh::STAGE + BM * 8 + bc * CH;
      u4 ah[TM], al[TM];
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        ah[a] = at[(16 * a + c) * 8 + sa0];
        al[a] = at[(16 * a + c) * 8 + sa1];
      }
      // B's operands a group of TG tiles ahead of its products (the scheduling
      // barriers keep the reads there: left alone, the compiler reads each
      // group's operands just before its products and waits)
      u4 wv[2][TG][P];
      auto read = [&](auto set, int bg) {
        constexpr int X = decltype(set)::value;
#pragma unroll
        for (int j = 0; j < TG; ++j)
#pragma unroll
          for (int p = 0; p < P; ++p) wv[X][j][p] = bt[(16 * (TG * bg + j) + c) * CH + sb[p]];
      };
      using c0_ = std::integral_constant<int, 0>;
      using c1_ = std::integral_constant<int, 1>;
      read(c0_{}, 0);
      if constexpr (NG > 1) read(c1_{}, 1);
      __builtin_amdgcn_sched_barrier(0);
      if (s) add_group(last_{}, NG - 1, turn);
      if constexpr (AS != kExact) sg = __uint_as_float(0x3f800000u | (s & 1 ? alt : 0u));
      if constexpr (AS == kPairs) {
#pragma unroll
        for (int a = 0; a < TM; ++a) fac[a] = copysignf(fac[a], sg);
        if (kbs < steps) {
          if (left == 0) {  // a block begins: its factor, and the next one's scale on its way
            left = kbs, blk = min(blk + 1, steps / kbs - 1);
#pragma unroll
            for (int a = 0; a < TM; ++a) {
              fac[a] = sg * inext[a] * __uint_as_float((254 - (imax >> (8 * a) & 255)) << 23);
              inext[a] = inv_a[int64_t(blk) * M + min(m0 + 16 * a + c, M - 1)];
            }
          }
          --left;
        }
      } else {
        if constexpr (AS == kExact) {
          if (s == 0)
#pragma unroll
            for (int a = 0; a < TM; ++a) sa[a] = pet_split::pair_scale(smax[ar + 16 * a + c]);
        } else {
          float m[TM];
          bool over = false;
#pragma unroll
          for (int a = 0; a < TM; ++a) {
            m[a] = amax8(ah[a], al[a]);
            over |= m[a] > lim[a];
          }
          if (__builtin_amdgcn_ballot_w64(over) != 0) {  // a row outgrew its scale
#pragma unroll
            for (int a = 0; a < TM; ++a) {
              const float f = outgrow(m[a], sa[a], lim[a]);
#pragma unroll
              for (int b = 0; b < TN; ++b) acc[a][b] *= f;
            }
          }
        }
#pragma unroll
        for (int a = 0; a < TM; ++a) split8x(ah[a], al[a], P == 3 ? sg * sa[a] : sa[a]);
      }
      // the small products first, TG TM independent sums between two dependent
      // ones; a group's step is added under the next group's products
      auto products = [&](auto set, int bg) {
        constexpr int X = decltype(set)::value;
#pragma unroll
        for (int j = 0; j < TG; ++j)
#pragma unroll
          for (int a = 0; a < TM; ++a) ts[X][a][j] = f4{0.f, 0.f, 0.f, 0.f};
        auto prod = [&](int p, const u4* a_) {
#pragma unroll
          for (int j = 0; j < TG; ++j)
#pragma unroll
            for (int a = 0; a < TM; ++a) ts[X][a][j] = mfma_h(wv[X][j][p], a_[a], ts[X][a][j]);
        };
        if constexpr (P == 2) {
          prod(0, al), prod(1, ah), prod(0, ah);
        } else {
          prod(1, al), prod(2, ah), prod(0, al), prod(1, ah), prod(0, ah);
        }
        if (bg > 0) add_group(std::integral_constant<int, X ^ 1>{}, bg - 1, turn);
      };
#pragma unroll
      for (int bg = 0; bg < NG; bg += 2) {
        products(c0_{}, bg);
        if (bg + 2 < NG) read(c0_{}, bg + 2);
        __builtin_amdgcn_sched_barrier(0);
        if (bg + 1 < NG) {
          products(c1_{}, bg + 1);
          if (bg + 3 < NG) read(c1_{}, bg + 3);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      stage = stage + 1 == ST ? 0 : stage + 1;
    }
    add_group(last_{}, NG - 1, turn);
  };
  if (AS == kExact && alt) {
    k_loop(std::true_type{});
    if (!(steps & 1))  // the last step's sign (a zero stays +0)
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f} - acc[a][b];
  } else {
    k_loop(std::false_type{});
  }
  wait_vm<0>();  // no load into LDS outlives the loop
  if constexpr (AS == kOnline)
#pragma unroll
    for (int a = 0; a < TM; ++a)
      special_rows(
          acc[a], steps, c,
          [&](int c, int s) {
            return reinterpret_cast<const u4*>(static_cast<const char*>(A) + min(m0 + 16 * a + c, M - 1) * arow + 128 * int64_t(s) + 32 * g);
          },
          [&](int c, int b, int s, u4& h, u4& lo) {
            const u4* q = B + int64_t(min(nt + col_of(bc + 16 * b + c), N - 1)) * KG * P + s * CH + g * P;
            h = q[0], lo = q[P - 1];
          });

  // ---- epilogue
  float ia[TM];
#pragma unroll
  for (int a = 0; a < TM; ++a) ia[a] = AS == kPairs ? __uint_as_float((imax >> (8 * a) & 255) << 23) : 1.f / sa[a];
  rows_epilogue<TM, TN, OUT, P == 3 || OUT == kBlocks>(acc, ia, inv_b, m0, n0, c, g, M, N, C, ldc, epi);
}

// The same product with K split over a workgroup's waves, for launches of few
// tiles: wave w takes steps w, w + NW, ... of the whole 16 TM x 16 TN tile through
// an LDS slice of its own (its loads, its waits: no barrier), and the waves'
// sums meet in LDS once, in the order of the waves. A step of gemm_rows_kernel with
// one or two waves a SIMD is a chain of about 1000 cycles (barrier, LDS reads,
// scale, split, 330 cycles of products), and more stages in flight or the next
// step's split under this one's products did not shorten it (8096 x 128 x 1024:
// 20.3, 20.4, 19.0 us); this has a quarter of the steps (17.2; 648 rows: 18.7 -> 8.5).
template <int TM, int TN, int NW, int OUT>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
gemm_ksplit_kernel(int M, int N, int K, const void* A, int64_t lda, const u4* B, float* C, int64_t ldc, Epi epi, int,
                   int win) {
  constexpr int P = 3, BM = 16 * TM, BN = 16 * TN, CH = 4 * P, LA = BM / 8, LB = BN * CH / 64;
  constexpr int SLICE = BM * 8 + BN * CH;  // 16-byte chunks; the wave's sums (64 TM TN) fit in it
  static_assert(TN == 4 && TM <= NW && 64 * TM * TN + 4 * TM <= SLICE, "the epilogue's 64 columns; a row tile a wave");
  extern __shared__ u4 lds[];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, c = l & 15, g = l >> 4;
  const int KG = K / 8, steps = K / 32;
  const int NT = (N + BN - 1) / BN, RBk = (M + BM - 1) / BM;
  const int t = pet_attn::xcd_item(blockIdx.x, gridDim.x);
  const int wi = t / (win * NT), wr_ = min(win, RBk - wi * win), within = t - wi * win * NT;
  const int m0 = (wi * win + within % wr_) * BM, n0 = (within / wr_) * BN;
  u4* slice = lds + w * SLICE;
  const char* pa[LA];
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int e = 64 * q + l, r = e >> 3;
    pa[q] = static_cast<const char*>(A) + min(m0 + r, M - 1) * (4 * lda) + 16 * swizzle<2>(e & 7, r);
  }
  const u4* pb[LB];
#pragma unroll
  for (int q = 0; q < LB; ++q) {
    const int e = 64 * q + l, r = e / CH;
    pb[q] = B + int64_t(min(n0 + col_of(r), N - 1)) * KG * P + unswizzle<P>(e - r * CH, r);
  }
  auto issue = [&](int s) {
#pragma unroll
    for (int q = 0; q < LA; ++q) ring_load(reinterpret_cast<const u4*>(pa[q] + 128 * int64_t(s)), slice + 64 * q);
#pragma unroll
    for (int q = 0; q < LB; ++q) ring_load(pb[q] + s * CH, slice + BM * 8 + 64 * q);
  };
  f4 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};
  float sa[TM], lim[TM];
#pragma unroll
  for (int a = 0; a < TM; ++a) sa[a] = 1.f, lim[a] = 0.f;
  const int sa0 = swizzle<2>(2 * g, c), sa1 = swizzle<2>(2 * g + 1, c);
  int sb[P];
#pragma unroll
  for (int p = 0; p < P; ++p) sb[p] = swizzle<P>(g * P + p, c);
  const float sg = (w ^ (w >> 1)) & 1 ? -1.f : 1.f;  // waves 1 and 2 of four sum the negated rows (add_step's reason)
  if (w < steps) issue(w);
  for (int s = w; s < steps; s += NW) {
    wait_vm<0>();
    asm volatile("" ::: "memory");
    u4 ah[TM], al[TM], wv[TN][P];
    const u4* bt = slice + BM * 8;
#pragma unroll
    for (int a = 0; a < TM; ++a) ah[a] = slice[(16 * a + c) * 8 + sa0], al[a] = slice[(16 * a + c) * 8 + sa1];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int p = 0; p < P; ++p) wv[j][p] = bt[(16 * j + c) * CH + sb[p]];
    // the slice is read: the next step's loads into it
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    if (s + NW < steps) issue(s + NW);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    float m[TM];
    bool over = false;
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      m[a] = amax8(ah[a], al[a]);
      over |= m[a] > lim[a];
    }
    if (__builtin_amdgcn_ballot_w64(over) != 0) {  // as gemm_rows_kernel's
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        const float f = outgrow(m[a], sa[a], lim[a]);
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] *= f;
      }
    }
#pragma unroll
    for (int a = 0; a < TM; ++a) split8x(ah[a], al[a], sg * sa[a]);
    auto prod = [&](int p, const u4 (&a_)[TM]) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int a = 0; a < TM; ++a) acc[a][j] = mfma_h(wv[j][p], a_[a], acc[a][j]);
    };
    prod(1, al), prod(2, ah), prod(0, al), prod(1, ah), prod(0, ah);
  }
  // the waves' sums and their rows' inverse scales (0: nothing but zeros) into
  // their slices; a row's sums at the largest of those
#pragma unroll
  for (int a = 0; a < TM; ++a) {
#pragma unroll
    for (int b = 0; b < TN; ++b) slice[64 * (a * TN + b) + l] = __builtin_bit_cast(u4, f4(acc[a][b] * sg));
    if (g == 0) reinterpret_cast<float*>(slice + 64 * TM * TN)[16 * a + c] = lim[a] > 0.f ? 1.f / sa[a] : 0.f;
  }
  __syncthreads();
  if (w >= TM) return;
  float inv[NW], top = 0x1p-126f;
#pragma unroll
  for (int v = 0; v < NW; ++v)
    inv[v] = reinterpret_cast<const float*>(lds + v * SLICE + 64 * TM * TN)[16 * w + c], top = fmaxf(top, inv[v]);
  f4 sum[1][TN];
#pragma unroll
  for (int b = 0; b < TN; ++b) {
    sum[0][b] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      const f4 x = __builtin_bit_cast(f4, lds[v * SLICE + 64 * (w * TN + b) + l]);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[0][b][e] = fmaf(x[e], inv[v] * (1.f / top), sum[0][b][e]);
    }
  }
  special_rows(
      sum[0], steps, c,
      [&](int c, int s) {
        return reinterpret_cast<const u4*>(static_cast<const char*>(A) + min(m0 + 16 * w + c, M - 1) * (4 * lda) + 128 * int64_t(s) + 32 * g);
      },
      [&](int c, int b, int s, u4& h, u4& lo) {
        const u4* q = B + int64_t(min(n0 + col_of(16 * b + c), N - 1)) * KG * P + s * CH + g * P;
        h = q[0], lo = q[P - 1];
      });
  const float ia[1] = {top};
  rows_epilogue<1, TN, OUT, true>(sum, ia, reinterpret_cast<const float*>(B + int64_t(N) * KG * P), m0 + 16 * w, n0, c, g, M,
                            N, C, ldc, epi);
}

// The short contraction (K = 32 KB at most 128, three-part weights): a workgroup
// holds a strip of 16 TN columns' weights of all of K in LDS for its life, and
// its eight waves stream 16-row blocks of A past it, each on its own: a wave's
// block comes by its own loads into its own LDS slice (no barrier after the
// weights'), its rows' largest |x| and their split are made in registers, and
// the next block's loads run under this one's products, epilogue and stores.
// What bounds it: at K = 128 a block of 128 columns is 160 matrix instructions
// a wave against 16 KB of results written (with a kept pre-activation 16 + 8):
// about even, so neither the weights (once a workgroup) nor a barrier a block
// may stand between them. One workgroup a CU (96 KB of weights, 64 KB of
// slices at K = 128). XCD x takes rows [x M / 8, (x + 1) M / 8), its
// workgroups S a strip, so the strips re-read A from their L2.
template <int KB, int TN, int OUT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
gemm_strip_kernel(int M, int N, const float* A, int64_t lda, const u4* B, float* C, int64_t ldc, Epi epi, int S) {
  constexpr int BN = 16 * TN, CH = 12, KG = 4 * KB, NW = 8;
  constexpr int TG = TN < 4 ? TN : 4, NG = TN / TG;
  constexpr int BCH = KB * BN * CH, ACH = KB * 16 * 8;  // chunks of the strip's weights, of a block of A
  extern __shared__ u4 lds[];  // [KB][BN][CH] weights, then a slice [KB][16][8] a wave
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, c = l & 15, g = l >> 4;
  const int NT = (N + BN - 1) / BN, x = blockIdx.x & 7, li = blockIdx.x >> 3;
  const int n0 = (li % NT) * BN, rs = li / NT;
  const int xr0 = int(int64_t(x) * M / 8), xr1 = int(int64_t(x + 1) * M / 8), nb = (xr1 - xr0 + 15) / 16;
  // this wave's blocks: every (8 S)-th
  int blk = rs * NW + w;
  u4* slice = lds + BCH + w * ACH;
  const char* pa[ACH / 64];
#pragma unroll
  for (int q = 0; q < ACH / 64; ++q) {
    const int e = 64 * q + l, k = e >> 7, r = (e >> 3) & 15;
    pa[q] = reinterpret_cast<const char*>(A) + 128 * k + 16 * swizzle<2>(e & 7, r);
  }
  auto issue = [&](int b) {
#pragma unroll
    for (int q = 0; q < ACH / 64; ++q) {
      const int r = ((64 * q + l) >> 3) & 15;
      const int64_t row = min(xr0 + 16 * b + r, xr1 - 1);
      ring_load(reinterpret_cast<const u4*>(pa[q] + 4 * lda * row), slice + 64 * q);
    }
  };
  // the strip's weights: chunk e = (k, row, slot); a column's chunks of step k are 12 consecutive
#pragma unroll 1
  for (int i = w; i < BCH / 64; i += NW) {
    const int e = 64 * i + l, k = e / (BN * CH), r = (e / CH) % BN, ch = unswizzle<3>(e % CH, r);
    ring_load(B + (int64_t(min(n0 + col_of(r), N - 1)) * KG + 4 * k) * 3 + ch, lds + 64 * i);
  }
  if (blk < nb) issue(blk);
  wait_vm<0>();
  ring_barrier();
  const int s0 = swizzle<2>(2 * g, c), s1 = swizzle<2>(2 * g + 1, c);
  int sb[3];
#pragma unroll
  for (int p = 0; p < 3; ++p) sb[p] = swizzle<3>(3 * g + p, c);
  const float* inv_b = reinterpret_cast<const float*>(B + int64_t(N) * KG * 3);
  for (; blk < nb; blk += NW * S) {
    // (the block's loads are done: waited for after the last block's epilogue)
    u4 ah[KB], al[KB];
#pragma unroll
    for (int k = 0; k < KB; ++k) ah[k] = slice[(16 * k + c) * 8 + s0], al[k] = slice[(16 * k + c) * 8 + s1];
    float sa = 1.f, lim = 0.f, f[KB];  // the running scale, as gemm_rows_kernel's: the same bits
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const float m = amax8(ah[k], al[k]);
      f[k] = 1.f;
      if (__builtin_amdgcn_ballot_w64(m > lim) != 0) f[k] = outgrow(m, sa, lim);
      split8x(ah[k], al[k], k & 1 ? -sa : sa);
    }
    // the slice is read: the next block's loads into it
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    if (blk + NW * S < nb) issue(blk + NW * S);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    f4 acc[1][TN];
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[0][b] = f4{0.f, 0.f, 0.f, 0.f};
    u4 wv[2][TG][3];
    auto read = [&](auto set, int i) {  // group i: step i / NG, tiles TG (i % NG) ..
      constexpr int X = decltype(set)::value;
#pragma unroll
      for (int j = 0; j < TG; ++j)
#pragma unroll
        for (int p = 0; p < 3; ++p) wv[X][j][p] = lds[((i / NG) * BN + 16 * (TG * (i % NG) + j) + c) * CH + sb[p]];
    };
    f4 t[2][TG];  // a group's step, added under the next group's products
    auto add_group = [&](auto set, int i) {
      constexpr int X = decltype(set)::value;
#pragma unroll
      for (int j = 0; j < TG; ++j) add_step(acc[0][TG * (i % NG) + j], t[X][j], (i / NG) & 1 ? -1.f : 1.f);
    };
    auto products = [&](auto set, int i) {
      constexpr int X = decltype(set)::value;
      const int k = i / NG;
      if (k > 0 && i % NG == 0 && __builtin_amdgcn_ballot_w64(f[k] != 1.f) != 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[0][j] *= f[k];
#pragma unroll
        for (int j = 0; j < TG; ++j) t[X ^ 1][j] *= f[k];
      }
#pragma unroll
      for (int j = 0; j < TG; ++j) t[X][j] = f4{0.f, 0.f, 0.f, 0.f};
      auto prod = [&](int p, const u4& a) {
#pragma unroll
        for (int j = 0; j < TG; ++j) t[X][j] = mfma_h(wv[X][j][p], a, t[X][j]);
      };
      prod(1, al[k]), prod(2, ah[k]), prod(0, al[k]), prod(1, ah[k]), prod(0, ah[k]);
      if (i > 0) add_group(std::integral_constant<int, X ^ 1>{}, i - 1);
    };
    using c0_ = std::integral_constant<int, 0>;
    using c1_ = std::integral_constant<int, 1>;
    constexpr int G = KB * NG;
    read(c0_{}, 0);
    if constexpr (G > 1) read(c1_{}, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < G; i += 2) {
      products(c0_{}, i);
      if (i + 2 < G) read(c0_{}, i + 2);
      __builtin_amdgcn_sched_barrier(0);
      if (i + 1 < G) {
        products(c1_{}, i + 1);
        if (i + 3 < G) read(c1_{}, i + 3);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    add_group(std::integral_constant<int, (G - 1) & 1>{}, G - 1);
    special_rows(
        acc[0], KB, c,
        [&](int c, int s) {
          return reinterpret_cast<const u4*>(reinterpret_cast<const char*>(A) + min(xr0 + 16 * blk + c, xr1 - 1) * (4 * lda) + 128 * s + 32 * g);
        },
        [&](int c, int b, int s, u4& h, u4& lo) {
          const u4* q = lds + (s * BN + 16 * b + c) * CH;
          h = q[sb[0]], lo = q[sb[2]];
        });
    const float ia[1] = {1.f / sa};
    rows_epilogue<1, TN, OUT, true>(acc, ia, inv_b, xr0 + 16 * blk, n0, c, g, xr1, N, C, ldc, epi);
    // the next block's loads done: issued before the epilogue, whose last
    // stores (four at least: a run's results are one store or more) may still
    // be on their way
    if (n0 + BN <= N) wait_vm<TN / 2>();
    else wait_vm<0>();  // (a partial strip stores fewer)
    asm volatile("" ::: "memory");
  }
}

}  // namespace pet_gemm

using namespace pet_gemm;

namespace {
using RowsKernel = void (*)(int, int, int, const void*, int64_t, const u4*, float*, int64_t, Epi, int, int);
struct RowsShape {
  RowsKernel k = nullptr;
  int bm = 0, bn = 0, threads = 0;
  size_t lds = 0;
};
template <int TM, int TN, int WR, int WC, int P, int AS, int OUT>
RowsShape rows_shape() {
  using Sh = RowsTile<TM, TN, WR, WC, P>;
  return {gemm_rows_kernel<TM, TN, WR, WC, P, AS, OUT>, Sh::BM, Sh::BN, 64 * WR * WC, Sh::bytes};
}
template <int TM, int NW, int OUT>
RowsShape ksplit_shape() {
  return {gemm_ksplit_kernel<TM, 4, NW, OUT>, 16 * TM, 64, 64 * NW, size_t(NW) * (16 * TM * 8 + 64 * 12) * 16};
}
// The shapes: 1 256 x 256 of 64 x 128 a wave, 2 128 x 128 of 64 x 64 (both two
// parts), 3 64 x 128 of 32 x 64, 4 64 x 64 and 5 32 x 64 of 16 x 64; 7, 8 and 9 64,
// 32 and 16 x 64 with the steps split over four waves (three parts); block
// pairs out (a wave 128 columns, a block of the output): 1, and 6 128 x 128 of
// 32 x 128. With block pairs out shape 1 needs more than its 256 registers: it spills
// 69 (120 bytes a lane) in the epilogue; the 128-column strip spills 16.
template <int P, int AS, int OUT>
RowsShape rows_pick(int cfg) {
  if constexpr (OUT == kBlocks) {
    if (cfg == 1) return rows_shape<4, 8, 4, 2, P, AS, OUT>();
    return rows_shape<2, 8, 4, 1, P, AS, OUT>();
  } else {
    if constexpr (P == 2) {
      if constexpr (OUT == kVec)
        if (cfg == 1) return rows_shape<4, 8, 4, 2, P, AS, OUT>();
      if (cfg <= 2) return rows_shape<4, 4, 2, 2, P, AS, OUT>();
    }
    if (cfg == 3) return rows_shape<2, 4, 2, 2, P, AS, OUT>();
    if (cfg == 4) return rows_shape<1, 4, 4, 1, P, AS, OUT>();
    if constexpr (AS == kOnline && P == 3) {
      if (cfg == 7) return ksplit_shape<4, 4, OUT>();
      if (cfg == 8) return ksplit_shape<2, 4, OUT>();
      if (cfg == 9) return ksplit_shape<1, 4, OUT>();
    }
    return rows_shape<1, 4, 2, 1, P, AS, OUT>();
  }
}
}  // namespace

// C = epi(A B^T) on gemm_rows_kernel. P parts of B's rows (pet_gemm_split_weights
// from K = 256: 2; pet_gemm_pair_weights: 3); as: how A comes (kOnline,
// kExact: fp32 rows, 16-byte aligned; kPairs: pair rows or blocks of kb
// columns). K a multiple of 32; e.pout: block pairs in place of C (N a multiple
// of 128, A as pairs, every operand 16-byte aligned). cfg: the shape (0, with two
// parts: chosen here).
int pet_gemm_nt_rows(int M, int N, int K, const void* A, int64_t lda, int as, int kb, const void* Bp, int P, float* C,
                     int64_t ldc, const Epi& e, hipStream_t st, int cfg) {
  if (M < 0 || N < 0 || K < 32 || K % 32 || (as == kPairs && (kb < 32 || kb % 32 || K % kb))) return PET_ATTN_EINVAL;
  if (M == 0 || N == 0) return PET_ATTN_OK;
  auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  if ((as != kPairs && lda % 4) || !a16(A) || !a16(Bp)) return PET_ATTN_EALIGN;
  if (e.act == 2 && N % 2) return PET_ATTN_EINVAL;
  const bool vec = N % 4 == 0;
  auto tiles = [&](int bm, int bn) { return int64_t((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (tiles(64, 32) >= (int64_t(1) << 31)) return PET_ATTN_EINDEX;
  if (P == 3 && (cfg < 3 || cfg == 6)) return PET_ATTN_EINVAL;
  if (!cfg) {
    // 256 x 256 tiles (one workgroup a CU) where their last round of 256 leaves
    // at most a sixth of the CUs idle over all rounds: full, they are 1.13 to 1.17 times
    // faster than 128 x 128 (62291 x 512 x 1024 from pairs: 176 against 204 us, 488
    // tiles, 95% of their rounds full; at 82%, 26670 x 1024 x 512 with SwiGLU, 102
    // against 94; at 83%, 217834 x 256 x 768, 281 against 291: the line could lie a
    // hundredth lower). An
    // activation's backward into block pairs is bound by its operand: 128 x 128
    // there (62291 x 1024 x 512, SwiGLU: 324 against 382). A width that is no
    // multiple of 4 keeps to 128 x 128: with its last columns one by one the
    // 256 x 256 epilogue does not fit the registers.
    const int64_t t256 = tiles(256, 256), rounds = (t256 + 255) / 256;
    const bool c1 = vec && N > 128 && 6 * t256 >= 5 * 256 * rounds;
    if (e.pout)
      cfg = c1 && N % 256 == 0 && e.act <= 2 ? 1 : 6;
    else
      cfg = c1 ? 1 : N > 64 && tiles(128, 128) >= 512 ? 2 : N > 64 && tiles(64, 128) > 256 ? 3 : tiles(64, 64) >= 256 ? 4 : 5;
  }
  RowsShape s;
  using std::integral_constant;
  auto pick = [&](auto p, auto a) {
    constexpr int P_ = decltype(p)::value, A_ = decltype(a)::value;
    if (e.pout) {
      if constexpr (P_ == 2 && A_ == kPairs) s = rows_pick<P_, A_, kBlocks>(cfg);
    } else {
      s = vec ? rows_pick<P_, A_, kVec>(cfg) : rows_pick<P_, A_, kAny>(cfg);
    }
  };
  if (P == 3 && as == kOnline) pick(integral_constant<int, 3>{}, integral_constant<int, kOnline>{});
  else if (P == 2 && as == kExact) pick(integral_constant<int, 2>{}, integral_constant<int, kExact>{});
  else if (P == 2 && as == kPairs) pick(integral_constant<int, 2>{}, integral_constant<int, kPairs>{});
  if (!s.k) return PET_ATTN_EINVAL;
  if (const int rc = pet_attn::raise_lds(reinterpret_cast<const void*>(s.k), s.lds)) return rc;
  // windows of row blocks where the weights pass an L2's share
  const int win = int64_t(N) * K * 2 * P > (2 << 20) ? 4 : 1;
  hipLaunchKernelGGL(s.k, dim3(unsigned(tiles(s.bm, s.bn))), dim3(s.threads), s.lds, st, M, N, K, A, lda,
                     static_cast<const u4*>(Bp), C, ldc, e, as == kPairs ? kb / 32 : 0, win);
  tally(P == 3 ? 3 : 2, M, N, K);
  return hipGetLastError() == hipSuccess ? PET_ATTN_OK : PET_ATTN_ELAUNCH;
}

// C = epi(A B^T) for K at most 128 from three-part weights (pet_gemm_pair_weights)
// on gemm_strip_kernel, where there are rows enough to fill it.
int pet_gemm_nt_strip(int M, int N, int K, const float* A, int64_t lda, const void* Bp, float* C, int64_t ldc,
                      const Epi& e, hipStream_t st) {
  if (M < 0 || N < 0 || K < 32 || K > 128 || K % 32) return PET_ATTN_EINVAL;
  if (M == 0 || N == 0) return PET_ATTN_OK;
  auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  if (lda % 4 || !a16(A) || !a16(Bp)) return PET_ATTN_EALIGN;
  if (e.act == 2 && N % 2) return PET_ATTN_EINVAL;
  // 64 or 128 columns a workgroup: the strips of an XCD's 32 CUs take
  // ceil(blocks / (8 S)) rounds of 16-row blocks, and a round of 64 columns takes
  // 0.55 of one of 128 (26670 x 512 x 128 with the SwiGLU backward: 44 us with
  // 64, 7 rounds, 51 with 128, 4; 27318 x 128 x 128: 12.4 with 64, 2 rounds,
  // 11.9 with 128, 1); a width no multiple of 4 takes 64 (with its last columns one
  // by one the epilogue of 128 does not fit the registers)
  const int KB = K / 32, nbx = ((M + 7) / 8 + 15) / 16;  // 16-row blocks an XCD
  auto ranges = [&](int bn) {  // row ranges a strip in an XCD
    return std::max(1, std::min(32 / std::min(32, (N + bn - 1) / bn), (nbx + 7) / 8));
  };
  auto rounds = [&](int bn) { return (nbx + 8 * ranges(bn) - 1) / (8 * ranges(bn)); };
  const bool vec = N % 4 == 0;
  const int BN = vec && N > 64 && rounds(128) <= 0.55 * rounds(64) ? 128 : 64, NT = (N + BN - 1) / BN, S = ranges(BN);
  if (int64_t(8) * NT * S >= (int64_t(1) << 31)) return PET_ATTN_EINDEX;
  using K_ = void (*)(int, int, const float*, int64_t, const u4*, float*, int64_t, Epi, int);
  K_ k = nullptr;
  auto pick = [&](auto kb, auto tn) {
    constexpr int KB_ = decltype(kb)::value, TN_ = decltype(tn)::value;
    if constexpr (TN_ == 4) k = vec ? gemm_strip_kernel<KB_, 4, kVec> : gemm_strip_kernel<KB_, 4, kAny>;
    else k = gemm_strip_kernel<KB_, TN_, kVec>;
  };
  auto by_k = [&](auto tn) {
    switch (KB) {
      case 1: pick(std::integral_constant<int, 1>{}, tn); break;
      case 2: pick(std::integral_constant<int, 2>{}, tn); break;
      case 3: pick(std::integral_constant<int, 3>{}, tn); break;
      default: pick(std::integral_constant<int, 4>{}, tn); break;
    }
  };
  if (BN == 128) by_k(std::integral_constant<int, 8>{});
  else by_k(std::integral_constant<int, 4>{});
  const size_t bytes = size_t(KB) * (BN * 12 + 8 * 128) * 16;
  if (const int rc = pet_attn::raise_lds(reinterpret_cast<const void*>(k), bytes)) return rc;
  hipLaunchKernelGGL(k, dim3(unsigned(8 * NT * S)), dim3(512), bytes, st, M, N, A, lda, static_cast<const u4*>(Bp), C, ldc, e, S);
  tally(3, M, N, K);
  return hipGetLastError() == hipSuccess ? PET_ATTN_OK : PET_ATTN_ELAUNCH;
}

// C = epi(A B^T) from three-part weights (pet_gemm_pair_weights), any K a
// multiple of 32: the kernel and its tile. Up to K = 224 every choice gives the
// same bits, so a row's results do not depend on M. Measured on MI355X (us, with
// about 3 of launch; the rocBLAS fp32 product it takes the place of in the
// model about 20 up to 8096 rows):
//  - short K, results enough for every CU to stream rows past resident weights
//    (M N >= 3 * 2^20): the strip (27318 rows, K 128: N 128 / 512 11.7 / 29.2
//    against 12.8 / 33.5 with 64 x 128 tiles; 8096 x 384 10.9 against 11.7);
//    below, 64 x 64 tiles (4000 x 512: 7.9 against 8.9 with 64 x 128), or
//    32 x 64 where those would leave half of the 256 CUs idle.
//  - K of 256 and more: 64 x 128 tiles where they fill the chip (27318 x 128:
//    K 512 23.6 against 26.5 with 64 x 64), else 64 x 64; with at most 256 of
//    those, the steps split over the waves: a tile is then a chain of K / 128
//    steps, not K / 32 (K 1024: 8096 x 128 17.2 against 19.9; 4000 x 128 at K 512 8.9
//    with 32-row tiles against 11.4; 648 x 128 x 1024 8.5 with 16-row tiles
//    against 19.0).
int pet_gemm_nt_p3(int M, int N, int K, const float* A, int64_t lda, const void* Bp, float* C, int64_t ldc,
                   const Epi& e, hipStream_t st) {
  auto tiles = [&](int bm, int bn) { return int64_t((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  int cfg;
  if (K < 256) {
    if (K <= 128 && int64_t(M) * N >= 3 << 20) return pet_gemm_nt_strip(M, N, K, A, lda, Bp, C, ldc, e, st);
    cfg = N > 64 && tiles(64, 128) >= 512 ? 3 : tiles(64, 64) >= 128 ? 4 : 5;
  } else if (tiles(64, 64) > 256) {
    cfg = N > 64 && tiles(64, 128) > 256 ? 3 : 4;
  } else if (tiles(64, 64) > 128) {
    cfg = K >= 768 ? 7 : 4;
  } else {
    cfg = tiles(32, 64) > 128 ? 8 : 9;
  }
  return pet_gemm_nt_rows(M, N, K, A, lda, kOnline, 0, Bp, 3, C, ldc, e, st, cfg);
}
int pet_gemm_nt_parts(int M, int N, int K, const float* A, int64_t lda, const void* Bp, float* C, int64_t ldc,
                      const float* row_scale, const float* bias, const float* cin, int64_t ldcin, float beta,
                      float* pre, int64_t ldpre, int act, hipStream_t st) {
  Epi e;
  e.row_scale = row_scale, e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta, e.pre = pre, e.ldpre = ldpre;
  e.act = act;
  return pet_gemm_nt_p3(M, N, K, A, lda, Bp, C, ldc, e, st);
}
