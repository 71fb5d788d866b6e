// fp32 contraction on the bf16 matrix cores (gfx950), for grids large enough to be
// bound by the fp32 MFMA rate.
//
//   C[M, N] = A[M, K] x B[N, K]^T
//
// Every operand value is split into three bf16 parts, each the nearest bf16 of what the
// parts before it leave: x = x0 + x1 + x2 exactly (8 + 8 + 8 significant bits against 24).
// The exponent range of bf16 is fp32's, so the lower parts of a small value would be subnormal,
// which the matrix cores read as zero: values are split times 2^24, which leaves the least part
// of the least subnormal at 2^-125, and the sums are multiplied by 2^-48 at the end.  A product
// is the sum of eight part products,
//   x0 y0 + (x0 y1 + x1 y0) + (x1 y1 + x0 y2 + x2 y0) + (x1 y2 + x2 y1),
// each exact; x2 y2, the ninth, is below 2^-32 of it.  They are summed in fp32 by
// v_mfma_f32_32x32x16_bf16: eight of these take 256 cycles for the 16 k steps that eight
// v_mfma_f32_32x32x2f32 take 512 for.  The x0 y0 products and the others have a sum of their own
// each, joined at the end: the low one is 2^-8 of the other, so its roundings do not count, and
// the high one rounds once per 16 k (the fp32 tiles: once per k that has a product).  Relative
// error (2-norm) against float64 on 9216 x 256 x 256, fp32 tiles / these: dense rows 2.9e-7 /
// 0.9e-7; rows of 16, 4, 2 and 1 nonzeros 7.4 / 3.4, 4.0 / 2.6, 3.1 / 2.6 and 2.5 / 2.5e-8.  (All
// products into one sum: 2.4e-7, 13.8, 7.3, 5.1 and 3.5e-8, with six, eight or nine of them: a row's
// few products are rounded up to nine times where the fp32 tiles round once.)
//
// B (a layer's weight) comes packed: its parts made once per weight (pack_parts_kernel), in
// the MFMA operand order, so that a stage's parts go straight from global memory to LDS.  A
// wave owns WTM rows and all BN columns of the tile.  Its A rows pass through LDS as they
// are (global_load_lds_dwordx4, private to the wave, so no barrier guards them) and it splits
// them once, in registers.  Stages are 16 k deep, three of A and two of B; one barrier each.
//
// A tile with a sum that is not finite (an operand that is not, a value of 2^103 or more, which
// has no parts, or a sum past 2^79) is computed again by v_mfma_f32_32x32x2f32 from the fp32
// values, so such operands give what they give on the fp32 tiles.
#pragma once

#include "bf_gemm_parts_epilogue.h"

namespace bf {

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));

// Packed parts of B: per 32-column block and 16-k stage 3 KB, part by part, lane l's eight
// values (column l % 32, k 8 (l / 32) .. + 7) at 16 l; columns and k past the end are zero.
// A value that has no parts lies there as the NaN PARTS_RAW and the two halves of its 32 bits: the
// NaN sends every tile that meets it to the fp32 MFMAs, which read it whole.
constexpr int PARTS_BLOCK = 3 * 64 * 4;   // floats of one block and stage
constexpr uint32_t PARTS_RAW = 0x7fff;
constexpr float PARTS_SCALE = 16777216.f;   // 2^24

// OCC: workgroups resident per CU (the two sums of a 32 x 128 wave tile are 128 registers).
template <int FM_, int FN_, int NWM_, int OCC_>
struct TileParts {
  static constexpr int FM = FM_, FN = FN_, NWM = NWM_, NWN = 1, OCC = OCC_;
  static constexpr int WTM = 32 * FM, WTN = 32 * FN;   // wave tile
  static constexpr int BM = WTM * NWM, BN = WTN, BK = 16, NT = 64 * NWM;
  static constexpr int A_STAGE = BM * BK;              // floats of a stage of A rows
  static constexpr int B_STAGE = FN * PARTS_BLOCK;     // floats of a stage of B parts
  static constexpr int B_COPIES = 3 * FN / NWM;        // 1 KB copies of a B stage per wave
  static_assert(B_COPIES * NWM == 3 * FN, "whole copies per wave");
};

// lds_copy16 from a scalar base and a byte offset per lane.
__device__ __forceinline__ void lds_copy16_at(const float* base, uint32_t byte_off, float* lds_dst) {
  const uint32_t off = (uint32_t)(uintptr_t)((lds_float*)lds_dst);
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(byte_off), "s"(base), "s"(off) : "memory");
}

// The same, four bytes a lane (256 of LDS in a row), from a scalar base or a lane's own address.
__device__ __forceinline__ void lds_copy4_at(const float* base, uint32_t byte_off, float* lds_dst) {
  const uint32_t off = (uint32_t)(uintptr_t)((lds_float*)lds_dst);
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" ::"v"(byte_off), "s"(base), "s"(off) : "memory");
}
__device__ __forceinline__ void lds_copy4(const float* src, float* lds_dst) {
  const uint32_t off = (uint32_t)(uintptr_t)((lds_float*)lds_dst);
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(off) : "memory");
}

// (x, y) -> the packed bf16 pair nearest to it, and what the pair leaves of both.
__device__ __forceinline__ uint32_t take_part(float& x, float& y) {
  const floatx2 xy = {x, y};
  const uint32_t pk = __builtin_bit_cast(uint32_t, __builtin_convertvector(xy, bf16x2));   // v_cvt_pk_bf16_f32
  x -= __uint_as_float(pk << 16);
  y -= __uint_as_float(pk & 0xffff0000u);
  return pk;
}

// VEC: coefficient rows of whole 16-byte aligned float4s; else they are copied float by float (a row
// length that is no multiple of four), the same stage in four times as many copies.
template <int EPI, class T, bool VEC>
__global__ void __launch_bounds__(T::NT, (T::OCC * T::NWM + 3) / 4) gemm_parts_kernel(GemmArgs p) {
  constexpr int FM = T::FM, FN = T::FN, GBM = T::BM, GBN = T::BN, GBK = T::BK;
  // three stages of A rows, two of B parts; the relaxation epilogue stages its operands over all of it
  constexpr int SMEM = 3 * T::A_STAGE + 2 * T::B_STAGE;
  __shared__ __attribute__((aligned(16))) float smem_ab[SMEM];
  __shared__ float red[T::NWN][GBM];
  float* const bs = smem_ab + 3 * T::A_STAGE;

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lrow = lane & 31;
  const int h = lane >> 5;   // lane half -> k 8 h .. 8 h + 7 of a stage, in A and B alike
  const int z = (int)blockIdx.y;
  const bool lower = p.z_lower_first ? (z == 0) : (z == 1);
  const int64_t M = p.M, N = p.N, K = p.K;
  const bool fits32 = M < (1LL << 31);
  // XCD-aware tile order, as in gemm_kernel
  const int64_t ntn = ceil_div(N, GBN);
  const int64_t ntiles = ceil_div(M, GBM) * ntn;
  const int64_t per_xcd = ceil_div(ntiles, 8);
  const int64_t tile = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= ntiles) return;
  const int64_t tile_n = tile % ntn;
  const int64_t m0 = (tile / ntn) * GBM;
  const int64_t n0 = tile_n * GBN;
  const int64_t cols = N - n0;
  const int fn_act = cols >= GBN ? FN : (int)ceil_div(cols, 32);   // 32-column blocks inside N
  const int nk = (int)ceil_div(K, (int64_t)GBK);

  // copy slots of this wave's A rows: chunk j holds its rows 16 j .. 16 j + 15, float4 kq of row r
  // at position 4 r + (kq ^ (r / 2 % 4)) of the chunk, as in gemm_kernel's direct-to-LDS loop.
  // Byte offsets from the tile's first domain (below 2^32, checked at launch): a stage advances
  // the scalar base alone.
  constexpr int CHUNKS = VEC ? T::WTM / 16 : T::WTM / 4;   // copies of a stage: of 16 rows, or of 4
  constexpr int CHUNK = VEC ? 256 : 64;                    // floats of one
  const int64_t d0 = div_rows(m0, p.S, fits32);
  const float* __restrict__ a_base = p.A[z] + d0 * p.lda_d;
  uint32_t a_off[CHUNKS];
  int a_k[VEC ? 1 : 2];   // this lane's k of a stage (float by float: of even and of odd chunks)
  if constexpr (VEC) {
    a_k[0] = 4 * ((lane & 3) ^ ((lane >> 3) & 3));
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j) a_k[j] = 4 * (((lane >> 2) & 3) ^ (2 * j + (lane >> 5))) + (lane & 3);
  }
#pragma unroll
  for (int j = 0; j < CHUNKS; ++j) {
    const int64_t mr = m0 + wave * T::WTM + (VEC ? 16 * j + (lane >> 2) : 4 * j + (lane >> 4));
    const int64_t m = mr < M ? mr : M - 1;
    const int64_t d = div_rows(m, p.S, fits32);
    a_off[j] = (uint32_t)(4 * ((d - d0) * p.lda_d + (m - d * p.S) * p.lda + a_k[VEC ? 0 : j & 1]));
  }
  float* const a_wave = smem_ab + wave * T::WTM * GBK;
  auto copy_a = [&](int slot, int kt) {
    float* dst = a_wave + slot * T::A_STAGE;
    const float* src = a_base + (int64_t)kt * GBK;
    const bool whole = kt * GBK + GBK <= K;
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
      // k past the end reads the row start: it meets the zeros that B's parts hold there
      const int k = kt * GBK + a_k[VEC ? 0 : j & 1];
      if constexpr (VEC) {
        if (whole) lds_copy16_at(src, a_off[j], dst + CHUNK * j);
        else lds_copy16(src + (int64_t)(a_off[j] / 4) - (k < K ? 0 : k), dst + CHUNK * j);
      } else {
        if (whole) lds_copy4_at(src, a_off[j], dst + CHUNK * j);
        else lds_copy4(src + (int64_t)(a_off[j] / 4) - (k < K ? 0 : k), dst + CHUNK * j);
      }
    }
  };
  // this wave's copies of a B stage: block * 3 + part = B_COPIES wave .. ; blocks past N copy the
  // last one inside
  const float* __restrict__ b_base = p.B + (n0 / 32) * nk * PARTS_BLOCK;
  int64_t b_src[T::B_COPIES];
#pragma unroll
  for (int c = 0; c < T::B_COPIES; ++c) {
    const int u = T::B_COPIES * wave + c, blk = u / 3 < fn_act ? u / 3 : fn_act - 1;
    b_src[c] = (int64_t)blk * nk * PARTS_BLOCK + (u % 3) * 256;
  }
  const uint32_t b_lane = 16 * lane;
  auto copy_b = [&](int slot, int kt) {
    const float* src = b_base + (int64_t)kt * PARTS_BLOCK;
    float* dst = bs + slot * T::B_STAGE + T::B_COPIES * wave * 256;
#pragma unroll
    for (int c = 0; c < T::B_COPIES; ++c) lds_copy16_at(src + b_src[c], b_lane, dst + 256 * c);
  };

  floatx16 acc[FM][FN], low[FM][FN];   // sums of the x0 y0 products and of the others
  auto clear = [&](floatx16 (&sum)[FM][FN]) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[i][j][r] = 0.f;
  };
  clear(acc);
  clear(low);

  // operand positions of this lane in its wave's A stage: row 32 i + lrow, k quads 2 h and 2 h + 1
  const int swz = (lrow >> 1) & 3;
  int a_pos[2];
#pragma unroll
  for (int jq = 0; jq < 2; ++jq) a_pos[jq] = 4 * (4 * lrow + ((2 * h + jq) ^ swz));

  // One stage: its MFMAs, between them the split of the next stage's A rows, a part of a pair of
  // values (five VALU instructions) at a time, in the cycles the matrix cores take for the MFMA
  // before it.  The fences pin that order and the B reads one column block ahead of their use; left
  // to itself the compiler puts every split before the first MFMA.
  auto main_loop = [&](auto full_c) {
    constexpr bool FULL = decltype(full_c)::value;
    uint32x4 ap[2][FM][3];   // the A parts of this stage and of the next
    float v[FM][8];
    auto read_a = [&](int slot) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const float* src = a_wave + slot * T::A_STAGE + 512 * i;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const float4 f = *reinterpret_cast<const float4*>(src + a_pos[q]);
          v[i][4 * q] = f.x; v[i][4 * q + 1] = f.y; v[i][4 * q + 2] = f.z; v[i][4 * q + 3] = f.w;
        }
      }
    };
    constexpr int SPLITS = 12 * FM;   // part u / 4 % 3 of value pair u % 4 of row block u / 12
    auto split = [&](uint32x4 (&part)[FM][3], int u) {
      float &x = v[u / 12][2 * (u % 4)], &y = v[u / 12][2 * (u % 4) + 1];
      if (u / 4 % 3 == 0) {
        x *= PARTS_SCALE;
        y *= PARTS_SCALE;
      }
      part[u / 12][u / 4 % 3][u % 4] = take_part(x, y);
    };
    copy_a(0, 0);
    copy_b(0, 0);
    if (nk > 1) copy_a(1, 1);
    if (nk > 2) copy_a(2, 2);
    if (nk > 2) wait_vmem<2 * CHUNKS>(); else if (nk > 1) wait_vmem<CHUNKS>(); else wait_vmem<0>();
    read_a(0);
#pragma unroll
    for (int u = 0; u < SPLITS; ++u) split(ap[0], u);
    int sa = 0;   // A slot of the stage
    auto stage = [&](int kt, auto parity) {
      constexpr int cur = decltype(parity)::value;
      // the next stage's A rows and this one's B parts have landed; the A rows after them may not have
      if (kt + 2 < nk) wait_vmem<CHUNKS>(); else wait_vmem<0>();
      lds_barrier();   // every wave's B parts are there; no wave reads the slots refilled next
      if (kt + 1 < nk) copy_b(cur ^ 1, kt + 1);
      if (kt + 3 < nk) copy_a(sa, kt + 3);
      sa = sa == 2 ? 0 : sa + 1;
      const float* __restrict__ bst = bs + cur * T::B_STAGE + 4 * lane;
      uint32x4 bp[2][3];
      auto read_b = [&](int j) {
#pragma unroll
        for (int q = 0; q < 3; ++q)
          bp[j & 1][q] = *reinterpret_cast<const uint32x4*>(bst + j * PARTS_BLOCK + 256 * q);
      };
      read_b(0);
      read_a(sa);   // (past the last stage: what the slot held, split for nothing)
      __builtin_amdgcn_sched_barrier(0);
      // the smallest products first
      constexpr int NP = 8;
      constexpr int PA[NP] = {2, 1, 2, 0, 1, 1, 0, 0}, PB[NP] = {1, 2, 0, 2, 1, 0, 1, 0};
      constexpr int MFMAS = NP * FM;   // of a column block
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const bool on = FULL || j < fn_act;
        if (j + 1 < FN && (FULL || j + 1 < fn_act)) read_b(j + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < MFMAS; ++m) {
          const int q = m / FM, i = m % FM;
          if (on) {
            floatx16& sum = q == NP - 1 ? acc[i][j] : low[i][j];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ap[cur][i][PA[q]]),
                                                          __builtin_bit_cast(bf16x8, bp[j & 1][PB[q]]), sum, 0, 0, 0);
          }
          // (the first block leaves the A reads time to land)
          constexpr int FIRST = FN > 2 ? 1 : 0;
          if (j >= FIRST) {
            constexpr int N = (FN - FIRST) * MFMAS;
            const int at = (j - FIRST) * MFMAS + m;
#pragma unroll
            for (int u = at * SPLITS / N; u < (at + 1) * SPLITS / N; ++u) split(ap[cur ^ 1], u);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    int kt = 0;
    for (; kt + 2 <= nk; kt += 2) {
      stage(kt, std::integral_constant<int, 0>{});
      stage(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < nk) stage(kt, std::integral_constant<int, 0>{});
  };
  if (fn_act == FN) main_loop(std::true_type{});
  else main_loop(std::false_type{});

  // a sum that is not finite leaves a NaN here
  float probe = 0.f;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] += low[i][j][r];
        probe = __builtin_fmaf(acc[i][j][r], 0.f, probe);
      }
  if (__any(probe != 0.f)) {
    clear(acc);
    const float* arow[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int64_t mr = m0 + wave * T::WTM + 32 * i + lrow;
      const int64_t m = mr < M ? mr : M - 1;
      const int64_t d = div_rows(m, p.S, fits32);
      arow[i] = p.A[z] + d * p.lda_d + (m - d * p.S) * p.lda;
    }
    for (int kt = 0; kt < nk; ++kt)
      for (int e = 0; e < 8; ++e) {
        const int64_t k = (int64_t)kt * GBK + 8 * h + e;
        float av[FM], bv[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) av[i] = k < K ? arow[i][k] : 0.f;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          // the fp32 value again: the sum of its parts, which is exact, or its bits
          const int blk = j < fn_act ? j : fn_act - 1;
          const uint16_t* src = reinterpret_cast<const uint16_t*>(b_base + ((int64_t)blk * nk + kt) * PARTS_BLOCK) +
                                8 * lane + e;
          const uint32_t q0 = src[0], q1 = src[512], q2 = src[1024];
          const float x0 = __uint_as_float(q0 << 16), x1 = __uint_as_float(q1 << 16), x2 = __uint_as_float(q2 << 16);
          bv[j] = q0 == PARTS_RAW ? __uint_as_float(q1 << 16 | q2) : ((x0 + x1) + x2) * (1.f / PARTS_SCALE);
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[j], acc[i][j], 0, 0, 0);
      }
  } else {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] *= 1.f / (PARTS_SCALE * PARTS_SCALE);
  }
  __syncthreads();   // every wave is done with the stages before an epilogue reuses them
  parts_epilogue<EPI, T, SMEM>(p, acc, smem_ab, red, m0, n0, tile_n, wave, 0, lane, z, lower);
}

// (a 64 x 128 tile of two waves, four workgroups per CU: 3 to 9 % slower on grids past 1000 tiles, and no
// better where 128 x 128 tiles leave a second round of workgroups mostly empty)
using TileP = TileParts<1, 4, 4, 2>;    // 128 x 128, 4 waves of 32 x 128, 2 workgroups per CU
using TilePS = TileParts<1, 2, 2, 6>;   // 64 x 64, 2 waves of 32 x 64, 6 workgroups per CU

int launch_parts(const GemmArgs& a, int epi, int nz, bool small, hipStream_t stream);

}  // namespace bf
