// The three-part contraction kernels (bf_gemm_parts.h) and the packing of their weights.

#include <cstring>

#include "bf_gemm_parts.h"

namespace bf {

constexpr int PACK_SEG_MAX = 16;  // weights per pack_parts_kernel launch

// Weight s owns blocks [bstart[s], bstart[s + 1]).
struct PackSegs {
  const float* B[PACK_SEG_MAX];
  uint32x4* out[PACK_SEG_MAX];
  int64_t ldb[PACK_SEG_MAX], N[PACK_SEG_MAX], K[PACK_SEG_MAX];
  int64_t bstart[PACK_SEG_MAX + 1];
  int trans_b[PACK_SEG_MAX];
  int count;
};

// One thread per lane of a column block and stage: its eight values of B, split (times PARTS_SCALE, as the
// kernels split theirs) and written as the MFMA operands of the three parts, or as PARTS_RAW and their bits
// where the first part is no finite bf16.  A weight is packed once: nothing here is worth more than its one
// launch (500 x 500: 4 us).
__global__ void pack_parts_kernel(PackSegs p) {
  int s = 0;
  while (s + 1 < p.count && (int64_t)blockIdx.x >= p.bstart[s + 1]) ++s;
  const int64_t N = p.N[s], K = p.K[s], ldb = p.ldb[s], nk = ceil_div(K, (int64_t)16);
  const float* __restrict__ B = p.B[s];
  const int64_t i = ((int64_t)blockIdx.x - p.bstart[s]) * blockDim.x + threadIdx.x;
  const int lane = (int)(i & 63);
  const int64_t kt = (i >> 6) % nk, blk = (i >> 6) / nk;
  if (blk * 32 >= N) return;
  const int64_t n = blk * 32 + (lane & 31), k0 = kt * 16 + 8 * (lane >> 5);
  uint32x4 part[3];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int64_t k = k0 + e;
    const float x = n < N && k < K ? (p.trans_b[s] ? B[n * ldb + k] : B[k * ldb + n]) : 0.f;
    float left = x * PARTS_SCALE;
    uint32_t bits[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      bits[q] = __builtin_bit_cast(uint16_t, (__bf16)left);
      left -= __uint_as_float(bits[q] << 16);
    }
    if ((bits[0] & 0x7fff) >= 0x7f80) {
      bits[0] = PARTS_RAW;
      bits[1] = __float_as_uint(x) >> 16;
      bits[2] = __float_as_uint(x) & 0xffff;
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) part[q][e / 2] = e & 1 ? part[q][e / 2] | bits[q] << 16 : bits[q];
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) p.out[s][(i >> 6) * 192 + 64 * q + lane] = part[q];
}

int64_t parts_floats(int64_t N, int64_t K) { return ceil_div(N, (int64_t)32) * ceil_div(K, (int64_t)16) * PARTS_BLOCK; }

int pack_parts(int count, const float* const* B, const int64_t* ldb, const int* trans_b, const int64_t* N,
               const int64_t* K, float* const* out, hipStream_t stream) {
  for (int base = 0; base < count; base += PACK_SEG_MAX) {
    PackSegs p;
    memset(&p, 0, sizeof(p));
    p.count = count - base < PACK_SEG_MAX ? count - base : PACK_SEG_MAX;
    int64_t blocks = 0;
    for (int q = 0; q < p.count; ++q) {
      const int j = base + q;
      p.B[q] = B[j];
      p.out[q] = reinterpret_cast<uint32x4*>(out[j]);
      p.ldb[q] = ldb[j];
      p.N[q] = N[j];
      p.K[q] = K[j];
      p.trans_b[q] = trans_b[j];
      p.bstart[q] = blocks;
      blocks += ceil_div(parts_floats(N[j], K[j]) / 12, (int64_t)256);   // 12 floats a thread
    }
    p.bstart[p.count] = blocks;
    BF_REQUIRE(blocks < (1LL << 31), "pack_parts: weights too large");
    hipLaunchKernelGGL(pack_parts_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, p);
    BF_LAUNCH_CHECK("pack_parts_kernel");
  }
  return BF_OK;
}

template <class T, bool VEC>
static int launch_tile(const GemmArgs& a, int epi, int nz, hipStream_t stream) {
  const int64_t ntiles = ceil_div(a.M, (int64_t)T::BM) * ceil_div(a.N, (int64_t)T::BN);
  BF_REQUIRE(ntiles + 8 < (1LL << 31), "gemm grid too large (M=%lld N=%lld)", (long long)a.M, (long long)a.N);
  const dim3 grid((unsigned)(ceil_div(ntiles, 8) * 8), (unsigned)nz), block(T::NT);
  if (epi == EPI_STORE) {
    hipLaunchKernelGGL((gemm_parts_kernel<EPI_STORE, T, VEC>), grid, block, 0, stream, a);
  } else if (epi == EPI_ABSSUM) {
    hipLaunchKernelGGL((gemm_parts_kernel<EPI_ABSSUM, T, VEC>), grid, block, 0, stream, a);
  } else {
    if constexpr (T::BN == NORM_BN) {
      hipLaunchKernelGGL((gemm_parts_kernel<EPI_RELAX, T, VEC>), grid, block, 0, stream, a);
    } else {
      set_error("gemm: the relaxation epilogue takes 128-column tiles");
      return BF_EINVAL;
    }
  }
  BF_LAUNCH_CHECK("gemm_parts_kernel");
  return BF_OK;
}

int launch_parts(const GemmArgs& a, int epi, int nz, bool small, hipStream_t stream) {
  bool vec = a.K % 4 == 0 && a.lda % 4 == 0 && a.lda_d % 4 == 0;
  for (int z = 0; z < nz; ++z) vec = vec && ((uintptr_t)a.A[z] & 15) == 0;
  if (vec) return small ? launch_tile<TilePS, true>(a, epi, nz, stream) : launch_tile<TileP, true>(a, epi, nz, stream);
  return small ? launch_tile<TilePS, false>(a, epi, nz, stream) : launch_tile<TileP, false>(a, epi, nz, stream);
}

}  // namespace bf
