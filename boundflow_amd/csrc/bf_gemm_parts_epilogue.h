// Epilogues of the three-part contraction kernels (bf_gemm_parts.h), over the 32 x 32 accumulator
// blocks of a wave (row 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32).
#pragma once

#include "bf_gemm_kernel.h"

namespace bf {

// Rows of a lane's 16 an epilogue takes at a time (their row operands stay in registers over
// the column blocks).
constexpr int EPI_GROUP = 4;

// Rows 32 i .. 32 i + 31 of a wave's sub-tile in a row-major output: element (r, j) of a lane's
// accumulators lies at a scalar row base plus one 32-bit lane offset (row 8 (r / 4) + r % 4
// and column block j in the scalar part), so a store needs no vector address arithmetic.
template <class T>
struct EpilogueRows {
  float* base;
  int64_t ld, row0;
  uint32_t lane_off;   // bytes: 4 (lane / 32) rows down, lane % 32 columns across
  int h;
  __device__ EpilogueRows(float* out, int64_t ld_, int64_t m0, int64_t n0, int wm, int wn, int i, int lane)
      : ld(ld_), row0(m0 + wm * T::WTM + 32 * i), h(lane >> 5) {
    base = out + row0 * ld + n0 + wn * T::WTN;
    lane_off = (uint32_t)(4 * (4 * h * ld + (lane & 31)));
  }
  __device__ int64_t row(int r) const { return row0 + 8 * (r >> 2) + 4 * h + (r & 3); }
  __device__ bool whole(int64_t M) const { return row0 + 32 <= M; }
  __device__ void put(int r, int j, float v) const {
    float* const at = base + (8 * (r >> 2) + (r & 3)) * ld + 32 * j;
    *reinterpret_cast<float*>(reinterpret_cast<char*>(at) + lane_off) = v;
  }
};

// The values of rows g .. g + EPI_GROUP - 1's vectors (ld floats a domain; one for all with ld 0, read with
// the first group) at a lane's columns col0 + 32 j.  Groups alternate between the two halves of v, so that
// one is read while the group before it is stored: the compiler moves no load over those stores.
// (bf_gemm_rank1_parts on 36864 x 256 x 256, between launches of other kernels: 13 us less than with the
// values read where they are used; 2457 x 64 x 64 1.3 us.)
template <class T>
__device__ __forceinline__ void row_vectors(const GemmArgs& p, const EpilogueRows<T>& rows, const float* vec, int64_t ld,
                                            int64_t col0, int g, bool fits32, float (&v)[2][EPI_GROUP][T::FN]) {
  float (&to)[EPI_GROUP][T::FN] = v[g / EPI_GROUP & 1];
#pragma unroll
  for (int e = 0; e < EPI_GROUP; ++e) {
    const int64_t row = rows.row(g + e) < p.M ? rows.row(g + e) : p.M - 1;
    const float* at = ld ? vec + div_rows(row, p.S, fits32) * ld : vec;
#pragma unroll
    for (int j = 0; j < T::FN; ++j) {
      const int64_t col = col0 + 32 * j;
      to[e][j] = g > 0 && !ld ? v[0][0][j] : at[col < p.N ? col : p.N - 1];
    }
  }
}

// A value of each of a lane's 16 rows.
template <class T>
__device__ __forceinline__ void row_scalars(const GemmArgs& p, const EpilogueRows<T>& rows, const float* of,
                                            float (&s)[16]) {
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = of[rows.row(r) < p.M ? rows.row(r) : p.M - 1];
}

// The store, norm or relaxation epilogue of one workgroup tile: gemm_kernel's arithmetic in its
// order, taken column block by column block so that a lane's store is one instruction.  A whole
// row block takes neither bounds nor 64-bit addresses per element: the relaxation epilogue's launch
// on 128000 x 500 x 500, both bounds, went from 914 to 833 us by it, on 36864 x 256 x 256 with
// the unrelaxed product stored too from 77.6 to 59.6 us.
// smem_ab: SMEM floats of LDS no wave reads any more; m0, n0: the tile's first row and column,
// tile_n its column tile; wm, wn: the wave's place in the tile.
template <int EPI, class T, int SMEM>
__device__ __forceinline__ void parts_epilogue(const GemmArgs& p, floatx16 (&acc)[T::FM][T::FN], float* smem_ab,
                                              float (*red)[T::BM], int64_t m0, int64_t n0, int64_t tile_n, int wm,
                                              int wn, int lane, int z, bool lower) {
  constexpr int GBM = T::BM, GBN = T::BN, GNT = T::NT, FM = T::FM, FN = T::FN;
  const int64_t M = p.M, N = p.N;
  const int t = threadIdx.x;
  const int lrow = lane & 31;
  const int h = lane >> 5;
  if constexpr (EPI == EPI_STORE) {
    float* __restrict__ C = p.C[z];
    const int64_t ldc = p.ldc;
    const bool r1 = p.r1_row != nullptr;
    const bool fits32 = M < (1LL << 31);
    auto store = [&](auto rank1) {
      constexpr bool R1 = decltype(rank1)::value;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const EpilogueRows<T> rows(C, ldc, m0, n0, wm, wn, i, lane);
        const int64_t col0 = n0 + wn * T::WTN + lrow;
        float rf[16], v[2][EPI_GROUP][FN];   // each row's rank-1 factor and vector
        if constexpr (R1) {
          row_scalars(p, rows, p.r1_row, rf);
          row_vectors(p, rows, p.r1_col, p.r1_ld, col0, 0, fits32, v);
        }
#pragma unroll
        for (int g = 0; g < 16; g += EPI_GROUP) {
          if constexpr (R1)
            if (g + EPI_GROUP < 16) row_vectors(p, rows, p.r1_col, p.r1_ld, col0, g + EPI_GROUP, fits32, v);
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            if (col0 + 32 * j >= N) continue;
#pragma unroll
            for (int e = 0; e < EPI_GROUP; ++e)
              if (rows.whole(M) || rows.row(g + e) < M) {
                if constexpr (R1)
                  rows.put(g + e, j, acc[i][j][g + e] + rf[g + e] * v[g / EPI_GROUP & 1][e][j]);
                else rows.put(g + e, j, acc[i][j][g + e]);
              }
          }
        }
      }
    };
    if (r1) store(std::true_type{});
    else store(std::false_type{});
  } else if constexpr (EPI == EPI_ABSSUM) {
    static_assert(GBN == NORM_BN || GBN == NORM_BN / 2, "the |C| epilogue takes 128- or 64-column tiles");
    // sum_n |C[m, n]| * w[d, n] over this block's columns, fixed order (norm kind 0);
    // max_n |C[m, n]| (1) or sum_n C[m, n]^2 (2) for the L1 and L2 balls.  The kind
    // is uniform over the launch: one specialisation of the epilogue per kind.
    const bool fits32 = M < (1LL << 31);
    auto norm_epilogue = [&](auto kind, auto weighted, auto seeded) {
      constexpr int NK = decltype(kind)::value;
      constexpr bool W = decltype(weighted)::value, H = decltype(seeded)::value;
      auto join = [](float a, float b) { return NK == 1 ? fmaxf(a, b) : a + b; };
      float rs[FM][16];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const EpilogueRows<T> rows(p.h_out, N, m0, n0, wm, wn, i, lane);
        const int64_t col0 = n0 + wn * T::WTN + lrow;
        float hs[16], w[2][EPI_GROUP][FN];   // each row's seed scale and column weights
        if constexpr (H && NK == 0) row_scalars(p, rows, p.h_scale, hs);
        if constexpr (W) row_vectors(p, rows, p.wvec, p.w_ld, col0, 0, fits32, w);
#pragma unroll
        for (int g = 0; g < 16; g += EPI_GROUP) {
          if constexpr (W)
            if (g + EPI_GROUP < 16) row_vectors(p, rows, p.wvec, p.w_ld, col0, g + EPI_GROUP, fits32, w);
#pragma unroll
          for (int e = 0; e < EPI_GROUP; ++e) rs[i][g + e] = 0.f;
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            if (col0 + 32 * j >= N) continue;   // columns past N hold products no one keeps
#pragma unroll
            for (int e = 0; e < EPI_GROUP; ++e) {
              const int r = g + e;
              const float a = acc[i][j][r];
              float v = NK == 2 ? a * a : fabsf(a);
              float wgt = 1.f;
              if constexpr (W) {
                wgt = w[g / EPI_GROUP & 1][e][j];
                v = v * wgt;
              }
              rs[i][r] = join(rs[i][r], v);
              if constexpr (H) {
                if (!lower || !(rows.whole(M) || rows.row(r) < M)) continue;
                if constexpr (NK != 0) {
                  rows.put(r, j, a);   // the L1/L2 seeds need the whole row's norm: made from C afterwards
                } else {
                  const float sg = (a > 0.f) ? 1.f : ((a < 0.f) ? -1.f : 0.f);
                  rows.put(r, j, W ? hs[r] * sg * wgt : hs[r] * sg);
                }
              }
            }
          }
        }
      }
      float rsum[FM];
#pragma unroll
      for (int i = 0; i < FM; ++i) rsum[i] = halve_rows16(rs[i], lrow, join);
      if ((lrow & 1) == 0) {
        const int r = lrow >> 1;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int rloc = wm * T::WTM + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
          red[wn][rloc] = rsum[i];
        }
      }
      __syncthreads();
      for (int rr = t; rr < GBM; rr += GNT) {
        const int64_t row = m0 + rr;
        if (row < M) {
          float s = 0.f;
#pragma unroll
          for (int q = 0; q < T::NWN; ++q) s = join(s, red[q][rr]);
          p.partial[z][tile_n * M + row] = s;
        }
      }
    };
    using TT = std::true_type;
    using FF = std::false_type;
    auto run = [&](auto kind) {
      if constexpr (decltype(kind)::value == 0) {
        if (p.wvec) {
          if (p.h_out) norm_epilogue(kind, TT{}, TT{});
          else norm_epilogue(kind, TT{}, FF{});
          return;
        }
      }
      if (p.h_out) norm_epilogue(kind, FF{}, TT{});
      else norm_epilogue(kind, FF{}, FF{});
    };
    if (p.norm_kind == 0) run(std::integral_constant<int, 0>{});
    else if (p.norm_kind == 1) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
  } else {
    // Relaxation of the next ReLU (crown_ibp.py:1261-1296) applied to C before
    // it is stored, so the next contraction reads A' directly; every coefficient
    // is relaxed once here instead of once per column tile of its consumer.
    static_assert(GBN == NORM_BN, "the relaxation epilogue needs BN == NORM_BN");
    // smem_ab, free by now, holds an entry per domain and column of the tile: the float4 relaxations of all
    // of them (Te), then the split terms (Ae), then the centers (Ce).  The bias of a column (Ke) and the
    // domain of a row (Re) have arrays of their own.
    constexpr int E_DOMS = SMEM / (6 * GBN);
    __shared__ float Ke[GBN];
    __shared__ int Re[GBM];
    __syncthreads();
    float4* Te = reinterpret_cast<float4*>(smem_ab);
    float* Ae = smem_ab + 4 * E_DOMS * GBN;
    float* Ce = Ae + E_DOMS * GBN;
    const int64_t m_last = (m0 + GBM < M ? m0 + GBM : M) - 1;
    const bool fits32 = M < (1LL << 31);
    const int e_first = (int)div_rows(m0, p.S, fits32);
    const int endom = (int)div_rows(m_last, p.S, fits32) - e_first + 1;
    const bool staged = endom <= E_DOMS;   // uniform; otherwise entries are read from global memory
    const bool add_e = lower && (p.e_add != nullptr);
    const bool kb_e = p.e_kbias != nullptr;
    const bool cv_e = p.e_cvec != nullptr;
    if (staged) {
      for (int q = t; q < endom * GBN; q += GNT) {
        const int dd = q / GBN, c = q % GBN;
        const int64_t n = n0 + c, d = (int64_t)e_first + dd;
        const bool ok = n < N;
        // {slope, intercept} of a nonnegative, then of a negative coefficient
        const float4 e = ok ? p.e_relax[d * N + n] : make_float4(1.f, 0.f, 1.f, 0.f);
        Te[q] = lower ? make_float4(e.z, e.w, e.x, e.y) : e;
        if (add_e) Ae[q] = ok ? p.e_add[d * p.e_add_ld + n] : 0.f;
        if (cv_e) Ce[q] = ok ? p.e_cvec[d * p.e_cvec_ld + n] : 0.f;
      }
      for (int c = t; c < GBN; c += GNT) Ke[c] = (kb_e && n0 + c < N) ? p.e_kbias[n0 + c] : 0.f;
      for (int rl = t; rl < GBM; rl += GNT) {
        const int64_t m = m0 + rl;
        Re[rl] = (m < M ? (int)div_rows(m, p.S, fits32) : e_first) - e_first;
      }
    }
    __syncthreads();
    float* __restrict__ C = p.C[z];
    float* __restrict__ Cpre = p.C_pre[z];
    float pb[FM][16], pc[FM][16];
    // LDS: staged entries, else read from global memory; X: a split term or the unrelaxed product
    // to store; CV: center sums.
    auto relax = [&](auto from_lds, auto extra, auto center) {
      constexpr bool LDS = decltype(from_lds)::value, X = decltype(extra)::value, CV = decltype(center)::value;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const EpilogueRows<T> rows(C, p.ldc, m0, n0, wm, wn, i, lane);
        const EpilogueRows<T> pre(X ? Cpre : C, p.ldc, m0, n0, wm, wn, i, lane);
#pragma unroll
        for (int g = 0; g < 16; g += EPI_GROUP) {
          int dom[EPI_GROUP];   // the row's domain: its block of LDS entries, or its rows of the global operands
#pragma unroll
          for (int e = 0; e < EPI_GROUP; ++e) {
            const int64_t row = rows.row(g + e) < M ? rows.row(g + e) : M - 1;
            if constexpr (LDS) dom[e] = Re[(int)(rows.row(g + e) - m0)] * GBN;
            else dom[e] = (int)div_rows(row, p.S, fits32);
            pb[i][g + e] = 0.f;
            pc[i][g + e] = 0.f;
          }
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const int cloc = wn * T::WTN + j * 32 + lrow;
            const int64_t col = n0 + cloc;
            if (col >= N) continue;
            const float kb = kb_e ? (LDS ? Ke[cloc] : p.e_kbias[col]) : 0.f;
#pragma unroll
            for (int q = 0; q < EPI_GROUP; ++q) {
              const int r = g + q;
              const float a = acc[i][j][r];
              const bool keep = rows.whole(M) || rows.row(r) < M;
              float4 e;
              if constexpr (LDS) {
                e = Te[dom[q] + cloc];
              } else {
                const float4 t4 = p.e_relax[(int64_t)dom[q] * N + col];
                e = lower ? make_float4(t4.z, t4.w, t4.x, t4.y) : t4;
              }
              if constexpr (X)
                if (Cpre && keep) pre.put(r, j, a);
              float out = a * (a >= 0.f ? e.x : e.z);
              if constexpr (X)
                if (add_e) out = out + (LDS ? Ae[dom[q] + cloc] : p.e_add[dom[q] * p.e_add_ld + col]);
              pb[i][r] += a * (a >= 0.f ? e.y : e.w);
              if (kb_e) pb[i][r] += out * kb;
              if constexpr (CV) pc[i][r] += out * (LDS ? Ce[dom[q] + cloc] : p.e_cvec[dom[q] * p.e_cvec_ld + col]);
              if (keep) rows.put(r, j, out);
            }
          }
        }
      }
    };
    {
      using TT = std::true_type;
      using FF = std::false_type;
      if (!staged) { if (cv_e) relax(FF{}, TT{}, TT{}); else relax(FF{}, TT{}, FF{}); }
      else if (add_e || Cpre) { if (cv_e) relax(TT{}, TT{}, TT{}); else relax(TT{}, TT{}, FF{}); }
      else { if (cv_e) relax(TT{}, FF{}, TT{}); else relax(TT{}, FF{}, FF{}); }
    }
    // fixed-order reduction over the tile's columns: 32 lanes (halve_rows16), then the NWN waves
    const AddJoin add_f;
    float rb[FM], rc[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      rb[i] = halve_rows16(pb[i], lrow, add_f);
      rc[i] = cv_e ? halve_rows16(pc[i], lrow, add_f) : 0.f;
    }
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
      if (pass == 1 && !cv_e) break;   // uniform
      if ((lrow & 1) == 0) {
        const int r = lrow >> 1;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int rloc = wm * T::WTM + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
          red[wn][rloc] = pass == 0 ? rb[i] : rc[i];
        }
      }
      __syncthreads();
      float* __restrict__ dst = pass == 0 ? p.partial[z] : p.partial_c[z];
      for (int rr = t; rr < GBM; rr += GNT) {
        const int64_t row = m0 + rr;
        if (row < M) {
          float v = 0.f;
#pragma unroll
          for (int q = 0; q < T::NWN; ++q) v += red[q][rr];
          dst[tile_n * M + row] = v;
        }
      }
      __syncthreads();
    }
  }
}

}  // namespace bf
