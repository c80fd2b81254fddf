// fp32 products on gfx950: C[M][N] = R + sum_k A[m][k] B[k][n], every operand, sum and
// result fp32 (fp32 inputs of the fused linear cross entropy and of the decoder layer).
//
// v_mfma_f32_16x16x4_f32 (64 FLOP per cycle and SIMD, 157 TFLOP/s on the chip): lane l
// gives row l%16, k = l/16 of its first operand, column l%16, same k, of its second, and
// holds column l%16, rows 4(l/16) + r of the result. The first operand is B^T, so a lane
// ends with four columns of one row of C. At that rate a wave's operands need a few bytes
// per cycle only, so they come straight from global memory (L1, L2) into registers, one
// block of k ahead of their use; there is no LDS staging and no barrier in the k loop.
// Per 16-deep block of k, with g = l/16:
//   k-contiguous operand: row l%16 of each 16-row block, k = 4g .. +3 as one 16-byte load;
//   k-major operand: rows k = 4g + e, TW columns TW (l%16) .. as one load, column
//     TW (l%16) + j being row l%16 of block j.
// Both put k = 4g + e in MFMA step e. Operands whose rows or sizes are not whole aligned
// 16-byte pieces take the same loads unaligned, and single elements in the last block of k
// only (Run): element by element throughout, such products ran slower than one fed from LDS
// (1435 x 1571 x 1933 644 us, now 178; 1577 x 4454 x 79 59, now 27).
//
// What bounds it: the MFMA rate where the output fills the chip, else the length of one
// wave's k chain. Three tilings of a 256-thread workgroup, by the output's size alone:
//   128 x 128: 2 x 2 waves of 64 x 64, from kF32Tiles (one per CU) such tiles on;
//   64 x 64:   2 x 2 waves of 32 x 32, from kF32Tiles such tiles on;
//   32 x 32:   the four waves cut each k block among them (added through LDS in wave
//              order); below kF32Tiles tiles k is also cut over workgroups when the
//              caller's workspace holds the partials (splitk_reduce_kernel adds them).
// Measured (TFLOP/s over the three layouts in use): 4096^3 84-109, 2048^3 89-96,
// 512 x 16000 x 512 78-92, 512 x 1408 x 512 42-46; 256^3 5.5 us. The fp32 fused loss
// forward and backward at [512, 512, 16000] takes 407 us against 2819 us with 64 x 64
// tiles of VALU FMAs fed from LDS, and [17, 128, 1001] 56 against 183 us.
#include "gemm_kernel.hpp"

namespace eg {
namespace gk {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One operand of a product: [rows][ld], k along the rows (k-contiguous) or down them.
struct F32Op {
  const float* p;
  int64_t ld, rows;  // rows at or past `rows` read as zero
};

// How a run of an operand's elements is read: as one aligned load, as one load of any
// alignment that may run up to three elements past a row's columns (into the rest of the
// operand, so not in its last row: f32_whole), or element by element.
enum class Run { kAligned, kAny, kElements };
template <int W>
using F32Run = float __attribute__((ext_vector_type(W)));
template <int W, Run RUN>
__device__ __forceinline__ F32Run<W> f32_run(const float* p) {
  typedef F32Run<W> __attribute__((aligned(4))) any;
  if constexpr (RUN == Run::kAligned) return *reinterpret_cast<const F32Run<W>*>(p);
  else return *reinterpret_cast<const any*>(p);
}

// The 16 TW rows (or columns) of an operand from r0, k block k0 .. k0 + 15, as MFMA
// operand values: f[j][e] for block j, step e. `ext` is M or N. kAligned: 16-byte aligned rows,
// with K (k-contiguous) or ext (k-major) a multiple of 4, so every load lies inside or
// outside the operand as a whole. What is read past ext is no output's operand.
template <bool KC, int TW, Run RUN>
__device__ __forceinline__ void f32_block(const F32Op& o, int r0, int k0, int ext, int K, int m16,
                                          int g, float (&f)[TW][4]) {
  constexpr bool AL = RUN == Run::kAligned;
  if constexpr (KC) {
    const int k = k0 + 4 * g;
#pragma unroll
    for (int j = 0; j < TW; ++j) {
      const int64_t r = r0 + 16 * j + m16;
      const bool in = r < o.rows;
      const float* row = o.p + (in ? r : 0) * o.ld;
      if constexpr (RUN != Run::kElements) {
        const bool ok = in && (!AL || k < K);
        const f32x4 x = f32_run<4, RUN>(row + (!AL || k < K ? k : 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) f[j][e] = ok ? x[e] : 0.f;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool kin = k + e < K;
          const float x = row[kin ? k + e : 0];
          f[j][e] = in && kin ? x : 0.f;
        }
      }
    }
  } else {
    const int c = r0 + TW * m16;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t k = k0 + 4 * g + e;
      const bool in = k < o.rows;
      const float* row = o.p + (in ? k : 0) * o.ld;
      if constexpr (RUN != Run::kElements) {
        const F32Run<TW> x = f32_run<TW, RUN>(row + (c < ext ? c : 0));
#pragma unroll
        for (int j = 0; j < TW; ++j) f[j][e] = in ? x[j] : 0.f;
      } else {
#pragma unroll
        for (int j = 0; j < TW; ++j) {
          const bool cin = c + j < ext;
          const float x = row[cin ? c + j : 0];
          f[j][e] = in && cin ? x : 0.f;
        }
      }
    }
  }
}

// Depth up to which an operand can be read as Run::kAny: a k-contiguous one to its last whole
// run, a k-major one up to its last row, whose columns end the operand.
template <bool KC>
__device__ __forceinline__ int64_t f32_whole(const F32Op& o, int ext, int K) {
  if (KC) return K;
  return o.ld >= 4 && ext >= 4 ? (o.rows < K ? o.rows : (int64_t)K) - 1 : 0;
}

// Four columns of row `row` from `col`, plus the residual's.
__device__ __forceinline__ void f32_store(float* C, int64_t ldc, const float* R,
                                          int64_t ldr, int M, int N, int row, int col, f32x4 v) {
  typedef f32x4 __attribute__((aligned(4))) any4;
  if (row >= M) return;
  float* c = C + (int64_t)row * ldc + col;
  const float* r = R ? R + (int64_t)row * ldr + col : nullptr;
  if (col + 3 < N) {
    if (r) v += *reinterpret_cast<const any4*>(r);
    *reinterpret_cast<any4*>(c) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < N) c[e] = r ? v[e] + r[e] : v[e];
  }
}

// TW: 16-row blocks per side of a wave's tile. CUT: the waves cut k (tile 16 TW), else they
// tile 2 x 2 (tile 32 TW). Workgroup row blockIdx.y takes k blocks [y per, (y + 1) per)
// and, with part non-null, writes its sums to the [M][N] slab part[y].
template <bool AKC, bool BKC, int TW, bool CUT, bool VEC>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(F32Op a, F32Op b, float* C, int M, int N,
                                                          int K, int64_t ldc, const float* R,
                                                          int64_t ldr, int tiles_n, int per,
                                                          float* part) {
  constexpr int KU = TW == 2 ? 2 : 1;  // 16-deep k blocks per step
  constexpr int BT = CUT ? 16 * TW : 32 * TW;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m16 = lane & 15, g = lane >> 4;
  const int m0 = (int)(blockIdx.x / tiles_n) * BT, n0 = (int)(blockIdx.x % tiles_n) * BT;
  const int wm = m0 + (CUT ? 0 : (w >> 1) * 16 * TW), wn = n0 + (CUT ? 0 : (w & 1) * 16 * TW);
  // k blocks of 16 KU: this workgroup's range, dealt over the waves when they cut k
  const int nk = min((K + 16 * KU - 1) / (16 * KU), ((int)blockIdx.y + 1) * per);
  const int first = (int)blockIdx.y * per + (CUT ? w : 0);
  constexpr int STEP = CUT ? 4 : 1;
  f32x4 acc[TW][TW];
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int j = 0; j < TW; ++j) acc[i][j] = f32x4{};
  float fa[2][KU][TW][4], fb[2][KU][TW][4];
  auto load_as = [&](auto run, int set, int kb) {
    constexpr Run R = decltype(run)::value;
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      f32_block<AKC, TW, R>(a, wm, 16 * (KU * kb + u), M, K, m16, g, fa[set][u]);
      f32_block<BKC, TW, R>(b, wn, 16 * (KU * kb + u), N, K, m16, g, fb[set][u]);
    }
  };
  // without VEC: the k blocks before `whole` in unaligned loads, the last ones by elements
  const int64_t depth = VEC ? 0 : min(f32_whole<AKC>(a, M, K), f32_whole<BKC>(b, N, K));
  const int whole = (int)(depth / (16 * KU));
  auto load = [&](int set, int kb) {
    if constexpr (VEC) load_as(std::integral_constant<Run, Run::kAligned>{}, set, kb);
    else if (kb < whole) load_as(std::integral_constant<Run, Run::kAny>{}, set, kb);
    else load_as(std::integral_constant<Run, Run::kElements>{}, set, kb);
  };
  auto mul = [&](int set) {
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TW; ++i)
#pragma unroll
          for (int j = 0; j < TW; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[set][u][j][e], fa[set][u][i][e],
                                                             acc[i][j], 0, 0, 0);
  };
  if (first < nk) load(0, first);
  for (int kb = first; kb < nk; kb += 2 * STEP) {  // two register sets, by turns
    if (kb + STEP < nk) load(1, kb + STEP);
    mul(0);
    if (kb + STEP >= nk) break;
    if (kb + 2 * STEP < nk) load(0, kb + 2 * STEP);
    mul(1);
  }
  float* out = part ? part + (int64_t)blockIdx.y * M * N : C;
  const int64_t ldo = part ? N : ldc;
  const float* res = part ? nullptr : R;
  // row of block i in this lane, and the four columns of result index 4g + r
  auto rowof = [&](int i) { return AKC ? 16 * i + m16 : TW * m16 + i; };
  if constexpr (CUT) {
    __shared__ __align__(16) float buf[4][16 * TW][16 * TW + 4];
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
      for (int j = 0; j < TW; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          buf[w][rowof(i)][BKC ? 16 * j + 4 * g + r : TW * (4 * g + r) + j] = acc[i][j][r];
    __syncthreads();
    constexpr int CPR = 4 * TW;  // four-column chunks per row
    for (int c = threadIdx.x; c < 16 * TW * CPR; c += 256) {
      const int r = c / CPR, d = 4 * (c % CPR);
      f32x4 s = *reinterpret_cast<const f32x4*>(&buf[0][r][d]);
#pragma unroll
      for (int k = 1; k < 4; ++k) s += *reinterpret_cast<const f32x4*>(&buf[k][r][d]);
      f32_store(out, ldo, res, ldr, M, N, m0 + r, n0 + d, s);
    }
  } else {
#pragma unroll
    for (int i = 0; i < TW; ++i) {
      const int row = wm + rowof(i);
      if constexpr (BKC) {
#pragma unroll
        for (int j = 0; j < TW; ++j)
          f32_store(out, ldo, res, ldr, M, N, row, wn + 16 * j + 4 * g, acc[i][j]);
      } else {
        // columns TW (4g + r) + j: 4 TW consecutive ones from 4 TW g
#pragma unroll
        for (int c = 0; c < TW; ++c) {
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][(4 * c + e) % TW][(4 * c + e) / TW];
          f32_store(out, ldo, res, ldr, M, N, row, wn + 4 * TW * g + 4 * c, v);
        }
      }
    }
  }
}

// Tiling of an M x N x K product (see the file comment) and its k split over workgroups.
// Both wide tilings add k in the same order, one chain of MFMAs per output; the 32-wide one
// and each split have orders of their own.
constexpr int64_t kF32Tiles = 256, kF32MaxSplits = 8, kF32MinSteps = 8;
struct F32Plan {
  int64_t tile, tiles, splits;
};
F32Plan f32_plan(int64_t M, int64_t N, int64_t K) {
  auto tiles = [&](int64_t t) { return ((M + t - 1) / t) * ((N + t - 1) / t); };
  for (int64_t t : {128, 64})
    if (tiles(t) >= kF32Tiles) return {t, tiles(t), 1};
  const int64_t nt = tiles(32), nk = (K + 31) / 32;
  // enough splits for two workgroups per CU, each wave keeping kF32MinSteps / 4 k blocks
  const int64_t s = std::min({(2 * kF32Tiles + nt - 1) / nt, nk / kF32MinSteps, kF32MaxSplits});
  if (nt >= kF32Tiles || s < 2) return {32, nt, 1};
  const int64_t per = (nk + s - 1) / s;
  return {32, nt, (nk + per - 1) / per};
}

// The tiling of M rows of a product of `rows` rows, with the whole product's order of sums:
// its k split, and its 32-wide tiles or the wide ones that suit M.
F32Plan f32_plan_rows(int64_t M, int64_t rows, int64_t N, int64_t K) {
  F32Plan p = f32_plan(rows, N, K);
  auto tiles = [&](int64_t t) { return ((M + t - 1) / t) * ((N + t - 1) / t); };
  if (p.tile == 128 && tiles(128) < kF32Tiles) p.tile = 64;
  p.tiles = tiles(p.tile);
  return p;
}

}  // namespace
}  // namespace gk

using namespace gk;

int gemm_f32_splits(int64_t M, int64_t N, int64_t K) { return (int)f32_plan(M, N, K).splits; }

size_t gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int64_t s = f32_plan(M, N, K).splits;
  return s > 1 ? (size_t)s * M * N * sizeof(float) : 0;
}

int gemm_f32_launch(const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K,
                    int64_t lda, int64_t ldb, int64_t ldc, bool a_kc, bool b_kc, int64_t a_rows,
                    int64_t b_rows, hipStream_t st, const char* name, const float* R, int64_t ldr,
                    void* ws, size_t ws_bytes, int splits, int64_t plan_rows) {
  F32Plan p = f32_plan_rows(M, plan_rows > 0 ? plan_rows : M, N, K);
  if (splits > 0) p.splits = splits;
  if (p.splits > 1 &&
      !(ws && aligned16(ws) && ws_bytes >= (size_t)p.splits * M * N * sizeof(float)))
    p.splits = 1;
  if (p.tiles >= ((int64_t)1 << 24)) {
    set_error("%s: too many tiles", name);
    return 1;
  }
  const int ku = p.tile == 128 ? 16 : 32;  // depth of one k step
  const int64_t nk = (K + ku - 1) / ku, per = (nk + p.splits - 1) / p.splits;
  const int tiles_n = (int)((N + p.tile - 1) / p.tile);
  const bool va = aligned16(A) && lda % 4 == 0 && (a_kc ? K : M) % 4 == 0;
  const bool vb = aligned16(B) && ldb % 4 == 0 && (b_kc ? K : N) % 4 == 0;
  float* part = p.splits > 1 ? (float*)ws : nullptr;
  const bool vr = !R || (aligned16(R) && ldr % 4 == 0);
  auto go = [&](auto akc, auto bkc, auto tw, auto cut, auto vec) {
    EG_LAUNCH((gemm_f32_kernel<decltype(akc)::value, decltype(bkc)::value, decltype(tw)::value,
                               decltype(cut)::value, decltype(vec)::value>),
              dim3((unsigned)p.tiles, (unsigned)p.splits), dim3(256), 0, st,
              F32Op{A, lda, a_rows}, F32Op{B, ldb, b_rows}, C, (int)M, (int)N, (int)K, ldc, R, ldr,
              tiles_n, (int)per, part);
  };
  using TT = std::true_type;
  using FF = std::false_type;
  auto by_vec = [&](auto akc, auto bkc, auto tw, auto cut) {
    if (va && vb) go(akc, bkc, tw, cut, TT{});
    else go(akc, bkc, tw, cut, FF{});
  };
  auto by_tile = [&](auto akc, auto bkc) {
    if (p.tile == 128) by_vec(akc, bkc, std::integral_constant<int, 4>{}, FF{});
    else if (p.tile == 64) by_vec(akc, bkc, std::integral_constant<int, 2>{}, FF{});
    else by_vec(akc, bkc, std::integral_constant<int, 2>{}, TT{});
  };
  if (a_kc && b_kc) by_tile(TT{}, TT{});
  else if (a_kc) by_tile(TT{}, FF{});
  else if (b_kc) by_tile(FF{}, TT{});
  else by_tile(FF{}, FF{});
  if (int e = check_launch(name)) return e;
  if (!part) return 0;
  const bool v4 = N % 4 == 0 && aligned16(C) && ldc % 4 == 0 && vr;
  const int64_t n = M * N / (v4 ? 4 : 1);
  const dim3 rg((unsigned)((n + 255) / 256));
  if (v4)
    EG_LAUNCH((splitk_reduce_kernel<float, 4>), rg, dim3(256), 0, st, part, (int)p.splits, (int)M,
              (int)N, C, ldc, (const void*)R, ldr, 0, SegArgs{});
  else
    EG_LAUNCH((splitk_reduce_kernel<float, 1>), rg, dim3(256), 0, st, part, (int)p.splits, (int)M,
              (int)N, C, ldc, (const void*)R, ldr, 0, SegArgs{});
  return check_launch(name);
}

}  // namespace eg
