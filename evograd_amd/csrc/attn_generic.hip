// Causal (grouped-query) attention for the shapes the 16-bit MFMA kernels do not take:
// fp32 tensors, and head sizes other than 64 and 128 in any dtype.
//
// Same contract as attention.hip (F.scaled_dot_product_attention(q, k, v,
// is_causal=True) as called by src/evograd/ops/level3/llama3_decoder_layer/
// forward_ref.py:107, with the kv head of query head h being h / (H / Hkv), the
// repeat_interleave of :101-105): o = softmax(q k^T * scale + causal mask) v, lse =
// logsumexp of the scaled, masked scores (natural log, fp32), and the backward
// dq, dk, dv with P recomputed from lse and delta = rowsum(do * o). The reference's
// decoder layer gates its algebra at fp32 with head_dim 32 and 16
// (src/evograd/ops/level3/llama3_decoder_layer/__init__.py:55-65).
//
// Every product runs in fp32 on v_mfma_f32_16x16x4_f32 (16-bit tensors are widened as
// they are loaded), whose operands are one value per lane: A holds row l%16, k = l/16;
// B column l%16, k = l/16; the 16 x 16 result has column l%16 in lane l and row
// 4(l/16) + r in register r. Two register layouts of a 16-row tile feed them:
//   rows (load_rows): lane l holds columns 16j + 4(l/16) + e of row l%16: MFMA step
//     4j + e takes those of each lane as its four k, for A and B alike;
//   columns (load_cols): lane l holds, of row 4(l/16) + r, the columns dcol(l%16, t),
//     the A operand of a product over the tile's rows. Its k order (row 4(l/16) + r in
//     step r) is the order in which a result tile already holds its rows, so a tile of
//     P or dS is the B operand of the next product as it stands.
// So no product needs a shuffle or LDS: operands come from global memory (L2) in
// 16-byte loads, each tile's loads issued one product ahead of their use.
//
// What bounds it: with few heads the work is one long chain per row block, so the walk
// over the other side is cut over the kGenWaves waves of a workgroup (tile t to wave
// t % kGenWaves), which add their parts through LDS in wave order; the dK/dV walk is
// also cut over `parts` workgroups whose fp32 slabs attn_gen_reduce_kernel adds in
// order. At fp32 [1, 8 / 2 kv, 1024, 64] a kernel trace has 21.1 us (forward), 32.2 (dQ) and
// 41.7 + 4.7 (dK/dV and its reduction), with the matrix cores busy for 38% of the cycles of
// each, against 6031, 6316 and 30931 us for one wave per
// 64 rows on VALU FMAs (128 waves on the chip's 1024 SIMDs, about 6 us per key of the
// longest row: one dependent chain with its operands broadcast from LDS).
// No atomics: every sum has a fixed order.
//
// A masked score's weight is an exact 0, but 0 times an infinite or NaN value is NaN:
// the tiles that hold masked pairs look for such values in the operand that meets the
// zeros and, where there is one, add their products pair by pair (add_pairs).
#include "eg_common.hpp"

#include <algorithm>
#include <initializer_list>
#include <type_traits>

namespace eg {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kGenWaves = 4;
constexpr int kGenThreads = kGenWaves * 64;
constexpr int64_t kGenTarget = 512;  // workgroups: two per CU
constexpr float kGenLog2e = 1.4426950408889634f;
constexpr float kGenLn2 = 0.6931471805599453f;

__device__ __forceinline__ f32x4 gmma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Columns per lane and load of the column layout, and the column of lane index m
// (0..15), tile t: runs of kRun<DM> consecutive columns.
template <int DM> constexpr int kRun = DM >= 64 ? 4 : DM / 16;
template <int DM> __device__ __forceinline__ int dcol(int m, int t) {
  return (t / kRun<DM>) * (16 * kRun<DM>) + m * kRun<DM> + t % kRun<DM>;
}

// W consecutive columns c .. c + W - 1 of a row of D, zero past D. VEC: W | D and
// aligned rows, so one load; the address of a column past D is replaced by column 0.
template <typename T, int W, bool VEC>
__device__ __forceinline__ void load_run(const T* __restrict__ row, int c, int D, float (&x)[W]) {
  if constexpr (VEC) {
    const bool in = c < D;
    load_f32<T, W>(row + (in ? c : 0), x);
#pragma unroll
    for (int i = 0; i < W; ++i) x[i] = in ? x[i] : 0.f;
  } else {
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const bool in = c + i < D;
      const float y = to_f32(row[in ? c + i : 0]);
      x[i] = in ? y : 0.f;
    }
  }
}

// Row layout: this lane's columns of `row` (the row l%16 of the tile).
template <typename T, int DM, bool VEC>
__device__ __forceinline__ void load_rows(const T* __restrict__ row, int D, int g,
                                          float (&f)[DM / 4]) {
#pragma unroll
  for (int j = 0; j < DM / 16; ++j) {
    float x[4];
    load_run<T, 4, VEC>(row, 16 * j + 4 * g, D, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * j + e] = x[e];
  }
}

// Column layout: rows r0 + 4g + r (clamped to the slice's last row) of a [S, D] slice.
template <typename T, int DM, bool VEC>
__device__ __forceinline__ void load_cols(const T* __restrict__ slice, int r0, int S, int D, int g,
                                          int m, float (&f)[4][DM / 16]) {
  constexpr int W = kRun<DM>;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const T* row = slice + (int64_t)min(r0 + 4 * g + r, S - 1) * D;
#pragma unroll
    for (int t0 = 0; t0 < DM / 16; t0 += W) {
      float x[W];
      load_run<T, W, VEC>(row, dcol<DM>(m, t0), D, x);
#pragma unroll
      for (int i = 0; i < W; ++i) f[r][t0 + i] = x[i];
    }
  }
}

template <int DT>
__device__ __forceinline__ bool all_finite(const float (&f)[4][DT]) {
  bool ok = true;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int t = 0; t < DT; ++t) ok &= __builtin_fabsf(f[r][t]) < INFINITY;
  return __builtin_amdgcn_ballot_w64(!ok) == 0;
}

// acc += (column-layout tile f)^T w over the tile's 16 rows.
template <int DT>
__device__ __forceinline__ void add_tile(f32x4 (&acc)[DT], const float (&f)[4][DT], f32x4 w) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = gmma(f[r][t], w[r], acc[t]);
}

// The same sum pair by pair, leaving masked pairs out: bit 4G + r of `on` says whether
// row 4G + r of the tile counts for this lane's column.
template <int DT>
__device__ __forceinline__ void add_pairs(f32x4 (&acc)[DT], const float (&f)[4][DT], f32x4 w,
                                          unsigned on, int lane) {
  const int m = lane & 15, g = lane >> 4;
  for (int G = 0; G < 4; ++G)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float wr = __shfl(w[r], 16 * G + m, 64);
      const bool in = (on >> (4 * G + r)) & 1;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = __shfl(f[r][t], 16 * G + 4 * g + e, 64);
          acc[t][e] = in ? __builtin_fmaf(wr, x, acc[t][e]) : acc[t][e];
        }
    }
}

// Sum over the workgroup's waves of a 16-row result (acc tiles: this lane's row l%16,
// columns dcol(4g + e, t)), through LDS in wave order: rows row0 .. row0 + 15 below
// `rows` of dst, row stride D, times f. Every wave calls it; `buf` holds one [16][DM + 4]
// tile per wave.
template <typename TO, int DM>
__device__ __forceinline__ void store_sum(float (*buf)[16][DM + 4], const f32x4 (&acc)[DM / 16],
                                          TO* __restrict__ dst, int row0, int rows, int D,
                                          float f) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m = lane & 15, g = lane >> 4;
  __syncthreads();  // the buffer's last use is over
#pragma unroll
  for (int t = 0; t < DM / 16; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) buf[w][m][dcol<DM>(4 * g + e, t)] = acc[t][e];
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * DM; i += kGenThreads) {
    const int r = i / DM, d = i % DM;
    float s = buf[0][r][d];
#pragma unroll
    for (int k = 1; k < kGenWaves; ++k) s += buf[k][r][d];
    if (row0 + r < rows && d < D) dst[(int64_t)(row0 + r) * D + d] = from_f32<TO>(s * f);
  }
}

// Row blocks lie along y and, past what y can hold, z (gen_grid).
constexpr int64_t kGenGridY = 32768;
__device__ __forceinline__ int block_index() { return blockIdx.z * gridDim.y + blockIdx.y; }
inline dim3 gen_grid(int64_t x, int64_t blocks) {
  const int64_t y = std::min(blocks, kGenGridY);
  return dim3((unsigned)x, (unsigned)y, (unsigned)((blocks + y - 1) / y));
}

// Order in which the blocks of a triangle are taken, 0 = the longest walk. Longest first,
// so that what a CU takes last is short. PAIR, for kernels with two workgroups on a CU:
// where the whole grid is resident at once (kGenTarget), nothing is taken last and the
// second workgroup of each CU comes shortest first, so that every CU holds a long and a
// short walk. fp32 calls, longest first against paired: [1, 8 / 2 kv, 1024, 64] forward 26.2 ->
// 22.1 us, backward 91.5 -> 77.0 (the longest CU had 1.5 times the mean work), [1, 8 / 2,
// 1000, 128] forward 45.9 -> 36.9; the backward there has registers for one workgroup on
// a CU and would go 176.6 -> 189.9.
template <bool PAIR>
__device__ __forceinline__ int walk_order(int blk, int n) {
  const int first = kGenTarget / 2 / gridDim.x;  // blocks of the first workgroup on each CU
  return PAIR && (int64_t)gridDim.x * n <= kGenTarget && blk >= first ? n - 1 - (blk - first)
                                                                      : blk;
}

__device__ __forceinline__ float over_groups(float v, bool is_max) {
#pragma unroll
  for (int off = 16; off <= 32; off <<= 1) {
    const float o = __shfl_xor(v, off, 64);
    v = is_max ? fmaxf(v, o) : v + o;
  }
  return v;
}

// Forward: workgroup = 16 query rows of one head, its waves cutting the keys in tiles of
// 16 KT. The workgroups with the most keys come first.
template <typename T, int DM, bool VEC>
__global__ __launch_bounds__(kGenThreads, 2) void attn_gen_fwd_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, T* __restrict__ o,
    float* __restrict__ lse, int S, int D, int nqb, int group, float scale_log2) {
  constexpr int NS = DM / 4, DT = DM / 16, KT = DM > 64 ? 1 : 2;
  __shared__ float buf[kGenWaves][16][DM + 4];
  __shared__ float wm[kGenWaves][16], wl[kGenWaves][16];
  const int bh = blockIdx.x, blk = block_index();
  if (blk >= nqb) return;
  const int q0 = (nqb - 1 - walk_order<true>(blk, nqb)) * 16;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m16 = lane & 15, g = lane >> 4;
  const T* qs = q + (int64_t)bh * S * D;
  const T* ks = k + (int64_t)(bh / group) * S * D;
  const T* vs = v + (int64_t)(bh / group) * S * D;
  const int query = q0 + m16;
  float qf[NS];
  load_rows<T, DM, VEC>(qs + (int64_t)min(query, S - 1) * D, D, g, qf);
#pragma unroll
  for (int i = 0; i < NS; ++i) qf[i] *= scale_log2;
  f32x4 acc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) acc[t] = f32x4{};
  float m = -INFINITY, l = 0.f;
  const int nt = (min(S, q0 + 16) + 16 * KT - 1) / (16 * KT);
  float kf[KT][NS];
  auto load_k = [&](int tile) {
#pragma unroll
    for (int i = 0; i < KT; ++i)
      load_rows<T, DM, VEC>(ks + (int64_t)min(16 * (KT * tile + i) + m16, S - 1) * D, D, g, kf[i]);
  };
  if (w < nt) load_k(w);
  for (int tile = w; tile < nt; tile += kGenWaves) {
    const int key0 = 16 * KT * tile;
    float vf[KT][4][DT];
#pragma unroll
    for (int i = 0; i < KT; ++i) load_cols<T, DM, VEC>(vs, key0 + 16 * i, S, D, g, m16, vf[i]);
    f32x4 s[KT];
#pragma unroll
    for (int i = 0; i < KT; ++i) s[i] = f32x4{};
#pragma unroll
    for (int st = 0; st < NS; ++st)
#pragma unroll
      for (int i = 0; i < KT; ++i) s[i] = gmma(kf[i][st], qf[st], s[i]);
    if (tile + kGenWaves < nt) load_k(tile + kGenWaves);
    const bool masked = key0 + 16 * KT - 1 > q0;
    if (masked) {
#pragma unroll
      for (int i = 0; i < KT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (key0 + 16 * i + 4 * g + r > query) s[i][r] = -INFINITY;
    }
    float mt = -INFINITY;
#pragma unroll
    for (int i = 0; i < KT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) mt = fmaxf(mt, s[i][r]);
    const float mn = fmaxf(m, over_groups(mt, true));
    const float ref = mn == -INFINITY ? 0.f : mn;
    const float alpha = __builtin_amdgcn_exp2f(m - ref);
    l *= alpha;
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] *= alpha;
    m = mn;
#pragma unroll
    for (int i = 0; i < KT; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[i][r] = __builtin_amdgcn_exp2f(s[i][r] - ref);
        l += s[i][r];
      }
      if (masked && !all_finite<DT>(vf[i])) {
        const int n = query - (key0 + 16 * i) + 1;  // keys of the tile this query sees
        add_pairs<DT>(acc, vf[i], s[i], n >= 16 ? 0xffffu : n <= 0 ? 0u : (1u << n) - 1, lane);
      } else {
        add_tile<DT>(acc, vf[i], s[i]);
      }
    }
  }
  // The waves' maxima and sums, then their outputs, each scaled to the common maximum.
  l = over_groups(l, false);
  if (g == 0) { wm[w][m16] = m; wl[w][m16] = l; }
  __syncthreads();
  float M = wm[0][m16];
#pragma unroll
  for (int i = 1; i < kGenWaves; ++i) M = fmaxf(M, wm[i][m16]);
  const float ref = M == -INFINITY ? 0.f : M;
  float L = 0.f;
#pragma unroll
  for (int i = 0; i < kGenWaves; ++i) L += wl[i][m16] * __builtin_amdgcn_exp2f(wm[i][m16] - ref);
  const float f = __builtin_amdgcn_exp2f(m - ref) / L;
#pragma unroll
  for (int t = 0; t < DT; ++t) acc[t] *= f;
  store_sum<T, DM>(buf, acc, o + (int64_t)bh * S * D, q0, S, D, 1.f);
  if (w == 0 && g == 0 && query < S) lse[(int64_t)bh * S + query] = (M + __log2f(L)) * kGenLn2;
}

// dQ (and delta = rowsum(do * o) for the dK/dV kernel): workgroup and waves as above,
// key tiles of 16 KT.
template <typename T, int DM, bool VEC>
__global__ __launch_bounds__(kGenThreads, DM > 64 ? 1 : 2) void attn_gen_dq_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
    const T* __restrict__ dout, const T* __restrict__ o, const float* __restrict__ lse,
    float* __restrict__ delta, T* __restrict__ dq, int S, int D, int nqb, int group,
    float scale) {
  constexpr int NS = DM / 4, DT = DM / 16, KT = DM > 64 ? 1 : 2;
  __shared__ float buf[kGenWaves][16][DM + 4];
  const int bh = blockIdx.x, blk = block_index();
  if (blk >= nqb) return;
  const int q0 = (nqb - 1 - walk_order<(DM <= 64)>(blk, nqb)) * 16;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m16 = lane & 15, g = lane >> 4;
  const int query = q0 + m16, qc = min(query, S - 1);
  const int64_t row = ((int64_t)bh * S + qc) * D;
  const T* ks = k + (int64_t)(bh / group) * S * D;
  const T* vs = v + (int64_t)(bh / group) * S * D;
  const float sl2 = scale * kGenLog2e;
  float qf[NS], df[NS], dl = 0.f;
  load_rows<T, DM, VEC>(q + row, D, g, qf);
  load_rows<T, DM, VEC>(dout + row, D, g, df);
  {
    float of[NS];
    load_rows<T, DM, VEC>(o + row, D, g, of);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      dl = __builtin_fmaf(df[i], of[i], dl);
      qf[i] *= sl2;
    }
  }
  dl = over_groups(dl, false);
  const float l2 = lse[(int64_t)bh * S + qc] * kGenLog2e;
  if (w == 0 && g == 0 && query < S) delta[(int64_t)bh * S + query] = dl;
  f32x4 acc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) acc[t] = f32x4{};
  const int nt = (min(S, q0 + 16) + 16 * KT - 1) / (16 * KT);
  float kf[KT][NS], vf[KT][NS];
  auto load_kv = [&](int tile) {
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int64_t at = (int64_t)min(16 * (KT * tile + i) + m16, S - 1) * D;
      load_rows<T, DM, VEC>(ks + at, D, g, kf[i]);
      load_rows<T, DM, VEC>(vs + at, D, g, vf[i]);
    }
  };
  if (w < nt) load_kv(w);
  for (int tile = w; tile < nt; tile += kGenWaves) {
    const int key0 = 16 * KT * tile;
    float kc[KT][4][DT];
#pragma unroll
    for (int i = 0; i < KT; ++i) load_cols<T, DM, VEC>(ks, key0 + 16 * i, S, D, g, m16, kc[i]);
    f32x4 s[KT], dp[KT];
#pragma unroll
    for (int i = 0; i < KT; ++i) { s[i] = f32x4{}; dp[i] = f32x4{}; }
#pragma unroll
    for (int st = 0; st < NS; ++st)
#pragma unroll
      for (int i = 0; i < KT; ++i) {
        s[i] = gmma(kf[i][st], qf[st], s[i]);
        dp[i] = gmma(vf[i][st], df[st], dp[i]);
      }
    if (tile + kGenWaves < nt) load_kv(tile + kGenWaves);
    const bool masked = key0 + 16 * KT - 1 > q0;
#pragma unroll
    for (int i = 0; i < KT; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float ds = __builtin_amdgcn_exp2f(s[i][r] - l2) * (dp[i][r] - dl);
        s[i][r] = key0 + 16 * i + 4 * g + r > query ? 0.f : ds;
      }
      if (masked && !all_finite<DT>(kc[i])) {
        const int n = query - (key0 + 16 * i) + 1;
        add_pairs<DT>(acc, kc[i], s[i], n >= 16 ? 0xffffu : n <= 0 ? 0u : (1u << n) - 1, lane);
      } else {
        add_tile<DT>(acc, kc[i], s[i]);
      }
    }
  }
  store_sum<T, DM>(buf, acc, dq + (int64_t)bh * S * D, q0, S, D, scale);
}

// dK, dV: workgroup = 16 keys of one kv head, part pi of `parts`; the walk over the
// group's query heads and their 16-row tiles from the diagonal on is dealt out step by
// step over the parts' waves. With parts > 1 the sums go to fp32 slabs, part[pi] for dK
// and part[parts + pi] for dV ([BHkv][S][D] each).
template <typename T, int DM, bool VEC>
__global__ __launch_bounds__(kGenThreads, DM > 64 ? 1 : 2) void attn_gen_dkdv_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
    const T* __restrict__ dout, const float* __restrict__ lse, const float* __restrict__ delta,
    T* __restrict__ dk, T* __restrict__ dv, int S, int D, int BHkv, int group, float scale,
    int parts, float* __restrict__ part) {
  constexpr int NS = DM / 4, DT = DM / 16;
  __shared__ float buf[kGenWaves][16][DM + 4];
  const int bhk = blockIdx.x % BHkv, pi = blockIdx.x / BHkv;
  const int nkb = (S + 15) / 16, blk = block_index();
  if (blk >= nkb) return;
  const int k0 = walk_order<(DM <= 64)>(blk, nkb) * 16;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m16 = lane & 15, g = lane >> 4;
  const int key = k0 + m16;
  const int64_t slice = (int64_t)S * D;
  const float sl2 = scale * kGenLog2e;
  float kf[NS], vf[NS];
  load_rows<T, DM, VEC>(k + bhk * slice + (int64_t)min(key, S - 1) * D, D, g, kf);
  load_rows<T, DM, VEC>(v + bhk * slice + (int64_t)min(key, S - 1) * D, D, g, vf);
#pragma unroll
  for (int i = 0; i < NS; ++i) kf[i] *= sl2;
  f32x4 adk[DT], adv[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) { adk[t] = f32x4{}; adv[t] = f32x4{}; }
  const int ntq = (S - k0 + 15) / 16, nsteps = group * ntq, stride = parts * kGenWaves;
  float qf[NS], df[NS];
  auto load_qd = [&](int step) {
    const int64_t at = ((int64_t)bhk * group + step / ntq) * slice +
                       (int64_t)min(k0 + 16 * (step % ntq) + m16, S - 1) * D;
    load_rows<T, DM, VEC>(q + at, D, g, qf);
    load_rows<T, DM, VEC>(dout + at, D, g, df);
  };
  const int first = pi * kGenWaves + w;
  if (first < nsteps) load_qd(first);
  for (int step = first; step < nsteps; step += stride) {
    const int64_t bh = (int64_t)bhk * group + step / ntq;
    const int q0 = k0 + 16 * (step % ntq);
    float qc[4][DT], dc[4][DT];
    load_cols<T, DM, VEC>(dout + bh * slice, q0, S, D, g, m16, dc);
    load_cols<T, DM, VEC>(q + bh * slice, q0, S, D, g, m16, qc);
    float lr[4], er[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t at = bh * S + min(q0 + 4 * g + r, S - 1);
      lr[r] = lse[at] * kGenLog2e;
      er[r] = delta[at];
    }
    f32x4 s = f32x4{}, dp = f32x4{};
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      s = gmma(qf[st], kf[st], s);
      dp = gmma(df[st], vf[st], dp);
    }
    if (step + stride < nsteps) load_qd(step + stride);
    unsigned on = 0;  // this lane's rows
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = q0 + 4 * g + r;
      const bool in = row >= key && row < S;
      on |= (unsigned)in << (4 * g + r);
      const float p = __builtin_amdgcn_exp2f(s[r] - lr[r]);
      dp[r] = in ? p * (dp[r] - er[r]) : 0.f;
      s[r] = in ? p : 0.f;
    }
    if ((q0 < k0 + 16 || q0 + 16 > S) && !(all_finite<DT>(qc) && all_finite<DT>(dc))) {
      on |= __shfl_xor(on, 16, 64);
      on |= __shfl_xor(on, 32, 64);
      add_pairs<DT>(adv, dc, s, on, lane);
      add_pairs<DT>(adk, qc, dp, on, lane);
    } else {
      add_tile<DT>(adv, dc, s);
      add_tile<DT>(adk, qc, dp);
    }
  }
  if (parts > 1) {
    const int64_t slab = (int64_t)BHkv * slice;
    store_sum<float, DM>(buf, adk, part + pi * slab + bhk * slice, k0, S, D, scale);
    store_sum<float, DM>(buf, adv, part + (parts + pi) * slab + bhk * slice, k0, S, D, 1.f);
  } else {
    store_sum<T, DM>(buf, adk, dk + bhk * slice, k0, S, D, scale);
    store_sum<T, DM>(buf, adv, dv + bhk * slice, k0, S, D, 1.f);
  }
}

// dK (blockIdx.y = 0) and dV (1) of a cut walk: the parts' slabs in order, rounded once.
template <typename T>
__global__ __launch_bounds__(256) void attn_gen_reduce_kernel(const float* __restrict__ part,
                                                              int parts, int64_t n,
                                                              T* __restrict__ dk,
                                                              T* __restrict__ dv) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float* p = part + blockIdx.y * parts * n + i;
  float s = p[0];
  for (int j = 1; j < parts; ++j) s += p[j * n];
  (blockIdx.y ? dv : dk)[i] = from_f32<T>(s);
}

// f(type, DM, VEC): DM the smallest of 16, 32, 64, 128 that holds D; VEC when rows can
// be read four columns at a time (D % 4 == 0 and every tensor aligned to four elements).
template <typename F>
int gen_dispatch(int dtype, int64_t D, std::initializer_list<const void*> ptrs, const char* name,
                 F&& f) {
  auto by_vec = [&](auto tag, auto dm) -> int {
    bool vec = D % 4 == 0;
    for (const void* p : ptrs) vec = vec && (uintptr_t)p % (4 * sizeof(tag)) == 0;
    return vec ? f(tag, dm, std::true_type{}) : f(tag, dm, std::false_type{});
  };
  auto by_dim = [&](auto tag) -> int {
    if (D <= 16) return by_vec(tag, std::integral_constant<int, 16>{});
    if (D <= 32) return by_vec(tag, std::integral_constant<int, 32>{});
    if (D <= 64) return by_vec(tag, std::integral_constant<int, 64>{});
    return by_vec(tag, std::integral_constant<int, 128>{});
  };
  switch (dtype) {
    case EG_F32: return by_dim(float{});
    case EG_F16: return by_dim(f16_t{});
    case EG_BF16: return by_dim(bf16_t{});
    default: set_error("%s: unsupported dtype %d", name, dtype); return 1;
  }
}

// Parts of the dK/dV walk: at least kGenTarget workgroups (two per CU), while the
// longest walk still gives every wave kGenMinSteps steps. From the shape only.
constexpr int64_t kGenMaxParts = 8, kGenMinSteps = 2;
int64_t gen_parts(int64_t BHkv, int64_t group, int64_t S) {
  const int64_t nkb = (S + 15) / 16;
  const int64_t want = (kGenTarget + BHkv * nkb - 1) / (BHkv * nkb);
  const int64_t most = group * nkb / (kGenWaves * kGenMinSteps);
  return std::max<int64_t>(1, std::min({want, most, kGenMaxParts}));
}

}  // namespace

size_t attn_generic_part_bytes(int64_t B, int64_t H, int64_t Hkv, int64_t S, int64_t D) {
  const int64_t parts = gen_parts(B * Hkv, H / Hkv, S);
  return parts > 1 ? (size_t)2 * parts * B * Hkv * S * D * sizeof(float) : 0;
}

int attn_generic_fwd(const void* q, const void* k, const void* v, void* o, float* lse, int64_t B,
                     int64_t H, int64_t Hkv, int64_t S, int64_t D, float scale, int dtype,
                     hipStream_t st) {
  const int64_t nqb = (S + 15) / 16;
  const int group = (int)(H / Hkv);
  return gen_dispatch(dtype, D, {q, k, v}, "eg_attn_fwd", [&](auto tag, auto dm, auto vec) {
    using T = decltype(tag);
    EG_LAUNCH((attn_gen_fwd_kernel<T, decltype(dm)::value, decltype(vec)::value>),
              gen_grid(B * H, nqb), dim3(kGenThreads), 0, st, (const T*)q, (const T*)k,
              (const T*)v, (T*)o, lse, (int)S, (int)D, (int)nqb, group, scale * kGenLog2e);
    return check_launch("eg_attn_fwd(generic)");
  });
}

int attn_generic_bwd(const void* dout, const void* q, const void* k, const void* v,
                     const void* o, const float* lse, void* dq, void* dk, void* dv, float* delta,
                     float* part, int64_t B, int64_t H, int64_t Hkv, int64_t S, int64_t D,
                     float scale, int dtype, hipStream_t st) {
  const int64_t nb = (S + 15) / 16;
  const int group = (int)(H / Hkv);
  const int parts = (int)gen_parts(B * Hkv, group, S);
  return gen_dispatch(dtype, D, {dout, q, k, v, o}, "eg_attn_bwd", [&](auto tag, auto dm,
                                                                       auto vec) {
    using T = decltype(tag);
    constexpr int DM = decltype(dm)::value;
    constexpr bool VEC = decltype(vec)::value;
    EG_LAUNCH((attn_gen_dq_kernel<T, DM, VEC>), gen_grid(B * H, nb), dim3(kGenThreads), 0, st,
              (const T*)q, (const T*)k, (const T*)v, (const T*)dout, (const T*)o, lse, delta,
              (T*)dq, (int)S, (int)D, (int)nb, group, scale);
    if (int e = check_launch("eg_attn_bwd(generic dq)")) return e;
    EG_LAUNCH((attn_gen_dkdv_kernel<T, DM, VEC>), gen_grid(B * Hkv * parts, nb),
              dim3(kGenThreads), 0, st, (const T*)q, (const T*)k, (const T*)v, (const T*)dout, lse,
              delta, (T*)dk, (T*)dv, (int)S, (int)D, (int)(B * Hkv), group, scale, parts, part);
    if (int e = check_launch("eg_attn_bwd(generic dkdv)")) return e;
    if (parts == 1) return 0;
    const int64_t n = B * Hkv * S * D;
    EG_LAUNCH((attn_gen_reduce_kernel<T>), dim3((unsigned)((n + 255) / 256), 2u), dim3(256), 0, st,
              (const float*)part, parts, n, (T*)dk, (T*)dv);
    return check_launch("eg_attn_bwd(generic dkdv reduce)");
  });
}

}  // namespace eg
