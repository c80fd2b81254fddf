// Causal scaled-dot-product attention forward/backward for gfx950 (bf16/fp16
// operands, fp32 accumulation on MFMA).
//
// Semantics: F.scaled_dot_product_attention(q, k, v, is_causal=True) as used by
// src/evograd/ops/level3/llama3_decoder_layer/forward_ref.py:107:
//   o = softmax(q k^T * scale + causal mask) v,   lse = logsumexp(q k^T * scale + mask)
// Backward recomputes P = exp(q k^T * scale - lse) and, with delta = rowsum(do * o):
//   dv = P^T do,  dS = P * (dP - delta) with dP = do v^T,  dq = scale * dS k,
//   dk = scale * dS^T q.
//
// Layout: q, o, do, dq are [B, H, S, D] row-major (D contiguous); k, v, dk, dv
// are [B, Hkv, S, D] with H a multiple of Hkv (grouped-query attention: query
// head h reads kv head h / (H / Hkv), the repeat_interleave of
// src/evograd/ops/level3/llama3_decoder_layer/forward_ref.py:101-105 without the
// copy; Hkv = H is ordinary multi-head attention); lse and delta are fp32 [B, H, S].
//
// MFMA: v_mfma_f32_32x32x16_{bf16,f16}. Lane l of a wave holds, for an M x K
// operand A, row l%32 and k = 8*(l/32) .. +7; for B (K x N), column l%32 and the
// same k; the 32 x 32 fp32 result C gives lane l column l%32 and, in register r,
// row (r/4)*8 + (l/32)*4 + r%4. Every product is arranged so that its result is
// the B operand of the next one without a shuffle: the k order of that product is
// permuted to C's register order (rows 8j + 4*(l/32) + i), and its A operand is
// read from LDS in the same order.
//
// LDS tiles are row-major ([rows][D], 16-byte chunks XOR-swizzled per row) and
// are filled by direct buffer->LDS loads (no VGPR staging). One tile serves both
// operand shapes:
//   rows as A (k along D): one 16-byte ds_read_b128 per lane;
//   transposed as A (rows = D index, k along the tile's rows): two
//   ds_read_b64_tr_b16, each giving a lane 4 consecutive tile rows of one column.
// gfx950 LDS serves 256 bytes per cycle; the swizzle 4*(r%4) + (r/4)%4 puts the
// 16 rows of a b128 read in 16 distinct bank groups and the 4 rows of a
// transpose read in 4 distinct 64-byte quarters (conflict-free at D = 128).
//
// Kernels (all deterministic, no atomics):
//   attn_fwd:   workgroup = 8 waves x 32 query rows (4 waves on grids of fewer than
//               512 8-wave workgroups; 2 x 4 waves cutting the keys between them on
//               small grids of long rows, split_keys); double-buffered 64-key K and
//               V tiles; online softmax in the log2 domain against a running
//               reference max, refreshed only when a P term could exceed 2^8 (a
//               lane's sum of P terms bounds each term, so no per-tile max is
//               formed; exact: the reference point cancels in o = sum / l);
//               S^T = K Q^T, O^T += V^T P^T.
//   attn_dq:    (runs first) workgroup = 4 waves x 32 query rows (or 2 x 4 waves, as
//               above); also computes
//               delta = rowsum(do * o) for its rows into the workspace;
//               double-buffered 64-key K, V tiles; S^T = K Q^T, dP^T = V dO^T,
//               dQ^T += K^T dS^T.
//   attn_dkdv:  workgroup = NW waves x 32 keys (K in registers, the workgroup's V
//               in LDS); double-buffered 32-row Q and dO tiles from the diagonal
//               down; S = Q K^T, dP = dO V^T, dV^T += dO^T P, dK^T += Q^T dS.
// The dQ pass recomputes S and dP (7 products executed where the causal
// FLOP convention counts 5) so that no atomics are needed.
//
// Workgroup order: workgroup i runs on XCD i % 8 and every block of one (b, h)
// is mapped to the same XCD, so K/V (or Q/dO) tiles of a head are shared in
// that XCD's L2; the blocks with the most work are dispatched first.
#include "eg_common.hpp"

#include <initializer_list>
#include <type_traits>

namespace eg {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
#define EG_LDS __attribute__((address_space(3)))

template <typename T> struct MM;
template <> struct MM<bf16_t> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) { return pack2_bf16(lo, hi); }
};
template <> struct MM<f16_t> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) { return pack2_f16(lo, hi); }
};

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kRescaleBound = 256.0f;  // largest P term kept without a max refresh
constexpr int kFwdPrefetch = 4;            // forward S operand reads in flight
constexpr int kDqPrefetch = 2;             // dQ S / dP operand reads in flight

// Eight fp32 values (registers off..off+7 of a result tile) rounded and packed
// as one MFMA operand.
template <typename T>
__device__ __forceinline__ typename MM<T>::v8 pack8(const f32x16& c, int off) {
  uint4 u;
  u.x = MM<T>::pack2(c[off + 0], c[off + 1]);
  u.y = MM<T>::pack2(c[off + 2], c[off + 3]);
  u.z = MM<T>::pack2(c[off + 4], c[off + 5]);
  u.w = MM<T>::pack2(c[off + 6], c[off + 7]);
  typename MM<T>::v8 r;
  __builtin_memcpy(&r, &u, 16);
  return r;
}

// The two 16-bit values of a packed word, widened to fp32 (element 0 is bits 0..15).
template <typename T> __device__ __forceinline__ float half_lo(uint32_t u);
template <typename T> __device__ __forceinline__ float half_hi(uint32_t u);
template <> __device__ __forceinline__ float half_lo<bf16_t>(uint32_t u) { return __uint_as_float(u << 16); }
template <> __device__ __forceinline__ float half_hi<bf16_t>(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
template <> __device__ __forceinline__ float half_lo<f16_t>(uint32_t u) {
  const uint16_t b = (uint16_t)(u & 0xffffu);
  f16_t h;
  __builtin_memcpy(&h, &b, 2);
  return (float)h;
}
template <> __device__ __forceinline__ float half_hi<f16_t>(uint32_t u) {
  const uint16_t b = (uint16_t)(u >> 16);
  f16_t h;
  __builtin_memcpy(&h, &b, 2);
  return (float)h;
}

// Writes the rows of a transposed 32 x 32 result (lane = row of the output, its
// registers = 32 consecutive columns in C's order), scaled, as 8-byte stores.
template <typename T>
__device__ __forceinline__ void store_rows(uint16_t* __restrict__ row, const f32x16& c, int t,
                                           int hh, float f) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    uint2 u;
    u.x = MM<T>::pack2(c[4 * g + 0] * f, c[4 * g + 1] * f);
    u.y = MM<T>::pack2(c[4 * g + 2] * f, c[4 * g + 3] * f);
    *reinterpret_cast<uint2*>(row + 32 * t + 8 * g + 4 * hh) = u;
  }
}

// The same rows as fp32 (16-byte stores), for a split walk's partial sums.
__device__ __forceinline__ void store_rows_f32(float* __restrict__ row, const f32x16& c, int t,
                                               int hh, float f) {
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *reinterpret_cast<float4*>(row + 32 * t + 8 * g + 4 * hh) =
        make_float4(c[4 * g + 0] * f, c[4 * g + 1] * f, c[4 * g + 2] * f, c[4 * g + 3] * f);
}

// RoPE on a query row held as MFMA operands (the decoder layer's q rotation,
// src/evograd/ops/level3/llama3_decoder_layer/forward_ref.py:42-51, fused into the
// forward's Q load): f[kk] holds columns 16kk + 8hh .. +7, so f[kk] and
// f[kk + KSTEPS/2] are the two halves of the same 8 rotation pairs.
//   y1 = x1 cos1 - x2 sin1,  y2 = x2 cos2 + x1 sin2   (fp32, rounded once)
template <typename T, int D>
__device__ __forceinline__ void rotate_row(typename MM<T>::v8* f, const float* __restrict__ cr,
                                           const float* __restrict__ sr, int hh) {
  constexpr int H2 = D / 32;  // KSTEPS / 2
#pragma unroll
  for (int kk = 0; kk < H2; ++kk) {
    const int col = 16 * kk + 8 * hh;
    uint4 u1, u2;
    __builtin_memcpy(&u1, &f[kk], 16);
    __builtin_memcpy(&u2, &f[kk + H2], 16);
    const uint32_t w1[4] = {u1.x, u1.y, u1.z, u1.w}, w2[4] = {u2.x, u2.y, u2.z, u2.w};
    float c1[8], s1[8], c2[8], s2[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float4 a = *reinterpret_cast<const float4*>(cr + col + 4 * h);
      const float4 b = *reinterpret_cast<const float4*>(sr + col + 4 * h);
      const float4 c = *reinterpret_cast<const float4*>(cr + col + D / 2 + 4 * h);
      const float4 d = *reinterpret_cast<const float4*>(sr + col + D / 2 + 4 * h);
      c1[4 * h] = a.x; c1[4 * h + 1] = a.y; c1[4 * h + 2] = a.z; c1[4 * h + 3] = a.w;
      s1[4 * h] = b.x; s1[4 * h + 1] = b.y; s1[4 * h + 2] = b.z; s1[4 * h + 3] = b.w;
      c2[4 * h] = c.x; c2[4 * h + 1] = c.y; c2[4 * h + 2] = c.z; c2[4 * h + 3] = c.w;
      s2[4 * h] = d.x; s2[4 * h + 1] = d.y; s2[4 * h + 2] = d.z; s2[4 * h + 3] = d.w;
    }
    uint32_t o1[4], o2[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x1l = half_lo<T>(w1[e]), x1h = half_hi<T>(w1[e]);
      const float x2l = half_lo<T>(w2[e]), x2h = half_hi<T>(w2[e]);
      const int i = 2 * e;
      o1[e] = MM<T>::pack2(x1l * c1[i] - x2l * s1[i], x1h * c1[i + 1] - x2h * s1[i + 1]);
      o2[e] = MM<T>::pack2(x2l * c2[i] + x1l * s2[i], x2h * c2[i + 1] + x1h * s2[i + 1]);
    }
    u1 = make_uint4(o1[0], o1[1], o1[2], o1[3]);
    u2 = make_uint4(o2[0], o2[1], o2[2], o2[3]);
    __builtin_memcpy(&f[kk], &u1, 16);
    __builtin_memcpy(&f[kk + H2], &u2, 16);
  }
}

// The transpose of RoPE applied to a gradient held as transposed result tiles
// (lane = one row of the output, register r of tile t = column 32t + 8(r/4) +
// 4hh + r%4; tiles t and t + DT/2 hold the two halves): with a the first-half and
// b the second-half entries,
//   a' = a cos1 + b sin2,  b' = b cos2 - a sin1
// the gradient of the rotation above (cr, sr: this row of the tables).
template <int D>
__device__ __forceinline__ void unrotate_rows(f32x16* acc, const float* __restrict__ cr,
                                              const float* __restrict__ sr, int hh) {
  constexpr int H2 = D / 64;  // DT / 2
#pragma unroll
  for (int t = 0; t < H2; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * t + 8 * g + 4 * hh;
      const float4 c1 = *reinterpret_cast<const float4*>(cr + d);
      const float4 s1 = *reinterpret_cast<const float4*>(sr + d);
      const float4 c2 = *reinterpret_cast<const float4*>(cr + d + D / 2);
      const float4 s2 = *reinterpret_cast<const float4*>(sr + d + D / 2);
      const float cv1[4] = {c1.x, c1.y, c1.z, c1.w}, sv1[4] = {s1.x, s1.y, s1.z, s1.w};
      const float cv2[4] = {c2.x, c2.y, c2.z, c2.w}, sv2[4] = {s2.x, s2.y, s2.z, s2.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = acc[t][4 * g + i], b = acc[t + H2][4 * g + i];
        acc[t][4 * g + i] = a * cv1[i] + b * sv2[i];
        acc[t + H2][4 * g + i] = b * cv2[i] - a * sv1[i];
      }
    }
}

template <int D>
__device__ __forceinline__ int swz(int row) {
  return (((row & 3) << 2) | ((row >> 2) & 3)) & (D / 8 - 1);
}
template <int D>
__device__ __forceinline__ int toff(int row, int chunk) {
  return row * D + ((chunk ^ swz<D>(row)) << 3);
}

__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// A operand from the rows of a tile (row `row`, k = D columns 16kk + 8hh ..+7).
template <typename V, int D>
__device__ __forceinline__ V rd_rows(const uint16_t* lds, int row, int kk, int hh) {
  return *reinterpret_cast<const V*>(lds + toff<D>(row, 2 * kk + hh));
}

// A operand of a transposed tile: rows = D index dd0 + l%32, k = 16 tile rows
// from r16 in the permuted order r16 + 4hh + {0..3}, r16 + 8 + 4hh + {0..3}.
// ds_read_b64_tr_b16: within each 16-lane group, lane j receives element j%4 of
// the 8 bytes addressed by lanes 4i + j/4 (i = 0..3), so lane j points at row
// 4hh + j/4, columns 4*(j%4) .. +3 and receives column j of rows +0..3.
template <typename V, int D>
__device__ __forceinline__ V rd_tr(const uint16_t* lds, int r16, int dd0, int lane) {
  const int m = lane & 15, gs = (lane >> 4) & 1, hh = lane >> 5;
  const int col = dd0 + 16 * gs + 4 * (m & 3);
  const int chunk = col >> 3, sub = col & 7;
  const int r0 = r16 + 4 * hh + (m >> 2);
  const i16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((EG_LDS i16x4*)(lds + toff<D>(r0, chunk) + sub));
  const i16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((EG_LDS i16x4*)(lds + toff<D>(r0 + 8, chunk) + sub));
  V r;
  __builtin_memcpy(&r, &a, 8);
  __builtin_memcpy(reinterpret_cast<char*>(&r) + 8, &b, 8);
  return r;
}

// Copies rows [row0, row0 + ROWS) of a [nrows, D] slice into a swizzled LDS tile
// with 16-byte buffer->LDS loads. Each lane's offset inside the tile is fixed;
// the buffer resource starts at row0 and ends at the slice's last row, so rows
// past the slice are not fetched: their LDS rows are written with zeros (the
// bounded-access rules in eg_common.hpp).
template <int ROWS, int D, int NW>
struct TileLoader {
  static constexpr int CPR = D / 8;
  static constexpr int ITER = ROWS * CPR / (64 * NW);
  static_assert(ITER >= 1 && ITER * 64 * NW == ROWS * CPR, "tile must split evenly over the waves");
  int voff[ITER], w;  // w: this wave among the NW that load the tile
  __device__ __forceinline__ void init(int wave) {
    const int lane = threadIdx.x & 63;
    w = wave;
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
      const int p = (it * NW + w) * 64 + lane;
      const int r = p / CPR;
      const int c = (p % CPR) ^ swz<D>(r);
      voff[it] = (r * D + c * 8) * 2;
    }
  }
  __device__ __forceinline__ void load(const uint16_t* slice, int row0, int nrows,
                                       uint16_t* lds) const {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(slice + (int64_t)row0 * D), (short)0, (nrows - row0) * D * 2,
        0x00020000);
#pragma unroll
    for (int it = 0; it < ITER; ++it)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (EG_LDS void*)(lds + (it * NW + w) * 64 * 8), 16,
                                               voff[it], 0, 0, 0);
  }
};

__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int NT>
__device__ __forceinline__ void zero_lds(void* p, int bytes) {
  uint4* z = reinterpret_cast<uint4*>(p);
  for (int e = threadIdx.x; e < bytes / 16; e += NT) z[e] = make_uint4(0, 0, 0, 0);
}

// Workgroup i -> (head, block index): XCD i % 8 holds heads xcd, xcd + 8, ...;
// block index 0 is dispatched first for every head.
__device__ __forceinline__ void block_coords(int BH, int& bh, int& blk) {
  const int i = blockIdx.x;
  const int xcd = i % 8, rest = i / 8;
  const int groups = (BH + 7) / 8;
  bh = xcd + 8 * (rest % groups);
  blk = rest / groups;
}

// Grouped-query attention: query head `bh_q` (flat over batch x heads) reads key/
// value head bh_q / group. A virtual head index v (the one block_coords spreads
// over the XCDs) maps to bh_q = (v % BHkv) * group + v / BHkv, so the `group`
// query heads that share a kv head have the same v % 8, i.e. the same XCD and L2,
// whenever BHkv is a multiple of 8. With group = 1 this is the identity.
__device__ __forceinline__ int query_head(int v, int BHkv, int group) {
  return (v % BHkv) * group + v / BHkv;
}

// ------------------------------------------------------------------ forward
// KG = 2: two groups of NW waves share the workgroup's rows and take the key tiles by
// turns, each with tile buffers, a reference max, sums and an output of its own; group 1
// hands these to group 0 through LDS at the end. Halves the chain of tiles of a row block,
// which is what bounds a grid that leaves the chip's SIMDs with one wave or less.
template <typename T, int D, int NW, int KG, bool ROPE>
__global__ __launch_bounds__(NW * KG * 64, 2) void attn_fwd_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, uint16_t* __restrict__ o, float* __restrict__ lse, int S,
    float scale_log2, int nqb, int BH, int group, const float* __restrict__ rope_cos,
    const float* __restrict__ rope_sin) {
  using v8 = typename MM<T>::v8;
  constexpr int BM = 32 * NW, BN = 64;
  constexpr int KSTEPS = D / 16, DT = D / 32;
  // One __shared__ object per buffer (see the file comment): LDS reads of one
  // buffer never wait for the loads in flight into the other.
  __shared__ __align__(16) uint16_t Ks0[KG * BN * D], Ks1[KG * BN * D];
  __shared__ __align__(16) uint16_t Vs0[KG * BN * D], Vs1[KG * BN * D];

  int vh, blk;
  block_coords(BH, vh, blk);
  if (vh >= BH) return;
  const int bh = query_head(vh, BH / group, group);
  const int q0 = (nqb - 1 - blk) * BM;  // longest rows first
  const int lane = threadIdx.x & 63;
  const int w = KG == 1 ? wave_id() : wave_id() % NW, kg = KG == 1 ? 0 : wave_id() / NW;
  const int kvo = kg * BN * D;  // this group's tile buffers
  const int l32 = lane & 31, hh = lane >> 5;
  const int64_t base = (int64_t)bh * S * D;
  const int64_t kvbase = (int64_t)(bh / group) * S * D;
  const uint16_t* kp = k + kvbase;
  const uint16_t* vp = v + kvbase;

  const int qrow = q0 + 32 * w + l32;
  const int qrc = qrow < S ? qrow : S - 1;
  v8 qf[KSTEPS];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk)
    qf[kk] = *reinterpret_cast<const v8*>(q + base + (int64_t)qrc * D + kk * 16 + 8 * hh);

  // Element offsets of this lane's operand reads inside a tile, computed once: the
  // S reads (row l32, chunk 2kk + hh; the second 32-row half adds 32 * D) and the
  // transposed V reads (rows 4hh + m/4 and +8 of each 16-row step, column block t;
  // step ms adds 16 * D). With the tile loop unrolled over the two buffers, each
  // read is one of these registers plus an immediate.
  int offS[KSTEPS], offV[DT][2];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) offS[kk] = toff<D>(l32, 2 * kk + hh);
  {
    const int mq = lane & 15, gs = (lane >> 4) & 1, r0 = 4 * hh + (mq >> 2);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int col = 32 * t + 16 * gs + 4 * (mq & 3);
      offV[t][0] = toff<D>(r0, col >> 3) + (col & 7);
      offV[t][1] = toff<D>(r0 + 8, col >> 3) + (col & 7);
    }
  }

  f32x16 acc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) acc[t] = f32x16{};
  float m = -INFINITY, lsum = 0.f;
  const int kv_end = min(S, q0 + BM);
  const int ntiles = (kv_end + BN - 1) / BN;
  const int nturns = (ntiles + KG - 1) / KG;  // tile KG * j + kg in turn j
  const int wave_first_row = q0 + 32 * w;

  zero_lds<NW * KG * 64>(Ks0, sizeof(Ks0));
  zero_lds<NW * KG * 64>(Ks1, sizeof(Ks1));
  zero_lds<NW * KG * 64>(Vs0, sizeof(Vs0));
  zero_lds<NW * KG * 64>(Vs1, sizeof(Vs1));
  __syncthreads();
  TileLoader<BN, D, NW> ld;
  ld.init(w);
  if (kg < ntiles) {
    ld.load(kp, kg * BN, S, Ks0 + kvo);
    ld.load(vp, kg * BN, S, Vs0 + kvo);
  }
  // The rotation waits for q and the tables, so it comes after the first tile's
  // loads are issued: those are in flight meanwhile.
  if constexpr (ROPE)
    rotate_row<T, D>(qf, rope_cos + (int64_t)qrc * D, rope_sin + (int64_t)qrc * D, hh);
  auto tile = [&](auto bufc, int j) {
    constexpr int buf = decltype(bufc)::value;
    wait_loads();
    __syncthreads();
    const int next = KG * (j + 1) + kg;
    if (next < ntiles) {
      ld.load(kp, next * BN, S, (buf ? Ks0 : Ks1) + kvo);
      ld.load(vp, next * BN, S, (buf ? Vs0 : Vs1) + kvo);
    }
    const int k0 = (KG * j + kg) * BN;
    // every key of the tile is above this wave's rows (a tile past the last one too)
    if (k0 > wave_first_row + 31) return;
    if (KG > 1 && k0 >= kv_end) return;
    const uint16_t* Kb = (buf ? Ks1 : Ks0) + kvo;
    const uint16_t* Vb = (buf ? Vs1 : Vs0) + kvo;
    f32x16 s[2];
    // S^T = K Q^T with the K operand reads kFwdPrefetch MFMAs ahead of their use
    // (MFMA i takes (kk, T2) = (i / 2, i % 2)); the scheduling groups keep that
    // order, which the default schedule would collapse to one read ahead. Keys past
    // the diagonal (and past S) are set to -inf (diagonal tiles only).
    auto scores = [&]() {
      s[0] = f32x16{};
      s[1] = f32x16{};
      constexpr int NM = 2 * KSTEPS, PF = kFwdPrefetch;
      v8 ring[PF];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < PF; ++i)
        ring[i] = *reinterpret_cast<const v8*>(Kb + offS[i >> 1] + 32 * D * (i & 1));
#pragma unroll
      for (int i = 0; i < NM; ++i) {
        s[i & 1] = MM<T>::mma(ring[i % PF], qf[i >> 1], s[i & 1]);
        if (i + PF < NM)
          ring[i % PF] =
              *reinterpret_cast<const v8*>(Kb + offS[(i + PF) >> 1] + 32 * D * ((i + PF) & 1));
      }
      __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);  // the first PF LDS reads
#pragma unroll
      for (int i = 0; i < NM; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        if (i + PF < NM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one read
      }
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + BN - 1 > wave_first_row) {
#pragma unroll
        for (int T2 = 0; T2 < 2; ++T2)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = k0 + 32 * T2 + (r >> 2) * 8 + 4 * hh + (r & 3);
            if (key > qrow) s[T2][r] = -INFINITY;
          }
      }
    };
    auto exps = [&](float nm) {
      float sum = 0.f;
#pragma unroll
      for (int T2 = 0; T2 < 2; ++T2)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[T2][r], scale_log2, nm));
          s[T2][r] = p;
          sum += p;
        }
      return sum;
    };
    scores();
    // P against the running reference max m (log2 units), in place. A lane's sum of
    // its 32 terms bounds each of them, so a sum <= 2^8 shows that no score of its
    // row grew past m + 8. Otherwise (and on the first tile, where m is -inf, or
    // on overflow) the tile's scores are formed again, the row max is taken, the
    // running sums are rescaled to it and P is recomputed.
    float ps = 0.f;
    bool refresh = j == 0;
    if (!refresh) {
      ps = exps(-m);
      refresh = __builtin_amdgcn_ballot_w64(!(ps <= kRescaleBound)) != 0;
      if (refresh) scores();
    }
    if (refresh) {
      float mt = -INFINITY;
#pragma unroll
      for (int T2 = 0; T2 < 2; ++T2)
#pragma unroll
        for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[T2][r]);
      mt = fmaxf(mt, __shfl_xor(mt, 32, 64)) * scale_log2;
      const float m_new = fmaxf(m, mt);
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      lsum *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t) acc[t] *= alpha;
      m = m_new;
      ps = exps(m == -INFINITY ? 0.f : -m);
    }
    lsum += ps;
#pragma unroll
    for (int ms = 0; ms < BN / 16; ++ms) {
      const v8 pb = pack8<T>(s[ms >> 1], 8 * (ms & 1));
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (EG_LDS i16x4*)(Vb + offV[t][0] + 16 * D * ms));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (EG_LDS i16x4*)(Vb + offV[t][1] + 16 * D * ms));
        v8 va;
        __builtin_memcpy(&va, &lo, 8);
        __builtin_memcpy(reinterpret_cast<char*>(&va) + 8, &hi, 8);
        acc[t] = MM<T>::mma(va, pb, acc[t]);
      }
    }
  };
  for (int j = 0; j < nturns; j += 2) {
    tile(std::integral_constant<int, 0>{}, j);
    if (j + 1 < nturns) tile(std::integral_constant<int, 1>{}, j + 1);
  }
  if constexpr (KG > 1) {
    // Group 1's values in the lane that holds the same rows in group 0, half of the output
    // tiles in each K buffer.
    constexpr int HT = DT / 2, STRIDE = NW * 64;
    static_assert(HT * 16 * STRIDE * 4 <= (int)sizeof(Ks0), "half the output fits a buffer");
    float* half0 = reinterpret_cast<float*>(Ks0);
    float* half1 = reinterpret_cast<float*>(Ks1);
    float* ml = reinterpret_cast<float*>(Vs0);
    const int at = w * 64 + lane;
    __syncthreads();  // the last tiles are consumed
    if (kg == 1) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          (t < HT ? half0 : half1)[((t % HT) * 16 + r) * STRIDE + at] = acc[t][r];
      ml[at] = m;
      ml[STRIDE + at] = lsum;
    }
    __syncthreads();
    if (kg == 1) return;
    const float m1 = ml[at], mx = fmaxf(m, m1), ref = mx == -INFINITY ? 0.f : mx;
    const float a0 = __builtin_amdgcn_exp2f(m - ref), a1 = __builtin_amdgcn_exp2f(m1 - ref);
    lsum = lsum * a0 + ml[STRIDE + at] * a1;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[t][r] = acc[t][r] * a0 +
                    (t < HT ? half0 : half1)[((t % HT) * 16 + r) * STRIDE + at] * a1;
    m = mx;
  }

  const float ltot = lsum + __shfl_xor(lsum, 32, 64);
  if (qrow < S) {
    const float inv = 1.0f / ltot;
    uint16_t* op = o + base + (int64_t)qrow * D;
#pragma unroll
    for (int t = 0; t < DT; ++t) store_rows<T>(op, acc[t], t, hh, inv);
    if (hh == 0) lse[(int64_t)bh * S + qrow] = (m + log2f(ltot)) * kLn2;
  }
}

// ------------------------------------------------------------ dK, dV
template <typename T, int D, int NW, int BQ, bool ROPE>
__global__ __launch_bounds__(NW * 64, 2) void attn_dkdv_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, const uint16_t* __restrict__ dout,
    const float* __restrict__ lse, const float* __restrict__ delta, uint16_t* __restrict__ dk,
    uint16_t* __restrict__ dv, int S, float scale, float scale_log2, int BHkv, int group,
    const float* __restrict__ rope_cos, const float* __restrict__ rope_sin, int parts,
    float* __restrict__ part) {
  using v8 = typename MM<T>::v8;
  constexpr int BK = 32 * NW;
  constexpr int KSTEPS = D / 16, DT = D / 32;
  static_assert(BQ == 32, "one 32-row Q / dO tile per step");
  __shared__ __align__(16) uint16_t Qs0[BQ * D], Qs1[BQ * D];  // one object per buffer
  __shared__ __align__(16) uint16_t Ds0[BQ * D], Ds1[BQ * D];
  // V of the workgroup's keys: the B operand of dP = dO V^T, read from LDS so
  // that its 64 registers per wave stay free for operand staging.
  __shared__ __align__(16) uint16_t Vk[BK * D];
  __shared__ __align__(16) float Ls[2][BQ];
  __shared__ __align__(16) float Es[2][BQ];

  // Workgroup (kv head, part of the walk, key block); with parts > 1 the walk
  // below is cut into `parts` ranges of steps, each summed into its own fp32 slab
  // of `part` (attn_dkdv_reduce_kernel adds the slabs in order). The parts of a
  // kv head share its XCD when BHkv is a multiple of 8.
  int vh, kb;
  block_coords(BHkv * parts, vh, kb);  // kb = 0 (the longest walk) first
  if (vh >= BHkv * parts) return;
  const int kvh = vh % BHkv, pi = vh / BHkv;
  const int k0 = kb * BK;
  const int lane = threadIdx.x & 63, w = wave_id();
  const int l32 = lane & 31, hh = lane >> 5;
  const int64_t base = (int64_t)kvh * S * D;  // k, v, dk, dv

  const int key = k0 + 32 * w + l32;
  const int krc = key < S ? key : S - 1;
  v8 kf[KSTEPS];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk)
    kf[kk] = *reinterpret_cast<const v8*>(k + base + (int64_t)krc * D + kk * 16 + 8 * hh);
  f32x16 dka[DT], dva[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) { dka[t] = f32x16{}; dva[t] = f32x16{}; }

  // Operand read offsets as one register per read family. The fields of toff() are
  // disjoint bit ranges (row * D, chunk ^ swizzle in bits 3-6, the 4-column
  // sub-offset in bit 2), and the swizzle depends on the row's low 4 bits only, so
  //   rows as A operand, row l32 (+32 for this wave's V rows), chunk 2kk + hh:  R0 ^ 16kk
  //   transposed reads, column block t, rows r0 / r0 + 8 (+16 per ms step):    T0[j] ^ 32t
  const int R0 = toff<D>(l32, hh);
  int T0[2];
  {
    const int mq = lane & 15, gs = (lane >> 4) & 1, r0 = 4 * hh + (mq >> 2);
    const int col = 16 * gs + 4 * (mq & 3);
    T0[0] = toff<D>(r0, col >> 3) + (col & 7);
    T0[1] = toff<D>(r0 + 8, col >> 3) + (col & 7);
  }
  const uint16_t* Vw = Vk + 32 * w * D;  // this wave's 32 keys

  zero_lds<NW * 64>(Qs0, sizeof(Qs0));
  zero_lds<NW * 64>(Qs1, sizeof(Qs1));
  zero_lds<NW * 64>(Ds0, sizeof(Ds0));
  zero_lds<NW * 64>(Ds1, sizeof(Ds1));
  zero_lds<NW * 64>(Vk, sizeof(Vk));
  // The walk: for each query head of the group (in order), the q tiles from the
  // diagonal block to S. dK and dV accumulate over all of them in registers, so
  // the kv-head gradient is the group sum without atomics or a second pass.
  const int i_first = k0 / BQ;
  const int ntq = (S + BQ - 1) / BQ - i_first;
  const int nsteps = group * ntq;
  const int per = (nsteps + parts - 1) / parts;
  const int s_begin = min(nsteps, pi * per), s_end = min(nsteps, s_begin + per);
  const int wave_first_key = k0 + 32 * w;
  TileLoader<BQ, D, NW> ld;
  ld.init(w);
  auto qhead = [&](int step) { return kvh * group + step / ntq; };
  auto qtile = [&](int step) { return i_first + step % ntq; };
  // lse and delta of a tile's rows: wave 0 loads them when the tile is requested
  // and converts and stores them to LDS only after the current step's compute, so
  // that waiting for them does not hold that compute behind the tile loads.
  float lraw = 0.f, eraw = 0.f;
  bool lrow = false;
  auto load_stats = [&](int step) {
    if (w == 0 && lane < BQ) {
      const int64_t hb = (int64_t)qhead(step) * S;
      const int row = qtile(step) * BQ + lane;
      const int rc = row < S ? row : S - 1;
      lraw = lse[hb + rc];
      eraw = delta[hb + rc];
      lrow = row < S;
    }
  };
  auto store_stats = [&](float* ls, float* es) {
    if (w == 0 && lane < BQ) {
      ls[lane] = lrow ? lraw * kLog2e : INFINITY;  // rows past S: p = 0
      es[lane] = lrow ? eraw : 0.f;
    }
  };
  __syncthreads();
  {
    TileLoader<BK, D, NW> lv;  // keys past S stay zero
    lv.init(w);
    lv.load(v + base, k0, S, Vk);
  }
  if (s_begin < s_end) {
    const int64_t hb = (int64_t)qhead(s_begin) * S * D;
    ld.load(q + hb, qtile(s_begin) * BQ, S, Qs0);
    ld.load(dout + hb, qtile(s_begin) * BQ, S, Ds0);
    load_stats(s_begin);
    store_stats(Ls[0], Es[0]);
  }
  auto step_fn = [&](auto bufc, int step) {
    constexpr int buf = decltype(bufc)::value;
    wait_loads();
    __syncthreads();
    const bool more = step + 1 < s_end;
    if (more) {
      const int64_t hb = (int64_t)qhead(step + 1) * S * D;
      ld.load(q + hb, qtile(step + 1) * BQ, S, buf ? Qs0 : Qs1);
      ld.load(dout + hb, qtile(step + 1) * BQ, S, buf ? Ds0 : Ds1);
      load_stats(step + 1);
    }
    const int qi0 = qtile(step) * BQ;
    if (qi0 + BQ - 1 >= wave_first_key) {  // some row of the tile sees some key of this wave
      const uint16_t* Qb = buf ? Qs1 : Qs0;
      const uint16_t* Db = buf ? Ds1 : Ds0;
      // Opaque copies of the offset registers: the XORs are redone in each step
      // instead of being hoisted out of the loop into 24 live registers.
      int r0 = R0, t0 = T0[0], t1 = T0[1];
      asm volatile("" : "+v"(r0), "+v"(t0), "+v"(t1));
      auto offR = [&](int kk) { return r0 ^ (16 * kk); };
      auto offT = [&](int t, int j) { return (j ? t1 : t0) ^ (32 * t); };
      // S = Q K^T and dP = dO V^T, the three operand reads of step kk + 1 issued
      // before the two MFMAs of step kk (scheduling groups keep that order).
      f32x16 s = f32x16{}, dp = f32x16{};
      {
        v8 qa[2], da[2], vb[2];
        __builtin_amdgcn_sched_barrier(0);
        qa[0] = *reinterpret_cast<const v8*>(Qb + offR(0));
        da[0] = *reinterpret_cast<const v8*>(Db + offR(0));
        vb[0] = *reinterpret_cast<const v8*>(Vw + offR(0));
#pragma unroll
        for (int kk = 0; kk < KSTEPS; ++kk) {
          if (kk + 1 < KSTEPS) {
            qa[(kk + 1) & 1] = *reinterpret_cast<const v8*>(Qb + offR(kk + 1));
            da[(kk + 1) & 1] = *reinterpret_cast<const v8*>(Db + offR(kk + 1));
            vb[(kk + 1) & 1] = *reinterpret_cast<const v8*>(Vw + offR(kk + 1));
          }
          s = MM<T>::mma(qa[kk & 1], kf[kk], s);
          dp = MM<T>::mma(da[kk & 1], vb[kk & 1], dp);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
        for (int kk = 0; kk < KSTEPS; ++kk) {
          if (kk + 1 < KSTEPS) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // P = exp(S * scale - lse); register r holds row 8(r/4) + 4hh + r%4.
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 l4 = *reinterpret_cast<const float4*>(&Ls[buf][8 * g + 4 * hh]);
        const float lv[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          s[4 * g + i4] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * g + i4], scale_log2, -lv[i4]));
      }
      // Causal mask, in the diagonal steps only (a wave-uniform branch): row
      // qi0 + 8g + 4hh + i4 sees this lane's key iff 8g + i4 >= key - qi0 - 4hh.
      if (qi0 < wave_first_key + 31) {
        const int mask_below = key - qi0 - 4 * hh;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + (r & 3) < mask_below) s[r] = 0.f;
      }
      // dS = P (dP - delta)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 e4 = *reinterpret_cast<const float4*>(&Es[buf][8 * g + 4 * hh]);
        const float ev[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          dp[4 * g + i4] = s[4 * g + i4] * (dp[4 * g + i4] - ev[i4]);
      }
      // dV^T += dO^T P and dK^T += Q^T dS in the order (ms, t, dV then dK), each
      // MFMA's transposed operand read one MFMA ahead (two ds_read_b64_tr_b16); the
      // scheduling groups keep that order, which the default schedule collapses to
      // a wait before every MFMA.
      constexpr int NM = 2 * DT * (BQ / 16);
      auto rd = [&](int i) {
        const int ms = i / (2 * DT), t = (i / 2) % DT;
        const uint16_t* tb = (i & 1) ? Qb : Db;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (EG_LDS i16x4*)(tb + offT(t, 0) + 16 * D * ms));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (EG_LDS i16x4*)(tb + offT(t, 1) + 16 * D * ms));
        v8 r;
        __builtin_memcpy(&r, &lo, 8);
        __builtin_memcpy(reinterpret_cast<char*>(&r) + 8, &hi, 8);
        return r;
      };
      v8 op[2], pb, sb;
      __builtin_amdgcn_sched_barrier(0);
      op[0] = rd(0);
#pragma unroll
      for (int i = 0; i < NM; ++i) {
        if (i + 1 < NM) op[(i + 1) & 1] = rd(i + 1);
        const int ms = i / (2 * DT), t = (i / 2) % DT;
        if (i % (2 * DT) == 0) {
          pb = pack8<T>(s, 8 * ms);
          sb = pack8<T>(dp, 8 * ms);
        }
        if (i & 1) dka[t] = MM<T>::mma(op[i & 1], sb, dka[t]);
        else dva[t] = MM<T>::mma(op[i & 1], pb, dva[t]);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
      for (int i = 0; i < NM; ++i) {
        if (i + 1 < NM) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) store_stats(Ls[buf ^ 1], Es[buf ^ 1]);
  };
  // Unrolled over the two buffers, so every LDS address is a register plus an
  // immediate and the buffers are distinct objects at compile time.
  for (int step = s_begin; step < s_end; step += 2) {
    step_fn(std::integral_constant<int, 0>{}, step);
    if (step + 1 < s_end) step_fn(std::integral_constant<int, 1>{}, step + 1);
  }

  if (key < S) {
    uint16_t* dkp = dk + base + (int64_t)key * D;
    uint16_t* dvp = dv + base + (int64_t)key * D;
    float fk = scale;
    if constexpr (ROPE) {  // dk of the pre-rotation keys: the rotation's transpose
#pragma unroll
      for (int t = 0; t < DT; ++t) dka[t] *= scale;
      unrotate_rows<D>(dka, rope_cos + (int64_t)key * D, rope_sin + (int64_t)key * D, hh);
      fk = 1.0f;
    }
    if (part) {  // this part's sums, scaled (and unrotated) like the direct store
      const int64_t slab = (int64_t)BHkv * S * D;
      float* pk = part + pi * slab + base + (int64_t)key * D;
      float* pv = part + (parts + pi) * slab + base + (int64_t)key * D;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        store_rows_f32(pk, dka[t], t, hh, fk);
        store_rows_f32(pv, dva[t], t, hh, 1.0f);
      }
    } else {
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        store_rows<T>(dkp, dka[t], t, hh, fk);
        store_rows<T>(dvp, dva[t], t, hh, 1.0f);
      }
    }
  }
}

// dK, dV of a split walk: the parts' fp32 slabs ([2][parts][BHkv][S][D], dK slabs
// first) added in part order and rounded once; 4 consecutive elements of each per
// thread (D is a multiple of 4).
template <typename T>
__global__ __launch_bounds__(256) void attn_dkdv_reduce_kernel(const float* __restrict__ part,
                                                               int parts, int64_t n,
                                                               uint16_t* __restrict__ dk,
                                                               uint16_t* __restrict__ dv) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  float4 a = *reinterpret_cast<const float4*>(part + i);
  float4 b = *reinterpret_cast<const float4*>(part + parts * n + i);
  for (int p = 1; p < parts; ++p) {
    const float4 x = *reinterpret_cast<const float4*>(part + p * n + i);
    const float4 y = *reinterpret_cast<const float4*>(part + (parts + p) * n + i);
    a.x += x.x, a.y += x.y, a.z += x.z, a.w += x.w;
    b.x += y.x, b.y += y.y, b.z += y.z, b.w += y.w;
  }
  uint2 u;
  u.x = MM<T>::pack2(a.x, a.y);
  u.y = MM<T>::pack2(a.z, a.w);
  *reinterpret_cast<uint2*>(dk + i) = u;
  u.x = MM<T>::pack2(b.x, b.y);
  u.y = MM<T>::pack2(b.z, b.w);
  *reinterpret_cast<uint2*>(dv + i) = u;
}

// ------------------------------------------------------------------- dQ
// KG as in the forward.
template <typename T, int D, int NW, int KG, bool ROPE>
__global__ __launch_bounds__(NW * KG * 64, 2) void attn_dq_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, const uint16_t* __restrict__ dout,
    const uint16_t* __restrict__ o, const float* __restrict__ lse, float* __restrict__ delta,
    uint16_t* __restrict__ dq, int S, float scale, float scale_log2, int nqb, int BH,
    int group, const float* __restrict__ rope_cos, const float* __restrict__ rope_sin) {
  using v8 = typename MM<T>::v8;
  constexpr int BM = 32 * NW, BN = 64;
  constexpr int KSTEPS = D / 16, DT = D / 32;
  // one object per buffer
  __shared__ __align__(16) uint16_t Ks0[KG * BN * D], Ks1[KG * BN * D];
  __shared__ __align__(16) uint16_t Vs0[KG * BN * D], Vs1[KG * BN * D];

  int vh, blk;
  block_coords(BH, vh, blk);
  if (vh >= BH) return;
  const int bh = query_head(vh, BH / group, group);
  const int q0 = (nqb - 1 - blk) * BM;
  const int lane = threadIdx.x & 63;
  const int w = KG == 1 ? wave_id() : wave_id() % NW, kg = KG == 1 ? 0 : wave_id() / NW;
  const int kvo = kg * BN * D;  // this group's tile buffers
  const int l32 = lane & 31, hh = lane >> 5;
  const int64_t base = (int64_t)bh * S * D;
  const int64_t kvbase = (int64_t)(bh / group) * S * D;

  const int qrow = q0 + 32 * w + l32;
  const int qrc = qrow < S ? qrow : S - 1;
  v8 qf[KSTEPS], df[KSTEPS];
  // delta = rowsum(do * o) for this row: the lane pair (l, l + 32) holds the
  // row's D columns between them; summed in a fixed order and written for the
  // dK/dV kernel, which runs after this one.
  float dsum = 0.f;
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) {
    const int64_t off = base + (int64_t)qrc * D + kk * 16 + 8 * hh;
    qf[kk] = *reinterpret_cast<const v8*>(q + off);
    df[kk] = *reinterpret_cast<const v8*>(dout + off);
    const uint4 ou = *reinterpret_cast<const uint4*>(o + off);
    uint4 du;
    __builtin_memcpy(&du, &df[kk], 16);
    const uint32_t ow[4] = {ou.x, ou.y, ou.z, ou.w}, dw[4] = {du.x, du.y, du.z, du.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dsum += half_lo<T>(dw[e]) * half_lo<T>(ow[e]);
      dsum += half_hi<T>(dw[e]) * half_hi<T>(ow[e]);
    }
  }
  dsum += __shfl_xor(dsum, 32, 64);
  const float lv = lse[(int64_t)bh * S + qrc];
  const float l2 = qrow < S ? lv * kLog2e : INFINITY;
  const float dl = qrow < S ? dsum : 0.f;
  if (qrow < S && hh == 0 && kg == 0) delta[(int64_t)bh * S + qrow] = dsum;

  f32x16 acc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) acc[t] = f32x16{};
  const int kv_end = min(S, q0 + BM);
  const int ntiles = (kv_end + BN - 1) / BN;
  const int nturns = (ntiles + KG - 1) / KG;
  const int wave_first_row = q0 + 32 * w;
  const uint16_t* kp = k + kvbase;
  const uint16_t* vp = v + kvbase;

  // Element offsets of this lane's operand reads inside a tile, computed once (as in
  // the forward): rows for S and dP (the K and V tiles share the layout), transposed
  // rows of K for dQ; the tile loop is unrolled over the two buffers.
  int offS[KSTEPS], offV[DT][2];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) offS[kk] = toff<D>(l32, 2 * kk + hh);
  {
    const int mq = lane & 15, gs = (lane >> 4) & 1, r0 = 4 * hh + (mq >> 2);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int col = 32 * t + 16 * gs + 4 * (mq & 3);
      offV[t][0] = toff<D>(r0, col >> 3) + (col & 7);
      offV[t][1] = toff<D>(r0 + 8, col >> 3) + (col & 7);
    }
  }
  zero_lds<NW * KG * 64>(Ks0, sizeof(Ks0));
  zero_lds<NW * KG * 64>(Ks1, sizeof(Ks1));
  zero_lds<NW * KG * 64>(Vs0, sizeof(Vs0));
  zero_lds<NW * KG * 64>(Vs1, sizeof(Vs1));
  __syncthreads();
  TileLoader<BN, D, NW> ld;
  ld.init(w);
  if (kg < ntiles) {
    ld.load(kp, kg * BN, S, Ks0 + kvo);
    ld.load(vp, kg * BN, S, Vs0 + kvo);
  }
  auto tile = [&](auto bufc, int j) {
    constexpr int buf = decltype(bufc)::value;
    wait_loads();
    __syncthreads();
    const int next = KG * (j + 1) + kg;
    if (next < ntiles) {
      ld.load(kp, next * BN, S, (buf ? Ks0 : Ks1) + kvo);
      ld.load(vp, next * BN, S, (buf ? Vs0 : Vs1) + kvo);
    }
    const int k0 = (KG * j + kg) * BN;
    if (k0 > wave_first_row + 31) return;
    if (KG > 1 && k0 >= kv_end) return;
    const uint16_t* Kb = (buf ? Ks1 : Ks0) + kvo;
    const uint16_t* Vb = (buf ? Vs1 : Vs0) + kvo;
    f32x16 s[2] = {f32x16{}, f32x16{}}, dp[2] = {f32x16{}, f32x16{}};
    // S^T = K Q^T and dP^T = V dO^T interleaved, each operand read kDqPrefetch MFMAs
    // ahead (read i: kk = i / 4, T2 = (i / 2) % 2, K for even i and V for odd i);
    // the scheduling groups keep that order.
    {
      constexpr int NR = 4 * KSTEPS, PF = kDqPrefetch;
      auto rd = [&](int i) {
        const uint16_t* tb = (i & 1) ? Vb : Kb;
        return *reinterpret_cast<const v8*>(tb + offS[i >> 2] + 32 * D * ((i >> 1) & 1));
      };
      v8 ring[PF];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < PF; ++i) ring[i] = rd(i);
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int kk = i >> 2, T2 = (i >> 1) & 1;
        if (i & 1) dp[T2] = MM<T>::mma(ring[i % PF], df[kk], dp[T2]);
        else s[T2] = MM<T>::mma(ring[i % PF], qf[kk], s[T2]);
        if (i + PF < NR) ring[i % PF] = rd(i + PF);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);  // the first PF LDS reads
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        if (i + PF < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one read
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int T2 = 0; T2 < 2; ++T2)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[T2][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[T2][r], scale_log2, -l2));
    // Keys past the diagonal only in the diagonal tiles: a wave-uniform branch
    // around the per-element selects, so the other tiles skip them.
    if (k0 + BN - 1 > wave_first_row) {
#pragma unroll
      for (int T2 = 0; T2 < 2; ++T2)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kkey = k0 + 32 * T2 + (r >> 2) * 8 + 4 * hh + (r & 3);
          if (kkey > qrow) s[T2][r] = 0.f;
        }
    }
#pragma unroll
    for (int T2 = 0; T2 < 2; ++T2)
#pragma unroll
      for (int r = 0; r < 16; ++r) dp[T2][r] = s[T2][r] * (dp[T2][r] - dl);
#pragma unroll
    for (int ms = 0; ms < BN / 16; ++ms) {
      const v8 sb = pack8<T>(dp[ms >> 1], 8 * (ms & 1));
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (EG_LDS i16x4*)(Kb + offV[t][0] + 16 * D * ms));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (EG_LDS i16x4*)(Kb + offV[t][1] + 16 * D * ms));
        v8 ka;
        __builtin_memcpy(&ka, &lo, 8);
        __builtin_memcpy(reinterpret_cast<char*>(&ka) + 8, &hi, 8);
        acc[t] = MM<T>::mma(ka, sb, acc[t]);
      }
    }
  };
  for (int j = 0; j < nturns; j += 2) {
    tile(std::integral_constant<int, 0>{}, j);
    if (j + 1 < nturns) tile(std::integral_constant<int, 1>{}, j + 1);
  }
  if constexpr (KG > 1) {
    constexpr int HT = DT / 2, STRIDE = NW * 64;
    static_assert(HT * 16 * STRIDE * 4 <= (int)sizeof(Ks0), "half of dQ fits a buffer");
    float* half0 = reinterpret_cast<float*>(Ks0);
    float* half1 = reinterpret_cast<float*>(Ks1);
    const int at = w * 64 + lane;
    __syncthreads();  // the last tiles are consumed
    if (kg == 1) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          (t < HT ? half0 : half1)[((t % HT) * 16 + r) * STRIDE + at] = acc[t][r];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[t][r] += (t < HT ? half0 : half1)[((t % HT) * 16 + r) * STRIDE + at];
  }

  if (qrow < S) {
    uint16_t* op = dq + base + (int64_t)qrow * D;
    float fq = scale;
    if constexpr (ROPE) {  // dq of the pre-rotation queries: the rotation's transpose
#pragma unroll
      for (int t = 0; t < DT; ++t) acc[t] *= scale;
      unrotate_rows<D>(acc, rope_cos + (int64_t)qrow * D, rope_sin + (int64_t)qrow * D, hh);
      fq = 1.0f;
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) store_rows<T>(op, acc[t], t, hh, fq);
  }
}

// --------------------------------------------------------------- launchers
// Forward workgroup width: 8 waves (256 query rows), two per SIMD, each K/V tile
// serving 256 rows (interleaved at [4, 32, 4096, 128]: 590-597 us with 4 waves,
// 565-571 us with 8). dQ keeps 4 waves (8: 3.5% slower).
constexpr int kFwdWaves = 8;
// Forward grids of fewer than two 8-wave workgroups per CU (few heads or short
// sequences: the decoder layer's B = 1, 32 heads at T <= 2048) take 4-wave workgroups
// instead, twice as many of them; the rows each wave computes are the same, so the
// results are identical.
constexpr int kFwdSmallWaves = 4, kFwdFullGrid = 512;
constexpr int kDqWaves = 4;
constexpr int kDkdvRows = 32;
// dK/dV workgroup width: 4 waves (128 keys), one per SIMD, so that two workgroups
// share a CU and one's barrier waits overlap the other's work (at D = 128, 8-wave
// workgroups of 256 keys are 3-4% slower).
template <int D> constexpr int dkdv_waves() { return 4; }

// Split walk of the dK/dV kernel: with fewer than kDkdvTarget workgroups (kv heads
// x key blocks of 128 keys: small batches, few kv heads, short sequences), each key
// block's walk over the query tiles of its group is cut into `parts` (at most
// kDkdvMaxParts) whose fp32 sums go to workspace slabs, added in part order by
// attn_dkdv_reduce_kernel. The choice depends on the shape only, so results are
// the same on every run and device.
constexpr int kDkdvTarget = 1024, kDkdvMaxParts = 8;
int dkdv_parts(int64_t BHkv, int64_t S, int64_t D) {
  if (D != 64 && D != 128) return 1;
  const int64_t nkb = (S + 32 * dkdv_waves<128>() - 1) / (32 * dkdv_waves<128>());
  const int64_t wgs = BHkv * nkb;
  if (wgs <= 0 || wgs >= kDkdvTarget) return 1;
  return (int)std::min<int64_t>(kDkdvMaxParts, (kDkdvTarget + wgs - 1) / wgs);
}
// Parts to take, up to that bound: each shortens the longest
// walk until the chip is full (two workgroups per CU) and costs its slabs' write and read.
// In us, 1.1 (D = 128) or 0.9 (64) per 32-row step, 1.6 per million elements of dK and
// part, and 5 for the reduction: fitted over 48 shapes timed at every number of parts; the
// backward at the bound against at the choice: bf16 [2, 12, 1000, 64] 54.7 -> 46.4 us (6 parts,
// 3), [4, 8, 512, 128] 72.1 -> 44.4 (8, 1), [1, 8, 2048, 128] 107.7 -> 92.2 (8, 5), [8, 16, 256, 64]
// 40.9 -> 22.0 (4, 1); [1, 32 / 8, 512, 128] stays at 8 parts, [1, 4, 8192, 64] at 4.
int dkdv_split(int64_t BHkv, int64_t group, int64_t S, int64_t D) {
  const int most = dkdv_parts(BHkv, S, D);
  const double step = D == 128 ? 1.1 : 0.9;
  const double steps = (double)group * (double)((S + 31) / 32);  // the longest walk
  const double wgs = (double)BHkv * (double)((S + 127) / 128);
  const double full = wgs * steps / 2 / 512, slab = 1.6e-6 * (double)BHkv * (double)(S * D);
  int best = 1;
  double least = 0;
  for (int p = 1; p <= most; ++p) {
    const double c = step * std::max(steps / p, full) + (p > 1 ? slab * p + 5.0 : 0.0);
    if (p == 1 || c < least) least = c, best = p;
  }
  return best;
}
// Backward workspace after delta (fp32 [BH, S], rounded up to 256 bytes): the split
// walk's slabs, 2 x parts x BHkv x S x D fp32 (none without a split).
size_t attn_delta_bytes(int64_t BH, int64_t S) { return ((size_t)(BH * S) * 4 + 255) / 256 * 256; }
size_t attn_part_bytes(int64_t BHkv, int64_t group, int64_t S, int64_t D) {
  const int parts = dkdv_split(BHkv, group, S, D);
  return parts > 1 ? (size_t)2 * parts * BHkv * S * D * 4 : 0;
}

// The MFMA kernels take 16-bit tensors with head_dim 64 or 128; everything else
// (fp32, other even head sizes up to 128) runs on the generic kernels
// (attn_generic.hip).
bool mfma_shape(int64_t D, int dtype) {
  return (D == 64 || D == 128) && (dtype == EG_BF16 || dtype == EG_F16);
}

int check_attn(const char* what, int64_t B, int64_t H, int64_t Hkv, int64_t S, int64_t D,
               int dtype, bool mfma_only = false) {
  if (B < 0 || H < 0 || S < 0) { set_error("%s: negative size", what); return 1; }
  if (H > 0 && (Hkv <= 0 || H % Hkv != 0)) {
    set_error("%s: heads (%lld) must be a positive multiple of kv_heads (%lld)", what,
              (long long)H, (long long)Hkv);
    return 1;
  }
  if (mfma_only) {
    if (D != 64 && D != 128) { set_error("%s: head_dim must be 64 or 128, got %lld", what, (long long)D); return 1; }
    if (dtype != EG_BF16 && dtype != EG_F16) { set_error("%s: dtype must be bf16 or fp16", what); return 1; }
  } else {
    if (D < 2 || D > 128 || D % 2) { set_error("%s: head_dim must be even and at most 128, got %lld", what, (long long)D); return 1; }
    if (dtype != EG_BF16 && dtype != EG_F16 && dtype != EG_F32) { set_error("%s: dtype must be fp32, bf16 or fp16", what); return 1; }
  }
  // One (b, h) slice is addressed with 32-bit buffer offsets: S * D * 2 < 2^31.
  if (S > ((int64_t)1 << 22) || B * H > ((int64_t)1 << 24)) {
    set_error("%s: size out of range (seq <= 4194304, batch*heads <= 16777216)", what);
    return 1;
  }
  return 0;
}

inline unsigned grid_for(int64_t BH, int nblocks) {
  return (unsigned)(((BH + 7) / 8) * 8 * nblocks);
}

// Two key groups per workgroup (KG = 2) in the forward and dQ: for grids of at most 512
// 128-row workgroups, where the chain of key tiles of the last rows sets the time, from
// 768 positions (12 tiles) on. bf16 forward / backward, one group against two: [1, 16 / 4,
// 2000, 128] 38.0 / 114.4 -> 30.7 / 108.5 us, [1, 4, 900, 128] 19.7 / 51.3 -> 17.7 / 50.7, [1, 8,
// 768, 64] 13.0 / 33.9 -> 12.0 / 34.0; shorter rows only pay for the exchange ([1, 2 / 1, 200,
// 128] 8.2 -> 9.0 us, [4, 8, 512, 128] 12.8 -> 13.3).
// A CU holds one workgroup of two groups or two of one, so past 256 workgroups the second
// round has to be won back by longer rows. Forward: at D = 128 from 2048 positions ([1, 64 / 8,
// 1000] 28.0 -> 30.1, [1, 32 / 8, 2048] 47.8 -> 44.5), at 64 always ([1, 64 / 8, 800] 16.2 -> 15.8,
// [1, 40 / 8, 1152] 19.5 -> 17.9). dQ, backward: up to 384 workgroups at 128 from 2048 ([1, 24 /
// 8, 2048] 150.4 -> 144.4, [1, 16 / 4, 2500] 146.3 -> 135.5, [1, 48 / 12, 903] 90.5 -> 97.0), at 64
// from 1152 ([3, 16, 900] 50.4 -> 53.8, [2, 24, 780] 44.3 -> 47.3, [1, 40 / 8, 1152] 60.7 -> 60.6,
// [1, 24 / 8, 2048] 86.0 -> 81.8); up to 512 from 4096 ([1, 32 / 8, 2048, 128] 173.4 -> 171.7 but
// 178.1 -> 180.9 on another card, [1, 16 / 4, 4096, 128] 287.6 -> 273.5).
// A head's result is a sum in the order its grid takes, so it may differ in its last bits
// between calls with few and with many heads.
constexpr int64_t kSplitKeysGrid = 512, kSplitKeysSeq = 768;
inline bool split_keys(int64_t BH, int64_t S, int64_t D, bool dq) {
  const int64_t grid = grid_for(BH, (int)((S + 127) / 128));
  if (S < kSplitKeysSeq || grid > kSplitKeysGrid) return false;
  if (grid <= 256) return true;
  if (!dq) return D == 64 || S >= 2048;
  return S >= 4096 || (grid <= 384 && S >= (D == 64 ? 1152 : 2048));
}

// With ROPE, q is rotated in registers by the fp32 tables rc/rs [S, D] as it is
// loaded (k must already be rotated).
template <typename T, int D, bool ROPE = false>
int attn_fwd_launch(const void* q, const void* k, const void* v, void* o, float* lse, int64_t BH,
                    int64_t S, int group, float scale, hipStream_t st,
                    const float* rc = nullptr, const float* rs = nullptr) {
  auto go = [&](auto nwc, auto kgc) {
    constexpr int NW = decltype(nwc)::value, KG = decltype(kgc)::value;
    const int nqb = (int)((S + 32 * NW - 1) / (32 * NW));
    EG_LAUNCH((attn_fwd_kernel<T, D, NW, KG, ROPE>), dim3(grid_for(BH, nqb)), dim3(NW * KG * 64), 0, st,
              (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (uint16_t*)o, lse,
              (int)S, scale * kLog2e, nqb, (int)BH, group, rc, rs);
    return check_launch("eg_attn_fwd");
  };
  const int nqb_full = (int)((S + 32 * kFwdWaves - 1) / (32 * kFwdWaves));
  using One = std::integral_constant<int, 1>;
  if (split_keys(BH, S, D, false))
    return go(std::integral_constant<int, kFwdSmallWaves>{}, std::integral_constant<int, 2>{});
  if (grid_for(BH, nqb_full) < (unsigned)kFwdFullGrid)
    return go(std::integral_constant<int, kFwdSmallWaves>{}, One{});
  return go(std::integral_constant<int, kFwdWaves>{}, One{});
}

// BH counts query heads (x batch); the key/value tensors hold BH / group heads.
// With ROPE, q and k are the rotated tensors and dq, dk are written for the
// pre-rotation ones (the rotation's transpose applied to the results in registers).
template <typename T, int D, bool ROPE = false>
int attn_bwd_launch(const void* dout, const void* q, const void* k, const void* v, const void* o,
                    const float* lse, void* dq, void* dk, void* dv, float* delta, int64_t BH,
                    int64_t S, int group, float scale, hipStream_t st,
                    const float* rc = nullptr, const float* rs = nullptr) {
  // The split walk's slabs follow delta in the workspace.
  float* part = (float*)((char*)delta + attn_delta_bytes(BH, S));
  // dQ first: it also computes delta = rowsum(do * o) for its rows, which the
  // dK/dV kernel reads.
  constexpr int NQ = kDqWaves;
  const int nqb = (int)((S + 32 * NQ - 1) / (32 * NQ));
  auto run_dq = [&](auto kgc) {
    constexpr int KG = decltype(kgc)::value;
    EG_LAUNCH((attn_dq_kernel<T, D, NQ, KG, ROPE>), dim3(grid_for(BH, nqb)), dim3(NQ * KG * 64), 0,
              st, (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v,
              (const uint16_t*)dout, (const uint16_t*)o, lse, delta, (uint16_t*)dq, (int)S, scale,
              scale * kLog2e, nqb, (int)BH, group, rc, rs);
  };
  if (split_keys(BH, S, D, true)) run_dq(std::integral_constant<int, 2>{});
  else run_dq(std::integral_constant<int, 1>{});
  if (int rc = check_launch("eg_attn_bwd(dq)")) return rc;
  constexpr int NK = dkdv_waves<D>();
  const int nkb = (int)((S + 32 * NK - 1) / (32 * NK));
  const int64_t BHkv = BH / group;
  static_assert(NK == dkdv_waves<128>(), "dkdv_parts assumes one key-block width");
  const int parts = dkdv_split(BHkv, group, S, D);
  EG_LAUNCH((attn_dkdv_kernel<T, D, NK, kDkdvRows, ROPE>), dim3(grid_for(BHkv * parts, nkb)),
            dim3(NK * 64), 0, st, (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v,
            (const uint16_t*)dout, lse, delta, (uint16_t*)dk, (uint16_t*)dv, (int)S, scale,
            scale * kLog2e, (int)BHkv, group, rc, rs, parts, parts > 1 ? part : nullptr);
  if (int e = check_launch("eg_attn_bwd(dkdv)")) return e;
  if (parts == 1) return 0;
  const int64_t n = BHkv * S * D;
  EG_LAUNCH((attn_dkdv_reduce_kernel<T>), dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, st,
            (const float*)part, parts, n, (uint16_t*)dk, (uint16_t*)dv);
  return check_launch("eg_attn_bwd(dkdv reduce)");
}

// Explicit instantiations: hip-clang leaves some implicitly instantiated kernel
// templates without a host launch stub (undefined symbol at load time); naming
// every kernel here makes the stubs certain.
#define EG_ATTN_INSTANTIATE(T, D, R)                                                         \
  template __global__ void attn_fwd_kernel<T, D, kFwdWaves, 1, R>(                           \
      const uint16_t*, const uint16_t*, const uint16_t*, uint16_t*, float*, int, float, int,   \
      int, int, const float*, const float*);                                                 \
  template __global__ void attn_fwd_kernel<T, D, kFwdSmallWaves, 1, R>(                      \
      const uint16_t*, const uint16_t*, const uint16_t*, uint16_t*, float*, int, float, int,   \
      int, int, const float*, const float*);                                                 \
  template __global__ void attn_fwd_kernel<T, D, kFwdSmallWaves, 2, R>(                      \
      const uint16_t*, const uint16_t*, const uint16_t*, uint16_t*, float*, int, float, int,   \
      int, int, const float*, const float*);                                                 \
  template __global__ void attn_dkdv_kernel<T, D, dkdv_waves<D>(), kDkdvRows, R>(            \
      const uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*, const float*,        \
      const float*, uint16_t*, uint16_t*, int, float, float, int, int, const float*,           \
      const float*, int, float*);                                                            \
  template __global__ void attn_dq_kernel<T, D, kDqWaves, 1, R>(                                \
      const uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*,     \
      const float*, float*, uint16_t*, int, float, float, int, int, int, const float*,         \
      const float*);                                                                      \
  template __global__ void attn_dq_kernel<T, D, kDqWaves, 2, R>(                                \
      const uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*,     \
      const float*, float*, uint16_t*, int, float, float, int, int, int, const float*,         \
      const float*);
EG_ATTN_INSTANTIATE(bf16_t, 128, false)
EG_ATTN_INSTANTIATE(bf16_t, 64, false)
EG_ATTN_INSTANTIATE(f16_t, 128, false)
EG_ATTN_INSTANTIATE(f16_t, 64, false)
EG_ATTN_INSTANTIATE(bf16_t, 128, true)
EG_ATTN_INSTANTIATE(bf16_t, 64, true)
EG_ATTN_INSTANTIATE(f16_t, 128, true)
EG_ATTN_INSTANTIATE(f16_t, 64, true)
#undef EG_ATTN_INSTANTIATE

bool attn_aligned(std::initializer_list<const void*> ptrs) {
  for (const void* p : ptrs)
    if (!aligned16(p)) return false;
  return true;
}

}  // namespace
}  // namespace eg

using namespace eg;

extern "C" size_t eg_attn_gqa_workspace_bytes(int64_t batch, int64_t heads, int64_t kv_heads,
                                              int64_t seq, int64_t head_dim) {
  if (batch <= 0 || heads <= 0 || seq <= 0 || kv_heads <= 0) return 0;
  // the dtype is not known here: the larger of the MFMA and the generic kernels' slabs
  return attn_delta_bytes(batch * heads, seq) +
         std::max(attn_part_bytes(batch * kv_heads, heads / kv_heads, seq, head_dim),
                  attn_generic_part_bytes(batch, heads, kv_heads, seq, head_dim));
}

extern "C" size_t eg_attn_workspace_bytes(int64_t batch, int64_t heads, int64_t seq,
                                          int64_t head_dim) {
  return eg_attn_gqa_workspace_bytes(batch, heads, heads, seq, head_dim);
}

extern "C" int eg_attn_gqa_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                               int64_t batch, int64_t heads, int64_t kv_heads, int64_t seq,
                               int64_t head_dim, float scale, int dtype, void* stream) {
  clear_error();
  if (check_attn("eg_attn_fwd", batch, heads, kv_heads, seq, head_dim, dtype)) return 1;
  if (batch == 0 || heads == 0 || seq == 0) return 0;
  if (!q || !k || !v || !o || !lse) { set_error("eg_attn_fwd: null pointer"); return 1; }
  hipStream_t st = as_stream(stream);
  if (!mfma_shape(head_dim, dtype))
    return attn_generic_fwd(q, k, v, o, lse, batch, heads, kv_heads, seq, head_dim, scale, dtype,
                            st);
  if (!attn_aligned({q, k, v, o})) { set_error("eg_attn_fwd: tensors must be 16-byte aligned"); return 1; }
  const int64_t BH = batch * heads;
  const int group = (int)(heads / kv_heads);
  if (dtype == EG_BF16)
    return head_dim == 128 ? attn_fwd_launch<bf16_t, 128>(q, k, v, o, lse, BH, seq, group, scale, st)
                           : attn_fwd_launch<bf16_t, 64>(q, k, v, o, lse, BH, seq, group, scale, st);
  return head_dim == 128 ? attn_fwd_launch<f16_t, 128>(q, k, v, o, lse, BH, seq, group, scale, st)
                         : attn_fwd_launch<f16_t, 64>(q, k, v, o, lse, BH, seq, group, scale, st);
}

extern "C" int eg_attn_gqa_bwd(const void* dout, const void* q, const void* k, const void* v,
                               const void* o, const float* lse, void* dq, void* dk, void* dv,
                               void* workspace, int64_t batch, int64_t heads, int64_t kv_heads,
                               int64_t seq, int64_t head_dim, float scale, int dtype,
                               void* stream) {
  clear_error();
  if (check_attn("eg_attn_bwd", batch, heads, kv_heads, seq, head_dim, dtype)) return 1;
  if (batch == 0 || heads == 0 || seq == 0) return 0;
  if (!dout || !q || !k || !v || !o || !lse || !dq || !dk || !dv || !workspace) {
    set_error("eg_attn_bwd: null pointer");
    return 1;
  }
  hipStream_t st = as_stream(stream);
  float* delta = (float*)workspace;
  if (!mfma_shape(head_dim, dtype))
    return attn_generic_bwd(dout, q, k, v, o, lse, dq, dk, dv, delta,
                            (float*)((char*)delta + attn_delta_bytes(batch * heads, seq)), batch,
                            heads, kv_heads, seq, head_dim, scale, dtype, st);
  if (!attn_aligned({dout, q, k, v, o, dq, dk, dv})) {
    set_error("eg_attn_bwd: tensors must be 16-byte aligned");
    return 1;
  }
  const int64_t BH = batch * heads;
  const int group = (int)(heads / kv_heads);
  if (dtype == EG_BF16)
    return head_dim == 128
               ? attn_bwd_launch<bf16_t, 128>(dout, q, k, v, o, lse, dq, dk, dv, delta, BH, seq, group, scale, st)
               : attn_bwd_launch<bf16_t, 64>(dout, q, k, v, o, lse, dq, dk, dv, delta, BH, seq, group, scale, st);
  return head_dim == 128
             ? attn_bwd_launch<f16_t, 128>(dout, q, k, v, o, lse, dq, dk, dv, delta, BH, seq, group, scale, st)
             : attn_bwd_launch<f16_t, 64>(dout, q, k, v, o, lse, dq, dk, dv, delta, BH, seq, group, scale, st);
}

extern "C" int eg_attn_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                           int64_t batch, int64_t heads, int64_t seq, int64_t head_dim,
                           float scale, int dtype, void* stream) {
  return eg_attn_gqa_fwd(q, k, v, o, lse, batch, heads, heads, seq, head_dim, scale, dtype, stream);
}

extern "C" int eg_attn_bwd(const void* dout, const void* q, const void* k, const void* v,
                           const void* o, const float* lse, void* dq, void* dk, void* dv,
                           void* workspace, int64_t batch, int64_t heads, int64_t seq,
                           int64_t head_dim, float scale, int dtype, void* stream) {
  return eg_attn_gqa_bwd(dout, q, k, v, o, lse, dq, dk, dv, workspace, batch, heads, heads, seq,
                         head_dim, scale, dtype, stream);
}

// ----------------------------------------- RoPE(q, k) -> grouped causal attention
// The attention half of the Llama-3 decoder layer
// (src/evograd/ops/level3/llama3_decoder_layer/forward_ref.py:93-107): q and k
// rotated by fp32 tables cos/sin [S, D], then causal GQA attention. The forward
// rotates k into the workspace (one small pass over the kv heads) and q in the
// attention kernel's registers as it loads them; the backward rotates q and k into
// the workspace again (the saved state holds the pre-rotation inputs only) and
// applies the rotation's transpose to dq and dk in the kernels' registers before
// the stores. Backward workspace: q_r [B, H, S, D], k_r [B, Hkv, S, D] (dtype),
// delta [B, H, S] fp32, in that order; the forward's holds only its k_r.
static size_t llama3_ws_qr(int64_t B, int64_t H, int64_t S, int64_t D) { return (size_t)(B * H * S * D) * 2; }
static size_t llama3_ws_kr(int64_t B, int64_t Hkv, int64_t S, int64_t D) { return (size_t)(B * Hkv * S * D) * 2; }

extern "C" size_t eg_llama3_attn_workspace_bytes(int64_t batch, int64_t heads, int64_t kv_heads,
                                                 int64_t seq, int64_t head_dim) {
  if (batch <= 0 || heads <= 0 || kv_heads <= 0 || seq <= 0 || head_dim <= 0) return 0;
  return llama3_ws_qr(batch, heads, seq, head_dim) + llama3_ws_kr(batch, kv_heads, seq, head_dim) +
         attn_delta_bytes(batch * heads, seq) +
         attn_part_bytes(batch * kv_heads, heads / kv_heads, seq, head_dim);
}

template <typename F>
static int llama3_dispatch(int dtype, int64_t head_dim, F&& f) {
  if (dtype == EG_BF16)
    return head_dim == 128 ? f(bf16_t{}, std::integral_constant<int, 128>{})
                           : f(bf16_t{}, std::integral_constant<int, 64>{});
  return head_dim == 128 ? f(f16_t{}, std::integral_constant<int, 128>{})
                         : f(f16_t{}, std::integral_constant<int, 64>{});
}

extern "C" int eg_llama3_attn_fwd(const void* q, const void* k, const void* v, const float* cos,
                                  const float* sin, void* o, float* lse, void* workspace,
                                  int64_t batch, int64_t heads, int64_t kv_heads, int64_t seq,
                                  int64_t head_dim, float scale, int dtype, void* stream) {
  static const char* name = "eg_llama3_attn_fwd";
  clear_error();
  if (check_attn(name, batch, heads, kv_heads, seq, head_dim, dtype, true)) return 1;
  if (batch == 0 || heads == 0 || seq == 0) return 0;
  if (!q || !k || !v || !cos || !sin || !o || !lse || !workspace) {
    set_error("%s: null pointer", name);
    return 1;
  }
  if (!attn_aligned({q, k, v, o, cos, sin, workspace})) {
    set_error("%s: tensors, tables and workspace must be 16-byte aligned", name);
    return 1;
  }
  hipStream_t st = as_stream(stream);
  void* k_r = workspace;
  if (int rc = rope_apply(nullptr, k, nullptr, k_r, cos, sin, batch, 0, kv_heads, seq, head_dim,
                          dtype, EG_F32, false, st))
    return rc;
  const int64_t BH = batch * heads;
  const int group = (int)(heads / kv_heads);
  return llama3_dispatch(dtype, head_dim, [&](auto tc, auto dc) {
    using T = decltype(tc);
    return attn_fwd_launch<T, decltype(dc)::value, true>(q, k_r, v, o, lse, BH, seq, group, scale,
                                                         st, cos, sin);
  });
}

extern "C" int eg_llama3_attn_bwd(const void* dout, const void* q, const void* k, const void* v,
                                  const void* o, const float* lse, const float* cos,
                                  const float* sin, void* dq, void* dk, void* dv, void* workspace,
                                  int64_t batch, int64_t heads, int64_t kv_heads, int64_t seq,
                                  int64_t head_dim, float scale, int dtype, void* stream) {
  static const char* name = "eg_llama3_attn_bwd";
  clear_error();
  if (check_attn(name, batch, heads, kv_heads, seq, head_dim, dtype, true)) return 1;
  if (batch == 0 || heads == 0 || seq == 0) return 0;
  if (!dout || !q || !k || !v || !o || !lse || !cos || !sin || !dq || !dk || !dv || !workspace) {
    set_error("%s: null pointer", name);
    return 1;
  }
  if (!attn_aligned({dout, q, k, v, o, cos, sin, dq, dk, dv, workspace})) {
    set_error("%s: tensors, tables and workspace must be 16-byte aligned", name);
    return 1;
  }
  hipStream_t st = as_stream(stream);
  char* ws = (char*)workspace;
  void* q_r = ws;
  void* k_r = ws + llama3_ws_qr(batch, heads, seq, head_dim);
  float* delta = (float*)((char*)k_r + llama3_ws_kr(batch, kv_heads, seq, head_dim));
  if (int rc = rope_apply(q, k, q_r, k_r, cos, sin, batch, heads, kv_heads, seq, head_dim, dtype,
                          EG_F32, false, st))
    return rc;
  const int64_t BH = batch * heads;
  const int group = (int)(heads / kv_heads);
  return llama3_dispatch(dtype, head_dim, [&](auto tc, auto dc) {
    using T = decltype(tc);
    return attn_bwd_launch<T, decltype(dc)::value, true>(dout, q_r, k_r, v, o, lse, dq, dk, dv,
                                                         delta, BH, seq, group, scale, st, cos,
                                                         sin);
  });
}
