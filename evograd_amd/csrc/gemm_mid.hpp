// The 16-bit product of gemm_kernel.hpp on 128 x 128 x 64 tiles, for outputs that are too
// small to occupy the chip in 256 x 256 tiles (the choice: gemm.hip, gemm_plan).
//
// Same operands, layouts, segments, bounds and k order as gemm_kernel: fp32 accumulation on
// v_mfma_f32_32x32x16 over 64-deep slices in increasing k, so a product's bits depend on
// its split of k only and not on which of the two kernels ran. 4 waves of 64 x 64 (four
// accumulators). What bounds a small product is the latency of its chain of slices: one
// workgroup per CU runs at most a few of them, so kMidStages slices (32 KB each) are in
// LDS or on their way, kMidStages - 1 steps ahead of their use. One barrier per step: after
// it every wave has read the previous slice, whose buffer takes the next loads.
// The whole tile leaves through LDS in fp32 (64 KB), so ragged tiles, residuals and partials
// are stored as row segments too.
#pragma once

#include "gemm_kernel.hpp"

namespace eg {
namespace gk {

constexpr int kMT = 128;                    // tile width and height
constexpr int kMidElems = kMT * kBK;        // one operand slice: 16 KB
constexpr int kMidStages = 4;

// One 128 x 64 operand slice (SliceLoader of gemm_kernel.hpp at half the width).
template <bool KC>
struct MidLoader {
  int voff[4];
  __device__ __forceinline__ void init(int64_t ld) {
    const int w = gwave(), lane = threadIdx.x & 63;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int p = (it * 4 + w) * 64 + lane;
      const int r = KC ? p >> 3 : p >> 4;
      const int c = KC ? (p & 7) ^ swz_kc(r) : (p & 15) ^ swz_km(r);
      voff[it] = (int)(((int64_t)r * ld + c * 8) * 2);
    }
  }
  __device__ __forceinline__ void load(const uint16_t* base, int64_t bytes,
                                       uint16_t* lds) const {
    const __amdgpu_buffer_rsrc_t rs = rsrc(base, bytes);
    const int w = gwave();
#pragma unroll
    for (int it = 0; it < 4; ++it)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (EG_LDS void*)(lds + (it * 4 + w) * 512), 16,
                                               voff[it], 0, 0, 0);
  }
};

// MFMA operands of a slice (OperandReader of gemm_kernel.hpp): blocks i of 32 rows from w0.
template <bool KC>
struct MidReader {
  int off[KC ? 4 : 2];
  __device__ __forceinline__ void init(int w0, int lane) {
    const int l32 = lane & 31, hh = lane >> 5;
    if constexpr (KC) {
      const int row = w0 + l32;
#pragma unroll
      for (int s = 0; s < 4; ++s) off[s] = row * 64 + (((2 * s + hh) ^ swz_kc(row)) << 3);
    } else {
      const int m = lane & 15, gs = (lane >> 4) & 1;
      const int k0 = 8 * hh + (m >> 2);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int col = w0 + 32 * i + 16 * gs + 4 * (m & 3);
        off[i] = k0 * kMT + (((col >> 3) ^ swz_km(k0)) << 3) + (col & 7);
      }
    }
  }
  template <typename V>
  __device__ __forceinline__ V read(const uint16_t* lds, int i, int s) const {
    if constexpr (KC) {
      return *reinterpret_cast<const V*>(lds + off[s] + i * 2048);
    } else {
      const uint16_t* p = lds + off[i] + s * 16 * kMT;
      const i16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((EG_LDS i16x4*)p);
      const i16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((EG_LDS i16x4*)(p + 4 * kMT));
      V r;
      __builtin_memcpy(&r, &a, 8);
      __builtin_memcpy(reinterpret_cast<char*>(&r) + 8, &b, 8);
      return r;
    }
  }
};

// Where one operand's slices lie: its buffer, or under segments along k (SEG == 2) the
// segment that holds slice k0 (slices are asked for in increasing k).
template <bool KC, int SEG>
struct MidOperand {
  OpView v;
  int64_t ld, rows;
  int si, next;
  __device__ __forceinline__ void init(const uint16_t* p, int64_t rows_, int64_t ld_,
                                       const SegArgs& g, const void* const* tab, int idx) {
    ld = ld_;
    rows = rows_;
    si = 0;
    next = 0x7fffffff;
    v = OpView{p, 0, rows * ld};
    if constexpr (SEG == 1) v = seg_view<KC>(p, rows, ld, g, tab, false, idx);
    if constexpr (SEG == 2) {
      if (tab[0]) {
        v.base = (const uint16_t*)tab[0];
        v.end = KC ? rows * ld : (int64_t)g.start[1] * ld;
        if (g.n > 1) next = g.start[1];
      }
    }
  }
  // first element of the slice at (r0, k0), and the bytes from there to the view's end
  __device__ __forceinline__ const uint16_t* at(int r0, int k0, const SegArgs& g,
                                                const void* const* tab, int64_t& bytes) {
    if constexpr (SEG == 2) {
      while (k0 >= next) {
        ++si;
        const int64_t st = g.start[si], en = g.start[si + 1];
        v.base = (const uint16_t*)tab[si];
        v.shift = KC ? st : st * ld;
        v.end = KC ? rows * ld : (en - st) * ld;
        next = si + 1 < g.n ? g.start[si + 1] : 0x7fffffff;
      }
    }
    const int64_t o = (KC ? (int64_t)r0 * ld + k0 : (int64_t)k0 * ld + r0) - v.shift;
    bytes = (v.end - o) * 2;
    return v.base + o;
  }
};

template <typename T, bool AKC, bool BKC, typename TC, int SEG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_mid_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, TC* C, int M,
                     int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int64_t a_rows,
                     int64_t b_rows, int tiles_m, int tiles, int vec_c, const void* R, int64_t ldr,
                     int r_f32, int kt_per, float* __restrict__ part, SegArgs seg) {
  using v8 = typename GM<T>::v8;
  // separate objects, selected at compile time: a read of one never waits for the loads
  // into another
  __shared__ __align__(16) uint16_t A0[kMidElems], A1[kMidElems], A2[kMidElems], A3[kMidElems];
  __shared__ __align__(16) uint16_t B0[kMidElems], B1[kMidElems], B2[kMidElems], B3[kMidElems];
  int kpart;
  const int t_idx = tile_index(tiles, 0, kpart);
  if (t_idx < 0) return;
  int tm, tn;
  tile_decode(t_idx, tiles_m, tiles, tm, tn);
  const int m0 = tm * kMT, n0 = tn * kMT;
  const int lane = threadIdx.x & 63, w = gwave();
  const int wm = (w >> 1) * 64, wn = (w & 1) * 64;
  MidLoader<AKC> la;
  MidLoader<BKC> lb;
  la.init(lda);
  lb.init(ldb);
  MidOperand<AKC, SEG> oa;
  MidOperand<BKC, SEG> ob;
  oa.init(A, a_rows, lda, seg, seg.a, m0);
  ob.init(B, b_rows, ldb, seg, seg.b, n0);
  MidReader<AKC> ra;
  MidReader<BKC> rb;
  ra.init(wm, lane);
  rb.init(wn, lane);
  const int nk_all = (K + kBK - 1) / kBK;
  const int kb = part ? (int)blockIdx.y * kt_per : 0;
  const int nk = part ? min(nk_all, kb + kt_per) : nk_all;
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
  auto bufA = [&](auto c) {
    constexpr int b = decltype(c)::value % kMidStages;
    if constexpr (b == 0) return A0;
    else if constexpr (b == 1) return A1;
    else if constexpr (b == 2) return A2;
    else return A3;
  };
  auto bufB = [&](auto c) {
    constexpr int b = decltype(c)::value % kMidStages;
    if constexpr (b == 0) return B0;
    else if constexpr (b == 1) return B1;
    else if constexpr (b == 2) return B2;
    else return B3;
  };
  // A slice at or past nk loads through an empty range (zeros), so that every step has
  // the same number of loads in flight.
  auto load = [&](auto c, int kt) {
    int64_t na = 0, nb = 0;
    const uint16_t* pa = A;
    const uint16_t* pb = B;
    if (kt < nk) {
      pa = oa.at(m0, kt * kBK, seg, seg.a, na);
      pb = ob.at(n0, kt * kBK, seg, seg.b, nb);
    }
    la.load(pa, na, bufA(c));
    lb.load(pb, nb, bufB(c));
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  static_assert(kMidStages == 4, "the waits and the unrolled loop below are for four stages");
  load(I0{}, kb);
  load(I1{}, kb + 1);
  load(I2{}, kb + 2);
  auto step = [&](auto c, int kt) {
    constexpr int b = decltype(c)::value;
    // this wave's 8 loads of slice kt are in (two later slices are in flight), and its
    // reads of the previous slice
    asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load(std::integral_constant<int, b + 3>{}, kt + 3);
    const uint16_t* as = bufA(c);
    const uint16_t* bs = bufB(c);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      v8 a[2], bb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = ra.template read<v8>(as, i, s);
#pragma unroll
      for (int j = 0; j < 2; ++j) bb[j] = rb.template read<v8>(bs, j, s);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = GM<T>::mma(bb[j], a[i], acc[i][j]);
    }
  };
  for (int kt = kb; kt < nk; kt += 4) {
    step(I0{}, kt);
    if (kt + 1 < nk) step(I1{}, kt + 1);
    if (kt + 2 < nk) step(I2{}, kt + 2);
    if (kt + 3 < nk) step(I3{}, kt + 3);
  }
  // No load may still be on its way into the buffers when the tile goes there.
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();
  // The tile in fp32, 32 rows per buffer pair A0|.. (32 rows x 512 B = one slice buffer);
  // 16-byte chunks XOR row % 32, as in gemm_kernel's staging.
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int hh = lane >> 5, l32 = lane & 31;
  auto rows32 = [&](int q) {
    return reinterpret_cast<float*>(q == 0 ? A0 : q == 1 ? A1 : q == 2 ? A2 : A3);
  };
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float* lrow = rows32((wm >> 5) + i) + l32 * kMT;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int chunk = (wn + 32 * j + 8 * q + 4 * hh) >> 2;
        *reinterpret_cast<f32x4*>(lrow + ((chunk ^ l32) << 2)) =
            f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                  acc[i][j][4 * q + 3]};
      }
  }
  __syncthreads();
  auto put_rows = [&](auto tag, auto* base, int64_t ld, bool vec, const void* res) {
    using TO = decltype(tag);
    constexpr int W = 16 / sizeof(TO);  // columns per 16-byte store
    constexpr int CPR = kMT / W;
#pragma unroll 2
    for (int e = threadIdx.x; e < kMT * CPR; e += 256) {
      const int r = e / CPR, c = (e % CPR) * W;
      const int row = m0 + r, col = n0 + c;
      if (row >= M || col >= N) continue;
      float v[W];
      const float* lrow = rows32(r >> 5) + (r & 31) * kMT;
#pragma unroll
      for (int q = 0; q < W / 4; ++q) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(lrow + ((((c >> 2) + q) ^ (r & 31)) << 2));
#pragma unroll
        for (int k = 0; k < 4; ++k) v[4 * q + k] = x[k];
      }
      TO* dst = base + (int64_t)row * ld + col;
      const TO* r16 = res ? (const TO*)res + (int64_t)row * ldr + col : nullptr;
      const float* r32 = res ? (const float*)res + (int64_t)row * ldr + col : nullptr;
      if (vec && col + W <= N) {
        if (res) {
          float x[W];
          if (r_f32) {
#pragma unroll
            for (int q = 0; q < W / 4; ++q) {
              const f32x4 y = *reinterpret_cast<const f32x4*>(r32 + 4 * q);
#pragma unroll
              for (int k = 0; k < 4; ++k) x[4 * q + k] = y[k];
            }
          } else {
            load_f32<TO, W>(r16, x);
          }
#pragma unroll
          for (int k = 0; k < W; ++k) v[k] += x[k];
        }
        store_f32<TO, W>(dst, v);
      } else {
#pragma unroll
        for (int k = 0; k < W; ++k)
          if (col + k < N) {
            if (res) v[k] += r_f32 ? r32[k] : to_f32(r16[k]);
            put<TO>(dst + k, v[k]);
          }
      }
    }
  };
  if (part) {
    put_rows(float{}, part + (int64_t)blockIdx.y * M * N, N, (N & 3) == 0, nullptr);
    return;
  }
  TC* cb = C;
  int64_t cshift = 0;
  if (SEG == 1) {
    const int sg = seg_of(seg, seg.dim == kSegM ? m0 : n0);
    if (seg.c[sg]) {
      cb = (TC*)seg.c[sg];
      cshift = seg.dim == kSegM ? (int64_t)seg.start[sg] * ldc : seg.start[sg];
    }
  }
  // vec_c allows 4-element pieces; the stores here are of 16 bytes
  const bool vec = vec_c && (ldc * (int)sizeof(TC)) % 16 == 0 &&
                   (!R || (ldr * (r_f32 ? 4 : (int)sizeof(TC))) % 16 == 0);
  put_rows(TC{}, cb - cshift, ldc, vec, R);
}

#define EG_MID_KERNEL(KIND, T, AKC, BKC, TC, SEG)                                               \
  KIND __global__ void gemm_mid_kernel<T, AKC, BKC, TC, SEG>(                                   \
      const uint16_t*, const uint16_t*, TC*, int, int, int, int64_t, int64_t, int64_t, int64_t,   \
      int64_t, int, int, int, const void*, int64_t, int, int, float*, SegArgs);
#define EG_MID_LAYOUTS(KIND, T, TC, SEG)      \
  EG_MID_KERNEL(KIND, T, true, true, TC, SEG)  \
  EG_MID_KERNEL(KIND, T, true, false, TC, SEG) \
  EG_MID_KERNEL(KIND, T, false, true, TC, SEG) \
  EG_MID_KERNEL(KIND, T, false, false, TC, SEG)
#define EG_MID_ALL_KERNELS(KIND, T) \
  EG_MID_LAYOUTS(KIND, T, T, 0)     \
  EG_MID_LAYOUTS(KIND, T, float, 0) \
  EG_MID_LAYOUTS(KIND, T, T, 1)     \
  EG_MID_LAYOUTS(KIND, T, T, 2)

}  // namespace gk
}  // namespace eg
