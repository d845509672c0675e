// Pieces shared by the W8A8 GEMM kernels (gemm_w8a8.hip: one persistent workgroup
// per CU on 256 x 256 tiles; gemm_tile.hip: smaller tiles): the arguments, the
// operand kinds' MFMA wrappers, the LDS-DMA load and the LDS row layout.
#pragma once

#include "fastdiv.h"
#include "xgen_common.h"

namespace xgen {

constexpr int BK = 64;  // K bytes per pipeline stage
// Output tiles of 256 x 256, one persistent workgroup per CU.
constexpr int kTileM = 256, kTileN = 256;

struct GemmArgs {
  const uint8_t *a;
  const uint8_t *w;
  int lda, ldw;  // bytes
  int M, N, K;
  const float *sa;
  int sa_stride;
  const float *sw;
  int sw_stride;
  const void *bias;
  int bias_dtype;
  int act, out_dtype;  // (the tile kernels; the 256 x 256 kernel has them as template arguments)
  void *out;
  int64_t ldo;  // elements
  void *acc_out;
  int tiles_m, tiles_n, per_xcd;
  int group_m;  // tile-rows per group of the tile order
  int kt4;      // stages per tile of the 256 x 256 kernel (a multiple of 4)
  uint32_t out_bytes;  // bytes of the output rows: (M - 1) * ldo * 2 + N * 2
  uint32_t a_bytes, w_bytes;
  // gated residual epilogue (GATED kernels only)
  const uint8_t *residual;
  int64_t ld_residual;  // elements
  const uint8_t *gate;
  int64_t gate_stride;  // elements
  int64_t gate_rows;
  const int64_t *indices;
  uint32_t seq, seq_magic, seq_shift;  // m % seq = m - ((mulhi(m, magic) + m) >> shift) * seq
  uint32_t residual_bytes, gate_bytes;  // (M - 1) * ld_residual * 2 + N * 2, (gate_rows - 1) * gate_stride * 2 + N * 2
};

// Operand kinds of the kernel template.
enum Kind { kInt8 = 0, kFp8 = 1, kFp8Exact = 2 };

// The smaller tile that a call runs on, or -1: the 256 x 256 kernel (gemm_tile.hip).
int choose_gemm_tile(int kind, int64_t M, int64_t N, int64_t K, bool gated, bool accumulators);
// Launches the call on that tile.  g: filled as for the 256 x 256 kernel.
void launch_gemm_tile(int kind, int tile, const GemmArgs &g, hipStream_t stream);

// Operand traits per kind: accumulator and fragment types (one fragment = 32
// rows of one 64-byte K step, as the fragment reads deliver them), MFMA steps per
// 64-byte K step, 16-byte LDS reads per fragment, accumulator to float.
template <int KIND>
struct Mfma;

template <>
struct Mfma<kFp8> {
  typedef f32x16 acc_t;
  typedef i32x8 frag_t;
  static constexpr int kSteps = BK / 64;  // 32x32x64: one step per stage
  static constexpr int kReads = 2;        // ds_read_b128 per fragment
  static __device__ __forceinline__ float to_f32(float v) { return v; }
};

// The exact kind reads the FP8 kind's fragments and multiplies them as bf16.
// The conversion is exact (bf16 holds every e4m3fn value, subnormals included).
template <>
struct Mfma<kFp8Exact> {
  typedef f32x16 acc_t;
  typedef i32x8 frag_t;
  static constexpr int kSteps = 1;
  static constexpr int kReads = 2;
  static __device__ __forceinline__ bf16x8 widen(int lo, int hi) {
    const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
    const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
    const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
    const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
    return bf16x8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
  }
  static __device__ __forceinline__ float to_f32(float v) { return v; }
};

template <>
struct Mfma<kInt8> {
  typedef i32x16 acc_t;
  typedef i32x4 frag_t;
  static constexpr int kSteps = BK / 32;  // 32x32x32: two steps per stage
  static constexpr int kReads = 1;        // ds_read_b128 per fragment
  static __device__ __forceinline__ float to_f32(int v) { return (float)v; }
};

// One 16-byte-per-lane buffer load on the LDS-DMA path: lane l's 16 bytes land
// at lds + 16 * l.  (A plain device function: called directly from the kernel
// template, the device-only builtin would keep the host pass from emitting the
// kernel's launch stub.)
__device__ __forceinline__ void dma_load16(__amdgpu_buffer_rsrc_t rsrc, uint8_t *lds, uint32_t offset) {
  typedef __attribute__((address_space(3))) void *lds_ptr_t;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)lds, 16, offset, 0, 0, 0);
}

// Workgroup barrier that orders LDS accesses without waiting for the vector
// memory counter: __syncthreads' fence would also wait for the DMA loads still
// in flight for later stages.  The empty asm statements keep the compiler from
// moving memory accesses across it; the caller waits lgkmcnt for its own LDS
// accesses first.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// s_waitcnt constraining only the vector-memory counter (gfx9 encoding: vmcnt
// in bits [3:0] and [15:14]; expcnt [6:4] and lgkmcnt [11:8] left at max).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// v rounded to the output dtype, as the stored output is rounded.  For f16 the
// empty asm keeps v an f32 value: the fma producing it would otherwise be
// selected with the f16 rounding as one v_fma_mixlo_f16 (one rounding of the
// exact a*b+c, where the store rounds the f32 result).
template <int OUT_DT>
__device__ __forceinline__ float round_out(float v) {
  if constexpr (OUT_DT == XGEN_DTYPE_BF16) {
    return round_bf16(v);
  } else {
    asm volatile("" : "+v"(v));
    return (float)(_Float16)v;
  }
}
template <int OUT_DT>
__device__ __forceinline__ uint32_t pack_out(float a, float b) {
  if constexpr (OUT_DT == XGEN_DTYPE_BF16) return pack_bf16x2(a, b);
  else return pack_f16x2(a, b);
}

// Output tile -> (m0, n0): tiles are walked in groups of group_m tile-rows.
template <int BM, int BN>
__device__ __forceinline__ void tile_origin(int pid, int tiles_m, int tiles_n, int group_m, int &m0, int &n0) {
  const int group_size = group_m * tiles_n;
  const int group = pid / group_size;
  const int first_m = group * group_m;
  const int gm = min(tiles_m - first_m, group_m);
  const int in_group = pid - group * group_size;
  m0 = (first_m + in_group % gm) * BM;
  n0 = (in_group / gm) * BN;
}

// Loads [first(s), first(s + 1)) of n loads spread over `slots` MFMA slots.
__host__ __device__ constexpr int spread_first(int s, int n, int slots) { return (s * n + slots - 1) / slots; }

// The kernels' MFMAs, with their accumulators pinned
// to AGPRs ("+a"): left to the register allocator, 256 accumulators plus the
// double-buffered fragments are shuffled between the register files and
// spilled.  The compiler sees these as opaque, so the kernel itself keeps the
// MFMA result hazards: a tile's first MFMA per accumulator adds an
// inline-constant zero (no VALU writes to accumulators at all; the tile kernels
// zero them long before the first MFMA), and the
// epilogue reads accumulators only after 24 wait states behind the
// tile's last MFMA.  Operand registers are written only by LDS loads, which
// the compiler's wait counts order before the MFMA that reads them; a buffer
// is reloaded only after the barrier that follows its last MFMA.
template <int KIND>
struct MfmaA;
template <>
struct MfmaA<kFp8> {
  static __device__ __forceinline__ void mma(f32x16 &c, const i32x8 &w, const i32x8 &x) {
    asm volatile("v_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
  }
  // c = w x (the accumulator's first product: an inline-constant zero addend)
  static __device__ __forceinline__ void mma0(f32x16 &c, const i32x8 &w, const i32x8 &x) {
    asm volatile("v_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, 0" : "=a"(c) : "v"(w), "v"(x));
  }
};
template <>
struct MfmaA<kInt8> {
  static __device__ __forceinline__ void mma(i32x16 &c, const i32x4 &w, const i32x4 &x) {
    asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
  }
  static __device__ __forceinline__ void mma0(i32x16 &c, const i32x4 &w, const i32x4 &x) {
    asm volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, 0" : "=a"(c) : "v"(w), "v"(x));
  }
};
// The exact kind: e4m3fn fragments in the FP8 kind's layout, widened to bf16
// (exact for every code) and multiplied by four 32x32x16 bf16 MFMAs, step s on
// bytes 8s..8s+7 of each lane's 32 from both operands, so every product pairs
// the same K index.  The activation fragment is widened once per block row
// (widen_x) and reused by its blocks; the weight fragment per call.
template <>
struct MfmaA<kFp8Exact> {
  struct xw_t {
    bf16x8 s[4];
  };
  static __device__ __forceinline__ xw_t widen_x(const i32x8 &x) {
    xw_t r;
#pragma unroll
    for (int k = 0; k < 4; ++k) r.s[k] = Mfma<kFp8Exact>::widen(x[2 * k], x[2 * k + 1]);
    return r;
  }
  template <bool ZERO>
  static __device__ __forceinline__ void run(f32x16 &c, const i32x8 &w, const xw_t &xb) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bf16x8 wb = Mfma<kFp8Exact>::widen(w[2 * k], w[2 * k + 1]);
      // the operands were just written by VALU conversions: 2 wait states before
      // an MFMA reads them (the compiler cannot see the MFMA inside the assembly)
      if (ZERO && k == 0)
        asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(wb), "v"(xb.s[k]));
      else
        asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(wb), "v"(xb.s[k]));
    }
  }
  static __device__ __forceinline__ void mma(f32x16 &c, const i32x8 &w, const xw_t &xb) { run<false>(c, w, xb); }
  // both operands already widened
  static __device__ __forceinline__ void mma(f32x16 &c, const xw_t &wb, const xw_t &xb) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(wb.s[k]), "v"(xb.s[k]));
  }
  static __device__ __forceinline__ void mma0(f32x16 &c, const i32x8 &w, const xw_t &xb) { run<true>(c, w, xb); }
  static __device__ __forceinline__ void mma(f32x16 &c, const i32x8 &w, const i32x8 &x) { run<false>(c, w, widen_x(x)); }
  static __device__ __forceinline__ void mma0(f32x16 &c, const i32x8 &w, const i32x8 &x) { run<true>(c, w, widen_x(x)); }
};

// 128-byte rows: 16-byte chunk c of row r at c ^ ((r >> 1) & 7); the 16 lanes of
// one 128-bit access (rows r..r+15, one chunk) hit 16 distinct bank groups.
__device__ __forceinline__ int swz128(int row, int chunk) { return row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4); }
template <int KIND>
__device__ __forceinline__ typename Mfma<KIND>::frag_t load_pair(const uint8_t *tile, int row, int half, int ks, int lane) {
  if constexpr (KIND == kInt8) {
    const u32x4 v = *reinterpret_cast<const u32x4 *>(tile + swz128(row, half * 4 + ks * 2 + (lane >> 5)));
    return typename Mfma<KIND>::frag_t{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
  } else {
    const int c0 = half * 4 + (lane >> 5) * 2;
    const u32x4 lo = *reinterpret_cast<const u32x4 *>(tile + swz128(row, c0));
    const u32x4 hi = *reinterpret_cast<const u32x4 *>(tile + swz128(row, c0 + 1));
    return typename Mfma<KIND>::frag_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w,
                                       (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  }
}

}  // namespace xgen
