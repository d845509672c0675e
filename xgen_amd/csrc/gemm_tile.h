// The W8A8 GEMM on tiles below 256 x 256 (gfx950): one output tile per
// workgroup, for calls whose 256 x 256 tiles would leave compute units idle.
//
// A workgroup of WM x WN waves computes a (32 WM FM) x (32 WN FN) output tile;
// each wave owns FM x FN MFMA fragments of 32 x 32.  K advances in pairs of
// 64-byte sub-stages as in the 256 x 256 kernel (128 bytes of K per row and DMA
// load, the same swizzled LDS rows, the same MFMA and K order: an output's
// accumulator is the same bits in every kernel), through a ring of SLOTS pair
// slots, one barrier per pair:
//
//   sub-stage 0 of pair p: MFMAs on buffer 0; the fragments of sub-stage 1 are read
//   wait for this thread's DMA of pair p + 1; barrier (publishes pair p + 1 and
//     retires every wave's reads of pair p)
//   sub-stage 1 of pair p: MFMAs on buffer 1; the fragments of pair p + 1's
//     sub-stage 0 are read; the DMA of pair p + SLOTS goes into pair p's slot
//
// so a pair's DMA has SLOTS - 1 pairs of work in front of it.
//
// What bounds it: a tile's K steps are a serial chain, so a few hundred tokens
// cost K / 128 steps whatever the number of workgroups below the CUs'.  On 32 x 64
// with the weights in the last-level cache a step takes 0.16 us, 0.34 in the exact
// kind (from memory: kTileCosts); 256 x 1,024 x 1,024 so takes 4.7 us on 128 such
// tiles, 15 on 4 tiles of 256 x 256 (exact kind 6.2 and 24).  From about one 128 x 192 tile per CU on it is the board's
// power: M = 1,955, N = 3,072, K = 12,288 on 256 tiles takes 62 us (2.37 PFLOP/s;
// 104 us on 96 tiles of 256 x 256), 49 us with all operands zero, and 59 us with
// the fragment reads taken out.  Per flop a smaller tile moves more data through
// L2 and LDS (128 bytes of both operands' rows per pair, 64 B per clock and CU at
// most), which is why the 256 x 256 kernel keeps the calls that fill it.
//
// Epilogue: the ring is free by then; the tile's outputs are rounded into it as
// rows, and stored from there as whole 16-byte pieces of rows.  GATED: the gated
// residual is applied at the store; its residual rows and table indices are read
// in front of the last sub-stage, its gate rows one group of pieces ahead (all of
// them read at the store: 3,906 x 3,072 x 3,072 FP8 43.2 us, 40.6 so).
#pragma once

#include "gemm_w8a8.h"

namespace xgen {

template <int WM, int WN, int FM, int FN, int SLOTS>
struct TileCfg {
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kM = 32 * WM * FM, kN = 32 * WN * FN;
  // 1 KB DMA loads (8 rows of 128 bytes) per wave and pair; load q of wave w fills
  // rows 8 (q kWaves + w) .. + 7 of its operand's tile
  static constexpr int kLoadsA = kM / 8 / kWaves, kLoadsW = kN / 8 / kWaves, kLoads = kLoadsA + kLoadsW;
  static constexpr int kSlotBytes = (kM + kN) * 128;
  static constexpr int kRing = SLOTS * kSlotBytes;
  // output rows in LDS: 16 bytes of padding move consecutive rows 4 banks on
  static constexpr int kRowPitch = kN * 2 + 16;
  static constexpr int kOutBytes = kM * kRowPitch;
  // the tile's scales and bias as f32, behind the output rows
  static constexpr int kParamBase = kOutBytes, kParamBytes = (kM + 2 * kN) * 4;
  static constexpr int kLdsBytes = kRing > kParamBase + kParamBytes ? kRing : kParamBase + kParamBytes;
  static_assert(kM % (8 * kWaves) == 0 && kN % (8 * kWaves) == 0 && kM <= 256 && kN <= 256, "DMA split");
  static_assert((SLOTS - 1) * kLoads < 64, "vmcnt range");
  static_assert(kLdsBytes <= 160 * 1024, "LDS");
};

template <int KIND, int WM, int WN, int FM, int FN, int SLOTS, bool GATED>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * WM * WN, 64 * WM * WN), amdgpu_waves_per_eu(1)))
void gemm_tile_kernel(GemmArgs p) {
  typedef TileCfg<WM, WN, FM, FN, SLOTS> C;
  typedef Mfma<KIND> T;
  typedef typename T::frag_t frag_t;
  constexpr int KS = T::kSteps;
  constexpr int kMfmas = KS * FM * FN;     // per sub-stage per wave (64-byte steps of the exact kind count once)
  // three slots or more: a pair's DMA loads are spread over two sub-stages (all in one queue
  // up in the address unit ahead of the MFMAs: 3% to 11% slower)
  constexpr bool kSpread = SLOTS > 2;
  // exact kind: both operands' fragments widened once, where a wave's activation fragments
  // fit the registers widened
  constexpr bool kWeightsOuter = FM <= 2;
  constexpr int kFrags = KS * (FM + FN);   // fragment reads per sub-stage per wave
  __shared__ __attribute__((aligned(1024))) uint8_t smem[C::kLdsBytes];

  // --- this workgroup's tile: consecutive workgroup ids go to the 8 XCDs round-robin,
  // XCD x owns a contiguous range of tiles ---
  const int t = (blockIdx.x & 7) * p.per_xcd + (blockIdx.x >> 3);
  if (t >= p.tiles_m * p.tiles_n) return;
  int m0, n0;
  tile_origin<C::kM, C::kN>(t, p.tiles_m, p.tiles_n, p.group_m, m0, n0);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;

  auto rsrc = [](const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, kBufferFlags);
  };
  const __amdgpu_buffer_rsrc_t ra = rsrc(p.a, p.a_bytes), rw = rsrc(p.w, p.w_bytes);

  // --- the epilogue's scales and bias: thread t holds token m0 + t's and feature n0 + t's
  // from here to the epilogue, which shares them through LDS ---
  static_assert(C::kM <= C::kThreads && C::kN <= C::kThreads, "one token and one feature per thread");
  const int pm = min(m0 + tid, p.M - 1), pn = min(n0 + tid, p.N - 1);
  const float sa_t = p.sa[p.sa_stride ? pm : 0], sw_t = p.sw[p.sw_stride ? pn : 0];
  float bias_t = 0.0f;
  if (p.bias) {  // uniform
    if (p.bias_dtype == XGEN_DTYPE_F32) bias_t = static_cast<const float *>(p.bias)[pn];
    else if (p.bias_dtype == XGEN_DTYPE_F16) bias_t = (float)static_cast<const _Float16 *>(p.bias)[pn];
    else bias_t = Half2<XGEN_DTYPE_BF16>::lo(static_cast<const uint16_t *>(p.bias)[pn]);
  }

  // --- global -> LDS DMA: lane l fills row (l >> 3) of an 8-row load, physical chunk
  // l & 7, i.e. logical chunk (l & 7) ^ ((row >> 1) & 7); a wave's loads all start at
  // rows of the same parity of row / 8 (kWaves is 1 or even) ---
  static_assert(C::kWaves % 2 == 0, "one chunk per lane for all of a wave's loads");
  const int ch = ((lane & 7) ^ (((wave & 1) << 2) | (lane >> 4))) * 16;
  const uint32_t offa = (uint32_t)(m0 + wave * 8 + (lane >> 3)) * (uint32_t)p.lda + ch;
  const uint32_t offw = (uint32_t)(n0 + wave * 8 + (lane >> 3)) * (uint32_t)p.ldw + ch;
  int dma_k = 0;             // K byte of the next pair to load
  uint32_t dma_slot = 0;     // its slot's LDS offset
  uint32_t oa = 0, ow = 0;   // its offsets, or out of range
  // (kOutOfRange + rows * ld stays out of range: the host keeps (M + 512) * lda below 2^32)
  auto issue_begin = [&]() {
    const bool live = dma_k + ch < p.K;
    oa = live ? offa + dma_k : kOutOfRange;
    ow = live ? offw + dma_k : kOutOfRange;
    asm volatile("" : "+v"(oa), "+v"(ow));
  };
  auto issue_load = [&](int q) {
    uint8_t *dst = smem + dma_slot + wave * 1024;
    if (q < C::kLoadsA) dma_load16(ra, dst + q * C::kWaves * 1024, oa + (uint32_t)(q * C::kWaves * 8 * p.lda));
    else {
      const int r = q - C::kLoadsA;
      dma_load16(rw, dst + C::kM * 128 + r * C::kWaves * 1024, ow + (uint32_t)(r * C::kWaves * 8 * p.ldw));
    }
  };
  auto issue_end = [&]() {
    dma_k += 128;
    dma_slot = dma_slot + C::kSlotBytes == C::kRing ? 0 : dma_slot + C::kSlotBytes;
  };

  // --- fragments: [register buffer = sub-stage][k step][fragment] ---
  const int row_x = wm * 32 * FM + (lane & 31), row_w = wn * 32 * FN + (lane & 31);
  frag_t xf[2][KS][FM], wf[2][KS][FN];
  uint32_t rd_slot = 0;  // LDS offset of the pair being multiplied
  auto read_frag = [&](int b, uint32_t slot, int r) {  // fragment r of sub-stage b, weights first
    const int ks = r / (FM + FN), f = r % (FM + FN);
    if (f < FN) wf[b][ks][f] = load_pair<KIND>(smem + slot + C::kM * 128, row_w + f * 32, b, ks, lane);
    else xf[b][ks][f - FN] = load_pair<KIND>(smem + slot, row_x + (f - FN) * 32, b, ks, lane);
  };

  typename T::acc_t acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      acc[i][j] = typename T::acc_t{};
      asm volatile("" : "+a"(acc[i][j]));
    }

  // one sub-stage: its MFMAs, with the next sub-stage's fragment reads (READ) and a share of
  // a later pair's DMA loads (LOAD) between them
  auto sub_stage = [&](auto B, auto LOAD, auto READ, uint32_t next_slot) {
    constexpr int b = decltype(B)::value;
    constexpr bool load = decltype(LOAD)::value, read = decltype(READ)::value;
    if constexpr (b == 1 && load) issue_begin();
    // the MFMAs are volatile asm statements: the loads written between them stay there
    // (the exact kind widens each activation fragment once per sub-stage and, weights
    // outermost, each weight fragment once too)
    [[maybe_unused]] typename std::conditional<KIND == kFp8Exact, MfmaA<kFp8Exact>::xw_t, int>::type xw[FM] = {}, ww{};
#pragma unroll
    for (int s = 0; s < kMfmas; ++s) {
      const int ks = s / (FM * FN);
      if constexpr (KIND == kFp8Exact && kWeightsOuter) {
        const int i = s / FM, j = s % FM;
        if (j == 0) ww = MfmaA<KIND>::widen_x(wf[b][ks][i]);
        if (i == 0) xw[j] = MfmaA<KIND>::widen_x(xf[b][ks][j]);
        MfmaA<KIND>::mma(acc[i][j], ww, xw[j]);
      } else if constexpr (KIND == kFp8Exact) {
        const int j = s / FN, i = s % FN;
        if (i == 0) xw[0] = MfmaA<KIND>::widen_x(xf[b][ks][j]);
        MfmaA<KIND>::mma(acc[i][j], wf[b][ks][i], xw[0]);
      } else {
        const int j = (s / FN) % FM, i = s % FN;
        MfmaA<KIND>::mma(acc[i][j], wf[b][ks][i], xf[b][ks][j]);
      }
      if constexpr (read) {
#pragma unroll
        for (int r = spread_first(s, kFrags, kMfmas); r < spread_first(s + 1, kFrags, kMfmas); ++r)
          read_frag(b ^ 1, next_slot, r);
      }
      if constexpr (load && kSpread) {
        // sub-stage 1 takes the first half of a pair's loads, the next sub-stage 0 the rest
        constexpr int kFirst = (C::kLoads + 1) / 2, n = b == 1 ? kFirst : C::kLoads - kFirst, q0 = b == 1 ? 0 : kFirst;
#pragma unroll
        for (int q = spread_first(s, n, kMfmas); q < spread_first(s + 1, n, kMfmas); ++q) issue_load(q0 + q);
      } else if constexpr (load && b == 1) {
#pragma unroll
        for (int q = spread_first(s, C::kLoads, kMfmas); q < spread_first(s + 1, C::kLoads, kMfmas); ++q) issue_load(q);
      }
    }
    if constexpr (load && b == (kSpread ? 0 : 1)) issue_end();
  };
  typedef std::integral_constant<int, 0> B0;
  typedef std::integral_constant<int, 1> B1;
  typedef std::integral_constant<bool, true> Yes;
  typedef std::integral_constant<bool, false> No;

  // --- prologue: SLOTS pairs in flight, pair 0's first fragments in registers ---
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    issue_begin();
#pragma unroll
    for (int q = 0; q < (kSpread && s == SLOTS - 1 ? (C::kLoads + 1) / 2 : C::kLoads); ++q) issue_load(q);
    if (!(kSpread && s == SLOTS - 1)) issue_end();
  }
  wait_vmcnt<(SLOTS - 1) * C::kLoads - (kSpread ? C::kLoads / 2 : 0)>();
  lds_barrier();
#pragma unroll
  for (int r = 0; r < kFrags; ++r) read_frag(0, 0, r);

  // pairs past K are zeros: the ring is filled once at least
  const int pairs = (p.K + 127) / 128 > SLOTS ? (p.K + 127) / 128 : SLOTS;
  // waits for this thread's loads of the next pair (`newer` pairs were issued after them),
  // then publishes every wave's and retires the reads of this one
  auto publish = [&](auto NEWER) {
    wait_vmcnt<decltype(NEWER)::value * C::kLoads>();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    lds_barrier();
  };
  auto next_slot = [&]() { return rd_slot + C::kSlotBytes == C::kRing ? 0u : rd_slot + C::kSlotBytes; };
  for (int k = 0; k < pairs - SLOTS; ++k) {
    sub_stage(B0(), Yes(), Yes(), rd_slot);
    publish(std::integral_constant<int, SLOTS - 2>());
    // (the DMA slot of sub-stage 1 is rd_slot: both advance once per pair)
    const uint32_t next = next_slot();
    sub_stage(B1(), Yes(), Yes(), next);
    rd_slot = next;
  }
  // the last SLOTS pairs: their loads are issued (but for the first one's share of a spread
  // pair), so fewer and fewer stay in flight
  auto tail = [&](auto LEFT) {  // LEFT pairs after this one
    constexpr int left = decltype(LEFT)::value;
    if constexpr (left == SLOTS - 1) sub_stage(B0(), Yes(), Yes(), rd_slot);
    else sub_stage(B0(), No(), Yes(), rd_slot);
    if constexpr (left > 0) {
      publish(std::integral_constant<int, left - 1>());
      const uint32_t next = next_slot();
      sub_stage(B1(), No(), Yes(), next);
      rd_slot = next;
    }
  };
  static_assert(SLOTS >= 2 && SLOTS <= 6, "tail");
  if constexpr (SLOTS > 5) tail(std::integral_constant<int, 5>());
  if constexpr (SLOTS > 4) tail(std::integral_constant<int, 4>());
  if constexpr (SLOTS > 3) tail(std::integral_constant<int, 3>());
  if constexpr (SLOTS > 2) tail(std::integral_constant<int, 2>());
  tail(std::integral_constant<int, 1>());
  tail(std::integral_constant<int, 0>());

  // the gated residual's inputs, in front of the last MFMAs and the rounding: this thread's
  // pieces of the residual rows, and their token's table indices
  constexpr int kChunks = C::kN / 8, kPieces = C::kM * kChunks, kSteps = kPieces / C::kThreads;
  static_assert(kPieces % C::kThreads == 0, "store split");
  [[maybe_unused]] u32x4 res[GATED ? kSteps : 1];
  [[maybe_unused]] u32x2 gidx[GATED ? kSteps : 1];
  auto piece = [&](int q, uint32_t &row, uint32_t &col) {  // piece q of this thread: 8 columns of a row
    const int c = q * C::kThreads + tid;
    row = (uint32_t)(m0 + c / kChunks), col = (uint32_t)(n0 + c % kChunks * 8);
    return row < (uint32_t)p.M && col < (uint32_t)p.N;
  };
  // (the rest, past what the registers hold beside the fragments, behind the rounding)
  constexpr int kResAhead = kSteps <= 16 ? kSteps : 8;
  [[maybe_unused]] auto load_res = [&](int q0, int q1) {
    const __amdgpu_buffer_rsrc_t rres = rsrc(p.residual, p.residual_bytes), rind = rsrc(p.indices, p.seq * 8);
#pragma unroll
    for (int q = q0; q < q1; ++q) {
      uint32_t row, col;
      const bool in = piece(q, row, col);
      const uint32_t mq = (__umulhi(row, p.seq_magic) + row) >> p.seq_shift;
      gidx[q] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rind, (row - mq * p.seq) * 8, 0, 0));
      res[q] = __builtin_amdgcn_raw_buffer_load_b128(
          rres, in ? (row * (uint32_t)p.ld_residual + col) * 2 : kOutOfRange, 0, 0);
    }
  };
  if constexpr (GATED) load_res(0, kResAhead);
  sub_stage(B1(), No(), No(), rd_slot);

  // --- epilogue --------------------------------------------------------------------
  // 24 wait states behind the last MFMAs before any accumulator is read
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+a"(acc[0][0]));
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) asm volatile("" : "+a"(acc[i][j]));
  // (every DMA load has landed: the last publish waited for all; the barrier retires the
  // other waves' fragment reads before the ring is written)
  lds_barrier();
  float *prm = reinterpret_cast<float *>(smem + C::kParamBase);  // [sa of kM][sw of kN][bias of kN]
  if (tid < C::kM) prm[tid] = sa_t;
  if (tid < C::kN) prm[C::kM + tid] = sw_t, prm[C::kM + C::kN + tid] = bias_t;
  __syncthreads();
  const int half = lane >> 5;
  // acc[i][j] element e: feature n0 + wn*32*FN + i*32 + (e/4)*8 + (lane/32)*4 + e%4,
  //                      token   m0 + wm*32*FM + j*32 + lane%32
  auto round_tile = [&](auto OUT, auto ACT) {
    constexpr int kOut = decltype(OUT)::value, kAct = decltype(ACT)::value;
    float sam[FM];
#pragma unroll
    for (int j = 0; j < FM; ++j) sam[j] = prm[wm * 32 * FM + j * 32 + (lane & 31)];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int nl = wn * 32 * FN + i * 32 + gq * 8 + half * 4;  // this lane's 4 features
        const f32x4 swr = *reinterpret_cast<const f32x4 *>(prm + C::kM + nl);
        const f32x4 bir = *reinterpret_cast<const f32x4 *>(prm + C::kM + C::kN + nl);
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          const int ml = wm * 32 * FM + j * 32 + (lane & 31);
          float y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            y[e] = __builtin_fmaf(T::to_f32(acc[i][j][gq * 4 + e]), sam[j] * swr[e], bir[e]);
            if constexpr (kAct == XGEN_ACT_GELU_TANH) y[e] = gelu_tanh(round_out<kOut>(y[e]));
          }
          *reinterpret_cast<u32x2 *>(smem + ml * C::kRowPitch + nl * 2) =
              u32x2{pack_out<kOut>(y[0], y[1]), pack_out<kOut>(y[2], y[3])};
          if (p.acc_out) {
            const int m = m0 + ml, n = n0 + nl;
            if (m < p.M && n < p.N) {
              typedef typename std::conditional<KIND == kInt8, i32x4, f32x4>::type acc4_t;
              *reinterpret_cast<acc4_t *>(static_cast<uint8_t *>(p.acc_out) + ((int64_t)m * p.N + n) * 4) = acc4_t{
                  acc[i][j][gq * 4 + 0], acc[i][j][gq * 4 + 1], acc[i][j][gq * 4 + 2], acc[i][j][gq * 4 + 3]};
            }
          }
        }
      }
  };
  typedef std::integral_constant<int, XGEN_DTYPE_BF16> Bf16;
  typedef std::integral_constant<int, XGEN_DTYPE_F16> F16;
  typedef std::integral_constant<int, XGEN_ACT_NONE> NoAct;
  typedef std::integral_constant<int, XGEN_ACT_GELU_TANH> Gelu;
  if (p.out_dtype == XGEN_DTYPE_BF16) {
    if (p.act == XGEN_ACT_NONE) round_tile(Bf16(), NoAct());
    else round_tile(Bf16(), Gelu());
  } else {
    if (p.act == XGEN_ACT_NONE) round_tile(F16(), NoAct());
    else round_tile(F16(), Gelu());
  }
  if constexpr (GATED) load_res(kResAhead, kSteps);
  __syncthreads();

  // rows of 16-byte pieces, consecutive lanes on consecutive pieces of a row; rows past M
  // and columns past N are dropped (N is a multiple of 16)
  const __amdgpu_buffer_rsrc_t ro = rsrc(p.out, p.out_bytes);
  constexpr int kUnroll = kSteps % 4 == 0 ? 4 : kSteps % 3 == 0 ? 3 : kSteps % 2 == 0 ? 2 : 1;
  [[maybe_unused]] u32x4 gt[GATED ? 2 : 1][kUnroll];  // the gate rows' pieces, one group ahead
  [[maybe_unused]] auto load_gate = [&](int q0) {
    const __amdgpu_buffer_rsrc_t rgate = rsrc(p.gate, p.gate_bytes);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      uint32_t row, col;
      const bool in = piece(q0 + u, row, col);
      const u32x2 g = gidx[q0 + u];
      const bool ok = g.y == 0 && g.x < (uint32_t)p.gate_rows;  // an int64 index in [0, gate_rows)
      gt[(q0 / kUnroll) & 1][u] = __builtin_amdgcn_raw_buffer_load_b128(
          rgate, in && ok ? (g.x * (uint32_t)p.gate_stride + col) * 2 : kOutOfRange, 0, 0);
    }
  };
  if constexpr (GATED) load_gate(0);
#pragma unroll
  for (int q0 = 0; q0 < kSteps; q0 += kUnroll) {
    if constexpr (GATED) {
      __builtin_amdgcn_sched_barrier(0);  // (a later group's reads stay behind this one's: registers)
      if (q0 + kUnroll < kSteps) load_gate(q0 + kUnroll);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int c = (q0 + u) * C::kThreads + tid;
      uint32_t row, col;
      const bool in = piece(q0 + u, row, col);
      u32x4 v = *reinterpret_cast<const u32x4 *>(smem + c / kChunks * C::kRowPitch + c % kChunks * 16);
      if constexpr (GATED) {
        const u32x2 g = gidx[q0 + u];
        v = g.y == 0 && g.x < (uint32_t)p.gate_rows
                ? gate_residual8(res[q0 + u], v, gt[(q0 / kUnroll) & 1][u])
                : u32x4{0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u};  // outside the table: NaN
      }
      __builtin_amdgcn_raw_buffer_store_b128(v, ro, in ? (row * (uint32_t)p.ldo + col) * 2 : kOutOfRange, 0, 0);
    }
  }
}

}  // namespace xgen
