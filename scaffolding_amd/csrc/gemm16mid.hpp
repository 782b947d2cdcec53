// gemm16mid.hpp — 16-bit GEMM for the sizes between the skinny stream (M <=
// 16) and full rounds of 256 x 256 tiles, and for operands at any 2-byte
// alignment:
//
//   C[b] = epi(alpha * op(A[b]) . op(B[b]) (+ bias) (+ R[b]))
//
// What bounds such a launch is latency: a few hundred short workgroups, each
// a serial chain of k slices.  So the tile is small (128 x 128, 64 x 64 or
// 32 x 64, picked with the k split by the host's estimate in abi.hip), two or
// three workgroups share a CU, and NST - 1 slices of 64 k are in flight while
// one is consumed.  Per slice: wait for this wave's loads of it, one barrier,
// issue the loads of slice t + NST - 1 into the stage that slice t - 1 left,
// read both halves' fragments, 2 FM FN MFMAs.
//
// Stages hold 128-byte lines in the layouts of gemm16nt_pp.hpp: rows of 64 k
// with 16-byte chunk h at slot h ^ (row & 7) for a K-contiguous operand, 64
// k-rows of 64 columns each with chunk c at slot c ^ fmn(k) for an
// M/N-contiguous one (fragments by ds_read_b64_tr_b16); both conflict-free.
// DMA: aligned operands move by buffer_load ... lds, chunks past an edge
// sent out of the buffer's range (zeros).  Otherwise the chunks are loaded
// into registers one slice ahead, 16 bytes at any 2-byte alignment, and
// written to the same layout; only a chunk across the edge is read element
// by element.
//
// k split (batch 1): the parts of a tile run on one XCD, park their fp32
// partials there, and the last to arrive sums all of them in part order
// (split_arrive_xcd: one atomic; the shared sum of the persistent kernel,
// with its chain of four, measured 1-4 us slower at these tile sizes).
//
// Measured (bf16, one MI355X, before -> after; before: register-staged 64 x
// 64 up to 256 x 128 tiles without a split, element-wise loads where
// unaligned):
//   226 x 1920 x 4096 NT    40.3 -> 13.3 us   64 x 64, 4 parts
//    64 x 4096 x 4096 NT    40.0 -> 11.6 us   32 x 64, 4 parts
//  1350 x 5760 x 1920 NT    81.4 -> 31.7 us   128 x 128 (940 TFLOP/s)
//  1350 x 1920 x 7680 NT    90.3 -> 50.0 us   128 x 128, 3 parts
//   603 x 1024 x 3200 NN    43.1 -> 15.1 us   64 x 64, 3 parts
//  2048 x 1920 x 7680 NN    82.8 -> 64.6 us   128 x 128, 2 parts
//  1920 x 1920 x 2048 TN    50.2 -> 26.2 us   128 x 128
//   777 x 1283 x 1001 NT    47.2 -> 14.7 us   64 x 64, unaligned
//   515 x 4097 x 2001 TN   217   -> 33.6 us   128 x 128, 3 parts, unaligned
// (Two, three or four unaligned slices held in registers instead of one:
// within 3 %; the unaligned accesses themselves are the limit.)
#pragma once

#include "gemm16nt_pp.hpp"

namespace sf {

// A 16-byte chunk at any 2-byte alignment (one global_load_dwordx4: global
// accesses need no alignment on this target).
struct __attribute__((packed, aligned(2))) Chunk16 {
  u32x4 v;
};

template <typename TIn, typename TOut, int BM, int BN, int WVM, int WVN, int NST, bool A_KM, bool B_KM, bool DMA,
          int OCC>
__global__ __launch_bounds__(WVM* WVN * 64, OCC) void gemm16mid_kernel(GemmParams p) {
  constexpr int NW = WVM * WVN;
  constexpr int BK = 64;
  constexpr int WM = BM / WVM, WN = BN / WVN;
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int A_BYTES = BM * 128, STAGE = (BM + BN) * 128;
  constexpr int IA = BM / 8 / NW, IB = BN / 8 / NW;  // 1 KB load instructions per wave and slice
  static_assert(WM % 16 == 0 && WN % 16 == 0 && IA * NW * 8 == BM && IB * NW * 8 == BN, "tile and wave grid");
  static_assert((A_KM || BM % 64 == 0) && (B_KM || BN % 64 == 0), "k-row blocks of 64 columns");
  static_assert(DMA || NST == 2, "register-staged loads run one slice ahead");
  constexpr int PITCH = WN * 2 + 16;  // staged output row
  constexpr int SMEM = NST * STAGE > NW * 16 * PITCH ? NST * STAGE : NW * 16 * PITCH;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WVN, wn = wave % WVN;
  const int M = p.M, N = p.N, K = p.K;
  const int KT = (K + BK - 1) / BK;

  // Workgroup -> (tile, k part).  XCD x (workgroup id mod 8) owns a
  // contiguous range of tiles with all their parts.
  const int xcd = blockIdx.x % kNumXcd, xo = blockIdx.x / kNumXcd;
  const int tiles = p.tiles_m * p.tiles_n;
  int tile, part = -1, t0 = 0, t1 = KT;
  if (p.split > 0) {
    const int first = (int)((int64_t)tiles * xcd / kNumXcd), last = (int)((int64_t)tiles * (xcd + 1) / kNumXcd);
    tile = first + xo / p.split;
    if (tile >= last) return;  // workgroup-uniform
    part = xo % p.split;
    t0 = (int)((int64_t)KT * part / p.split);
    t1 = (int)((int64_t)KT * (part + 1) / p.split);
  } else {
    tile = xcd_remap(blockIdx.x, gridDim.x);
  }
  int tm, tn;
  group_tile(tile, p.tiles_m, p.tiles_n, 8, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int64_t b = blockIdx.y;
  const uint16_t* __restrict__ A = static_cast<const uint16_t*>(p.A) + b * p.sA;
  const uint16_t* __restrict__ B = static_cast<const uint16_t*>(p.B) + b * p.sB;

  // ---- loads ----------------------------------------------------------------
  // Instruction i of wave w fills the 8 lines 8 (i NW + w) .. + 7 of its
  // operand.  K-contiguous: line = row, chunk h (8 k) at slot h ^ (row & 7).
  // M/N-contiguous: lines are the 64 k-rows of one 64-column block after the
  // other, chunk c (8 columns) of k-row k at slot c ^ fmn(k).
  const int l3 = lane >> 3;
  auto line_row = [&](int i) { return (i * NW + wave) * 8 + l3; };
  auto mn_chunk = [&](int krow) { return (lane & 7) ^ (2 * ((krow >> 1) & 1) + 4 * ((krow >> 3) & 1)); };
  constexpr uint32_t OOB = 0x80000000u;  // past every buffer's range: reads zeros
  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(
      (void*)A, (short)0, DMA ? (int)((uint32_t)(A_KM ? M : K) * (uint32_t)p.lda * 2u) : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t rB = __builtin_amdgcn_make_buffer_rsrc(
      (void*)B, (short)0, DMA ? (int)((uint32_t)(B_KM ? N : K) * (uint32_t)p.ldb * 2u) : 0, 0x00020000);
  uint32_t vo[IA + IB];  // per-lane offsets (slice 0 for an M/N-contiguous operand)
  if constexpr (DMA) {
    static_for<IA + IB>([&](auto i_c) {
      constexpr int I = decltype(i_c)::value;
      constexpr bool ISA = I < IA;
      constexpr int J = ISA ? I : I - IA;
      constexpr bool KM = ISA ? A_KM : B_KM;
      const int r = line_row(J), base = ISA ? m0 : n0, lim = ISA ? M : N;
      const uint32_t ld2 = (uint32_t)(ISA ? p.lda : p.ldb) * 2u;
      if constexpr (KM) {
        vo[I] = base + r < lim ? (uint32_t)(base + r) * ld2 + (uint32_t)(((lane & 7) ^ l3) * 16) : OOB;
      } else {
        const int col = base + (r >> 6) * 64 + mn_chunk(r & 63) * 8;
        vo[I] = col < lim ? (uint32_t)(r & 63) * ld2 + (uint32_t)col * 2u : OOB;
      }
    });
  }
  // Slice t into stage s.  Chunks past K (the last slice of a K that is no
  // multiple of 64) are sent out of range and read as zeros.
  auto issue = [&](int t, int s) {
    uint8_t* st = smem + s * STAGE;
    const bool tail = (t + 1) * BK > K;  // uniform
    static_for<IA + IB>([&](auto i_c) {
      constexpr int I = decltype(i_c)::value;
      constexpr bool ISA = I < IA;
      constexpr int J = ISA ? I : I - IA;
      constexpr bool KM = ISA ? A_KM : B_KM;
      uint32_t o = vo[I];
      int so = 0;
      if constexpr (KM) {
        so = t * BK * 2;
        if (tail && t * BK + ((lane & 7) ^ l3) * 8 >= K) o = OOB;
      } else {
        const uint32_t step = (uint32_t)t * (uint32_t)BK * (uint32_t)(ISA ? p.lda : p.ldb) * 2u;
        if ((tail && t * BK + (line_row(J) & 63) >= K) || o == OOB) o = OOB;
        else o += step;
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ISA ? rA : rB, (lds_ptr_t)(st + (ISA ? 0 : A_BYTES) + (J * NW + wave) * 1024),
                                               16, o, so, 0, 0);
    });
  };
  // Register-staged loads at any 2-byte alignment: whole chunks in one
  // load, the chunk that straddles the end element by element.
  u32x4 rg[DMA ? 1 : IA + IB];
  auto fetch = [&](int t) {
    static_for<IA + IB>([&](auto i_c) {
      constexpr int I = decltype(i_c)::value;
      constexpr bool ISA = I < IA;
      constexpr int J = ISA ? I : I - IA;
      constexpr bool KM = ISA ? A_KM : B_KM;
      const int r = line_row(J), base = ISA ? m0 : n0, lim = ISA ? M : N;
      const uint16_t* P = ISA ? A : B;
      const int64_t ld = ISA ? p.lda : p.ldb;
      // row (of ld elements), first element in it, elements valid from there
      int row, col, n_ok;
      if constexpr (KM) {
        row = base + r;
        col = t * BK + ((lane & 7) ^ l3) * 8;
        n_ok = row < lim ? K - col : 0;
      } else {
        row = t * BK + (r & 63);
        col = base + (r >> 6) * 64 + mn_chunk(r & 63) * 8;
        n_ok = row < K ? lim - col : 0;
      }
      u32x4 v = {0u, 0u, 0u, 0u};
      if (n_ok >= 8) {
        v = reinterpret_cast<const Chunk16*>(P + (int64_t)row * ld + col)->v;
      } else if (n_ok > 0) {
        const uint16_t* e = P + (int64_t)row * ld + col;
#pragma unroll
        for (int q = 0; q < 7; ++q)
          if (q < n_ok) v[q >> 1] |= (uint32_t)e[q] << ((q & 1) * 16);
      }
      rg[DMA ? 0 : I] = v;
    });
  };
  auto park = [&](int s) {
    static_for<IA + IB>([&](auto i_c) {
      constexpr int I = decltype(i_c)::value;
      constexpr bool ISA = I < IA;
      constexpr int J = ISA ? I : I - IA;
      *reinterpret_cast<u32x4*>(smem + s * STAGE + (ISA ? 0 : A_BYTES) + (J * NW + wave) * 1024 + lane * 16) =
          rg[DMA ? 0 : I];
    });
  };

  // ---- fragments ------------------------------------------------------------
  const int fkm = (lane & 15) * 128 + (((lane >> 4) ^ (lane & 7)) << 4);
  const int mn_g = lane >> 4, mn_e = (lane >> 2) & 3, mn_a = lane & 3;
  const int mn_f = 2 * ((mn_e >> 1) & 1) + 4 * (mn_g & 1);
  const int fmn = (8 * mn_g + mn_e) * 128 + ((mn_f | (mn_a >> 1)) << 4) + (mn_a & 1) * 8;
  // 16-row block J of a wave tile that starts at row w0, k half H.
  auto frag = [&](auto km_c, auto j_c, auto h_c, uint32_t base, int w0) -> u32x4 {
    constexpr bool KM = decltype(km_c)::value;
    constexpr int J = decltype(j_c)::value, H = decltype(h_c)::value;
    if constexpr (KM) {
      return ds_read16<J * 2048>((base + (uint32_t)(w0 * 128 + fkm)) ^ (H ? 64u : 0u));
    } else {
      const int blk = (w0 >> 4) + J;  // 16-column block of the tile
      const uint32_t ad = base + (uint32_t)((blk >> 2) * 8192) + ((uint32_t)fmn ^ (uint32_t)((blk & 3) << 5));
      const u32x2 lo = ds_read_tr16<H * 4096>(ad);
      const u32x2 hi = ds_read_tr16<H * 4096 + 512>(ad);
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  constexpr int HALF_READS = FM * (A_KM ? 1 : 2) + FN * (B_KM ? 1 : 2);

  f32x4 acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int s) {
    const uint32_t la = lds_addr(smem) + (uint32_t)(s * STAGE), lb = la + (uint32_t)A_BYTES;
    u32x4 ya[2][FM], xb[2][FN];
    __builtin_amdgcn_sched_barrier(0);
    static_for<2>([&](auto h_c) {
      constexpr int H = decltype(h_c)::value;
      static_for<FM>([&](auto j_c) {
        ya[H][decltype(j_c)::value] = frag(std::integral_constant<bool, A_KM>{}, j_c, h_c, la, wm * WM);
      });
      static_for<FN>([&](auto i_c) {
        xb[H][decltype(i_c)::value] = frag(std::integral_constant<bool, B_KM>{}, i_c, h_c, lb, wn * WN);
      });
    });
    static_for<2>([&](auto h_c) {
      constexpr int H = decltype(h_c)::value;
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, H ? 0 : (HALF_READS < 15 ? HALF_READS : 15)));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = Mfma16<TIn>::run(xb[H][i], ya[H][j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // ---- main loop --------------------------------------------------------------
  if constexpr (DMA) {
#pragma unroll
    for (int i = 0; i < NST - 1; ++i)
      if (t0 + i < t1) issue(t0 + i, i);
    int s = 0, sn = NST - 1;
    for (int t = t0; t < t1; ++t) {
      __builtin_amdgcn_sched_barrier(0);
      // this wave's loads of slice t landed; NST - 2 later slices in flight
      if (t + NST - 2 < t1)
        __builtin_amdgcn_s_waitcnt(waitcnt_imm((NST - 2) * (IA + IB), 0));
      else
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      // every wave has read slice t - 1, whose stage takes slice t + NST - 1
      if (t + NST - 1 < t1) issue(t + NST - 1, sn);
      __builtin_amdgcn_sched_barrier(0);
      compute(s);
      s = s + 1 == NST ? 0 : s + 1;
      sn = sn + 1 == NST ? 0 : sn + 1;
    }
  } else if (t0 < t1) {
    fetch(t0);
    park(0);
    __syncthreads();
    for (int t = t0; t < t1; ++t) {
      const int s = (t - t0) & 1;
      if (t + 1 < t1) fetch(t + 1);
      compute(s);
      if (t + 1 < t1) park(s ^ 1);
      __syncthreads();
    }
  }
  __syncthreads();

  const int tid = threadIdx.x;
  // ---- split tile: park the partial; the last part sums all in part order ------
  if (part >= 0) {
    constexpr int NT = NW * 64;
    float* mine = p.ws + (size_t)(tile * p.split + part) * (BM * BN);
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j)
        *reinterpret_cast<f32x4*>(mine + (size_t)((i * FM + j) * NT + tid) * 4) = acc[i][j];
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int* arrived = reinterpret_cast<int*>(smem);  // the operand stages are done with
    if (tid == 0) *arrived = split_arrive_xcd(&p.counters[tile], p.split, (xcd + p.xcd_shift) & (kNumXcd - 1));
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(*arrived) != p.split - 1) return;  // workgroup-uniform
    __syncthreads();  // read by every wave before the epilogue stages over it
    const float* all = p.ws + (size_t)tile * p.split * (BM * BN) + (size_t)tid * 4;
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int q = 0; q < p.split; ++q) {
      f32x4 v[FN][FM];
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
          v[i][j] = *reinterpret_cast<const f32x4*>(all + ((size_t)q * (FN * FM) + i * FM + j) * NT * 4);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] += v[i][j];
    }
    if (tid == 0) __hip_atomic_store(&p.counters[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // ---- epilogue: alpha, bias, activation, residual; staged through LDS --------
  const bool has_bias = epi_has_bias(p.epi);
  const float alpha = p.alpha;
  float bv[FN][4];
#pragma unroll
  for (int i = 0; i < FN; ++i) {
#pragma unroll
    for (int q = 0; q < 4; ++q) bv[i][q] = 0.f;
    if (has_bias) load_bias4<TIn>(p.bias, n0 + wn * WN + i * 16 + 4 * (lane >> 4), N, bv[i]);
  }
  uint8_t* stage = smem + wave * (16 * PITCH);
  uint16_t* C = static_cast<uint16_t*>(p.C) + b * p.sC;
  const void* R = p.res != nullptr ? static_cast<const uint16_t*>(p.res) + b * p.sR : nullptr;
  const bool rvec = R != nullptr && res_vec_ok<TOut>(R, p.ldr);
  constexpr int LROW = WN / 8;       // lanes per staged row (16 bytes each)
  constexpr int RPI = 64 / LROW;     // rows per store instruction
  constexpr int NSTO = RPI >= 16 ? 1 : 16 / RPI;
  with_act(epi_act(p.epi), [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int gmr = m0 + wm * WM + j * 16 + (lane & 15);
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const int n = n0 + wn * WN + i * 16 + 4 * (lane >> 4);
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = act_t<ACT>(acc[i][j][q] * alpha + bv[i][q]);
        if (R != nullptr && gmr < M) {
          float rr[4];
          Res4<TOut>::load(R, (int64_t)gmr * p.ldr, n, N, rvec, rr);
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] += rr[q];
        }
        *reinterpret_cast<u32x2*>(stage + (lane & 15) * PITCH + (i * 16 + 4 * (lane >> 4)) * 2) =
            u32x2{pack2<TOut>(v[0], v[1]), pack2<TOut>(v[2], v[3])};
      }
      wave_lds_sync();
#pragma unroll
      for (int rr = 0; rr < NSTO; ++rr) {
        const int r = rr * RPI + lane / LROW;
        const int cl = lane % LROW;
        if (RPI > 16 && r >= 16) continue;
        const u32x4 val = *reinterpret_cast<const u32x4*>(stage + r * PITCH + cl * 16);
        const int gm = m0 + wm * WM + j * 16 + r;
        const int gn = n0 + wn * WN + cl * 8;
        if (gm < M && gn < N) {
          uint16_t* crow = C + (int64_t)gm * p.ldc + gn;
          if (gn + 8 <= N) {
            reinterpret_cast<Chunk16*>(crow)->v = val;
          } else {
#pragma unroll
            for (int e = 0; e < 7; ++e)
              if (gn + e < N) crow[e] = static_cast<uint16_t>(val[e >> 1] >> ((e & 1) * 16));
          }
        }
      }
    }
  });
}

}  // namespace sf
