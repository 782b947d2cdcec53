// attention_wide.hpp — fused attention forward for head sizes up to 128 and
// with an additive mask, 16-bit Q/K/V/O, fp32 accumulation and softmax:
//
//   O[b] = softmax(scale * Q[b] K[b]^T + mask) V[b]
//
// attn64_kernel's scheme (attention.hpp: Q in registers, K and V blocks of 64
// keys through an LDS ring by direct loads, exponents out of the score MFMAs
// against lazily raised row references, P never between lanes) on tiles 64,
// 96 or 128 wide along d.  A wave holds 32 query rows instead of 64: at head
// size 128 the O accumulator alone would take 128 of the 256 registers that
// let two workgroups share a CU, and a mask block of 64 rows 64 more.  K and
// V rows longer than 64 d lie in two 128-byte halves; V's second half is read
// into the first half's registers once its products are issued.  Work items
// are 128 query rows; each XCD takes a contiguous range of them, so the
// blocks of one head share its L2 (K and V are read once per 128 rows, twice
// as often as by attn64_kernel).
//
// The mask block of the next 64 keys is loaded while P V runs.  Its values
// go into the score MFMAs' C operand (PRE), so a masked score costs two VALU
// operations more than an unmasked one.  Rows that have no reference yet, or
// one far down or up (a large finite mask so far), form their scores without
// a reference first ("deep"); rows that meet no key at all are finished by
// attn_special_rows, those that the exponent domain cannot hold by
// attn_exact_rows.
//
// Bound by VALU issue and MFMA alternating in two waves a SIMD, as
// attn64_kernel.  Measured (bf16, one MI355X; before: three launches with
// the scores in memory):
//   2 x 16 heads, 2048 x 2048, D 128          278 -> 64 us   (1080 TFLOP/s)
//   2 x 24 heads, 8192 x 8192, D 128             1.38 ms     (1200 TFLOP/s)
//   1 x 30 heads, 7239 x 7239, D 72        7.6 ms -> 0.56 ms
//   4 x 16 heads, 1024 x 1024, D 64, causal mask 127 -> 40 us
//   1 x 30 heads, 1350 x 1350, D 64           37.2 -> 30.4 us (attn64_kernel)
#pragma once

#include "attention.hpp"

namespace sf {

struct AttnWideParams {
  AttnParams a;
  const void* mask;            // NULL without one (MK == 0)
  int64_t mB, mH, mR;          // its batch, head and row strides, elements
};

// DW: tile width along d (64, 96 or 128).  Rows of 64 d (128 bytes) as in
// attn64_kernel, DW > 64 in two such halves.
template <int DW>
struct AttnWideCfg {
  static constexpr int MB = 2;                 // 16-row query blocks per wave
  static constexpr int ROWS = 4 * MB * 16;     // query rows per work item
  static constexpr int HALVES = (DW + 63) / 64;
  static constexpr int NS = DW > 64 ? 2 : 3;   // key blocks of 64 in LDS
  static constexpr int PART_O = 4 * MB * (DW / 16) * 64 * 4;
  static constexpr int PART = PART_O + 4 * MB * 64 * 2;  // floats of one split part
};

// Sixteen bits or fp32 mask values of four consecutive keys at any element
// alignment, as fp32.
struct __attribute__((packed, aligned(4))) MaskF4 {
  f32x4 v;
};
struct __attribute__((packed, aligned(2))) MaskH4 {
  u32x2 v;
};

template <typename T, int MK>
__device__ __forceinline__ float mask_at(const void* row, int64_t j) {
  if constexpr (MK == 1) return static_cast<const float*>(row)[j];
  else return Elem<T>::to_f32(static_cast<const uint16_t*>(row)[j]);
}

template <typename T, int MK>
__device__ __forceinline__ f32x4 mask4(const void* row, int64_t j) {
  if constexpr (MK == 1) {
    return reinterpret_cast<const MaskF4*>(static_cast<const float*>(row) + j)->v;
  } else {
    const u32x2 w = reinterpret_cast<const MaskH4*>(static_cast<const uint16_t*>(row) + j)->v;
    return f32x4{Elem<T>::to_f32((uint16_t)(w.x & 0xffffu)), Elem<T>::to_f32((uint16_t)(w.x >> 16)),
                 Elem<T>::to_f32((uint16_t)(w.y & 0xffffu)), Elem<T>::to_f32((uint16_t)(w.y >> 16))};
  }
}

// Output rows whose every key is masked to -inf or so far down that the mask
// overflowed in the exponent domain (below about -2e38), all scores finite.
// There mask + score is the mask itself in fp32, so the softmax is uniform
// over the keys that carry the row's largest mask value, and NaN where that
// is -inf: what softmax(scores + mask) gives.  (A row with a NaN or +inf
// score is not sent here: its exponents are NaN; one with a score of -inf
// goes to attn_exact_rows.)  `rows`: bit i for row q0 + i.  One wave; rows
// that share one mask row (mR == 0) share the sum.
template <typename T, int MK>
__device__ __forceinline__ void attn_special_rows(const AttnWideParams& wp, int64_t b, int64_t h, int q0,
                                                  uint64_t rows) {
  const AttnParams& p = wp.a;
  const int lane = threadIdx.x & 63;
  const uint16_t* Vb = static_cast<const uint16_t*>(p.V) + b * p.sV + h * p.hV;
  // Lane 16 g + c: columns 8 c .. 8 c + 7 of every fourth key from g.
  const int g = lane >> 4, d0 = 8 * (lane & 15);
  const bool dok = d0 < p.D;  // D % 8 == 0
  u32x4 out = {0u, 0u, 0u, 0u};
  bool have = false;
  while (rows != 0) {
    const int r = q0 + __builtin_ctzll(rows);
    rows &= rows - 1;
    if (!have || wp.mR != 0) {
      have = true;
      const int64_t mo = b * wp.mB + h * wp.mH + (int64_t)r * wp.mR;
      const void* mrow = MK == 1 ? (const void*)(static_cast<const float*>(wp.mask) + mo)
                                 : (const void*)(static_cast<const uint16_t*>(wp.mask) + mo);
      float mx = -INFINITY;
      for (int j = lane; j < p.Sk; j += 64) mx = fmaxf(mx, mask_at<T, MK>(mrow, j));
      mx = wave_max(mx);
      float n = 0.f, acc[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = 0.f;
      if (mx > -INFINITY) {
        for (int j0 = g; j0 < p.Sk; j0 += 32) {
          u32x4 v[8];
          bool in[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {  // eight keys' loads in flight
            const int j = j0 + 4 * u;
            const int jc = j < p.Sk ? j : p.Sk - 1;
            in[u] = j < p.Sk && mask_at<T, MK>(mrow, jc) == mx;
            v[u] = *reinterpret_cast<const u32x4*>(Vb + (int64_t)jc * p.ldv + (dok ? d0 : 0));
          }
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const float pu = in[u] ? 1.f : 0.f;  // times V: a NaN or infinite V reaches the row
            n += pu;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const uint32_t w = v[u][e >> 1];
              acc[e] = __builtin_fmaf(pu, Elem<T>::to_f32((uint16_t)(w >> ((e & 1) * 16))), acc[e]);
            }
          }
        }
      }
#pragma unroll
      for (int off = 16; off <= 32; off <<= 1) {
        n += __shfl_xor(n, off, 64);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
      }
      const float inv = 1.0f / n;  // no key: 0 * inf = NaN
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = pack2<T>(acc[2 * e] * inv, acc[2 * e + 1] * inv);
    }
    if (g == 0 && dok)
      *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p.O) + b * p.sO + h * p.hO + (int64_t)r * p.ldo + d0) = out;
  }
}

// Output rows that the exponent domain cannot hold: a mask value whose
// product with log2 e overflows upwards, a reference raised far up in one
// step, or a score of -inf in a row without a key in reach.  softmax(scores +
// mask) V term by term in fp32, scores from global memory: slow, for inputs
// that hold such values.  One wave.  Not inlined: its mere presence in the
// kernels cost launches of few blocks up to 7 % (4 x 8 heads, 77 x 77, D 128:
// 8.8 -> 9.4 us; called, 8.8 us).
template <typename T, int MK>
__device__ __attribute__((noinline)) void attn_exact_rows(const AttnWideParams& wp, int64_t b, int64_t h, int q0,
                                                          uint64_t rows) {
  constexpr float LN2 = 0.6931471805599453f, LOG2E = 1.4426950408889634f;
  const AttnParams& p = wp.a;
  const int lane = threadIdx.x & 63;
  const uint16_t* Kb = static_cast<const uint16_t*>(p.K) + b * p.sK + h * p.hK;
  const uint16_t* Vb = static_cast<const uint16_t*>(p.V) + b * p.sV + h * p.hV;
  const float scale = p.scale_log2e * LN2;
  const bool dok = 2 * lane < p.D;  // lane: columns 2 lane, 2 lane + 1
  while (rows != 0) {
    const int r = q0 + __builtin_ctzll(rows);
    rows &= rows - 1;
    const uint16_t* qrow = static_cast<const uint16_t*>(p.Q) + b * p.sQ + h * p.hQ + (int64_t)r * p.ldq;
    const int64_t mo = b * wp.mB + h * wp.mH + (int64_t)r * wp.mR;
    const void* mrow = MK == 1 ? (const void*)(static_cast<const float*>(wp.mask) + mo)
                               : (const void*)(static_cast<const uint16_t*>(wp.mask) + mo);
    auto score = [&](int j) {
      const uint16_t* krow = Kb + (int64_t)j * p.ldk;
      float dot = 0.f;
#pragma nounroll
      for (int d = 0; d < p.D; d += 8) {
        const u32x4 qv = *reinterpret_cast<const u32x4*>(qrow + d), kv = *reinterpret_cast<const u32x4*>(krow + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t qw = qv[e], kw = kv[e];
          dot = __builtin_fmaf(Elem<T>::to_f32((uint16_t)(qw & 0xffffu)), Elem<T>::to_f32((uint16_t)(kw & 0xffffu)), dot);
          dot = __builtin_fmaf(Elem<T>::to_f32((uint16_t)(qw >> 16)), Elem<T>::to_f32((uint16_t)(kw >> 16)), dot);
        }
      }
      return __builtin_fmaf(dot, scale, mask_at<T, MK>(mrow, j));
    };
    float mx = -INFINITY;
    bool bad = false;
#pragma nounroll
    for (int j = lane; j < p.Sk; j += 64) {
      const float x = score(j);
      bad |= x != x;
      mx = fmaxf(mx, x);
    }
    mx = wave_max(mx);
    // NaN scores, +inf (inf - inf) or nothing but -inf
    bad = __builtin_amdgcn_ballot_w64(bad) != 0 || !(mx > -INFINITY) || mx == INFINITY;
    float l = 0.f, a0 = 0.f, a1 = 0.f;
    if (!bad) {
#pragma nounroll
      for (int j0 = 0; j0 < p.Sk; j0 += 64) {
        const int n = p.Sk - j0 < 64 ? p.Sk - j0 : 64;
        const float pj = lane < n ? __builtin_amdgcn_exp2f((score(j0 + lane) - mx) * LOG2E) : 0.f;
        l += pj;
#pragma nounroll
        for (int u = 0; u < n; ++u) {
          const float pu = __shfl(pj, u, 64);
          const uint32_t w =
              *reinterpret_cast<const uint32_t*>(Vb + (int64_t)(j0 + u) * p.ldv + (dok ? 2 * lane : 0));
          a0 = __builtin_fmaf(pu, Elem<T>::to_f32((uint16_t)(w & 0xffffu)), a0);
          a1 = __builtin_fmaf(pu, Elem<T>::to_f32((uint16_t)(w >> 16)), a1);
        }
      }
      l = wave_sum(l);
    }
    const float inv = 1.0f / l;  // bad: 0 * inf = NaN
    if (dok)
      *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(p.O) + b * p.sO + h * p.hO + (int64_t)r * p.ldo + 2 * lane) =
          pack2<T>(a0 * inv, a1 * inv);
  }
}

// Rows of a 16-row block that need other means than its sums: bit i for row
// q0 + i.  special: no key within reach (attn_special_rows); exact:
// attn_exact_rows.  l: the row's sum; low: this lane met a score of -inf;
// far: the row's reference was raised by more than FAR.
template <typename T, int MK>
__device__ __forceinline__ void attn_odd_rows(const AttnWideParams& wp, int64_t b, int64_t h, int q0, int lane,
                                              float l, bool low, bool far, uint64_t& special, uint64_t& exact) {
  const bool in = q0 + (lane & 15) < wp.a.Sq;
  uint64_t lows = __builtin_amdgcn_ballot_w64(low);
  lows |= lows >> 32;
  lows |= lows >> 16;
  const uint64_t zero = __builtin_amdgcn_ballot_w64(in && l == 0.f) & 0xffffull;
  special = zero & ~lows;
  exact = (zero & lows) | (__builtin_amdgcn_ballot_w64(in && far) & 0xffffull);
  // NaN sums from a finite mask value past the exponent domain
  uint64_t nans = __builtin_amdgcn_ballot_w64(in && l != l) & 0xffffull;
  bool have = false, big = false;
  while (nans != 0) {
    const int i = __builtin_ctzll(nans);
    if (!have || wp.mR != 0) {
      have = true;
      const int64_t mo = b * wp.mB + h * wp.mH + (int64_t)(q0 + i) * wp.mR;
      const void* mrow = MK == 1 ? (const void*)(static_cast<const float*>(wp.mask) + mo)
                                 : (const void*)(static_cast<const uint16_t*>(wp.mask) + mo);
      big = false;
      for (int j = lane; j < wp.a.Sk; j += 64) {
        const float x = mask_at<T, MK>(mrow, j);
        big |= x > 2.0e38f && x < INFINITY;
      }
      big = __builtin_amdgcn_ballot_w64(big) != 0;
    }
    if (big) exact |= 1ull << i;
    nans &= nans - 1;
  }
}

// Stores one 16-row block but the rows in `skip`.
template <typename T, int DB>
__device__ __forceinline__ void attn_wide_store(const AttnParams& p, int64_t b, int64_t h, int q0, int lane,
                                                const f32x4 (&o)[DB], float l, uint64_t skip) {
  const int r = q0 + (lane & 15);
  if (r < p.Sq && ((skip >> (lane & 15)) & 1) == 0) {
    uint16_t* orow = static_cast<uint16_t*>(p.O) + b * p.sO + h * p.hO + (int64_t)r * p.ldo;
    const float inv = 1.0f / l;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int d = db * 16 + 4 * (lane >> 4);
      if (d < p.D)
        *reinterpret_cast<u32x2*>(orow + d) =
            u32x2{pack2<T>(o[db][0] * inv, o[db][1] * inv), pack2<T>(o[db][2] * inv, o[db][3] * inv)};
    }
  }
}

// The kernel's parameters where the launch put them: what a function that is
// not inlined can take by reference without a copy in scratch.  (Each kernel
// here has the one parameter, at the segment's start.)
__device__ __forceinline__ const AttnWideParams& kernel_params() {
  return *(const AttnWideParams*)__builtin_amdgcn_kernarg_segment_ptr();
}

// MK: 0 no mask, 1 an fp32 mask, 2 a mask of type T.  PRE: Q scaled by scale
// log2 e in registers (attn64_kernel's PRESCALE).
template <typename T, int DW, int MK, bool PRE>
__global__ __launch_bounds__(256, 2) void attn_wide_kernel(AttnWideParams wp) {
  using C = AttnWideCfg<DW>;
  constexpr int MB = C::MB, HV = C::HALVES, NS = C::NS;
  constexpr int KC = DW / 32, DB = DW / 16;
  constexpr int KB = 64;
  constexpr int HB = KB * 128;  // one half of a key block
  constexpr int LPB = 4 * HV;   // direct loads per wave and key block
  constexpr float THRESH = 8.0f, DEEP = 256.0f, FAR = 65536.0f, UNSET = -3.0e38f, LOG2E = 1.4426950408889634f;
  const AttnParams& p = wp.a;
  __shared__ __attribute__((aligned(1024))) uint8_t sK[NS][HV * HB];
  __shared__ __attribute__((aligned(1024))) uint8_t sV[NS][HV * HB];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int Sq = p.Sq, Sk = p.Sk;
  const int NB = (Sk + KB - 1) / KB;
  const int k_tail = Sk - (NB - 1) * KB;
  const AttnItem wi = attn_item(p, p.item0 + attn_slot(p), NB);
  const int64_t b = wi.b, h = wi.h;
  const int q0 = wi.qb * C::ROWS + wave * (MB * 16);
  const int kb0 = wi.kb0, kb1 = wi.kb1;
  const uint16_t* Qb = static_cast<const uint16_t*>(p.Q) + b * p.sQ + h * p.hQ;
  const uint16_t* Kb = static_cast<const uint16_t*>(p.K) + b * p.sK + h * p.hK;
  const uint16_t* Vb = static_cast<const uint16_t*>(p.V) + b * p.sV + h * p.hV;
  const __amdgpu_buffer_rsrc_t rK =
      __builtin_amdgcn_make_buffer_rsrc((void*)Kb, (short)0, (int)((uint32_t)Sk * (uint32_t)p.ldk * 2u), 0x00020000);
  const __amdgpu_buffer_rsrc_t rV =
      __builtin_amdgcn_make_buffer_rsrc((void*)Vb, (short)0, (int)((uint32_t)Sk * (uint32_t)p.ldv * 2u), 0x00020000);
  // Loads as attn64_kernel's, per half: 16-byte chunk hch of rows drow and
  // drow + 8; chunks at or past D are sent out of range (zeros).  The last
  // key row of a head that is not the last in its row may read up to 2 * D
  // bytes short of its end, never past it: every chunk lies below D.
  const int drow = wave * 16 + (lane >> 3);
  const int hch = (lane & 7) ^ (lane >> 3);
  uint32_t vk0[HV], vv0[HV];
#pragma unroll
  for (int hf = 0; hf < HV; ++hf) {
    const int d = hf * 64 + hch * 8;
    vk0[hf] = d < p.D ? (uint32_t)drow * (uint32_t)p.ldk * 2u + (uint32_t)d * 2u : 0x80000000u;
    vv0[hf] = d < p.D ? (uint32_t)drow * (uint32_t)p.ldv * 2u + (uint32_t)d * 2u : 0x80000000u;
  }
  const uint32_t k8 = 8u * (uint32_t)p.ldk * 2u, v8 = 8u * (uint32_t)p.ldv * 2u;
  auto issue = [&](int j) {
    const int s = (j - kb0) % NS;
    const uint32_t ko = (uint32_t)j * (uint32_t)(KB * p.ldk * 2), vo = (uint32_t)j * (uint32_t)(KB * p.ldv * 2);
#pragma unroll
    for (int hf = 0; hf < HV; ++hf) {
      uint8_t* k = &sK[s][0] + hf * HB + wave * 2048;
      uint8_t* v = &sV[s][0] + hf * HB + wave * 2048;
      // plain uint32_t arguments: with a template-dependent one the host
      // pass drops the kernel's stub
      const uint32_t ok = vk0[hf] + ko, ov = vv0[hf] + vo;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rK, (lds_ptr_t)k, 16, ok, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rK, (lds_ptr_t)(k + 1024), 16, ok + k8, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rV, (lds_ptr_t)v, 16, ov, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rV, (lds_ptr_t)(v + 1024), 16, ov + v8, 0, 0, 0);
    }
  };
  issue(kb0);
  if (NS > 2 && kb0 + 1 < kb1) issue(kb0 + 1);

  u32x4 qf[MB][KC];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    int r = q0 + mb * 16 + (lane & 15);
    r = r < Sq ? r : Sq - 1;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      const int d0 = kc * 32 + 8 * (lane >> 4);
      qf[mb][kc] = d0 < p.D ? *reinterpret_cast<const u32x4*>(Qb + (int64_t)r * p.ldq + d0) : u32x4{0u, 0u, 0u, 0u};
      if constexpr (PRE) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t w = qf[mb][kc][e];
          qf[mb][kc][e] = pack2<T>(Elem<T>::to_f32((uint16_t)(w & 0xffffu)) * p.scale_log2e,
                                   Elem<T>::to_f32((uint16_t)(w >> 16)) * p.scale_log2e);
        }
      }
    }
  }

  // Mask rows of this lane's queries, at this lane's keys of a block.
  const void* mrow[MB];
  f32x4 mk[MK != 0 ? MB : 1][4];
  auto load_mask = [&](int j) {
    if constexpr (MK != 0) {
      const bool whole = j * KB + KB <= Sk;  // uniform
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
          const int key = j * KB + nb * 16 + 4 * (lane >> 4);
          if (whole) {
            mk[mb][nb] = mask4<T, MK>(mrow[mb], key);
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) mk[mb][nb][q] = key + q < Sk ? mask_at<T, MK>(mrow[mb], key + q) : -INFINITY;
          }
        }
    }
  };
  if constexpr (MK != 0) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      int r = q0 + mb * 16 + (lane & 15);
      r = r < Sq ? r : Sq - 1;
      const int64_t mo = b * wp.mB + h * wp.mH + (int64_t)r * wp.mR;
      mrow[mb] = MK == 1 ? (const void*)(static_cast<const float*>(wp.mask) + mo)
                         : (const void*)(static_cast<const uint16_t*>(wp.mask) + mo);
    }
    load_mask(kb0);
  }

  f32x4 o[MB][DB], osum[MB], nq[MB];
  float th[MB];  // a row is raised when one of its exponents exceeds this
  // bit mb: a row without a reference met a score of -inf here; bit 8 + mb:
  // a row was raised by more than FAR (see below)
  uint32_t odd = 0;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    osum[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    nq[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    th[mb] = UNSET;
#pragma unroll
    for (int db = 0; db < DB; ++db) o[mb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t one2 = (uint32_t)Elem<T>::from_f32(1.0f) * 0x10001u;
  const u32x4 ones = u32x4{one2, one2, one2, one2};

  const uint32_t kfo = (uint32_t)((lane & 15) * 128 + (((lane >> 4) ^ (lane & 7)) << 4));
  const int vs = lane & 15, vg = lane >> 4;
  const int vrow0 = 4 * vg + (vs >> 2);
  const uint32_t vfo_base = (uint32_t)vrow0 * 128u + (uint32_t)((vs & 1) * 8);
  const int vch = (vs & 3) >> 1;
  const int vsw = vrow0 & 7;

  for (int j = kb0; j < kb1; ++j) {
    const int st = (j - kb0) % NS;
    __builtin_amdgcn_sched_barrier(0);
    // NS == 2: this block's loads are the newest but the mask's; NS == 3:
    // one later block may be in flight (older than the mask's).
    if (MK == 0 && NS == 3 && j + 1 < kb1)
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(LPB, 0));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (j + NS - 1 < kb1) issue(j + NS - 1);
    __builtin_amdgcn_sched_barrier(0);

    // ---- S = Q K^T (+ mask), from -m or the mask as the C operand ---------
    const uint32_t ka = lds_addr(&sK[st][0]) + kfo;
    f32x4 s[MB][4];
    auto read_k = [&](auto nb_c, u32x4 (&f)[KC]) {
      constexpr int NBK = decltype(nb_c)::value;
      static_for<KC>([&](auto kc_c) {
        constexpr int KCI = decltype(kc_c)::value;
        f[KCI] = ds_read16<(KCI >> 1) * HB + NBK * 2048>((KCI & 1) ? (ka ^ 64u) : ka);
      });
    };
    // REF: the exponents, against the row references (with PRE the mask and
    // the reference are the score MFMAs' C operand: one FMA, whose rounding
    // is that of the reference, at most 2^8).  Otherwise scores + mask,
    // rounded as one fp32 sum, without a reference.
    auto scores = [&](auto ref_c) {
      constexpr bool REF = decltype(ref_c)::value;
      u32x4 kf[KC];
      read_k(std::integral_constant<int, 0>{}, kf);
      static_for<4>([&](auto nbc) {
        constexpr int NBK = decltype(nbc)::value;
        u32x4 nk[KC];
        if constexpr (NBK < 3) {
          read_k(std::integral_constant<int, (NBK < 3 ? NBK + 1 : 0)>{}, nk);
          __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, KC));
        } else {
          __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          f32x4 c = {0.f, 0.f, 0.f, 0.f};
          if constexpr (PRE && REF) {
            c = nq[mb];
            if constexpr (MK != 0) {
#pragma unroll
              for (int q = 0; q < 4; ++q) c[q] = __builtin_fmaf(mk[mb][NBK][q], LOG2E, nq[mb][q]);
            }
          }
          s[mb][NBK] = Mfma16<T>::run(kf[0], qf[mb][0], c);
        }
#pragma unroll
        for (int kc = 1; kc < KC; ++kc)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) s[mb][NBK] = Mfma16<T>::run(kf[kc], qf[mb][kc], s[mb][NBK]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (NBK < 3) {
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) kf[kc] = nk[kc];
        }
      });
      if constexpr (MK != 0 && !REF) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          float mn = s[mb][0][0];
#pragma unroll
          for (int e = 1; e < 16; ++e) mn = __builtin_elementwise_minimum(mn, s[mb][e >> 2][e & 3]);  // NaN: NaN row
          odd |= (PRE ? mn : mn * p.scale_log2e) == -INFINITY ? 1u << mb : 0u;
        }
      }
      if constexpr (!PRE || !REF) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < 4; ++nb)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma clang fp contract(off)
              float add = REF ? nq[mb][q] : 0.f;
              if constexpr (MK != 0) {
                if constexpr (REF) {
                  add = __builtin_fmaf(mk[mb][nb][q], LOG2E, add);
                } else {
                  add = mk[mb][nb][q] * LOG2E;
                }
              }
              s[mb][nb][q] = PRE ? s[mb][nb][q] + add : __builtin_fmaf(s[mb][nb][q], p.scale_log2e, add);
            }
      }
    };
    // With a mask, a row that has met no key yet or only keys far down or
    // up (a large finite mask) has no reference that exponents could be
    // formed against: the scores, rounded in its magnitude as their fp32 sum
    // with the mask is, would be compared with scores that are not.
    bool deep = false;
    if constexpr (MK != 0) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) deep |= th[mb] < 0.f || fabsf(nq[mb][0]) > DEEP;
      deep = __builtin_amdgcn_ballot_w64(deep) != 0;
    }
    if (deep)
      scores(std::false_type{});
    else
      scores(std::true_type{});

    // ---- V fragments of d 0-63 (they land under the softmax) ---------------
    const uint32_t va = lds_addr(&sV[st][0]) + vfo_base;
    u32x4 vf[4][2];
    auto read_v = [&](auto h_c, auto n_c) {
      constexpr int H = decltype(h_c)::value;
      static_for<decltype(n_c)::value>([&](auto dbc) {
        constexpr int D4 = decltype(dbc)::value;
        const uint32_t a0 = va + (uint32_t)(((2 * D4 + vch) ^ vsw) << 4);
        const u32x2 t00 = ds_read_tr16<H * HB + 0>(a0);
        const u32x2 t01 = ds_read_tr16<H * HB + 16 * 128>(a0);
        const u32x2 t10 = ds_read_tr16<H * HB + 32 * 128>(a0);
        const u32x2 t11 = ds_read_tr16<H * HB + 48 * 128>(a0);
        vf[D4][0] = u32x4{t00.x, t00.y, t01.x, t01.y};
        vf[D4][1] = u32x4{t10.x, t10.y, t11.x, t11.y};
      });
    };
    __builtin_amdgcn_sched_barrier(0);
    read_v(std::integral_constant<int, 0>{}, std::integral_constant<int, 4>{});
    __builtin_amdgcn_sched_barrier(0);

    // Keys past Sk (with a mask they carry -inf already).
    if (MK == 0 && k_tail < KB && j == NB - 1) {
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (nb * 16 + 4 * (lane >> 4) + q >= k_tail)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) s[mb][nb][q] = -INFINITY;
    }

    // ---- lazy row references -----------------------------------------------
    bool need = false;
    float lmx[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float mx = s[mb][0][0];
#pragma unroll
      for (int e = 1; e < 16; ++e) mx = __builtin_elementwise_maximum(mx, s[mb][e >> 2][e & 3]);
      lmx[mb] = mx;
      need |= mx > th[mb];
    }
    if (deep || __builtin_amdgcn_ballot_w64(need) != 0) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        float mx = fmaxf(lmx[mb], __shfl_xor(lmx[mb], 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        // A row without a reference takes its first finite maximum (O and
        // its sum are still zero); later ones only raise it.
        const bool unset = th[mb] < 0.f;
        const bool found = mx > UNSET;
        const float old = nq[mb][0];
        float nm, sub, corr;  // new -m, what the scores still lack, 2^(m - m')
        if (deep) {
          sub = found ? (unset ? mx : fmaxf(mx, -old)) : -old;
          nm = -sub;
          corr = unset ? 1.0f : __builtin_amdgcn_exp2f(-old - sub);
        } else {
          sub = unset ? (found ? mx : 0.f) : fmaxf(mx, 0.f);
          nm = old - sub;
          corr = unset ? 1.0f : __builtin_amdgcn_exp2f(-sub);
          // A step that far (a large positive mask after smaller ones): this
          // block's exponents were rounded against the old reference, the
          // next blocks' ("deep") will be against the new one, an ulp of
          // sub apart.
          if (MK != 0 && sub > FAR) odd |= 256u << mb;
        }
        nq[mb] = f32x4{nm, nm, nm, nm};
        if (found) th[mb] = THRESH;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
          for (int q = 0; q < 4; ++q) s[mb][nb][q] -= sub;
        osum[mb] *= corr;
#pragma unroll
        for (int db = 0; db < DB; ++db) o[mb][db] *= corr;
      }
    }

    // ---- P = 2^x in 16 bits, O += P V, row sums -----------------------------
    u32x4 pf[MB][2];
    auto expo = [&](int mb) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        uint32_t w[4];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int q2 = 0; q2 < 2; ++q2)
            w[hh * 2 + q2] = pack2<T>(__builtin_amdgcn_exp2f(s[mb][2 * c + hh][2 * q2]),
                                      __builtin_amdgcn_exp2f(s[mb][2 * c + hh][2 * q2 + 1]));
        pf[mb][c] = u32x4{w[0], w[1], w[2], w[3]};
      }
    };
    auto sums = [&](int mb) {
      osum[mb] = Mfma16<T>::run(ones, pf[mb][0], osum[mb]);
      osum[mb] = Mfma16<T>::run(ones, pf[mb][1], osum[mb]);
    };
    auto pv = [&](int mb, auto h_c, auto n_c) {
      constexpr int H = decltype(h_c)::value, N = decltype(n_c)::value;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int d4 = 0; d4 < N; ++d4)
          o[mb][H * 4 + d4] = Mfma16<T>::run(vf[d4][c], pf[mb][c], o[mb][H * 4 + d4]);
    };
    constexpr std::integral_constant<int, 0> h0{};
    constexpr std::integral_constant<int, 4> n0{};
    expo(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));  // V fragments landed
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    sums(0);
    pv(0, h0, n0);
    expo(1);
#pragma unroll
    for (int g = 0; g < 10; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // The next block's mask, into registers whose scores are spent.
    if constexpr (MK != 0)
      if (j + 1 < kb1) load_mask(j + 1);
    __builtin_amdgcn_sched_barrier(0);
    sums(1);
    pv(1, h0, n0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (HV > 1) {
      constexpr std::integral_constant<int, 1> h1{};
      constexpr std::integral_constant<int, DB - 4> n1{};
      read_v(h1, n1);
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
      __builtin_amdgcn_sched_barrier(0);
      pv(0, h1, n1);
      pv(1, h1, n1);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
  }

  if (wi.part >= 0) {
    float* w = p.ws + wi.part * C::PART;
    f32x4* po = reinterpret_cast<f32x4*>(w) + wave * (MB * DB * 64) + lane;
    float2* pml = reinterpret_cast<float2*>(w + C::PART_O) + wave * (MB * 64) + lane;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
      for (int db = 0; db < DB; ++db) po[(mb * DB + db) * 64] = o[mb][db];
      // A row that met no key in this part weighs nothing in the merge; its
      // sum, zero then, tells whether it met a score of -inf.  A sum's sign
      // tells of a far raise.
      const bool none = th[mb] < 0.f;
      float l = osum[mb][0];
      if (none && l == 0.f && ((odd >> mb) & 1) != 0) l = 1.f;
      if (((odd >> (8 + mb)) & 1) != 0) l = -l;
      pml[mb * 64] = float2{none ? -INFINITY : -nq[mb][0], l};
    }
    return;
  }
  // Waves without an odd row end here, ahead of the code for those.
  bool any = odd != 0;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) any |= !(osum[mb][0] > 0.f);
  if (MK == 0 || __builtin_expect(__builtin_amdgcn_ballot_w64(any) == 0, 1)) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) attn_wide_store<T, DB>(p, b, h, q0 + mb * 16, lane, o[mb], osum[mb][0], 0);
    return;
  }
  if constexpr (MK != 0) {
    uint64_t special = 0, exact = 0;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      uint64_t sp = 0, ex = 0;
      attn_odd_rows<T, MK>(wp, b, h, q0 + mb * 16, lane, osum[mb][0], ((odd >> mb) & 1) != 0,
                           ((odd >> (8 + mb)) & 1) != 0, sp, ex);
      attn_wide_store<T, DB>(p, b, h, q0 + mb * 16, lane, o[mb], osum[mb][0], sp | ex);
      special |= sp << (16 * mb);
      exact |= ex << (16 * mb);
    }
    if (special != 0) attn_special_rows<T, MK>(wp, b, h, q0, special);
    if (exact != 0) attn_exact_rows<T, MK>(kernel_params(), b, h, q0, exact);
  }
}

// Merges the parts of split items in part order: one wave per 16 query rows.
template <typename T, int DW, int MK>
__global__ __launch_bounds__(64) void attn_wide_combine_kernel(AttnWideParams wp) {
  using C = AttnWideCfg<DW>;
  constexpr int MB = C::MB, DB = DW / 16;
  const AttnParams& p = wp.a;
  const int lane = threadIdx.x;
  const int blk = blockIdx.x % (4 * MB);  // wave and row block of the item
  const int64_t s = p.item0 + blockIdx.x / (4 * MB);
  const AttnItem wi = attn_item(p, p.full_items + s * p.parts, 1);
  const int q0 = wi.qb * C::ROWS + blk * 16;
  if (q0 >= p.Sq) return;
  const float* base = p.ws + s * p.parts * (int64_t)C::PART;
  const int ml_off = C::PART_O + (blk * 64 + lane) * 2;
  const int o_off = (blk * DB * 64 + lane) * 4;
  float mmax = -INFINITY;
#pragma unroll 8
  for (int q = 0; q < p.parts; ++q) mmax = fmaxf(mmax, base[(int64_t)q * C::PART + ml_off]);
  float l = 0.f;
  bool low = false, far = false;
  f32x4 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int q = 0; q < p.parts; ++q) {
    const float* pq = base + (int64_t)q * C::PART;
    const float2 ml = *reinterpret_cast<const float2*>(pq + ml_off);
    // (0 times the sums of a part that met only NaN scores stays NaN)
    const float w = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - mmax);
    low |= ml.x == -INFINITY && ml.y == 1.f;
    far |= ml.y < 0.f;
    l += w * fabsf(ml.y);
    const f32x4* po = reinterpret_cast<const f32x4*>(pq + o_off);
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] += w * po[db * 64];
  }
  if (MK == 0 || __builtin_expect(__builtin_amdgcn_ballot_w64(low || far || !(l > 0.f)) == 0, 1)) {
    attn_wide_store<T, DB>(p, wi.b, wi.h, q0, lane, o, l, 0);
    return;
  }
  if constexpr (MK != 0) {
    uint64_t special = 0, exact = 0;
    attn_odd_rows<T, MK>(wp, wi.b, wi.h, q0, lane, l, low, far, special, exact);
    attn_wide_store<T, DB>(p, wi.b, wi.h, q0, lane, o, l, special | exact);
    if (special != 0) attn_special_rows<T, MK>(wp, wi.b, wi.h, q0, special);
    if (exact != 0) attn_exact_rows<T, MK>(kernel_params(), wi.b, wi.h, q0, exact);
  }
}

}  // namespace sf
