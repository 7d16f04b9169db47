// kivi_quant.h -- the writer's device code: quantisation of a 32-token group
// by one wavefront, and one wavefront's share of a cache append.  Used by the
// writer kernel and by the fused write + decode step.
//
// Bit-exact with the reference (source_patch.py:1509-1640): fp32 min / max
// over the fp16 inputs, scale = (max - min) / 15 by IEEE division, scale <= 0
// -> 1, code = clamp(rint((x - min) / scale)), scale and min stored as fp16
// with round-to-nearest-even.
#pragma once

#include "kivi_kernels.h"

namespace jacq {

// 16-byte vector as a native vector type: arrays of it stay in registers
// (HIP's uint4 class does not).
typedef uint32_t w4 __attribute__((ext_vector_type(4)));
typedef short s16x2 __attribute__((ext_vector_type(2)));

// Stores of the append: plain, or (DEV) device-scope, for what wavefronts of
// the same launch on other XCDs read next.
template <bool DEV, typename T>
__device__ inline void st_out(T* p, T v) {
  if constexpr (DEV)
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else
    *p = v;
}
// Sixteen bytes.  A VALU write of the data registers of a store wider than 8
// bytes needs one wait state after it, which the compiler's hazard recognizer
// does not give an asm statement: the s_nop.
template <bool DEV>
__device__ inline void st_out16(void* p, w4 v) {
  if constexpr (DEV)
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
  else
    *(w4*)p = v;
}

// fp16 bits, two per dword, to and from integers of the same order (-0 below
// +0): packed signed 16-bit min / max then are min_num / max_num of values
// that are no NaN, ties of zeros included, two channels per instruction.
__device__ inline uint32_t order_key(uint32_t x) {
  const s16x2 s = __builtin_bit_cast(s16x2, x) >> (short)15;
  return x ^ (__builtin_bit_cast(uint32_t, s) & 0x7FFF7FFFu);
}
__device__ inline uint32_t pk_min(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(s16x2, a),
                                                                __builtin_bit_cast(s16x2, b)));
}
__device__ inline uint32_t pk_max(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(s16x2, a),
                                                                __builtin_bit_cast(s16x2, b)));
}
__device__ inline uint32_t swap_halves(uint32_t x) { return (x >> 16) | (x << 16); }
__device__ inline float half_of(uint32_t x, int k) { return h2f((uint16_t)(x >> (16 * k))); }

// The order keys of a NaN lie above +inf's or below -inf's, so a reduced
// minimum or maximum (of the low half, or of either) shows whether one was
// there.
__device__ inline bool nan_low(uint32_t mn, uint32_t mx) {
  return (int16_t)mx > 0x7C00 || (int16_t)mn < (int16_t)0x83FF;
}
__device__ inline bool nan_pair(uint32_t mn, uint32_t mx) {
  return nan_low(mn, mx) || nan_low(mn >> 16, mx >> 16);
}

// min / max of two dwords' fp16 pairs in fp32 with the reference's NaN rule:
// the general form of pk_min / pk_max on order keys, for tiles with a NaN.
// The result is again fp16 bits (min and max pick one of the inputs).
__device__ inline uint32_t num_min(uint32_t a, uint32_t b) {
  return (uint32_t)f2h(min_num(half_of(a, 0), half_of(b, 0))) |
         ((uint32_t)f2h(min_num(half_of(a, 1), half_of(b, 1))) << 16);
}
__device__ inline uint32_t num_max(uint32_t a, uint32_t b) {
  return (uint32_t)f2h(max_num(half_of(a, 0), half_of(b, 0))) |
         ((uint32_t)f2h(max_num(half_of(a, 1), half_of(b, 1))) << 16);
}

// Eight codes without a division (six instructions each): with inv =
// rcp(scale), q = (x - min) * inv is off the IEEE quotient by less than 4e-6
// (1 ulp of the reciprocal, half an ulp each of the difference's and the
// quotient's own rounding, at most 15 * 2^-22), so where q is further than
// 2^-16 from a rounding boundary it rounds to the quotient's integer.  q +
// 1.5 * 2^23 rounds it half to even into the low mantissa bits, so a code
// costs a subtraction (from the fp16 input), two fused multiply-adds, a
// subtraction, a maximum and a shift-add.  Returns the codes, and in `off` the largest
// |q - rint(q)| (NaN for infinities and NaNs).
__device__ inline float half_minus(uint32_t x, int k, float mn) {
  float d;
  if (k == 0)
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(x), "v"(mn));
  else
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=v"(d) : "v"(x), "v"(mn));
  return d;
}
constexpr float kRoundMagic = 12582912.0f;  // 1.5 * 2^23
constexpr uint32_t kMagicSum = 0x3F400000u;  // its bits shifted by 0, 4 .. 28, added
constexpr float kSure = 0.5f - 0x1p-16f;
__device__ inline uint32_t code_fast(uint32_t w, uint32_t x, int k, float mn, float inv, int shift,
                                     float* off) {
#pragma clang fp contract(off)
  const float d = half_minus(x, k, mn);
  const float t = __builtin_fmaf(d, inv, kRoundMagic);
  const float r = t - kRoundMagic;
  *off = __builtin_elementwise_maximum(*off, __builtin_fabsf(__builtin_fmaf(d, inv, -r)));
  return w + (__float_as_uint(t) << shift);
}

// Where a group's tokens are stored: per half of 16 rows the index of its first
// token row over all pages and heads, and whether its page may be written (an
// id outside the pool, or past the table, is not).
struct GroupRows {
  int64_t row[2];
  bool ok[2];
  __device__ GroupRows(const KiviGeo& g, int h, int p0, int p1) {
    const int P = g.page;
    row[0] = ((int64_t)p0 * g.nkv + h) * P;
    row[1] = P == kGroup ? row[0] + 16 : ((int64_t)p1 * g.nkv + h) * P;
    ok[0] = p0 >= 0 && p0 < g.num_pages;
    ok[1] = p1 >= 0 && p1 < g.num_pages;
  }
};

// The quantisation of one 32-token tile by one wavefront.  CH lanes hold one
// token row's channels, 8 each (16 bytes): lane = (row q = lane / CH, piece
// c = lane % CH), x[i] = row RQ i + q.  CH = 4 is a 32-channel slice of a
// head, CH = HD / 8 the whole row.  Results: codes[i], the 8 codes of x[i] (channel
// k in bits 4k), and the scales and zeros in fp16:
//   K (per channel over the 32 rows): sc / zr hold the lane's 8 channels;
//   V (per row over 32 channels = 4 lanes): sc / zr hold row i at half i.
template <int CH, bool IS_V>
struct QuantTile {
  static constexpr int RQ = 64 / CH, NI = kGroup / RQ;
  uint32_t codes[NI];
  w4 sc, zr;

  // scale of one min / max pair
  static __device__ float scale_of(float mn, float mx) {
#pragma clang fp contract(off)
    const float s = (mx - mn) / 15.0f;
    return s > 0.0f ? s : 1.0f;
  }

  // The lane's min and max keys or fp16 bits reduced over the lanes that share
  // a result.
  template <class Min, class Max>
  static __device__ __attribute__((always_inline)) void reduce(const w4 (&x)[NI], uint32_t (&mn)[IS_V ? NI : 4],
                                uint32_t (&mx)[IS_V ? NI : 4], Min fmn, Max fmx) {
    if constexpr (IS_V) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        uint32_t a = fmn(fmn(x[i][0], x[i][1]), fmn(x[i][2], x[i][3]));
        uint32_t b = fmx(fmx(x[i][0], x[i][1]), fmx(x[i][2], x[i][3]));
        a = fmn(a, swap_halves(a));
        b = fmx(b, swap_halves(b));
#pragma unroll
        for (int off = 1; off < 4; off <<= 1) {
          a = fmn(a, (uint32_t)__shfl_xor((int)a, off, 64));
          b = fmx(b, (uint32_t)__shfl_xor((int)b, off, 64));
        }
        mn[i] = a;
        mx[i] = b;
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint32_t a = x[0][k], b = x[0][k];
#pragma unroll
        for (int i = 1; i < NI; ++i) {
          a = fmn(a, x[i][k]);
          b = fmx(b, x[i][k]);
        }
#pragma unroll
        for (int off = CH; off < 64; off <<= 1) {
          a = fmn(a, (uint32_t)__shfl_xor((int)a, off, 64));
          b = fmx(b, (uint32_t)__shfl_xor((int)b, off, 64));
        }
        mn[k] = a;
        mx[k] = b;
      }
    }
  }

  __device__ __attribute__((always_inline)) void run(const w4 (&x)[NI]) {
#pragma clang fp contract(off)
    constexpr int M = IS_V ? NI : 4;  // dwords of min / max a lane holds
    uint32_t mn[M], mx[M];
    {
      w4 key[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) key[i][k] = order_key(x[i][k]);
      reduce(key, mn, mx, pk_min, pk_max);
    }
    bool nan = false;
#pragma unroll
    for (int k = 0; k < M; ++k) nan = nan || (IS_V ? nan_low : nan_pair)(mn[k], mx[k]);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(nan) != 0, 0)) {
      reduce(x, mn, mx, num_min, num_max);
      if constexpr (IS_V) {  // of several NaNs the reference keeps its first channel's
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int first = (int)(threadIdx.x & 60);
          mn[i] = (uint32_t)__shfl((int)mn[i], first, 64);
          mx[i] = (uint32_t)__shfl((int)mx[i], first, 64);
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < M; ++k) {
        mn[k] = order_key(mn[k]);  // its own inverse
        mx[k] = order_key(mx[k]);
      }
    }
    // scales: K of the lane's 8 channels, V of its NI rows
    constexpr int NS = IS_V ? NI : 8;
    float lo[NS], s[NS], inv[NS];
    sc = w4{0u, 0u, 0u, 0u};
    zr = w4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      lo[k] = IS_V ? half_of(mn[k], 0) : half_of(mn[k / 2], k & 1);
      const float hi = IS_V ? half_of(mx[k], 0) : half_of(mx[k / 2], k & 1);
      s[k] = scale_of(lo[k], hi);
      inv[k] = __builtin_amdgcn_rcpf(s[k]);
      sc[k / 2] |= (uint32_t)f2h(s[k]) << (16 * (k & 1));
      zr[k / 2] |= (uint32_t)f2h(lo[k]) << (16 * (k & 1));
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      float off = 0.0f;
      uint32_t w = 0u - kMagicSum;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int p = IS_V ? i : k;
        w = code_fast(w, x[i][k / 2], k & 1, lo[p], inv[p], 4 * k, &off);
      }
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(off < kSure)) != 0, 0)) {
        w = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int p = IS_V ? i : k;
          w |= (uint32_t)clamp_code((half_of(x[i][k / 2], k & 1) - lo[p]) / s[p]) << (4 * k);
        }
      }
      codes[i] = w;
    }
  }

  // Store the tile as channels [8 CH q0, 8 CH (q0 + 1)) of kv head h.
  template <int HD, bool DEV>
  __device__ __attribute__((always_inline)) void store(const KiviGeo& g, const AppendArgs& a, int h,
                                                       int q0, int p0, int p1, int lane) const {
    constexpr int HDP = HD / 2, HDG = HD / kGroup, HI = NI / 2;  // HI: rows of a half per lane
    const int c = lane % CH, q = lane / CH;
    const GroupRows to(g, h, p0, p1);
    uint8_t* const code = (IS_V ? a.v_code : a.k_code) + 4 * (CH * q0 + c) + q * HDP;
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (to.ok[i / HI])
        st_out<DEV>((uint32_t*)(code + (to.row[i / HI] + RQ * (i % HI)) * HDP), codes[i]);
    if constexpr (IS_V) {
      // the four lanes of a (row, 32 channels) hold the same scales: lane k
      // of them stores those of rows i = k, k + 4
#pragma unroll
      for (int ib = 0; ib < NI; ib += 4) {
        const int k = c & 3, i = ib + k;
        uint32_t s = 0, z = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (ib + e < NI && k == e) {
            s = (sc[(ib + e) / 2] >> (16 * (e & 1))) & 0xFFFFu;
            z = (zr[(ib + e) / 2] >> (16 * (e & 1))) & 0xFFFFu;
          }
        const bool second = i >= HI;
        const int64_t at = ((second ? to.row[1] + RQ * (i - HI) : to.row[0] + RQ * i) + q) * HDG +
                           (CH * q0 + c) / 4;
        if (i < NI && (second ? to.ok[1] : to.ok[0])) {
          st_out<DEV>(a.v_scale + at, (uint16_t)s);
          st_out<DEV>(a.v_zero + at, (uint16_t)z);
        }
      }
    } else if (q == 0) {
      // K scales live in every page of the group
#pragma unroll
      for (int pg = 0; pg < 2; ++pg) {
        const int p = pg == 0 ? p0 : p1;
        if (!to.ok[pg] || (pg == 1 && g.page == kGroup)) continue;
        const int64_t at = ((int64_t)p * g.nkv + h) * HD + 8 * (CH * q0 + c);
        st_out16<DEV>(a.k_scale + at, sc);
        st_out16<DEV>(a.k_zero + at, zr);
      }
    }
  }
};

// The new tokens of one sequence against its scratch (source_patch.py
// :1655-1697, :1737-1775): stream row p is scratch row p below r0 and new
// token p - r0 from there on; rows [0, D) age out as D / 32 groups.
struct AppendSpan {
  int old0, r0, r1, D;  // old tokens before; scratch rows before / after; rows that age out
  bool in_scratch;      // the reference's one-shift case: every new row fits the scratch
  __device__ AppendSpan(const KiviGeo& g, int start, int n) {
    old0 = split_old_tokens(start, g.residual);
    r0 = start - old0;
    const int old1 = split_old_tokens(start + n, g.residual);
    r1 = start + n - old1;
    D = old1 - old0;
    in_scratch = r0 + n <= g.rs;
  }
  __device__ int scratch_groups() const { return min(D, (r0 + kGroup - 1) / kGroup * kGroup) / kGroup; }
};

// Physical pages of aged group gi (read through the constant address space:
// wave-uniform scalar loads); -1 past the table.
__device__ inline void group_pages(const KiviGeo& g, const AppendArgs& a, int b, int group, int* p0,
                                   int* p1) {
  const int ppg = kGroup / g.page, fp = group * ppg;
  *p0 = *p1 = -1;
  if (fp + ppg <= g.max_pages) {
    const __attribute__((address_space(4))) int32_t* bt =
        (const __attribute__((address_space(4))) int32_t*)(a.block_tables + (int64_t)b * a.bt_stride);
    *p0 = bt[fp];
    *p1 = ppg == 2 ? bt[fp + 1] : *p0;
  }
}

// One wavefront's share of an append that ages groups out: channels [32 q, 32 q + 32) of K or V of
// (sequence b, kv head h) -- the aged groups that hold a scratch row, and the
// scratch itself.  K is quantised per channel and V per (row, 32 channels), so
// the slice needs no other bytes and slices need no order among themselves;
// all of a wavefront's scratch loads come before its scratch stores, so
// the append needs no barrier.  Aged groups of new tokens alone are not
// handled here.  What bounds it is latency (lengths, then rows and table,
// then stores): every row of a one-group age-out at R <= 128 is loaded in one
// round.
// landed() is called where everything the wavefront issued before this slice is
// complete.
template <int HD, bool IS_V, bool DEV, class Landed>
__device__ __attribute__((always_inline)) inline void append_slice(const KiviGeo& g,
                                                                   const AppendArgs& a, int b,
                                                                   int h, int q, int start, int n,
                                                                   int lane, Landed&& landed) {
  const AppendSpan sp(g, start, n);
  const int c = lane & 3, r = lane >> 2;
  uint16_t* xs = (IS_V ? a.v_scr : a.k_scr) + (int64_t)b * a.scr_stride + (int64_t)h * g.rs * HD +
                 kGroup * q + 8 * c;
  const uint16_t* nx = (IS_V ? a.new_v : a.new_k) + (int64_t)b * a.new_stride + (int64_t)h * HD +
                       kGroup * q + 8 * c;
  const int64_t tok_stride = (int64_t)g.nkv * HD;
  auto row = [&](int p) -> w4 {
    return *(const w4*)(p < sp.r0 ? xs + (int64_t)p * HD : nx + (int64_t)(p - sp.r0) * tok_stride);
  };
  constexpr int kPer = 10;  // rows of a shift pass: 16 per load, 160 = R + 32 at R = 128
  const int ng = sp.scratch_groups();
  QuantTile<4, IS_V> qt;
  w4 x[2], sh[kPer];
  int p0 = -1, p1 = -1;
  if (ng > 0) {
    group_pages(g, a, b, sp.old0 / kGroup, &p0, &p1);
    x[0] = row(r);
    x[1] = row(16 + r);
  }
  // every load unconditional (past the last row it re-reads that row): under a
  // branch the compiler waits for each before the next
#pragma unroll
  for (int k = 0; k < kPer; ++k) sh[k] = row(sp.D + min(r + 16 * k, sp.r1 - 1));
  for (int gi = 0; gi < ng; ++gi) {
    if (gi > 0) {
      group_pages(g, a, b, sp.old0 / kGroup + gi, &p0, &p1);
      x[0] = row(kGroup * gi + r);
      x[1] = row(kGroup * gi + 16 + r);
    }
    qt.run(x);
    qt.template store<HD, DEV>(g, a, h, q, p0, p1, lane);
  }
  // rows [0, r1) <- stream rows [D, D + r1).  A pass's loads land before its
  // stores, and a later pass reads rows above everything stored before it (D
  // >= 32 further up).
  for (int base = 0; base < sp.r1; base += 16 * kPer) {
    if (base > 0) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) sh[k] = row(sp.D + min(base + r + 16 * k, sp.r1 - 1));
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (base == 0) landed();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int d = base + r + 16 * k;
      if (d < sp.r1) st_out16<DEV>(xs + (int64_t)d * HD, sh[k]);
    }
  }
  // the reference's stale rows: appended, and above what the shift rewrote
  if (sp.in_scratch)
    for (int p = max(sp.r0, sp.r1) + r; p < sp.r0 + n; p += 16)
      st_out16<DEV>(xs + (int64_t)p * HD, *(const w4*)(nx + (int64_t)(p - sp.r0) * tok_stride));
}

// An append that ages no group out, by the HD / 32 wavefronts of a (sequence, kv head,
// K | V): the new rows into the scratch, whole rows side by side (a 32-channel slice per
// wavefront took 58 us, not 49, for 128 tokens to each of 256 sequences, 8 kv heads, HD 128).
template <int HD>
__device__ inline void append_rows(const KiviGeo& g, const AppendArgs& a, int b, int h, bool is_v,
                                   int wave, int r0, int n, int lane) {
  constexpr int CH = HD / 8, RQ = 64 / CH;  // lanes of a row; rows of a wavefront's load
  const int c = 8 * (lane % CH);
  uint16_t* xs = (is_v ? a.v_scr : a.k_scr) + (int64_t)b * a.scr_stride + (int64_t)h * g.rs * HD + c;
  const uint16_t* nx = (is_v ? a.new_v : a.new_k) + (int64_t)b * a.new_stride + (int64_t)h * HD + c;
  for (int t = RQ * wave + lane / CH; t < n; t += RQ * (HD / kGroup))
    *(w4*)(xs + (int64_t)(r0 + t) * HD) = *(const w4*)(nx + (int64_t)t * g.nkv * HD);
}

}  // namespace jacq
