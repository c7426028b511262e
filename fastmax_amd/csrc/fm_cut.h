// Forward pass on dense score tiles for fp32 tensors of up to 64 channels, on the bf16 matrix instruction: what
// dense_fwd_kernel (fm_dense.h) computes, for calls whose outputs no backward pass reads.
//
// Every operand is cut into three bf16 parts, each the nearest bf16 value of what the parts before it leave: 3 x 8
// significand bits and the signs of the parts hold all 24 bits of the float.  Of the nine products of parts the six
// largest are formed (accumulated in fp32, smallest first).  What is left out, x1 y2 + x2 y1 + x2 y2, is at most about
// 2^-24 of a product (x = y = 1.00388: 0.99 x 2^-24; root mean square 2^-27.5), where rounding the product to fp32 costs
// up to 2^-24, too; a step of 16 products then rounds the accumulator six times instead of sixteen.  Error against 64
// bits, fp32 instruction -> here: 2.2e-7 -> 1.8e-7 (256 heads x 1000 x 32, causal), 3.4e-7 -> 2.9e-7 (48 x 3000 x 64).
//
// What bounds it: six v_mfma_f32_32x32x16_bf16 take ~200 cycles where eight v_mfma_f32_32x32x2f32 take 512; around them
// the cutting of the weights (~5.5 VALU instructions a value) and the operand reads, three planes each.  The parts of
// streamed rows are formed once per block on their way into LDS, those of own rows once per wave, only those of the
// weights per tile.  Unmasked, 512 heads x 1000 x 64: 1164 us a pass on the fp32 instruction, 800-840 here (by box).
//
// Not for passes that are differentiated.  The gradients of the first rows are differences of nearly equal numbers,
// g . v - c with c formed from this output, and the row that carries the row-norm maximum takes the rounding of a whole
// head's sum: there fp32 rounding is 3e-5 to 9e-5 of the gradient's rms already, and every other rounding of the output
// moves the gradients by as much again.
#pragma once
#include "fm_dense.h"

namespace cut {

struct Frag {
  fm_u4 p[3];
};
__device__ __forceinline__ f16v mma1(const fm_u4& a, const fm_u4& b, const f16v& c) {
  return FM_MFMA_BF16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c);
}
__device__ __forceinline__ f16v mma(const Frag& a, const Frag& b, f16v c) {
  c = mma1(a.p[2], b.p[0], c);
  c = mma1(a.p[0], b.p[2], c);
  c = mma1(a.p[1], b.p[1], c);
  c = mma1(a.p[1], b.p[0], c);
  c = mma1(a.p[0], b.p[1], c);
  return mma1(a.p[0], b.p[0], c);
}
// the three parts of a pair of floats, packed
__device__ __forceinline__ void parts(float x, float y, uint32_t (&w)[3]) {
  w[0] = pack_bf2(x, y);
  x -= bf_lo(w[0]);
  y -= bf_hi(w[0]);
  w[1] = pack_bf2(x, y);
  x -= bf_lo(w[1]);
  y -= bf_hi(w[1]);
  w[2] = pack_bf2(x, y);
}
__device__ __forceinline__ Frag make(const float (&x)[8]) {
  Frag f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t w[3];
    parts(x[2 * e], x[2 * e + 1], w);
#pragma unroll
    for (int k = 0; k < 3; ++k) f.p[k][e] = w[k];
  }
  return f;
}
// an LDS row (column) holds its three planes one after another, `plane` elements apart
__device__ __forceinline__ Frag load(const uint16_t* p, int plane) {
  Frag f;
#pragma unroll
  for (int k = 0; k < 3; ++k) f.p[k] = *reinterpret_cast<const fm_u4*>(p + k * plane);
  return f;
}

constexpr int BN = 32;   // streamed rows per stage
constexpr int KF = 16, EPL = 8, NFA = 32 / KF;
template <int DP>
struct Lds {
  static constexpr int PR = 3 * DP + 8, PT = 3 * BN + 8;   // pitches: odd numbers of 16-byte words
  static constexpr int RM = BN * PR, TR = DP * PT;
  static constexpr size_t bytes(int own_rows) { return (size_t)2 * (RM + TR) * sizeof(uint16_t) + (own_rows + 4) * sizeof(float); }
};

// BN rows x DP channels on their way global -> registers -> LDS by NT threads, as dense::TileRegs
template <int DP, int NT>
struct Stage {
  static constexpr int TOTAL = BN * DP / 4, NV = TOTAL / NT;
  static_assert(TOTAL % NT == 0 || TOTAL < NT, "whole passes over the tile, or at most one piece a thread");
  static constexpr int N = NV > 0 ? NV : 1;
  float4 raw[N];
  __device__ __forceinline__ void load(const HeadRows<const float>& hr, int pos0, int pend, int d, int tid) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int idx = tid + u * NT, row = idx % BN, ch = idx / BN * 4, pos = pos0 + row;
      const bool live = idx < TOTAL && pos < pend && ch < d;
      const float4 t = *reinterpret_cast<const float4*>(hr.base + ((unsigned)(pos < pend ? pos : pend - 1) * hr.pitch + (unsigned)(live ? ch : 0)));
      raw[u] = live ? t : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  __device__ __forceinline__ void store_rows(uint16_t* l, int tid) const {
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int idx = tid + u * NT;
      if (idx < TOTAL) {
        uint32_t a[3], b[3];
        parts(raw[u].x, raw[u].y, a);
        parts(raw[u].z, raw[u].w, b);
#pragma unroll
        for (int k = 0; k < 3; ++k)
          *reinterpret_cast<uint2*>(l + (idx % BN) * Lds<DP>::PR + k * DP + idx / BN * 4) = make_uint2(a[k], b[k]);
      }
    }
  }
  // transposed, row x at column tpos(x)
  __device__ __forceinline__ void store_columns(uint16_t* l, int tid) const {
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int idx = tid + u * NT;
      if (idx < TOTAL) {
        uint32_t a[3], b[3];
        parts(raw[u].x, raw[u].y, a);
        parts(raw[u].z, raw[u].w, b);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          uint16_t* c = l + (idx / BN * 4) * Lds<DP>::PT + k * BN + dense::Mma<bf16_t>::tpos(idx % BN);
          c[0] = (uint16_t)a[k];
          c[Lds<DP>::PT] = (uint16_t)(a[k] >> 16);
          c[2 * Lds<DP>::PT] = (uint16_t)b[k];
          c[3 * Lds<DP>::PT] = (uint16_t)(b[k] >> 16);
        }
      }
    }
  }
};

// ---------------------------------------------------------------------------------------
// grid = (heads, query blocks of 32 NW positions from the one that holds position Q.lo), the walk of dense_fwd_kernel
// (which explains the mask): each wave has 32 own rows, the keys are streamed in stages that the waves share.
// ---------------------------------------------------------------------------------------
template <int DP, int NW>
__global__ __launch_bounds__(64 * NW, DP == 32 ? 4 : 2) void cut_fwd_kernel(
    Rows<const float> Q, Rows<const float> K, Rows<const float> V, const float* __restrict__ qscale,
    const float* __restrict__ kscale, Rows<float> O, RowScalarsOut den, int npos, int nk, int d, int masked, float a0,
    float a1, float a2, int ratio) {
  using L = Lds<DP>;
  constexpr int NF = DP / KF, CB = DP / 32, NT = 64 * NW, BM = 32 * NW, HC = DP == 64 ? 1 : 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char cut_smem[];
  uint16_t* Kl = reinterpret_cast<uint16_t*>(cut_smem);   // [2][BN][PR]
  uint16_t* Vt = Kl + 2 * L::RM;                          // [2][DP][PT]
  float* denl = reinterpret_cast<float*>(Vt + 2 * L::TR);   // [BM]
  int* seen = reinterpret_cast<int*>(denl + BM);            // 1: one of the block's sums is zero, 2: one of its values is subnormal

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int nb = gridDim.y, bx = blockIdx.y;
  const int head = blockIdx.x, hkv = head / ratio;
  const int tok0 = (Q.lo / BM + (masked ? nb - 1 - bx : bx)) * BM, q00 = tok0 + w * 32;   // (q00: the wave's first own position)
  const HeadRows<const float> Qh = Q.head(head), Kh = K.head(hkv), Vh = V.head(hkv);
  const float kq = qscale[head] * kscale[hkv];
  const int own = q00 + i;
  const bool own_live = own >= Qh.lo && own < npos;
  const float* qrow = Qh.base + (unsigned)max(own < npos ? own : npos - 1, Qh.lo) * Qh.pitch;

  bool qodd = false;
  if (tid == 0) *seen = 0;
  Frag qf[NF];
#pragma unroll
  for (int m = 0; m < NF; ++m) {
    float x[EPL];
#pragma unroll
    for (int u = 0; u < EPL; u += 4) {
      const int ch = KF * m + EPL * hh + u;
      const bool ok = own_live && ch < d;
      const float4 t = *reinterpret_cast<const float4*>(qrow + (ok ? ch : 0));
      x[u] = ok ? t.x * kq : 0.f;
      x[u + 1] = ok ? t.y * kq : 0.f;
      x[u + 2] = ok ? t.z * kq : 0.f;
      x[u + 3] = ok ? t.w * kq : 0.f;
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e) qodd |= fabsf(x[e]) > 0x1p60f || (fabsf(x[e]) < 0x1p-100f && x[e] != 0.f);
    qf[m] = make(x);
  }

  qodd = __any(qodd);

  const int kend = masked ? (tok0 + BM < nk ? tok0 + BM : nk) : nk;
  const int nst = (kend + BN - 1) / BN;
  // The first 32 positions of a causal head stay on the fp32 instruction: with one key in sight the output is that key's
  // value to the last bit but one, whichever kernel ran.  (They see a single tile.)
  const bool first = masked && q00 == 0;
  Stage<DP, NT> kt, vt;
  auto stage_load = [&](int st) {
    kt.load(Kh, st * BN, nk, d, tid);
    vt.load(Vh, st * BN, nk, d, tid);
  };
  auto stage_store = [&](int buf) {
    kt.store_rows(Kl + buf * L::RM, tid);
    vt.store_columns(Vt + buf * L::TR, tid);
  };
  f16v acc[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) acc[cb] = dense::kZero16;
  float dn = 0.f;

  // weights of a score tile (rows = keys kb + trow(r, hh), lanes = own queries)
  auto weights = [&](f16v& sc, int kb) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float s = sc[r];
      sc[r] = a0 + s * (a1 + a2 * s);
    }
    if (masked && kb == q00) {   // (wave-uniform) a key may not lie after the query
      FM_KEEP_BRANCH();
      int lim = i - 4 * hh;
      asm volatile("" : "+v"(lim));   // (compared here: sixteen comparisons kept across the walk are 32 registers)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (trow(r, 0) > lim) sc[r] = 0.f;
    }
    if (!masked && kb + 32 > nk) {   // (wave-uniform) keys past the end
      FM_KEEP_BRANCH();
      int lim = nk - kb - 4 * hh;
      asm volatile("" : "+v"(lim));
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (trow(r, 0) >= lim) sc[r] = 0.f;
    }
  };
  auto tile = [&](int kb, const uint16_t* kl, const uint16_t* vl) __attribute__((always_inline)) {
    // (the value fragments are requested first: they arrive under the score tile's work)
    Frag vb[NFA][CB];
#pragma unroll
    for (int f = 0; f < NFA; ++f)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) vb[f][cb] = load(vl + (cb * 32 + i) * L::PT + KF * f + EPL * hh, BN);
    f16v sc = dense::kZero16;
#pragma unroll
    for (int m0 = 0; m0 < NF; m0 += HC) {   // (HC operand fragments are read ahead of the instructions that use them)
      Frag ka[HC];
#pragma unroll
      for (int m = 0; m < HC; ++m) ka[m] = load(kl + i * L::PR + KF * (m0 + m) + EPL * hh, DP);
#pragma unroll
      for (int m = 0; m < HC; ++m) sc = mma(ka[m], qf[m0 + m], sc);
    }
    weights(sc, kb);
    static_for<NFA>([&](auto ftag) {
      constexpr int F = 8 * decltype(ftag)::value;
      const float x[8] = {sc[F], sc[F + 1], sc[F + 2], sc[F + 3], sc[F + 4], sc[F + 5], sc[F + 6], sc[F + 7]};
      const Frag wa = make(x);
      dn += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[cb] = mma(wa, vb[F / 8][cb], acc[cb]);
    });
  };

  stage_load(0);
  stage_store(0);
  __syncthreads();
  for (int st = 0; st < nst; ++st) {
    const int buf = st & 1, kb = st * BN;
    if (st + 1 < nst) stage_load(st + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (!first && !(masked && kb > q00)) tile(kb, Kl + buf * L::RM, Vt + buf * L::TR);
    if (st + 1 < nst) stage_store(buf ^ 1);
    __syncthreads();
  }

  // Whether the parts held what the wave's rows are made of.  An infinite first part (of an infinity, or of a finite value
  // above bf16's largest) makes a result that is not finite.  Values below 2^-102 lose what lies below 2^-133: of the
  // values that shows in a weighted sum below 2^-100 of the sum of weights (or below 2^-80, where products of parts
  // begin to underflow; a sum of zero is what it should be unless a value was subnormal), of the weights where their sum is
  // below 2^-80, of the scores where a query is as small or beyond 2^60.
  const float sum = dn + __shfl_xor(dn, 32, 64);
  if (hh == 0) denl[w * 32 + i] = sum;   // (read back by the wave itself)
  bool odd = own_live && !(fabsf(sum) >= 0x1p-80f && fabsf(sum) < __builtin_inff()), none = false;
  float top = fabsf(sum);
#pragma unroll
  for (int off = 16; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off, 64));
  const float least = fmaxf(0x1p-80f, 0x1p-100f * top);
  // (bits without the sign, doubled: in one comparison of unsigned numbers everything that is not in [least, inf))
  const uint32_t floor2 = __float_as_uint(least) << 1;
  uint32_t far = 0;
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int r = 0; r < 16; ++r) far = max(far, (__float_as_uint(acc[cb][r]) << 1) - floor2);
  if (!first && __any(far >= 0xff000000u - floor2)) {   // (or a zero, an absent row or column: looked at one by one)
    FM_KEEP_BRANCH();
    int li = i, lh = hh;
    asm volatile("" : "+v"(li), "+v"(lh));
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int pos = q00 + trow(r, lh);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        const float mag = fabsf(acc[cb][r]);
        const bool out = pos >= Qh.lo && pos < npos && cb * 32 + li < d;
        odd |= out && !(mag < __builtin_inff() && (mag >= least || mag == 0.f));
        none |= out && mag == 0.f;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (none) atomicOr(seen, 1);
  __syncthreads();
  if (*seen) {   // (block-uniform: nothing below writes bit 0)
    FM_KEEP_BRANCH();
    bool subnormal = false;
    for (unsigned idx = tid; idx < (unsigned)kend * (DP / 4); idx += NT) {
      const int ch = idx % (DP / 4) * 4;
      const float4 t = *reinterpret_cast<const float4*>(Vh.base + (idx / (DP / 4) * Vh.pitch + (unsigned)(ch < d ? ch : 0)));
      constexpr int CLASS = 0x90;   // negative or positive subnormal
      subnormal |= __builtin_amdgcn_classf(t.x, CLASS) || __builtin_amdgcn_classf(t.y, CLASS) || __builtin_amdgcn_classf(t.z, CLASS) ||
                   __builtin_amdgcn_classf(t.w, CLASS);
    }
    if (subnormal) atomicOr(seen, 2);
    __syncthreads();
    odd |= none && (*seen & 2);
  }
  const bool again = first || qodd || __any(odd);
  if (again) {   // (wave-uniform)
    // The wave's rows on the fp32 instruction, operands straight from memory and in the order of dense_fwd_kernel (the same
    // bits).  No barrier in here: the other waves do not come along.
    FM_KEEP_BRANCH();
    int li = i, lh = hh;
    asm volatile("" : "+v"(li), "+v"(lh));   // (addresses are formed here, not kept across the walk)
    const int lown = q00 + li;
    const bool llive = lown >= Qh.lo && lown < npos;
    const float* lq = Qh.base + (unsigned)max(lown < npos ? lown : npos - 1, Qh.lo) * Qh.pitch;
    const int last = masked ? (q00 + 32 < nk ? q00 + 32 : nk) : nk;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[cb] = dense::kZero16;
    dn = 0.f;
#pragma unroll 1
    for (int kb = 0; kb < last; kb += 32) {
      const float* krow = Kh.base + (unsigned)(kb + li < nk ? kb + li : nk - 1) * Kh.pitch;
      f16v sc = dense::kZero16;
#pragma unroll 1
      for (int g = 0; g < DP / 8; ++g) {
        const int ch = 8 * g + 4 * lh;
        const bool on = ch < d, qon = on && llive, kon = on && kb + li < nk;
        const float4 k4 = *reinterpret_cast<const float4*>(krow + (on ? ch : 0)), q4 = *reinterpret_cast<const float4*>(lq + (on ? ch : 0));
        sc = FM_MFMA(kon ? k4.x : 0.f, qon ? q4.x * kq : 0.f, sc);
        sc = FM_MFMA(kon ? k4.y : 0.f, qon ? q4.y * kq : 0.f, sc);
        sc = FM_MFMA(kon ? k4.z : 0.f, qon ? q4.z * kq : 0.f, sc);
        sc = FM_MFMA(kon ? k4.w : 0.f, qon ? q4.w * kq : 0.f, sc);
      }
      weights(sc, kb);
      static_for<4>([&](auto ftag) {
        constexpr int F = 4 * decltype(ftag)::value;
        dn += (sc[F] + sc[F + 1]) + (sc[F + 2] + sc[F + 3]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = kb + trow(F + e, lh);
          const float* vrow = Vh.base + (unsigned)(key < nk ? key : nk - 1) * Vh.pitch;
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) {
            const int c = cb * 32 + li;
            const float v = vrow[c < d ? c : 0];
            acc[cb] = FM_MFMA(sc[F + e], key < nk && c < d ? v : 0.f, acc[cb]);
          }
          __builtin_amdgcn_sched_barrier(0);   // (register pressure)
        }
      });
    }
    const float sum32 = dn + __shfl_xor(dn, 32, 64);
    if (hh == 0) denl[w * 32 + i] = sum32;   // (read back by the wave itself)
  }

  const HeadRows<float> Oh = O.head(head);
  float* denh = den.head(head);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = w * 32 + trow(r, hh), pos = tok0 + row;
    if (pos < npos && pos >= Qh.lo) {
      const float dsum = denl[row], inv = 1.0f / dsum;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
        if (cb * 32 + i < d) Oh.base[(unsigned)pos * Oh.pitch + (unsigned)(cb * 32 + i)] = acc[cb][r] * inv;
      if (i == 0) denh[(int64_t)pos * den.stride] = dsum;
    }
  }
}

}  // namespace cut
