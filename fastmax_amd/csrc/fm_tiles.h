// Dense score tiles of bf16 tensors at p = 2: the same sums as fm_dense.h, on a form of the polynomial that costs
// one multiply-add an element, with operands that reach LDS without passing through registers.
//
// What bounds these kernels is the matrix instruction -- as long as nothing else gets in its way.  Measured on
// the chip, v_mfma_f32_32x32x16_bf16 occupies the matrix unit for 32 cycles and leaves the SIMD's other ports
// free: one wave that issues one matrix instruction and five VALU instructions in turn takes 36 cycles a group,
// and two waves in different phases of their work (eight matrix instructions, then 32 VALU ones) 42 cycles a
// matrix instruction, not 32 + 20.  (The fp32 instruction is different: it does keep the VALU from issuing.)
// So the two sides are balanced against each other and against LDS:
//
//   * f(s) = a0 + a1 s + a2 s^2 = A [(t s + h)^2 + c]: t rides on an own operand and h is the value the score
//     accumulator starts from, so u = t s + h is what the matrix instruction delivers, f / A = u^2 + c is ONE
//     multiply-add of it, f'(s) = 2 A t u is that accumulator itself, and the constants go to the epilogues.
//     Coefficients it does not suit (a2 zero or small against a1) stay with fm_dense.h: see square_form.
//   * K, V, Q and grad_out tiles go global -> LDS directly, as stored, row-major only; the second contraction
//     reads them through the transposing LDS load.  The copies take no registers and no VALU work, and
//     a stage is under way while the stage before it is computed.  Rows are 16-byte chunks whose place in
//     the row is XORed with a function of the row number, so that row reads and transposing reads both touch every bank once.
//   * the second contraction is formed transposed (channels x own rows), so that a lane ends up with its own row's
//     channels: scales and 1 / den are one factor a lane, and rows go out in 8-byte pieces.
//   * LDS reads run a few steps ahead of the matrix instructions that use them, in an order the compiler is not left to
//     choose (see steps).
// What is left: the waits between a wave's phases (scores, polynomial, second contraction), which two or three waves a
// SIMD hide in part.  LDS delivers 256 bytes a cycle (an operand read takes a CU 4.1 cycles), one operand per matrix
// instruction is half of that, and the dk / dv kernel needs up to 0.8; two own tiles a wave would halve it, but their
// registers leave one wave a SIMD, whose VALU work nothing then hides (dq at d = 64: 153 us against 88).  Counters at 128
// heads x 4096 x 64, forward: matrix unit busy 58 % at 1.8 GHz, to which the chip slows down under this load (2.1 GHz with
// it 28 % busy).
// us a launch, fm_dense.h -> these, GPU clock as it comes:            forward        dq            dk, dv
//   96 heads x 2048 x 64, causal                                      86 -> 61     132 -> 84     187 -> 132
//   64 heads on 16 of keys x 2049 x 128, causal                      139 -> 79     275 -> 121    554 -> 199
//   64 heads x 1000 queries behind 3000 keys x 64                    122 -> 77
#pragma once
#include "fm_common.h"
#include "fm_dense.h"

namespace tiles {

using dense::kZero16;
using M = dense::Mma<bf16_t>;
using Frag = M::Frag;

// The polynomial as a shifted square (see above).  f's sign and any positive factor m^2 may go into A.
struct Square {
  float t, h, c, A;
};
// Whether the form suits the coefficients, and the form.  Its terms are of size h^2 against max |a|: up to 256 times that,
// the fp32 rounding of the square (2^-24) stays below 2^-16 of the polynomial's coefficients, where the weights' bf16
// rounding is 2^-9.  (A NaN or an infinity among the coefficients fails the comparison.)
// m: with normalised rows the scores are small and the weights near a0, so m^2 = 9/8 |a0| puts them just below 1, where a
// bf16 step is smallest against the value (half of what it is just above); without normalisation m makes the scale
// kq t of the own operand a power of two, which rounds nothing.
inline bool square_form(float a0, float a1, float a2, bool normalize, float kq, Square& sq) {
  const float top = __builtin_fmaxf(__builtin_fabsf(a0), __builtin_fmaxf(__builtin_fabsf(a1), __builtin_fabsf(a2)));
  const float sg = a2 < 0.f ? -1.f : 1.f, t = __builtin_sqrtf(__builtin_fabsf(a2)), h = sg * a1 / (2.0f * t);
  if (!(t > 0.f && top <= 1e18f && h * h <= 256.0f * top)) return false;
  float m = 1.0f;
  if (normalize) {
    if (__builtin_fabsf(a0) >= 0x1p-20f * top) m = __builtin_sqrtf(1.125f * __builtin_fabsf(a0));
  } else {
    int e;
    const float x = __builtin_fabsf(kq) * t;
    if (x >= 0x1p-60f && x <= 0x1p60f) m = 2.0f * __builtin_frexpf(x, &e);
  }
  sq = Square{t / m, h / m, (sg * a0 - h * h) / (m * m), sg * m * m};
  return true;
}

template <int DP>
struct Geo {
  static constexpr int BN = 64;                  // streamed rows a stage
  static constexpr int CPR = DP / 8;             // 16-byte chunks of a row
  static constexpr int PITCH = DP * 2;           // bytes of a row
  static constexpr int TILE = BN * PITCH;        // bytes of a staged tile
  // Chunk c of row r is kept at chunk c ^ key(r) of its row.  LDS delivers 256 bytes at a time: a row read takes one
  // chunk of 16 rows (16 lanes x 16 bytes), a transposing read four chunks of four rows r0 .. r0 + 3 (32 lanes x 8
  // bytes).  key sends both to 16 different chunks of the 256 bytes.
  static __device__ __forceinline__ int key(int r) {
    if (CPR == 16) return ((r & 3) << 2) | ((r >> 2) & 3);
    if (CPR == 8) return (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
    return (r >> 2) & 3;
  }
  static constexpr int KEYS = CPR == 16 ? 16 : CPR == 8 ? 8 : 4;   // chunks a key can move a chunk among
};

// waits until at most N transfers to LDS of this wave are under way and its LDS reads are done, then for the
// block: behind it every wave sees what all have staged, and buffers read before it may be overwritten
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
}

// One streamed tensor's share of a stage for this wave: chunk (u NW + wave) 64 + lane of the tile, u = 0..NI-1.
// Rows outside [lo, end) are fetched from the nearest row inside and channels past d from the row's last chunk:
// valid addresses whose products the kernels' masks, zero operands and stores leave out.
template <int DP, int NW>
struct Copy {
  using G = Geo<DP>;
  static constexpr int NI = G::BN * G::CPR / 64 / NW;
  static_assert(NI * 64 * NW == G::BN * G::CPR, "every lane moves whole chunks");
  uint32_t off[NI];   // bytes from the tile's first row to this lane's chunk in instruction u
  static __device__ __forceinline__ int row(int u, int w, int l) { return ((u * NW + w) * 64 + l) / G::CPR; }
  static __device__ __forceinline__ int channel(int u, int w, int l, int d) {
    const int c = (((u * NW + w) * 64 + l) % G::CPR ^ G::key(row(u, w, l))) * 8;
    return c < d ? c : d - 8;
  }
  __device__ __forceinline__ void init(int w, int l, int d, unsigned pitch) {
#pragma unroll
    for (int u = 0; u < NI; ++u) off[u] = ((unsigned)row(u, w, l) * pitch + (unsigned)channel(u, w, l, d)) * 2u;
  }
  static __device__ __forceinline__ void transfer(const void* base, uint32_t offset, uint32_t dst) {
    // (in asm: behind the builtin the compiler waits for the transfer at the next LDS read of any buffer.  The compiler does not
    // see a memory instruction in it, so the five wait states from a vector instruction that writes a scalar register, as reading
    // a spilled one back from a lane does, to a memory instruction that reads it are kept here.)
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(dst), "v"(offset), "s"(base) : "memory");
  }
  // the stage's rows pos0 .. pos0 + BN - 1 to the tile at byte address lds
  __device__ __forceinline__ void issue(const HeadRows<const bf16_t>& hr, int pos0, int end, int d, uint32_t lds, int w, int l) const {
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds + (uint32_t)(w * 1024));
    if (pos0 >= hr.lo && pos0 + G::BN <= end) {   // (uniform) nothing to clamp: the lane's offsets stand
      const bf16_t* base = hr.base + (uint64_t)((unsigned)pos0 * hr.pitch);
#pragma unroll
      for (int u = 0; u < NI; ++u) transfer(base, off[u], dst + u * NW * 1024);
    } else {
      asm volatile("" : "+v"(l));   // (rare: nothing of it is kept in registers)
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const int p = pos0 + row(u, w, l);
        const int ps = max(p < end ? p : end - 1, hr.lo);
        transfer(hr.base, ((unsigned)ps * hr.pitch + (unsigned)channel(u, w, l, d)) * 2u, dst + u * NW * 1024);
      }
    }
  }
};

// A tile of equal values that stays in vector registers: as a uniform value the compiler would keep it in scalar ones
// and copy it to the accumulator before every contraction, where the matrix instruction can take it as it is.
__device__ __forceinline__ f16v splat16(float v) {
  f16v t;
#pragma unroll
  for (int r = 0; r < 16; ++r) t[r] = v;
  asm volatile("" : "+v"(t));
  return t;
}

// Byte offsets, within a tile, of what a lane reads of it: one per place a key can move a chunk to, so that row
// blocks, steps beyond eight chunks and buffers are constants on top.
template <int DP>
struct Reads {
  using G = Geo<DP>;
  static constexpr int NF = DP / 16, CB = DP / 32;
  static constexpr int NR = G::KEYS / 2;   // fragment steps (two chunks) within a key's range
  static constexpr int NT = G::KEYS / 4;   // column blocks (four chunks), likewise
  int rm[NR], tr[NT];
  __device__ __forceinline__ void init(int l) {
    const int i = l & 31, hh = l >> 5, L = l & 15, g = (l >> 4) & 1;
#pragma unroll
    for (int m = 0; m < NR; ++m) rm[m] = i * G::PITCH + (((2 * m + hh) ^ G::key(i)) << 4);
    const int r = 4 * hh + L / 4;
#pragma unroll
    for (int cb = 0; cb < NT; ++cb) tr[cb] = r * G::PITCH + (((cb * 4 + 2 * g + ((L & 3) >> 1)) ^ G::key(r)) << 4) + (L & 1) * 8;
  }
  // moves every address by `bytes` (to another buffer, in place: no second set of registers)
  __device__ __forceinline__ void shift(int bytes) {
#pragma unroll
    for (int m = 0; m < NR; ++m) rm[m] += bytes;
#pragma unroll
    for (int cb = 0; cb < NT; ++cb) tr[cb] += bytes;
  }
  // keeps them registers of their own (or the compiler adds a uniform part anew before every read)
  __device__ __forceinline__ void pin() {
#pragma unroll
    for (int m = 0; m < NR; ++m) asm volatile("" : "+v"(rm[m]));
#pragma unroll
    for (int cb = 0; cb < NT; ++cb) asm volatile("" : "+v"(tr[cb]));
  }
  // fragment m (channels 16 m + 8 hh ..) of row t32 * 32 + l % 32
  __device__ __forceinline__ int at(int m) const { return rm[m % NR] + (m / NR) * (NR * 32); }
  __device__ __forceinline__ Frag row(const unsigned char* tile, int t32, int m) const {
    return *reinterpret_cast<const Frag*>(tile + at(m) + t32 * 32 * G::PITCH);
  }
  // channel cb * 32 + l % 32 of the rows an accumulator fragment f of row block t32 stands for
  __device__ __forceinline__ Frag col(const unsigned char* tile, int t32, int f, int cb) const {
    const unsigned char* p = tile + (cb / NT) * (NT * 64) + (t32 * 32 + 16 * f) * G::PITCH;
    const uint2 a = lds_read_tr16(reinterpret_cast<const uint16_t*>(p + tr[cb % NT]));
    // (eight rows on, the key differs in the bit that moves a chunk by two)
    const uint2 b = lds_read_tr16(reinterpret_cast<const uint16_t*>(p + (tr[cb % NT] ^ 32) + 8 * G::PITCH));
    return Frag{a.x, a.y, b.x, b.y};
  }
};

__device__ __forceinline__ uint32_t lds_address(const unsigned char* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)p;
}

// The fragments of one own row (position pos of the head), times `scale`: fragment m holds channels 16 m + 8 hh .. + 7.  A
// row outside [lo, end) gives zeros, and so do channels past d.  Uniform base, 32-bit lane offset, and the offset is made
// anew on every call: hoisted out of a loop, one 64-bit address per fragment would stay in registers.
template <int DP>
__device__ __forceinline__ void own_row(const HeadRows<const bf16_t>& hr, int pos, int end, int d, int hh, float scale,
                                        Frag (&f)[DP / 16]) {
  const bool live = pos >= hr.lo && pos < end;
  uint32_t off = ((unsigned)max(pos < end ? pos : end - 1, hr.lo) * hr.pitch + (unsigned)(8 * hh)) * 2u;
  asm volatile("" : "+v"(off));
#pragma unroll
  for (int m = 0; m < DP / 16; ++m) {
    const bool ok = 16 * m + 8 * hh < d;   // (d is a multiple of 8: with hh = 1 and d = 8 the row's first chunk serves)
    const uint32_t o = ok ? off + 32u * m : off - 16u * hh;
    const uint4 t = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(hr.base) + o);
    float x[8];
    M::unpack(t, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = live && ok ? x[e] * scale : 0.f;
    f[m] = __builtin_bit_cast(Frag, M::pack(x));
  }
}

// N steps of a contraction whose operands come from LDS: step I reads the operands of step I + AHEAD (load) before it
// uses its own (use).  A read takes as long as four or more matrix instructions, and the compiler's own order -- read, wait, one
// matrix instruction -- leaves the matrix unit idle most of that time; the fence keeps LDS reads and matrix instructions
// in the order written here and lets everything else move across.  The first AHEAD reads are issued by `prime`, so that they can
// be placed under the work before the contraction.
__device__ __forceinline__ void order_fence() { __builtin_amdgcn_sched_barrier(0); }
template <int N, int AHEAD, class Load>
__device__ __forceinline__ void prime(Load&& load) {
  if constexpr (AHEAD > 0) {
    static_for<(AHEAD < N ? AHEAD : N)>([&](auto itag) __attribute__((always_inline)) { load(itag); });
    order_fence();
  }
}
template <int N, int AHEAD, class Load, class Use>
__device__ __forceinline__ void steps(Load&& load, Use&& use) {
  static_for<N>([&](auto itag) __attribute__((always_inline)) {
    constexpr int I = decltype(itag)::value;
    if constexpr (I + AHEAD < N) load(std::integral_constant<int, I + AHEAD>{});
    if constexpr (AHEAD > 0) order_fence();
    use(itag);
    if constexpr (AHEAD > 0) order_fence();
  });
}

// ---------------------------------------------------------------------------------------
// Forward.  grid = (heads, query blocks of 32 RT NW positions from the one that holds position Q.lo); npos: positions of
// the queries end here (nk under the mask: query i sits at position i + nk - nq).  NBUF stages of LDS.
// ---------------------------------------------------------------------------------------
// RT own tiles a wave; OCC waves a SIMD.
template <int DP, int RT, int NW, int NBUF, int OCC>
__global__ __launch_bounds__(64 * NW, OCC) void tiles_fwd_kernel(
    Rows<const bf16_t> Q, Rows<const bf16_t> K, Rows<const bf16_t> V, const float* __restrict__ qscale,
    const float* __restrict__ kscale, Rows<bf16_t> O, RowScalarsOut den, int npos, int nk, int d, int masked, Square sq, int ratio,
    int o_words) {
  using G = Geo<DP>;
  using C = Copy<DP, NW>;
  constexpr int NF = DP / 16, CB = DP / 32, BM = 32 * RT * NW, BN = G::BN, PD = NBUF - 1;
  constexpr int STAGE = 2 * G::TILE;
  extern __shared__ __attribute__((aligned(1024))) unsigned char tiles_smem[];   // [NBUF][K tile, V tile]

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int nb = gridDim.y, bx = blockIdx.y;
  const int head = blockIdx.x, hkv = head / ratio;
  // (under the mask the blocks with the most keys go first: the short ones fill the last round)
  const int tok0 = (Q.lo / BM + (masked ? nb - 1 - bx : bx)) * BM;
  const HeadRows<const bf16_t> Qh = Q.head(head), Kh = K.head(hkv), Vh = V.head(hkv);
  const int kend = masked ? (tok0 + BM < nk ? tok0 + BM : nk) : nk;
  const int nst = (kend + BN - 1) / BN;
  const uint32_t lds0 = lds_address(tiles_smem);

  C ck, cv;
  ck.init(w, l, d, Kh.pitch);
  cv.init(w, l, d, Vh.pitch);
  auto issue = [&](int st, int buf) {
    ck.issue(Kh, st * BN, nk, d, lds0 + buf * STAGE, w, l);
    cv.issue(Vh, st * BN, nk, d, lds0 + buf * STAGE + G::TILE, w, l);
  };
  issue(0, 0);
  if (PD > 1 && nst > 1) issue(1, 1);

  const float kq = qscale[head] * kscale[hkv] * sq.t;
  Frag qf[RT][NF];
  const int q00 = tok0 + w * RT * 32;   // first position of the wave's own tile 0
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) own_row<DP>(Qh, q00 + rt * 32 + i, npos, d, hh, kq, qf[rt]);
  Reads<DP> rd;
  rd.init(l);
  const f16v start = splat16(sq.h);

  f16v acc[RT][CB];
  float dn[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    dn[rt] = 0.f;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[rt][cb] = kZero16;
  }

  // One 32-key tile against the wave's own tiles.  EDGE: rel = key tile base - first position of own tile 0: own
  // tile rt has the key tile on its diagonal when rel == 32 rt and wholly after its queries when rel > 32 rt;
  // keys left of the sequence's end: `left`.  Only these tiles pay for per-element tests.
  constexpr int RA = 3, CA = 2;   // operand steps read ahead
  auto scores = [&](const unsigned char* kl, int t32, f16v (&sc)[RT]) __attribute__((always_inline)) {
    Frag ka[RA + 1];
    auto rows = [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value;
      ka[I % (RA + 1)] = rd.row(kl, t32, I);
    };
    prime<NF, RA>(rows);
    steps<NF, RA>(rows, [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) sc[rt] = M::mma(ka[I % (RA + 1)], qf[rt][I], I == 0 ? start : sc[rt]);
    });
  };
  auto weights = [&](f16v (&sc)[RT]) __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[rt][r] = sc[rt][r] * sc[rt][r] + sq.c;
  };
  auto edge = [&](f16v (&sc)[RT], int rel, int left) __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int lim = masked ? (rel > 32 * rt ? -1 : rel == 32 * rt ? i : 31) : 31;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (trow(r, hh) > lim || trow(r, hh) >= left) sc[rt][r] = 0.f;
    }
  };
  auto values = [&](const unsigned char* vl, int t32, const f16v (&sc)[RT]) __attribute__((always_inline)) {
    Frag vc[CA + 1], wa[RT];
    auto cols = [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value;
      vc[I % (CA + 1)] = rd.col(vl, t32, I / CB, I % CB);
    };
    prime<2 * CB, CA>(cols);
    steps<2 * CB, CA>(cols, [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value, F = I / CB, cb = I % CB;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        if constexpr (cb == 0) {
          wa[rt] = M::template from_acc<F>(sc[rt]);
          dn[rt] = M::fsum(wa[rt], dn[rt]);
        }
        acc[rt][cb] = M::mma(vc[I % (CA + 1)], wa[rt], acc[rt][cb]);
      }
    });
  };

  int buf = 0;
  // the stage is in LDS, the one PD further on its way
  auto next_stage = [&](int st) __attribute__((always_inline)) -> const unsigned char* {
    if (PD > 1 && st + 1 < nst) stage_barrier<2 * C::NI>();
    else stage_barrier<0>();
    if (st + PD < nst) issue(st + PD, buf == 0 ? NBUF - 1 : buf - 1);
    const unsigned char* kl = tiles_smem + buf * STAGE;
    buf = buf + 1 == NBUF ? 0 : buf + 1;
    return kl;
  };
  // stages whose keys all exist and lie before every own query; then the rest (none of this diverges within a wave,
  // and every wave of the block passes nst barriers)
  const int n_in = (masked && q00 < nk ? q00 : nk) / BN < nst ? (masked && q00 < nk ? q00 : nk) / BN : nst;
  int st = 0;
  for (; st < n_in; ++st) {
    const unsigned char* kl = next_stage(st);
    const unsigned char* vl = kl + G::TILE;
    f16v s0[RT], s1[RT];
    scores(kl, 0, s0);
    weights(s0);
    scores(kl, 1, s1);
    values(vl, 0, s0);
    weights(s1);
    values(vl, 1, s1);
  }
  for (; st < nst; ++st) {
    const unsigned char* kl = next_stage(st);
    const unsigned char* vl = kl + G::TILE;
#pragma unroll 1
    for (int t32 = 0; t32 < 2; ++t32) {
      const int kt = st * BN + t32 * 32;
      if (kt >= nk || (masked && kt > q00 + 32 * (RT - 1))) continue;   // past the end, or after every own query
      f16v s[RT];
      scores(kl + t32 * 32 * G::PITCH, 0, s);
      weights(s);
      edge(s, kt - q00, nk - kt);
      values(vl + t32 * 32 * G::PITCH, 0, s);
    }
  }

  // lanes = own queries, registers 4 j .. 4 j + 3 of a column block = channels 8 j + 4 hh ..
  const HeadRows<bf16_t> Oh = O.head(head);
  float* denh = den.head(head);
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const float tot = dn[rt] + other_half(dn[rt], hh);
    const int pos = q00 + rt * 32 + i;
    if (pos < npos && pos >= Qh.lo) {
      const float inv = 1.0f / tot;
      bf16_t* row = Oh.base + (unsigned)pos * Oh.pitch + 4 * hh;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (cb * 32 + 8 * j < d) {
            const uint2 x = pack_bf4u(acc[rt][cb][4 * j] * inv, acc[rt][cb][4 * j + 1] * inv, acc[rt][cb][4 * j + 2] * inv,
                                      acc[rt][cb][4 * j + 3] * inv);
            bf16_t* to = row + cb * 32 + 8 * j;
            if (o_words) {
              *reinterpret_cast<uint2*>(to) = x;
            } else {   // (rows of o that do not start on 8-byte boundaries, e.g. d + 1 elements apart)
              to[0].x = (uint16_t)x.x;
              to[1].x = (uint16_t)(x.x >> 16);
              to[2].x = (uint16_t)x.y;
              to[3].x = (uint16_t)(x.y >> 16);
            }
          }
      if (hh == 0) denh[(int64_t)pos * den.stride] = sq.A * tot;
    }
  }
}

// ---------------------------------------------------------------------------------------
// dq.  The forward kernel's walk with two score tiles a step: u as there, and P = grad_out . v - grad_out . o,
// whose start value is the own row's -grad_out . o.  W = u P goes straight back as the operand of W . K; what is
// constant in a row -- scales, 1 / den, f' = 2 A t u -- waits for the epilogue.  c_i = grad_out_i . o_i / den_i
// is left in cprep for the dk / dv kernel.  rpart[head * gridDim.y + block] receives the block's sum of dq . q for
// the normalisation chain rule (when rpart is given).
// ---------------------------------------------------------------------------------------
template <int DP, int RT, int NW, int NBUF, int OCC>
__global__ __launch_bounds__(64 * NW, OCC) void tiles_dq_kernel(
    Rows<const bf16_t> Q, Rows<const bf16_t> GO, RowScalars den, Rows<const bf16_t> K, Rows<const bf16_t> V,
    Rows<const bf16_t> OUTF, const float* __restrict__ qscale, const float* __restrict__ kscale, Rows<bf16_t> DQ,
    float* __restrict__ rpart, RowScalarsOut cprep, int npos, int nk, int d, int masked, Square sq, int ratio) {
  using G = Geo<DP>;
  using C = Copy<DP, NW>;
  constexpr int NF = DP / 16, CB = DP / 32, BM = 32 * RT * NW, BN = G::BN, PD = NBUF - 1;
  constexpr int STAGE = 2 * G::TILE;
  extern __shared__ __attribute__((aligned(1024))) unsigned char tiles_smem[];   // [NBUF][K tile, V tile], [NW]
  float* red = reinterpret_cast<float*>(tiles_smem + NBUF * STAGE);

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int nb = gridDim.y, bx = blockIdx.y;
  const int head = blockIdx.x, hkv = head / ratio;
  const int tok0 = (Q.lo / BM + (masked ? nb - 1 - bx : bx)) * BM;
  const HeadRows<const bf16_t> Qh = Q.head(head), Kh = K.head(hkv), Vh = V.head(hkv);
  const int kend = masked ? (tok0 + BM < nk ? tok0 + BM : nk) : nk;
  const int nst = (kend + BN - 1) / BN;
  const uint32_t lds0 = lds_address(tiles_smem);

  C ck, cv;
  ck.init(w, l, d, Kh.pitch);
  cv.init(w, l, d, Vh.pitch);
  auto issue = [&](int st, int buf) {
    ck.issue(Kh, st * BN, nk, d, lds0 + buf * STAGE, w, l);
    cv.issue(Vh, st * BN, nk, d, lds0 + buf * STAGE + G::TILE, w, l);
  };
  issue(0, 0);
  if (PD > 1 && nst > 1) issue(1, 1);

  const float kq = qscale[head] * kscale[hkv];
  const int q00 = tok0 + w * RT * 32;
  Frag qf[RT][NF], gf[RT][NF];
  float rden[RT], craw[RT];
  {
    const HeadRows<const bf16_t> Gh = GO.head(head), OFh = OUTF.head(head);
    const float* denh = den.head(head);
    float* cw = cprep.head(head);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int pos = q00 + rt * 32 + i;
      const bool live = pos >= Qh.lo && pos < npos;
      const int ps = max(pos < npos ? pos : npos - 1, Qh.lo);
      rden[rt] = 1.0f / denh[(int64_t)ps * den.stride];
      own_row<DP>(Qh, pos, npos, d, hh, kq * sq.t, qf[rt]);
      const bf16_t* grow = Gh.base + (unsigned)ps * Gh.pitch;
      const bf16_t* orow = OFh.base + (unsigned)ps * OFh.pitch;
      float dot = 0.f;
#pragma unroll
      for (int m = 0; m < NF; ++m) {
        const int ch = 16 * m + 8 * hh;
        const bool ok = live && ch < d;
        uint4 tg = *reinterpret_cast<const uint4*>(grow + (ok ? ch : 0));
        const uint4 to = *reinterpret_cast<const uint4*>(orow + (ok ? ch : 0));
        if (!ok) tg = make_uint4(0u, 0u, 0u, 0u);
        float x[8], y[8];
        M::unpack(tg, x);
        M::unpack(to, y);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot += ok ? x[e] * y[e] : 0.f;
        gf[rt][m] = __builtin_bit_cast(Frag, tg);
      }
      craw[rt] = dot + other_half(dot, hh);
      if (live && hh == 0) cw[(int64_t)pos * cprep.stride] = craw[rt] * rden[rt];
    }
  }
  Reads<DP> rd;
  rd.init(l);
  constexpr bool TIGHT = DP > 96;   // no registers for the start values: they are added afterwards
  const f16v start = splat16(sq.h);
  f16v gstart[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) gstart[rt] = splat16(-craw[rt]);

  f16v acc[RT][CB];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[rt][cb] = kZero16;

  constexpr int RA = OCC > 2 ? 0 : 2, CA = OCC > 2 ? 0 : 2;   // operand steps read ahead
  auto weights = [&](const unsigned char* kl, const unsigned char* vl, int t32, f16v (&wt)[RT]) __attribute__((always_inline)) {
    f16v sc[RT];
    Frag ka[RA + 1], va[RA + 1];
    auto rows = [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value, X = I % (RA + 1);
      ka[X] = rd.row(kl, t32, I);
      va[X] = rd.row(vl, t32, I);
    };
    prime<NF, RA>(rows);
    steps<NF, RA>(rows, [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value, X = I % (RA + 1);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        sc[rt] = M::mma(ka[X], qf[rt][I], I == 0 ? (TIGHT ? kZero16 : start) : sc[rt]);
        wt[rt] = M::mma(va[X], gf[rt][I], I == 0 ? (TIGHT ? kZero16 : gstart[rt]) : wt[rt]);
      }
    });
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int r = 0; r < 16; ++r) wt[rt][r] = TIGHT ? (sc[rt][r] + sq.h) * (wt[rt][r] - craw[rt]) : sc[rt][r] * wt[rt][r];
  };
  // (as in the forward kernel)
  auto edge = [&](f16v (&wt)[RT], int rel, int left) __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int lim = masked ? (rel > 32 * rt ? -1 : rel == 32 * rt ? i : 31) : 31;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (trow(r, hh) > lim || trow(r, hh) >= left) wt[rt][r] = 0.f;
    }
  };
  auto keys = [&](const unsigned char* kl, int t32, const f16v (&wt)[RT]) __attribute__((always_inline)) {
    Frag kc[CA + 1], wa[RT];
    auto cols = [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value;
      kc[I % (CA + 1)] = rd.col(kl, t32, I / CB, I % CB);
    };
    prime<2 * CB, CA>(cols);
    steps<2 * CB, CA>(cols, [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value, F = I / CB, cb = I % CB;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        if constexpr (cb == 0) wa[rt] = M::template from_acc<F>(wt[rt]);
        acc[rt][cb] = M::mma(kc[I % (CA + 1)], wa[rt], acc[rt][cb]);
      }
    });
  };

  int buf = 0;
  auto next_stage = [&](int st) __attribute__((always_inline)) -> const unsigned char* {
    if (PD > 1 && st + 1 < nst) stage_barrier<2 * C::NI>();
    else stage_barrier<0>();
    if (st + PD < nst) issue(st + PD, buf == 0 ? NBUF - 1 : buf - 1);
    const unsigned char* kl = tiles_smem + buf * STAGE;
    buf = buf + 1 == NBUF ? 0 : buf + 1;
    return kl;
  };
  const int n_in = (masked && q00 < nk ? q00 : nk) / BN < nst ? (masked && q00 < nk ? q00 : nk) / BN : nst;
  int st = 0;
  for (; st < n_in; ++st) {
    const unsigned char* kl = next_stage(st);
    const unsigned char* vl = kl + G::TILE;
#pragma unroll
    for (int t32 = 0; t32 < 2; ++t32) {
      f16v wt[RT];
      weights(kl, vl, t32, wt);
      keys(kl, t32, wt);
    }
  }
  for (; st < nst; ++st) {
    const unsigned char* kl = next_stage(st);
    const unsigned char* vl = kl + G::TILE;
#pragma unroll 1
    for (int t32 = 0; t32 < 2; ++t32) {
      const int kt = st * BN + t32 * 32;
      if (kt >= nk || (masked && kt > q00 + 32 * (RT - 1))) continue;
      const int off = t32 * 32 * G::PITCH;
      f16v wt[RT];
      weights(kl + off, vl + off, 0, wt);
      edge(wt, kt - q00, nk - kt);
      keys(kl + off, 0, wt);
    }
  }

  // lanes = own queries, registers 4 j .. 4 j + 3 of a column block = channels 8 j + 4 hh ..
  const HeadRows<bf16_t> Dh = DQ.head(head);
  float rs = 0.f;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int pos = q00 + rt * 32 + i;
    if (pos < npos && pos >= Qh.lo) {
      const float fac = 2.0f * sq.A * sq.t * kq * rden[rt];
      const bf16_t* qrow = Qh.base + (unsigned)pos * Qh.pitch + 4 * hh;
      bf16_t* row = Dh.base + (unsigned)pos * Dh.pitch + 4 * hh;
      float qv[CB][4][4];
      if (rpart) {   // (requested before the first store: no load waits behind one)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int j = 0; j < 4; ++j) load4(qrow + (cb * 32 + 8 * j < d ? cb * 32 + 8 * j : 0), qv[cb][j]);
      }
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (cb * 32 + 8 * j < d) {
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              x[e] = acc[rt][cb][4 * j + e] * fac;
              if (rpart) rs += x[e] * qv[cb][j][e];
            }
            *reinterpret_cast<uint2*>(row + cb * 32 + 8 * j) = pack_bf4u(x[0], x[1], x[2], x[3]);
          }
    }
  }
  if (rpart) {
    rs = dense::block_sum<NW>(rs, red, tid);
    if (tid == 0) rpart[(int64_t)head * nb + bx] = rs;
  }
}

// ---------------------------------------------------------------------------------------
// dk and dv.  grid = (key/value heads, key blocks of 32 KW positions); the streamed rows are the queries at or after the
// block's first key (all of them when unmasked) of every query head of the group in turn.  A block is KW x SW
// waves: wave (x, y) owns key tile x and takes the query tiles y, y + SW, .. of every stage, so that the longest walk
// -- the first keys of a long causal sequence, every query of every head -- is shared; at the end the SW parts are
// added through LDS.  Four share stages of 128 rows, which with the own rows of two key tiles are all of a CU's LDS.
// q and grad_out rows go to LDS as they are, 1 / den is a factor of the weights in fp32: one rounding less than grad_out / den
// in bf16 (dk and dv 2.4e-3 of 64 bits, before 2.9e-3), and a stage's 32 more multiplications a wave replace about 50
// instructions that divided and stored it (96 heads x 2048 x 64: 136 -> 132 us; 64 on 16 x 2049 x 128, SW = 2: 263 -> 232).
// (1 / den and c both read behind the first contraction, P = g.v / den - c: 141 us instead of 132.)  A head's query scale is a factor of everything its walk adds to dk, so the accumulator is kept over the
// scale of the head at hand.  rpart[kvhead * gridDim.y + block] = sum of dk . k.
// ---------------------------------------------------------------------------------------
template <int DP, int KW, int SW>
struct DkDvLds {   // two buffers of a q and a g tile, their rows' scalars, the own rows; the parts of SW waves lie over all of it
  static constexpr int ROWS = SW == 4 ? 128 : 64;   // streamed rows of a stage
  static constexpr int TILE = ROWS * Geo<DP>::PITCH, SCALARS = 4 * TILE, OWN = SCALARS + 4 * ROWS * 4;
  // (with 128 rows the first fragment of the own k rows has no place: it stays in registers)
  static constexpr int KREG = SW == 4 ? 1 : 0, PARTS = SW == 4 ? 4 * KW * DP * 32 * 4 : SW == 2 ? 2 * KW * DP * 32 * 4 : 0;
  static constexpr int END = OWN + (DP > 64 ? (2 * DP / 16 - KREG) * KW * 1024 : 0);
  static constexpr size_t BYTES = END > PARTS ? END : PARTS;
  static_assert(BYTES <= 160 * 1024, "a CU's LDS");
};
template <int DP, int KW, int SW, int OCC>
__global__ __launch_bounds__(64 * KW * SW, OCC) void tiles_dkdv_kernel(
    Rows<const bf16_t> K, Rows<const bf16_t> V, Rows<const bf16_t> Q, Rows<const bf16_t> GO, RowScalars den, RowScalars cvec,
    const float* __restrict__ qscale, const float* __restrict__ kscale, Rows<bf16_t> DK, Rows<bf16_t> DV,
    float* __restrict__ rpart, int npos, int nk, int d, int masked, Square sq, int ratio) {
  using G = Geo<DP>;
  using LD = DkDvLds<DP, KW, SW>;
  constexpr int NW = KW * SW, NF = DP / 16, CB = DP / 32, BM = 32 * KW, BN = LD::ROWS, TILE = LD::TILE, KREG = LD::KREG;
  static_assert(SW == 1 || SW == 2 || (SW == 4 && DP > 64), "a stage holds two or four query tiles");
  using C = Copy<DP, NW>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char tiles_smem[];   // [2][q tile, g tile], [2][-go.o, 1 / den][BN], own rows
  unsigned char* Ql = tiles_smem;
  unsigned char* Gl = tiles_smem + TILE;
  float* Cl = reinterpret_cast<float*>(tiles_smem + LD::SCALARS);

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int kw = w % KW, sw = w / KW;
  const int nb = gridDim.y, bx = blockIdx.y;
  const int hkv = blockIdx.x;
  const int tok0 = bx * BM;   // (under the mask the first key blocks see the most queries: already first)
  const int k00 = tok0 + kw * 32;
  const HeadRows<const bf16_t> Kh = K.head(hkv), Vh = V.head(hkv);
  const HeadRows<bf16_t> DKh = DK.head(hkv), DVh = DV.head(hkv);   // (here: the strides need not be kept)
  const float ks = kscale[hkv];
  const int lo = Q.lo;
  const int nst = (npos + BN - 1) / BN;
  const int st0 = masked ? (tok0 > lo ? tok0 : lo) / BN : 0;
  const uint32_t lds0 = lds_address(tiles_smem);

  // the loading side runs one stage ahead of the computing one, across heads
  HeadRows<const bf16_t> Qh, Gh;
  const float *denh, *ch;
  C cq, cg;
  float dreg = 1.0f, creg = 0.f, lon = qscale[hkv * ratio] == 0.f ? 0.f : 1.0f;
  Qh = Q.head(hkv * ratio);
  Gh = GO.head(hkv * ratio);
  denh = den.head(hkv * ratio);
  ch = cvec.head(hkv * ratio);
  const int64_t qstep = Q.step(), gstep = GO.step();   // (the heads of a group are equally far apart)
  auto stage_load = [&](int st, int buf) __attribute__((always_inline)) {
    if (w < BN / 64) {
      const int pos = st * BN + tid, ps = max(pos < npos ? pos : npos - 1, lo);
      dreg = denh[(unsigned)ps * (unsigned)den.stride];
      creg = ch[(unsigned)ps * (unsigned)cvec.stride];
    }
#pragma unroll
    for (int g = 0; g < BN / G::BN; ++g) {
      cq.issue(Qh, st * BN + g * G::BN, npos, d, lds0 + buf * 2 * TILE + g * G::TILE, w, l);
      cg.issue(Gh, st * BN + g * G::BN, npos, d, lds0 + (buf * 2 + 1) * TILE + g * G::TILE, w, l);
    }
  };
  // (rows outside the range count for nothing: both scalars zero)
  auto stage_store = [&](int st, int buf) __attribute__((always_inline)) {
    if (w < BN / 64) {
      const int pos = st * BN + tid;
      const bool in = pos >= lo && pos < npos;
      float* s = Cl + buf * 2 * BN + tid;
      s[0] = in && creg != 0.f ? -creg * dreg * lon : 0.f;   // (c = go.o / den, which is 0 where den has overflowed)
      s[BN] = in ? __builtin_amdgcn_rcpf(dreg) : 0.f;   // (one unit in the last place of 24 bits, on its way to 8)
    }
  };

  Reads<DP> rd;   // (at the buffer being read)
  rd.init(l);
  if (SW > 1) rd.shift(sw * 32 * G::PITCH);
  rd.pin();
  // own rows: in registers up to 64 channels; beyond, where the accumulators take half of them, in LDS
  constexpr bool VLDS = DP > 64;
  Frag* Vl = reinterpret_cast<Frag*>(tiles_smem + LD::OWN) + kw * NF * 64 + l;
  Frag* Kl = Vl + (KW * NF - kw * KREG - KREG) * 64;   // (at fragment 0, held or not)
  Frag kf[NF], vf[NF];
  auto own_to_lds = [&](const HeadRows<const bf16_t>& hr, float scale, Frag* dst, auto from) __attribute__((always_inline)) {
    uint32_t off = (unsigned)(k00 + i < nk ? k00 + i : nk - 1) * hr.pitch;
    asm volatile("" : "+v"(off));
#pragma unroll 2
    for (int m = decltype(from)::value; m < NF; ++m) {
      const int ch = 16 * m + 8 * hh;
      const uint4 t = *reinterpret_cast<const uint4*>(hr.base + (off + (unsigned)(ch < d ? ch : 0)));
      float x[8];
      M::unpack(t, x);
      const bool ok = k00 + i < nk && ch < d;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = ok ? x[e] * scale : 0.f;
      dst[m * 64] = __builtin_bit_cast(Frag, M::pack(x));
    }
  };
  auto own_first = [&]() __attribute__((always_inline)) {
    const bool ok = k00 + i < nk;
    const uint4 t = *reinterpret_cast<const uint4*>(Kh.base + ((unsigned)(ok ? k00 + i : nk - 1) * Kh.pitch + 8u * hh));
    return __builtin_bit_cast(Frag, ok ? t : make_uint4(0u, 0u, 0u, 0u));
  };
  f16v dk[CB], dv[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) dk[cb] = dv[cb] = kZero16;
  const f16v start = splat16(sq.h);
  float T = 0.f;   // this head's scale

  cq.init(w, l, d, Qh.pitch);
  cg.init(w, l, d, Gh.pitch);
  if constexpr (KREG) kf[0] = own_first();
  if (st0 < nst) {
    stage_load(st0, 0);
    stage_store(st0, 0);
  }
  // One 32-query tile against the wave's own keys.  diag: the tile's queries before row `first` (the lane's own key when
  // they are the same positions) lie before the key and do not see it.
  auto tile = [&](int t, const float* cl, auto diag, int first) __attribute__((always_inline)) {
    const unsigned char* qt = Ql + t * 32 * G::PITCH;
    const unsigned char* gt = Gl + t * 32 * G::PITCH;
    // rows = queries, lanes = own keys: u and den P = g . v - g . o
    f16v sc, pt;
    constexpr int RA = VLDS ? 1 : 2, CA = VLDS ? 1 : 2;   // operand steps read ahead
    Frag qa[RA + 1], ga[RA + 1], ka[RA + 1], va[RA + 1];
    auto rows = [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value, X = I % (RA + 1);
      qa[X] = rd.row(qt, 0, I);
      if constexpr (VLDS && I >= KREG) ka[X] = Kl[I * 64];
      ga[X] = rd.row(gt, 0, I);
      if constexpr (VLDS) va[X] = Vl[I * 64];
    };
    prime<NF, RA>(rows);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 c4 = *reinterpret_cast<const float4*>(cl + 8 * j + 4 * hh);
      pt[4 * j] = c4.x; pt[4 * j + 1] = c4.y; pt[4 * j + 2] = c4.z; pt[4 * j + 3] = c4.w;
    }
    steps<NF, RA>(rows, [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value, X = I % (RA + 1);
      sc = M::mma(qa[X], VLDS && I >= KREG ? ka[X] : kf[I], I == 0 ? (VLDS ? kZero16 : start) : sc);
      pt = M::mma(ga[X], VLDS ? va[X] : vf[I], pt);
    });
    Frag gc[CA + 1], qc[CA + 1];
    auto cols = [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value, X = I % (CA + 1);
      gc[X] = rd.col(gt, 0, I / CB, I % CB);
      qc[X] = rd.col(qt, 0, I / CB, I % CB);
    };
    prime<2 * CB, CA>(cols);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 r4 = *reinterpret_cast<const float4*>(cl + BN + 8 * j + 4 * hh);
      const float rden[4] = {r4.x, r4.y, r4.z, r4.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * j + e;
        const float u = VLDS ? sc[r] * T + sq.h : sc[r];   // (own k rows in LDS are not scaled: no registers for a start value either)
        sc[r] = (u * u + sq.c) * rden[e];
        pt[r] = u * (pt[r] * rden[e]);
      }
    }
    if constexpr (decltype(diag)::value) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (trow(r, hh) < first) sc[r] = pt[r] = 0.f;
    }
    Frag fa, wa;
    steps<2 * CB, CA>(cols, [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value, X = I % (CA + 1), F = I / CB, cb = I % CB;
      if constexpr (cb == 0) {
        fa = M::template from_acc<F>(sc);
        wa = M::template from_acc<F>(pt);
      }
      dv[cb] = M::mma(gc[X], fa, dv[cb]);
      dk[cb] = M::mma(qc[X], wa, dk[cb]);
    });
  };

  float qs_at = 1.0f, was_on = 1.0f;   // dk holds its sum over qs_at
  int buf = 0;
  for (int hq = 0; hq < ratio; ++hq) {
    const float qs = qscale[hkv * ratio + hq];
    // (a scale of zero: nothing of this head reaches dk, whose sum stays over the scale before)
    const float on = qs == 0.f ? 0.f : 1.0f;
    if constexpr (!VLDS) {
      if (hq == 0 || on != was_on) own_row<DP>(Vh, k00 + i, nk, d, hh, on, vf);
      __builtin_amdgcn_sched_barrier(0);   // (one row after the other: registers)
      own_row<DP>(Kh, k00 + i, nk, d, hh, ks * qs * sq.t, kf);
    } else {
      T = ks * qs * sq.t;
      if (hq == 0 || on != was_on) {
        if (hq > 0) __syncthreads();   // (the other waves of this key tile are through with the head before)
        if (sw == 0) {
          if (hq == 0) own_to_lds(Kh, 1.0f, Kl, std::integral_constant<int, KREG>{});
          own_to_lds(Vh, on, Vl, std::integral_constant<int, 0>{});
        }
      }
    }
    was_on = on;
    if (on != 0.f) {
      if (hq > 0) {
        const float fac = qs_at / qs;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int r = 0; r < 16; ++r) dk[cb][r] *= fac;
      }
      qs_at = qs;
    }
    // one stage, from buffer buf, while the next one (of this head or the next) is on its way to the other
    auto stage = [&](auto edge, int st) __attribute__((always_inline)) {
      stage_barrier<0>();
      const bool more = st + 1 < nst || hq + 1 < ratio;
      const int next = st + 1 < nst ? st + 1 : st0;
      if (more) {
        if (st + 1 == nst) {
          Qh.base += qstep;
          Gh.base += gstep;
          denh += den.hs;
          ch += cvec.hs;
          lon = qscale[hkv * ratio + hq + 1] == 0.f ? 0.f : 1.0f;
        }
        stage_load(next, buf ^ 1);
      }
#pragma unroll
      for (int t = 0; t < BN / 32 / SW; ++t) {
        const int t32 = SW > 1 ? sw : t, qb = st * BN + t32 * 32;
        if (qb >= npos || (decltype(edge)::value && qb < k00)) continue;   // past the end, or before every own key
        __builtin_amdgcn_sched_barrier(0);
        tile(t, Cl + buf * 2 * BN + t32 * 32, edge, qb == k00 ? i : 0);
      }
      if (more) stage_store(next, buf ^ 1);
      rd.shift(buf ? -2 * TILE : 2 * TILE);
      buf ^= 1;
    };
    // stages with queries that lie before an own key or at the same position; then those wholly after (every wave passes
    // the same number of barriers)
    int st = st0;
    for (const int edge = masked ? (k00 / BN + 1 < nst ? k00 / BN + 1 : nst) : st0; st < edge; ++st) stage(std::true_type{}, st);
    for (; st < nst; ++st) stage(std::false_type{}, st);
  }

  // the parts of the SW waves: the last two give theirs to the first two; of these the first finish dk, the second dv
  if constexpr (SW > 1) {
    float4* part = reinterpret_cast<float4*>(tiles_smem) + (size_t)kw * (CB * 4 * 64) + l;
    float4* part2 = part + (size_t)KW * (CB * 4 * 64);
    auto leave = [&](float4* p, const f16v (&a)[CB]) __attribute__((always_inline)) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int j = 0; j < 4; ++j) p[(cb * 4 + j) * 64] = make_float4(a[cb][4 * j], a[cb][4 * j + 1], a[cb][4 * j + 2], a[cb][4 * j + 3]);
    };
    auto take = [&](const float4* p, f16v (&a)[CB]) __attribute__((always_inline)) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float4 t = p[(cb * 4 + j) * 64];
          a[cb][4 * j] += t.x; a[cb][4 * j + 1] += t.y; a[cb][4 * j + 2] += t.z; a[cb][4 * j + 3] += t.w;
        }
    };
    __syncthreads();
    if constexpr (SW == 4) {
      constexpr size_t HALF = (size_t)2 * KW * (CB * 4 * 64);   // (sw = 0 and 2, sw = 1 and 3)
      if (sw >= 2) {
        leave(part + (sw - 2) * HALF, dk);
        leave(part2 + (sw - 2) * HALF, dv);
      }
      __syncthreads();
      if (sw < 2) {
        take(part + sw * HALF, dk);
        take(part2 + sw * HALF, dv);
      }
      __syncthreads();
    }
    if (sw == 1) leave(part, dk);
    else if (sw == 0) leave(part2, dv);
    __syncthreads();
    if (sw == 1) take(part2, dv);
    else if (sw == 0) take(part, dk);
  }
  // lanes = own keys, registers 4 j .. 4 j + 3 of a column block = channels 8 j + 4 hh ..
  int lane = tid;
  asm volatile("" : "+v"(lane));   // (nothing below is prepared before the loops and kept through them)
  const int pos = k00 + (lane & 31);
  float rs = 0.f;
  if (pos < nk && sw == 0) {
    const float fac = 2.0f * sq.A * sq.t * ks * qs_at;
    const bf16_t* krow = Kh.base + (unsigned)pos * Kh.pitch + 4 * hh;
    bf16_t* row = DKh.base + (unsigned)pos * DKh.pitch + 4 * hh;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      float kv[4][4];
      if (rpart) {   // (requested before the block's first store)
#pragma unroll
        for (int j = 0; j < 4; ++j) load4(krow + (cb * 32 + 8 * j < d ? cb * 32 + 8 * j : 0), kv[j]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (cb * 32 + 8 * j < d) {
          float x[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[e] = dk[cb][4 * j + e] * fac;
            if (rpart) rs += x[e] * kv[j][e];
          }
          *reinterpret_cast<uint2*>(row + cb * 32 + 8 * j) = pack_bf4u(x[0], x[1], x[2], x[3]);
        }
    }
  }
  if (pos < nk && sw == (SW > 1 ? 1 : 0)) {
    bf16_t* row = DVh.base + (unsigned)pos * DVh.pitch + 4 * hh;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (cb * 32 + 8 * j < d)
          *reinterpret_cast<uint2*>(row + cb * 32 + 8 * j) =
              pack_bf4u(dv[cb][4 * j] * sq.A, dv[cb][4 * j + 1] * sq.A, dv[cb][4 * j + 2] * sq.A, dv[cb][4 * j + 3] * sq.A);
  }
  if (rpart) {
    __syncthreads();   // (the parts were just read)
    rs = dense::block_sum<NW>(rs, Cl, tid);
    if (tid == 0) rpart[(int64_t)hkv * nb + bx] = rs;
  }
}

}  // namespace tiles
