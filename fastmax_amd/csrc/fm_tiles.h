// Dense score tiles of bf16 tensors at p = 2: the sums of fm_dense.h bit for bit -- the same operands, rounded at the same
// places, added in the same order -- by kernels whose streamed operands reach LDS without passing through registers.
// (A kernel that rounds elsewhere can be as good and one multiply-add a score cheaper: f as a shifted square, with 1 / den on the
// weights.  But its weights lose what a0 holds where a0 is small against a1^2 / a2, and its results are others than those
// of a version before.)
//
// What bounds these kernels is the matrix instruction -- as long as nothing else gets in its way.  Measured on
// the chip, v_mfma_f32_32x32x16_bf16 occupies the matrix unit for 32 cycles and leaves the SIMD's other ports
// free: one wave that issues one matrix instruction and five VALU instructions in turn takes 36 cycles a group,
// and two waves in different phases of their work (eight matrix instructions, then 32 VALU ones) 42 cycles a
// matrix instruction, not 32 + 20.  (The fp32 instruction is different: it does keep the VALU from issuing.)
//
//   * K, V and Q tiles go global -> LDS directly, as stored, row-major only; the second contraction
//     reads them through the transposing LDS load.  The copies take no registers and no VALU work, and
//     a stage is under way while the stage before it is computed.  Rows are 16-byte chunks whose place in
//     the row is XORed with a function of the row number, so that row reads and transposing reads both touch every bank once.
//   * LDS reads run a few steps ahead of the matrix instructions that use them, in an order the compiler is not left to
//     choose (see steps).
//   * the forward kernel forms its second contraction transposed (channels x own rows), so that rows leave in 8-byte pieces; the
//     backward kernels do not: the order of a sum over their outputs is that of lanes = channels.
// What is left: the waits between a wave's phases (scores, polynomial, second contraction), which two to four waves a
// SIMD hide in part, and 4 to 9 VALU instructions a matrix instruction.  LDS delivers 256 bytes a cycle (an operand read takes a CU 4.1
// cycles) and is a quarter busy.  Without gain: one tile's polynomial placed between the next tile's matrix instructions
// (d = 64, 128 heads x 4096: dk / dv 710 us for 691, dq 444 for 431), one wave a SIMD with 512 registers in dk / dv at d = 128 (350
// for 319), blocks of four waves that take two 128-row parts in turn (dk / dv 720).
#pragma once
#include "fm_common.h"
#include "fm_dense.h"

namespace tiles {

using dense::kZero16;
using M = dense::Mma<bf16_t>;
using Frag = M::Frag;

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

// waits for this wave's transfers to LDS and its LDS reads, then for the block: behind it every wave sees what all have
// staged, and buffers read before it may be overwritten
__device__ __forceinline__ void stage_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// the lane number, made anew where it is called: what an epilogue derives from it is not prepared before the loops and kept through them
__device__ __forceinline__ int fresh_lane() {
  int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  asm volatile("" : "+v"(l));
  return l;
}

// what rows that do not exist are copied from
static __device__ const uint4 zero_chunk = {0u, 0u, 0u, 0u};

// One streamed tensor's share of a stage for this wave: chunk (u NW + wave) 64 + lane of the tile, u = 0..NI-1.
// Rows outside [lo, end) and channels past d are zeros.  (Copies of the nearest row or chunk would do for finite values, which the
// kernels' masks and zero operands leave out; but an infinity times zero is a NaN.)  Chunks past d are cleared once, and their lanes
// move nothing; a lane's place in LDS does not depend on the others'.
template <int DP, int NW, bool LEAN = false>
struct Copy {
  using G = Geo<DP>;
  static constexpr int ALL = G::BN * G::CPR / 64, NI = (ALL + NW - 1) / NW;
  static constexpr bool EVEN = ALL % NW == 0;   // (12 instructions of 96 channels on eight waves: four waves have a second one)
  static __device__ __forceinline__ bool has(int u, int w) { return EVEN || u * NW + w < ALL; }
  uint32_t off[NI];   // bytes from the tile's first row to this lane's chunk in instruction u
  static __device__ __forceinline__ int row(int u, int w, int l) { return ((u * NW + w) * 64 + l) / G::CPR; }
  static __device__ __forceinline__ int channel(int u, int w, int l) { return (((u * NW + w) * 64 + l) % G::CPR ^ G::key(row(u, w, l))) * 8; }
  static __device__ __forceinline__ uint32_t offset(int u, int w, int l, unsigned pitch) {
    return ((unsigned)row(u, w, l) * pitch + (unsigned)channel(u, w, l)) * 2u;
  }
  __device__ __forceinline__ void init(int w, int l, unsigned pitch) {
#pragma unroll
    for (int u = 0; u < NI; ++u) off[u] = offset(u, w, l, pitch);
  }
  static __device__ __forceinline__ void transfer(const void* base, uint32_t offset, uint32_t dst) {
    // (in asm: behind the builtin the compiler waits for the transfer at the next LDS read of any buffer.  The compiler does not
    // see a memory instruction in it, so the five wait states from a vector instruction that writes a scalar register, as reading
    // a spilled one back from a lane does, to a memory instruction that reads it are kept here.)
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(dst), "v"(offset), "s"(base) : "memory");
  }
  // this wave's chunks past d of the tile at `tile`
  static __device__ __forceinline__ void clear(unsigned char* tile, int d, int w) {
    const int l = fresh_lane();
#pragma unroll
    for (int u = 0; u < NI; ++u)
      if (has(u, w) && channel(u, w, l) >= d) *reinterpret_cast<uint4*>(tile + ((u * NW + w) * 64 + l) * 16) = make_uint4(0u, 0u, 0u, 0u);
  }
  static __device__ __forceinline__ void transfer_from(uint64_t address, uint32_t dst) {   // (an address of its own for every lane)
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(dst), "v"(address) : "memory");
  }
  // the stage's rows pos0 .. pos0 + BN - 1 to the tile at byte address lds
  __device__ __forceinline__ void issue(const HeadRows<const bf16_t>& hr, int pos0, int end, int d, uint32_t lds, int w, int l) const {
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds + (uint32_t)(w * 1024));
    uint64_t zeros = (uint64_t)reinterpret_cast<uintptr_t>(&zero_chunk);
    const bool inside = pos0 >= hr.lo && pos0 + G::BN <= end;   // (uniform)
    const bf16_t* base = hr.base + (int64_t)pos0 * hr.pitch;
    if (inside) {
#pragma unroll
      for (int u = 0; u < NI; ++u)
        if (has(u, w)) {
          const int k = LEAN ? fresh_lane() : l;   // (LEAN: no registers to keep what follows in)
          const uint32_t o = LEAN ? offset(u, w, k, hr.pitch) : off[u];
          if (d == DP || channel(u, w, k) < d) transfer(base, o, dst + u * NW * 1024);
        }
    } else {
      l = fresh_lane();   // (rare: nothing of it is kept in registers)
      asm volatile("" : "+s"(zeros));
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const int p = pos0 + row(u, w, l), c = channel(u, w, l);
        const uint64_t from = (uint64_t)reinterpret_cast<uintptr_t>(hr.base) + (uint64_t)(((unsigned)p * hr.pitch + (unsigned)c) * 2u);
        if (has(u, w)) transfer_from(p >= hr.lo && p < end && c < d ? from : zeros, dst + u * NW * 1024);
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

// Element c of row pos: uniform base, 32-bit lane offset in bytes (a head spans less than 4 GiB).
template <class T>
__device__ __forceinline__ T* element(const HeadRows<T>& hr, int pos, int c) {
  using Byte = typename std::conditional<std::is_const<T>::value, const char, char>::type;
  return reinterpret_cast<T*>(reinterpret_cast<Byte*>(hr.base) + ((unsigned)pos * hr.pitch + (unsigned)c) * 2u);
}

// 32 rows of a sum in accumulators (registers = rows r0 + trow, lanes = channels), times `scale`, to the rows inside
// [lo, end); `dot`: also this lane's part of their inner product with the rows of x, over rows and then channels as the
// fm_dense.h kernels take them.  All of x is requested at once and used before the first store: no load waits behind a store or on
// its own.  A block's epilogue is a tenth of a causal pass at 2048 tokens and bound by its instructions, so whole tiles go
// without tests (dk and dv of 256 rows x 64 channels with one stage of queries: 14.6 us a block with a test an element here and a
// select an element in own_row, 11.5 without; rows passed through LDS for 16-byte accesses: 12.4).
template <int DP>
__device__ __forceinline__ float store_rows(const f16v (&acc)[DP / 32], float scale, const HeadRows<bf16_t>& out, const HeadRows<const bf16_t>& x,
                                            bool dot, int r0, int lo, int end, int d) {
  constexpr int CB = DP / 32;
  const int lane = fresh_lane(), c0 = lane & 31, hh = lane >> 5;
  float rs = 0.f;
  auto run = [&](auto whole) __attribute__((always_inline)) {
    constexpr bool W = decltype(whole)::value;   // every row and channel exists
    auto in = [&](int r, int cb) { return W || (r0 + trow(r, hh) >= lo && r0 + trow(r, hh) < end && cb * 32 + c0 < d); };
    if (dot) {
      float xv[16][CB];
#pragma unroll
      for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {   // (clamped, not predicated)
          const int pos = r0 + trow(r, hh), c = cb * 32 + c0;
          xv[r][cb] = to_f32(*element(x, W ? pos : max(pos < end ? pos : end - 1, lo), W || c < d ? c : 0));
        }
#pragma unroll
      for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          const float t = __builtin_fmaf(acc[cb][r] * scale, xv[r][cb], rs);
          rs = in(r, cb) ? t : rs;
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
        if (in(r, cb)) *element(out, r0 + trow(r, hh), cb * 32 + c0) = bf16_t{M::to_elt(acc[cb][r] * scale)};
  };
  if (r0 >= lo && r0 + 32 <= end && d == DP) {   // (uniform)
    run(std::true_type{});
  } else {
    FM_KEEP_BRANCH();
    run(std::false_type{});
  }
  return rs;
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
    for (int e = 0; e < 8; ++e) x[e] *= scale;
    const Frag y = __builtin_bit_cast(Frag, M::pack(x));
    f[m] = live && ok ? y : M::zero();
  }
}

// N steps of a contraction whose operands come from LDS: step I reads the operands of step I + AHEAD (load) before it
// uses its own (use).  A read takes as long as four or more matrix instructions, and the compiler's own order -- read, wait, one
// matrix instruction -- leaves the matrix unit idle most of that time; the fences keep what a step holds in that step.  The
// first AHEAD reads are issued by `prime`, so that they can be placed under the work before the contraction.
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
// Forward.  grid = (heads, query blocks of 128 positions from the one that holds position Q.lo); npos: positions of
// the queries end here (nk under the mask: query i sits at position i + nk - nq).  Two stages of LDS.  (Eight waves, a third stage: no
// gain; two own tiles a wave, half the LDS reads: 72 us for 62 at 96 heads x 2048 x 64, 121 for 79 at 64 x 2049 x 128.)
// ---------------------------------------------------------------------------------------
template <int DP, int OCC>   // OCC: waves a SIMD
__global__ __launch_bounds__(256, OCC) void tiles_fwd_kernel(
    Rows<const bf16_t> Q, Rows<const bf16_t> K, Rows<const bf16_t> V, const float* __restrict__ qscale,
    const float* __restrict__ kscale, Rows<bf16_t> O, RowScalarsOut den, int npos, int nk, int d, int masked, float a0, float a1, float a2,
    int ratio, int o_words) {
  using G = Geo<DP>;
  constexpr int NW = 4, NF = DP / 16, CB = DP / 32, BM = 32 * NW, BN = G::BN, STAGE = 2 * G::TILE;
  using C = Copy<DP, NW>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char tiles_smem[];   // [2][K tile, V tile]

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
  ck.init(w, l, Kh.pitch);
  cv.init(w, l, Vh.pitch);
  auto issue = [&](int st, int buf) {
    ck.issue(Kh, st * BN, nk, d, lds0 + buf * STAGE, w, l);
    cv.issue(Vh, st * BN, nk, d, lds0 + buf * STAGE + G::TILE, w, l);
  };
  issue(0, 0);
  if (d < DP)
#pragma unroll
    for (int t = 0; t < 4; ++t) C::clear(tiles_smem + t * G::TILE, d, w);

  const float kq = qscale[head] * kscale[hkv];
  Frag qf[NF];
  const int q0 = tok0 + w * 32;   // first position of the wave's own tile
  own_row<DP>(Qh, q0 + i, npos, d, hh, kq, qf);
  Reads<DP> rd;
  rd.init(l);

  f16v acc[CB];
  float dn = 0.f;
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) acc[cb] = kZero16;

  constexpr int RA = 3, CA = 2;   // operand steps read ahead
  auto scores = [&](const unsigned char* kl, int t32, f16v& sc) __attribute__((always_inline)) {
    Frag ka[RA + 1];
    auto rows = [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value;
      ka[I % (RA + 1)] = rd.row(kl, t32, I);
    };
    prime<NF, RA>(rows);
    steps<NF, RA>(rows, [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value;
      sc = M::mma(ka[I % (RA + 1)], qf[I], I == 0 ? kZero16 : sc);
    });
  };
  auto weights = [&](f16v& sc) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float s = sc[r];
      sc[r] = a0 + s * (a1 + a2 * s);
    }
  };
  // a key tile on the own tile's diagonal, or with no more than `left` keys before the sequence's end: only these pay for
  // per-element tests
  auto edge = [&](f16v& sc, bool diagonal, int left) __attribute__((always_inline)) {
    const int lim = diagonal ? i : 31;
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (trow(r, hh) > lim || trow(r, hh) >= left) sc[r] = 0.f;
  };
  auto values = [&](const unsigned char* vl, int t32, const f16v& sc) __attribute__((always_inline)) {
    Frag vc[CA + 1], wa;
    auto cols = [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value;
      vc[I % (CA + 1)] = rd.col(vl, t32, I / CB, I % CB);
    };
    prime<2 * CB, CA>(cols);
    steps<2 * CB, CA>(cols, [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value, F = I / CB, cb = I % CB;
      if constexpr (cb == 0) {
        wa = M::template from_acc<F>(sc);
        dn = M::fsum(wa, dn);
      }
      acc[cb] = M::mma(vc[I % (CA + 1)], wa, acc[cb]);
    });
  };

  int buf = 0;
  // the stage is in LDS, the one after it on its way
  auto next_stage = [&](int st) __attribute__((always_inline)) -> const unsigned char* {
    stage_barrier();
    if (st + 1 < nst) issue(st + 1, buf ^ 1);
    const unsigned char* kl = tiles_smem + buf * STAGE;
    buf ^= 1;
    return kl;
  };
  // stages whose keys all exist and lie before every own query; then the rest (none of this diverges within a wave,
  // and every wave of the block passes nst barriers)
  const int n_in = (masked && q0 < nk ? q0 : nk) / BN < nst ? (masked && q0 < nk ? q0 : nk) / BN : nst;
  int st = 0;
  for (; st < n_in; ++st) {
    const unsigned char* kl = next_stage(st);
    const unsigned char* vl = kl + G::TILE;
    f16v s0, s1;
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
      if (kt >= nk || (masked && kt > q0)) continue;   // past the end, or after every own query
      f16v s;
      scores(kl + t32 * 32 * G::PITCH, 0, s);
      weights(s);
      edge(s, masked && kt == q0, nk - kt);
      values(vl + t32 * 32 * G::PITCH, 0, s);
    }
  }

  // lanes = own queries, registers 4 j .. 4 j + 3 of a column block = channels 8 j + 4 hh ..
  const HeadRows<bf16_t> Oh = O.head(head);
  float* denh = den.head(head);
  const float tot = dn + other_half(dn, hh);
  const int pos = q0 + i;
  if (pos < npos && pos >= Qh.lo) {
    const float inv = 1.0f / tot;
    bf16_t* row = Oh.base + (unsigned)pos * Oh.pitch + 4 * hh;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (cb * 32 + 8 * j < d) {
          const uint2 x = pack_bf4u(acc[cb][4 * j] * inv, acc[cb][4 * j + 1] * inv, acc[cb][4 * j + 2] * inv, acc[cb][4 * j + 3] * inv);
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
    if (hh == 0) denh[(int64_t)pos * den.stride] = tot;
  }
}

// ---------------------------------------------------------------------------------------
// dq.  The forward kernel's walk with two score tiles a step: the own rows carry q times 2 a2, so that the score
// accumulator, started at a1, is f'(s), and g = grad_out / den, whose accumulator starts at -c.  W = f'(s) (g . v - c) goes
// straight back as the operand of W . K.  c_i = grad_out_i . o_i / den_i is left in cprep for the dk / dv kernel.
// rpart[head * gridDim.y + block] receives the block's sum of dq . q for the normalisation chain rule (when rpart is
// given), a sum whose order is part of the result: that of the lanes and rows of dense_dq_kernel, blocks as wide as there.
// ---------------------------------------------------------------------------------------
template <int DP, int NW, int OCC>
__global__ __launch_bounds__(64 * NW, OCC) void tiles_dq_kernel(
    Rows<const bf16_t> Q, Rows<const bf16_t> GO, RowScalars den, Rows<const bf16_t> K, Rows<const bf16_t> V,
    Rows<const bf16_t> OUTF, const float* __restrict__ qscale, const float* __restrict__ kscale, Rows<bf16_t> DQ,
    float* __restrict__ rpart, RowScalarsOut cprep, int npos, int nk, int d, int masked, float a1, float a2, int ratio) {
  using G = Geo<DP>;
  using C = Copy<DP, NW, (OCC == 4)>;
  constexpr int NF = DP / 16, CB = DP / 32, BM = 32 * NW, BN = G::BN, STAGE = 2 * G::TILE;
  extern __shared__ __attribute__((aligned(1024))) unsigned char tiles_smem[];   // [2][K tile, V tile], [NW]
  float* red = reinterpret_cast<float*>(tiles_smem + 2 * STAGE);

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int nb = gridDim.y, bx = blockIdx.y;
  const int head = blockIdx.x, hkv = head / ratio;
  const int tok0 = (Q.lo / BM + (masked ? nb - 1 - bx : bx)) * BM;
  const HeadRows<const bf16_t> Qh = Q.head(head), Kh = K.head(hkv), Vh = V.head(hkv);
  const int kend = masked ? (tok0 + BM < nk ? tok0 + BM : nk) : nk;
  const int nst = (kend + BN - 1) / BN;
  const uint32_t lds0 = lds_address(tiles_smem);

  C ck, cv;
  ck.init(w, l, Kh.pitch);
  cv.init(w, l, Vh.pitch);
  auto issue = [&](int st, int buf) {
    ck.issue(Kh, st * BN, nk, d, lds0 + buf * STAGE, w, l);
    cv.issue(Vh, st * BN, nk, d, lds0 + buf * STAGE + G::TILE, w, l);
  };
  issue(0, 0);
  if (d < DP)
#pragma unroll
    for (int t = 0; t < 4; ++t) C::clear(tiles_smem + t * G::TILE, d, w);

  const float kq = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, qscale[head] * kscale[hkv])));   // (uniform, in a scalar register)
  const int q0 = tok0 + w * 32;
  Frag qf[NF], gf[NF];
  float c;
  {
    const HeadRows<const bf16_t> Gh = GO.head(head), OFh = OUTF.head(head);
    const int pos = q0 + i;
    const bool live = pos >= Qh.lo && pos < npos;
    const int ps = max(pos < npos ? pos : npos - 1, Qh.lo);
    const float rden = (live ? 1.0f : 0.f) / den.head(head)[(int64_t)ps * den.stride];
    own_row<DP>(Qh, pos, npos, d, hh, kq * 2.0f * a2, qf);
    const bf16_t* grow = Gh.base + (unsigned)ps * Gh.pitch;
    const bf16_t* orow = OFh.base + (unsigned)ps * OFh.pitch;
    float dot = 0.f;
#pragma unroll
    for (int m = 0; m < NF; ++m) {
      const int ch = 16 * m + 8 * hh;
      const bool ok = live && ch < d;
      const uint4 tg = *reinterpret_cast<const uint4*>(grow + (ok ? ch : 0));
      const uint4 to = *reinterpret_cast<const uint4*>(orow + (ok ? ch : 0));
      float x[8], y[8];
      M::unpack(ok ? tg : make_uint4(0u, 0u, 0u, 0u), x);
      M::unpack(ok ? to : make_uint4(0u, 0u, 0u, 0u), y);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        dot = __builtin_fmaf(x[e], y[e], dot);   // (a product of two bf16 numbers is exact)
        x[e] *= rden;
      }
      gf[m] = __builtin_bit_cast(Frag, M::pack(x));
    }
    c = (dot + other_half(dot, hh)) * rden;
    if (live && hh == 0) cprep.head(head)[(int64_t)pos * cprep.stride] = c;
  }
  Reads<DP> rd;
  rd.init(l);
  // no registers for tiles of the start values: they are moved into the accumulators each time
  constexpr bool TIGHT = DP > 96 || OCC == 4;
  f16v start, gstart;
  if constexpr (!TIGHT) {
    start = splat16(a1);
    gstart = splat16(-c);
  }

  f16v acc[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) acc[cb] = kZero16;

  constexpr int RA = OCC > 2 ? 0 : 2, CA = OCC > 2 ? 0 : 2;   // operand steps read ahead
  auto weights = [&](const unsigned char* kl, const unsigned char* vl, int t32, f16v& wt) __attribute__((always_inline)) {
    f16v sc;
    if constexpr (TIGHT) {
      float a = a1, b = -c;
      asm volatile("" : "+v"(a), "+v"(b));   // (or both tiles would be prepared before the loop and kept)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sc[r] = a;
        wt[r] = b;
      }
    }
    Frag ka[RA + 1], va[RA + 1];
    auto rows = [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value, X = I % (RA + 1);
      ka[X] = rd.row(kl, t32, I);
      va[X] = rd.row(vl, t32, I);
    };
    prime<NF, RA>(rows);
    steps<NF, RA>(rows, [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value, X = I % (RA + 1);
      sc = M::mma(ka[X], qf[I], I == 0 && !TIGHT ? start : sc);
      wt = M::mma(va[X], gf[I], I == 0 && !TIGHT ? gstart : wt);
    });
#pragma unroll
    for (int r = 0; r < 16; ++r) wt[r] = sc[r] * wt[r];
  };
  // (as in the forward kernel)
  auto edge = [&](f16v& wt, bool diagonal, int left) __attribute__((always_inline)) {
    const int lane = fresh_lane(), lim = diagonal ? lane & 31 : 31;
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (trow(r, lane >> 5) > lim || trow(r, lane >> 5) >= left) wt[r] = 0.f;
  };
  auto keys = [&](const unsigned char* kl, int t32, const f16v& wt) __attribute__((always_inline)) {
    Frag kc[CA + 1], wa;
    auto cols = [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value;
      kc[I % (CA + 1)] = rd.col(kl, t32, I / CB, I % CB);
    };
    prime<2 * CB, CA>(cols);
    steps<2 * CB, CA>(cols, [&](auto n) __attribute__((always_inline)) {
      constexpr int I = decltype(n)::value, F = I / CB, cb = I % CB;
      if constexpr (cb == 0) wa = M::template from_acc<F>(wt);
      acc[cb] = M::mma(wa, kc[I % (CA + 1)], acc[cb]);
    });
  };

  int buf = 0;
  auto next_stage = [&](int st) __attribute__((always_inline)) -> const unsigned char* {
    stage_barrier();
    if (st + 1 < nst) issue(st + 1, buf ^ 1);
    const unsigned char* kl = tiles_smem + buf * STAGE;
    buf ^= 1;
    return kl;
  };
  const int n_in = (masked && q0 < nk ? q0 : nk) / BN < nst ? (masked && q0 < nk ? q0 : nk) / BN : nst;
  int st = 0;
  for (; st < n_in; ++st) {
    const unsigned char* kl = next_stage(st);
    const unsigned char* vl = kl + G::TILE;
#pragma unroll
    for (int t32 = 0; t32 < 2; ++t32) {
      f16v wt;
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
      if (kt >= nk || (masked && kt > q0)) continue;
      const int off = t32 * 32 * G::PITCH;
      f16v wt;
      weights(kl + off, vl + off, 0, wt);
      edge(wt, masked && kt == q0, nk - kt);
      keys(kl + off, 0, wt);
    }
  }

  // dq = qs ks acc (the keys went in unscaled); sum of dqh . qh = qs ks sum acc . q
  float rs = store_rows<DP>(acc, kq, DQ.head(head), Qh, rpart != nullptr, q0, Qh.lo, npos, d);
  if (rpart) {
    const int t = w * 64 + fresh_lane();
    rs = dense::block_sum<NW>(rs, red, t);
    if (t == 0) rpart[(int64_t)head * nb + bx] = rs;
  }
}

// ---------------------------------------------------------------------------------------
// dk and dv.  grid = (key/value heads, key blocks of 32 KW positions); the streamed rows are the queries at or after the
// block's first key (all of them when unmasked) of every query head of the group in turn.  q rows go to LDS as they are;
// grad_out rows pass through registers and go there twice, times qs / den for the score side (so that W comes out times qs, the
// factor of qh in dkh = sum W qh) and times 1 / den for dv, the operands that dense_dkdv_kernel forms.
// Up to 64 channels a wave owns a key tile and both its sums.  Beyond, where one wave's accumulators and own rows take
// all the registers a lone wave of a SIMD has and nothing hides its VALU work, two waves share a key tile: the one sums dk, the other
// dv; of a stage's two query tiles each forms the weights of one, keeps those of its own sum and hands the others over through LDS.
// rpart[kvhead * gridDim.y + block] = sum of dkh . kh, added up in dense_dkdv_kernel's order over blocks as wide.
// ---------------------------------------------------------------------------------------
template <int DP>
struct DkDv {
  static constexpr bool PAIR = DP > 64;
  static constexpr int KW = DP == 64 ? 8 : 4, NW = PAIR ? 2 * KW : KW;   // key tiles and waves of a block
  static constexpr int BN = Geo<DP>::BN, TILE = Geo<DP>::TILE;
  // two buffers each of q, qs g, g; then -qs c of the streamed rows, the weights handed over, the block sum
  static constexpr int QG = 2 * TILE, GV = 4 * TILE, SCALARS = 6 * TILE, GIVE = SCALARS + 2 * BN * 4, RED = GIVE + (PAIR ? NW * 2048 : 0);
  static constexpr size_t BYTES = RED + NW * 4;
  static_assert(BYTES <= 160 * 1024, "a CU's LDS");
};

// One wave's share of a stage of grad_out rows on their way through registers (chunks as in Copy).
template <int DP, int NW>
struct Scaled {
  using G = Geo<DP>;
  using C = Copy<DP, NW>;
  uint4 raw[C::NI];
  float div[C::NI];
  static __device__ __forceinline__ int chunk(int u, int w, int l) {   // (a wave without a u-th share loads what its first one does)
    return (((C::has(u, w) ? u * NW + w : w) * 64 + l) % G::CPR ^ G::key(row(u, w, l))) * 8;
  }
  static __device__ __forceinline__ int row(int u, int w, int l) { return ((C::has(u, w) ? u * NW + w : w) * 64 + l) / G::CPR; }
  __device__ __forceinline__ void load(const HeadRows<const bf16_t>& hr, int pos0, int end, int d, const float* den, unsigned stride, int w, int l) {
#pragma unroll
    for (int u = 0; u < C::NI; ++u) {
      const int p = pos0 + row(u, w, l), c = chunk(u, w, l);
      const unsigned ps = (unsigned)max(p < end ? p : end - 1, hr.lo);
      raw[u] = *reinterpret_cast<const uint4*>(hr.base + (ps * hr.pitch + (unsigned)(c < d ? c : 0)));
      div[u] = den[ps * stride];
    }
  }
  // over den, times qs to the tile at qg, as it is to the tile at gv; zeros for rows outside [lo, end) and channels past d
  __device__ __forceinline__ void store(unsigned char* qg, unsigned char* gv, float qs, int pos0, int lo, int end, int d, int w, int l) const {
#pragma unroll
    for (int u = 0; u < C::NI; ++u) {
      if (!C::has(u, w)) continue;
      const int p = pos0 + row(u, w, l);
      // (as bits: a choice between the loaded registers and zero would become a branch)
      const uint32_t keep = p >= lo && p < end && chunk(u, w, l) < d ? ~0u : 0u;
      float x[8], y[8];
      M::unpack(make_uint4(raw[u].x & keep, raw[u].y & keep, raw[u].z & keep, raw[u].w & keep), x);
      const float inv = 1.0f / div[u], f = inv * qs;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        y[e] = x[e] * inv;
        x[e] *= f;
      }
      const int at = ((u * NW + w) * 64 + l) * 16;
      *reinterpret_cast<uint4*>(qg + at) = M::pack(x);
      *reinterpret_cast<uint4*>(gv + at) = M::pack(y);
    }
  }
};

// waits for this wave's LDS accesses, then for the block; what is under way to registers or LDS from memory stays so
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int DP>
__global__ __launch_bounds__(64 * DkDv<DP>::NW, 2) void tiles_dkdv_kernel(
    Rows<const bf16_t> K, Rows<const bf16_t> V, Rows<const bf16_t> Q, Rows<const bf16_t> GO, RowScalars den, RowScalars cvec,
    const float* __restrict__ qscale, const float* __restrict__ kscale, Rows<bf16_t> DK, Rows<bf16_t> DV,
    float* __restrict__ rpart, int npos, int nk, int d, int masked, float a0, float a1, float a2, int ratio) {
  using G = Geo<DP>;
  using LD = DkDv<DP>;
  constexpr bool PAIR = LD::PAIR;
  constexpr int KW = LD::KW, NW = LD::NW, NF = DP / 16, CB = DP / 32, BM = 32 * KW, BN = LD::BN, TILE = LD::TILE, NS = PAIR ? 1 : 2;
  static_assert(BN == 64, "a stage is two query tiles");
  using C = Copy<DP, NW>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char tiles_smem[];
  float* Cl = reinterpret_cast<float*>(tiles_smem + LD::SCALARS);
  float* red = reinterpret_cast<float*>(tiles_smem + LD::RED);

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int kw = w % KW, side = w / KW;   // side (of a pair): 0 sums dk, 1 sums dv
  const int nb = gridDim.y, bx = blockIdx.y;
  const int hkv = blockIdx.x;
  const int tok0 = bx * BM;   // (under the mask the first key blocks see the most queries: already first)
  const int k00 = tok0 + kw * 32;
  const HeadRows<const bf16_t> Kh = K.head(hkv), Vh = V.head(hkv);
  const float ks = kscale[hkv];
  const int lo = Q.lo;
  const int nst = (npos + BN - 1) / BN;
  const int st0 = masked ? (tok0 > lo ? tok0 : lo) / BN : 0;
  const uint32_t lds0 = lds_address(tiles_smem);

  // the loading side runs one stage ahead of the computing one, across heads
  HeadRows<const bf16_t> Qh = Q.head(hkv * ratio), Gh = GO.head(hkv * ratio);
  const float *denh = den.head(hkv * ratio), *ch = cvec.head(hkv * ratio);
  const int64_t qstep = Q.step(), gstep = GO.step();   // (the heads of a group are equally far apart)
  float lqs = qscale[hkv * ratio];
  C cq;
  cq.init(w, l, Qh.pitch);
  Scaled<DP, NW> sg;
  float creg = 0.f;
  auto stage_load = [&](int st, int buf) __attribute__((always_inline)) {
    sg.load(Gh, st * BN, npos, d, denh, (unsigned)den.stride, w, l);
    if (w == 0) {
      const int pos = st * BN + l;
      creg = ch[(unsigned)max(pos < npos ? pos : npos - 1, lo) * (unsigned)cvec.stride];
    }
    cq.issue(Qh, st * BN, npos, d, lds0 + buf * TILE, w, l);
  };
  auto stage_store = [&](int st, int buf) __attribute__((always_inline)) {
    sg.store(tiles_smem + LD::QG + buf * TILE, tiles_smem + LD::GV + buf * TILE, lqs, st * BN, lo, npos, d, w, l);
    if (w == 0) {
      const int pos = st * BN + l;
      Cl[buf * BN + l] = -creg * lqs * ((pos >= lo && pos < npos) ? 1.0f : 0.f);   // (-qs c: the tile's start value)
    }
  };

  Reads<DP> rd;   // (at the buffer being read)
  rd.init(l);
  rd.pin();
  Frag kf[NF], vf[NF];
  f16v acc[NS][CB];   // dk and dv, or the one this wave sums
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[s][cb] = kZero16;
  if (st0 < nst) stage_load(st0, 0);
  if (d < DP) {
    C::clear(tiles_smem, d, w);
    C::clear(tiles_smem + TILE, d, w);
  }
  own_row<DP>(Vh, k00 + i, nk, d, hh, 1.0f, vf);
  __builtin_amdgcn_sched_barrier(0);   // (one row after the other: registers)
  own_row<DP>(Kh, k00 + i, nk, d, hh, ks, kf);
  if (st0 < nst) stage_store(st0, 0);

  float c2, c1, b2;   // f and f' of s = qs sr, where sr = q . kh is what the score tile holds
  // The weights of query tile t: f(s) in sc, qs f'(s) (g . v - c) in pt; rows = queries, lanes = own keys.
  auto scores = [&](int t, const float* cl, f16v& sc, f16v& pt) __attribute__((always_inline)) {
    constexpr int RA = PAIR ? 1 : 2;   // operand steps read ahead
    const unsigned char *qt = tiles_smem, *gt = tiles_smem + LD::QG;
    Frag qa[RA + 1], ga[RA + 1];
    auto rows = [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value, X = I % (RA + 1);
      qa[X] = rd.row(qt + t * 32 * G::PITCH, 0, I);
      ga[X] = rd.row(gt + t * 32 * G::PITCH, 0, I);
    };
    prime<NF, RA>(rows);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 c4 = *reinterpret_cast<const float4*>(cl + 8 * j + 4 * hh);
      pt[4 * j] = c4.x; pt[4 * j + 1] = c4.y; pt[4 * j + 2] = c4.z; pt[4 * j + 3] = c4.w;
    }
    steps<NF, RA>(rows, [&](auto m) __attribute__((always_inline)) {
      constexpr int I = decltype(m)::value, X = I % (RA + 1);
      sc = M::mma(qa[X], kf[I], I == 0 ? kZero16 : sc);
      pt = M::mma(ga[X], vf[I], pt);
    });
  };
  // diag: the tile's queries before row `first` (the lane's own key when they are the same positions) do not see the key
  auto polynomial = [&](f16v& sc, f16v& pt, auto diag, int first) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float s = sc[r];
      sc[r] = a0 + s * (c1 + c2 * s);
      pt[r] = (a1 + b2 * s) * pt[r];
    }
    if constexpr (decltype(diag)::value) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (trow(r, hh) < first) sc[r] = pt[r] = 0.f;
    }
  };

  int buf = 0;
  for (int hq = 0; hq < ratio; ++hq) {
    const float qs = qscale[hkv * ratio + hq];
    c2 = a2 * qs * qs; c1 = a1 * qs; b2 = 2.0f * a2 * qs;
    // one stage, from buffer buf, while the next one (of this head or the next) is on its way to the other
    auto stage = [&](auto edge, int st) __attribute__((always_inline)) {
      stage_barrier();
      const bool more = st + 1 < nst || hq + 1 < ratio;
      const int next = st + 1 < nst ? st + 1 : st0;
      if (more) {
        if (st + 1 == nst) {
          Qh.base += qstep;
          Gh.base += gstep;
          denh += den.hs;
          ch += cvec.hs;
          lqs = qscale[hkv * ratio + hq + 1];
        }
        stage_load(next, buf ^ 1);
      }
      const float* cl = Cl + buf * BN;
      // (tiles past the end, or before every own key, count for nothing)
      auto live = [&](int t) { const int qb = st * BN + t * 32; return qb < npos && !(decltype(edge)::value && qb < k00); };
      auto first = [&](int t) { return st * BN + t * 32 == k00 ? i : 0; };
      constexpr int CA = 2;   // operand steps read ahead
      if constexpr (!PAIR) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if (!live(t)) continue;
          __builtin_amdgcn_sched_barrier(0);
          f16v sc, pt;
          scores(t, cl + t * 32, sc, pt);
          Frag gc[CA + 1], qc[CA + 1];
          auto cols = [&](auto n) __attribute__((always_inline)) {
            constexpr int I = decltype(n)::value, X = I % (CA + 1);
            gc[X] = rd.col(tiles_smem + LD::GV, t, I / CB, I % CB);
            qc[X] = rd.col(tiles_smem, t, I / CB, I % CB);
          };
          prime<2 * CB, CA>(cols);
          polynomial(sc, pt, edge, first(t));
          Frag fa, wa;
          steps<2 * CB, CA>(cols, [&](auto n) __attribute__((always_inline)) {
            constexpr int I = decltype(n)::value, X = I % (CA + 1), F = I / CB, cb = I % CB;
            if constexpr (cb == 0) {
              fa = M::template from_acc<F>(sc);
              wa = M::template from_acc<F>(pt);
            }
            acc[1][cb] = M::mma(fa, gc[X], acc[1][cb]);
            acc[0][cb] = M::mma(wa, qc[X], acc[0][cb]);
          });
        }
      } else {
        Frag* give = reinterpret_cast<Frag*>(tiles_smem + LD::GIVE);
        const unsigned char* mine = tiles_smem + (side ? LD::GV : 0);   // the streamed rows of this wave's sum
        Frag keep[2] = {M::zero(), M::zero()};
        __builtin_amdgcn_sched_barrier(0);
        if (live(side)) {
          f16v sc, pt;
          scores(side, cl + side * 32, sc, pt);
          polynomial(sc, pt, edge, first(side));
          const Frag f0 = M::template from_acc<0>(sc), f1 = M::template from_acc<1>(sc);
          const Frag w0 = M::template from_acc<0>(pt), w1 = M::template from_acc<1>(pt);
          keep[0] = side ? f0 : w0;
          keep[1] = side ? f1 : w1;
          give[w * 128 + l] = side ? w0 : f0;
          give[w * 128 + 64 + l] = side ? w1 : f1;
        }
        lds_barrier();
        const Frag* got = give + ((1 - side) * KW + kw) * 128 + l;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if (!live(t)) continue;
          Frag a[2], xc[CA + 1];
          a[0] = got[0];
          a[1] = got[64];
          auto cols = [&](auto n) __attribute__((always_inline)) {
            constexpr int I = decltype(n)::value;
            xc[I % (CA + 1)] = rd.col(mine, t, I / CB, I % CB);
          };
          prime<2 * CB, CA>(cols);
          if (t == side) {
            a[0] = keep[0];
            a[1] = keep[1];
          }
          steps<2 * CB, CA>(cols, [&](auto n) __attribute__((always_inline)) {
            constexpr int I = decltype(n)::value, F = I / CB, cb = I % CB;
            acc[0][cb] = M::mma(a[F], xc[I % (CA + 1)], acc[0][cb]);
          });
        }
      }
      if (more) stage_store(next, buf ^ 1);
      rd.shift(buf ? -TILE : TILE);
      buf ^= 1;
    };
    // stages with queries that lie before an own key or at the same position; then those wholly after (every wave passes
    // the same number of barriers)
    int st = st0;
    for (const int edge = masked ? (k00 / BN + 1 < nst ? k00 / BN + 1 : nst) : st0; st < edge; ++st) stage(std::true_type{}, st);
    for (; st < nst; ++st) stage(std::false_type{}, st);
  }

  // dk = ks dkh (dkh = the accumulated sum); sum of dkh . kh = ks sum acc . k
  float rs = 0.f;
  if (side == 0) rs = store_rows<DP>(acc[0], ks, DK.head(hkv), Kh, rpart != nullptr, k00, 0, nk, d);
  if (!PAIR || side == 1) store_rows<DP>(acc[NS - 1], 1.0f, DV.head(hkv), Kh, false, k00, 0, nk, d);
  if (rpart) {
    rs = dense::block_sum<NW>(rs, red, tid);
    if (tid == 0) rpart[(int64_t)hkv * nb + bx] = rs;
  }
}

}  // namespace tiles
