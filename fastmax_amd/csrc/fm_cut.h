// The state part of the moment form for fp32 tensors, d = 64, p = 2, with every contraction on the bf16 matrix
// instruction (three parts per operand, six products: MmaSplit in fm_dense.h).
//
//   cut_apply_kernel  MODE 0  num_i, den_i = phi(qh_i) . S      MODE 1  dv_j = phi(kh_j) . R
//   cut_grad_kernel   MODE 0  dq from S and [g_i, -c_i]         MODE 1  dk from R and [v_j, -1]
//
// Both work on the fp32 states of build_kernel and are the state halves of apply_kernel / grad_kernel (which
// explain the feature indexing, the windows of rotated partners and the credits).  Under the causal mask a block
// leaves its sums in the output tensors and the dense kernels, walking the tiles of their own 256-position chunk
// only, add theirs and finish the rows; blocks without a state (the first chunk in scan order) write nothing.
// Unmasked there is nothing to add and the rows are finished here.
//
// What bounds them: a slab (the 64 state rows of one shift) takes 48 bf16 instructions of ~33 cycles per wave
// instead of 64 (66) fp32 ones of 64, and around them the cutting of operands: ~5.5 VALU instructions per value.
// Eight waves (256 tokens, a whole chunk) therefore share one cut copy of the slab -- each thread cuts the eight
// values it carries from memory to LDS -- so that only the features (apply) or nothing (grad: its own rows are cut
// once) are cut per wave.  One block per CU, two waves per SIMD; a slab is loaded while the one before is worked
// on and there is one barrier per slab.
//
// Measured, 64 x 16 heads x 10000 x 64 causal, ms a step (fp32 instruction with its own-chunk tiles -> here + the dense
// kernels' share): two state builds 48.4 -> 39.8, forward 26.1 -> 17.4 + 4.2, dq 27.9 -> 15.7 + 5.7, dk and dv
// 28.1 + 25.4 -> 15.6 + 16.9 + 7.4.  The error against 64 bits is 5 to 20 % smaller.
#pragma once
#include "fm_dense.h"
#include "fm_grad.h"

namespace cut {

using M = dense::MmaSplit;
using Frag = M::Frag;
constexpr int D = 64, TB = 256, NT = 512, NSLAB = Geo<D>::NS + 1;   // shifts 0 .. 32, then the order-1 rows
constexpr int LD = Geo<D>::LD, SLF = D * LD;

// ---------------------------------------------------------------------------------------
// grid = (256-token blocks from the one that holds position X.lo, heads).
// LDS: own rows (scaled), two buffers of a cut slab as [part][a / 8][column][a % 8] -- a lane's eight k-slots of one
// column are one 128-bit read -- and of its extra column, the denominators.
// ---------------------------------------------------------------------------------------
constexpr int PLANE = D * D, APPLY_LDS = TB * LD * 4 + 2 * 3 * PLANE * 2 + 2 * D * 4 + TB * 4;

template <int MODE>
__global__ __launch_bounds__(NT, 2) void cut_apply_kernel(Rows<const float> X, const float* __restrict__ xscale,
                                                          const float* __restrict__ state, int nslots, Rows<float> OUT,
                                                          RowScalarsOut den, int n, int chunk, int masked, float a0,
                                                          float a1, float a2, int xdiv, int adiv) {
  constexpr bool FWD = MODE == 0;
  constexpr int H2 = D / 2, NS = Geo<D>::NS;
  extern __shared__ __attribute__((aligned(16))) unsigned char cut_smem[];
  float* Xl = reinterpret_cast<float*>(cut_smem);                 // [TB][LD]
  uint16_t* Pl = reinterpret_cast<uint16_t*>(Xl + TB * LD);       // [2][3][D / 8][D][8]
  float* Ex = reinterpret_cast<float*>(Pl + 2 * 3 * PLANE);       // [2][D]
  float* denl = Ex + 2 * D;                                       // [TB]

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int lid = xcd_logical_id(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int head = lid / gridDim.x, tok0 = ((X.lo >> 8) + lid % gridDim.x) * TB;
  const int c = tok0 / chunk, nc = (n + chunk - 1) / chunk;
  if (masked && (FWD ? c == 0 : c == nc - 1)) return;   // (the whole block: nothing before / after this chunk)
  const int hx = head / xdiv, ha = head / adiv;
  const HeadRows<const float> Xh = X.head(hx);
  const float xs = xscale[hx];
  const float* sbase = state + ((int64_t)ha * nslots + (masked ? c : nslots - 1)) * Geo<D>::state_floats(1);

  // wave w carries rows 8 w .. 8 w + 7 of a slab, lane l column l of them (and row 8 w + l % 8 of the extra column)
  float sv[8], se;
  auto slab_load = [&](int st) __attribute__((always_inline)) {
    const float* src = sbase + st * SLF + 8 * w * LD;
#pragma unroll
    for (int e = 0; e < 8; ++e) sv[e] = src[e * LD + l];
    if (FWD) se = src[(l & 7) * LD + D];
  };
  auto slab_store = [&](int buf) __attribute__((always_inline)) {
    const Frag f = M::make(sv);
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<fm_u4*>(Pl + (buf * 3 + k) * PLANE + (w * D + l) * 8) = f.p[k];
    if (FWD && l < 8) Ex[buf * D + 8 * w + l] = se;
  };
  slab_load(0);
  // the order-0 row of the state: value columns i and 32 + i, and the extra column
  const float* row0 = sbase + (NS * D + D) * LD;
  const float z0[2] = {a0 * row0[i], a0 * row0[32 + i]}, zd = FWD ? a0 * row0[D] : 0.f;
  {
    float4 t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int pos = tok0 + w * 32 + 4 * u + l / 16;
      t[u] = *reinterpret_cast<const float4*>(Xh.base + ((unsigned)max(pos < n ? pos : n - 1, Xh.lo) * Xh.pitch + (unsigned)(4 * (l % 16))));
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int row = w * 32 + 4 * u + l / 16, pos = tok0 + row;
      const bool live = pos >= Xh.lo && pos < n;
      *reinterpret_cast<float4*>(Xl + row * LD + 4 * (l % 16)) =
          live ? make_float4(t[u].x * xs, t[u].y * xs, t[u].z * xs, t[u].w * xs) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  slab_store(0);
  __syncthreads();

  const float* xrow = Xl + (w * 32 + i) * LD;
  float Xr[H2];   // the lane half's channels 32 hh + t
#pragma unroll
  for (int t = 0; t < H2; t += 4) {
    const float4 q4 = *reinterpret_cast<const float4*>(xrow + hh * H2 + t);
    Xr[t] = q4.x; Xr[t + 1] = q4.y; Xr[t + 2] = q4.z; Xr[t + 3] = q4.w;
  }
  f16v acc[2] = {dense::kZero16, dense::kZero16};
  float dn = 0.f;
  float Wn[H2 + 4];
  auto window_load = [&](int s0, float cf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < H2 / 4 + 1; ++j) {
      const float4 q4 = *reinterpret_cast<const float4*>(xrow + ((hh * H2 + s0 + 4 * j) & (D - 1)));
      Wn[4 * j] = q4.x * cf; Wn[4 * j + 1] = q4.y * cf; Wn[4 * j + 2] = q4.z * cf; Wn[4 * j + 3] = q4.w * cf;
    }
  };
  auto slab_compute = [&](int buf, auto tag, auto wo) __attribute__((always_inline)) {
    constexpr bool ORD2 = decltype(tag)::value;
    constexpr int WO = decltype(wo)::value;
    const uint16_t* pl = Pl + buf * 3 * PLANE;
#pragma unroll
    for (int m = 0; m < 4; ++m) {   // k-slots: channels 32 hh + 8 m .. + 7
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = Xr[8 * m + e] * (ORD2 ? Wn[WO + 8 * m + e] : a1);
      if (FWD) {
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
          const float4 x4 = *reinterpret_cast<const float4*>(Ex + buf * D + hh * H2 + 8 * m + e);
          dn += f[e] * x4.x; dn += f[e + 1] * x4.y; dn += f[e + 2] * x4.z; dn += f[e + 3] * x4.w;
        }
      }
      const Frag a = M::make_own(f);
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) acc[cb] = M::mma(a, M::load(pl + ((4 * hh + m) * D + cb * 32 + i) * 8, PLANE), acc[cb]);
      if (FWD) asm volatile("" : "+v"(dn));   // (keeps the denominator's sums where their features are)
    }
  };
  // slab st is in buffer st % 2; the next one arrives meanwhile and goes to the other buffer, which every wave is past
  auto slab_iter = [&](int st, auto par, auto tag, auto wo) __attribute__((always_inline)) {
    constexpr int PAR = decltype(par)::value;
    __builtin_amdgcn_sched_barrier(0);
    if (st + 1 < NSLAB) slab_load(st + 1);
    slab_compute(PAR, tag, wo);
    if (st + 1 < NSLAB) slab_store(PAR ^ 1);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  for (int st = 0; st < NS - 1; st += 4) {
    window_load(st, 2.0f * a2);
    slab_iter(st, P0{}, std::true_type{}, std::integral_constant<int, 0>{});
    if (st == 0) {   // shift 0 lists every pair once
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[cb][r] *= 0.5f;
      dn *= 0.5f;
    }
    slab_iter(st + 1, P1{}, std::true_type{}, std::integral_constant<int, 1>{});
    slab_iter(st + 2, P0{}, std::true_type{}, std::integral_constant<int, 2>{});
    slab_iter(st + 3, P1{}, std::true_type{}, std::integral_constant<int, 3>{});
  }
  window_load(NS - 1, a2);   // shift D/2 lists every pair once, too
  slab_iter(NS - 1, P0{}, std::true_type{}, std::integral_constant<int, 0>{});
  slab_iter(NS, P1{}, std::false_type{}, std::integral_constant<int, 0>{});

  if (FWD) {
    const float dtot = dn + __shfl_xor(dn, 32, 64) + zd;
    const int tok = tok0 + w * 32 + i;
    if (hh == 0) {
      denl[w * 32 + i] = masked ? 1.0f : dtot;
      if (tok < n && tok >= Xh.lo) den.head(head)[(int64_t)tok * den.stride] = dtot;
    }
    __syncthreads();
  }
  const HeadRows<float> Oh = OUT.head(head);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = w * 32 + trow(r, hh), tk = tok0 + row;
    if (tk < n && tk >= Xh.lo) {
      const float inv = FWD ? 1.0f / denl[row] : 1.0f;
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) Oh.base[(unsigned)tk * Oh.pitch + (unsigned)(cb * 32 + i)] = (acc[cb][r] + z0[cb]) * inv;
    }
  }
}

// ---------------------------------------------------------------------------------------
// Grid as above.  LDS: two buffers of a cut slab as [row][part][column] and of its extra column.
// rpart (unmasked only): [head * gridDim.x + block] = the block's sum of out . x_hat.
// ---------------------------------------------------------------------------------------
constexpr int GP = 3 * D + 8;   // row pitch: an odd number of 16-byte words

template <int MODE>
__global__ __launch_bounds__(NT, 2) void cut_grad_kernel(Rows<const float> X, Rows<const float> Y, RowScalars yden,
                                                         RowScalars cvec, const float* __restrict__ xscale,
                                                         const float* __restrict__ state, int nslots, Rows<float> OUT,
                                                         float* __restrict__ rpart, int n, int chunk, int masked,
                                                         float a1, float a2, int xdiv, int adiv) {
  constexpr bool DQ = MODE == 0;
  constexpr int H2 = D / 2, NS = Geo<D>::NS, NG = D / 8;
  __shared__ __attribute__((aligned(16))) uint16_t Pl[2 * D * GP];
  __shared__ float Ex[2 * D];
  __shared__ double red[8];

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int lid = xcd_logical_id(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int head = lid / gridDim.x, bidx = lid % gridDim.x, tok0 = ((X.lo >> 8) + bidx) * TB;
  const int c = tok0 / chunk, nc = (n + chunk - 1) / chunk;
  if (masked && (DQ ? c == 0 : c == nc - 1)) return;
  const int hx = head / xdiv, ha = head / adiv;
  const HeadRows<const float> Xh = X.head(hx), Yh = Y.head(hx);
  const float* ydh = yden.head(hx);
  const float* ch = cvec.head(head);
  const float xs = xscale[hx];
  const int tok = tok0 + w * 32 + i;   // the lane's own token
  const bool live = tok < n && tok >= Xh.lo;
  const int tokc = max(tok < n ? tok : n - 1, Xh.lo);
  const float* sbase = state + ((int64_t)ha * nslots + (masked ? c : nslots - 1)) * Geo<D>::state_floats(1);

  // thread tid carries columns 8 (tid % 8) .. + 7 of row tid / 8 of a slab
  const int srow = tid >> 3, spc = tid & 7;
  float4 sa, sb;
  float se;
  auto slab_load = [&](int st) __attribute__((always_inline)) {
    const float* src = sbase + st * SLF + srow * LD;
    sa = *reinterpret_cast<const float4*>(src + 8 * spc);
    sb = *reinterpret_cast<const float4*>(src + 8 * spc + 4);
    se = src[D];
  };
  auto slab_store = [&](int buf) __attribute__((always_inline)) {
    const float x[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
    const Frag f = M::make(x);
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<fm_u4*>(Pl + (buf * D + srow) * GP + k * D + 8 * spc) = f.p[k];
    if (spc == 0) Ex[buf * D + srow] = se;
  };
  slab_load(0);
  const float c_ld = DQ ? ch[(int64_t)tokc * cvec.stride] : 0.f;
  // x of the lane's own channels and of the four above each own group (as in grad_kernel); y cut for the B operand
  float xo[H2], xp[H2];
  Frag yf[4];
  {
    const float4* xr = reinterpret_cast<const float4*>(Xh.row(tokc));
    float4 xa[NG], xb[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      xa[g] = xr[2 * g + hh];
      xb[g] = xr[(2 * g + hh + 1) % (2 * NG)];
    }
    const float xsc = live ? xs : 0.f;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      xo[4 * g] = xa[g].x * xsc; xo[4 * g + 1] = xa[g].y * xsc; xo[4 * g + 2] = xa[g].z * xsc; xo[4 * g + 3] = xa[g].w * xsc;
      xp[4 * g] = xb[g].x * xsc; xp[4 * g + 1] = xb[g].y * xsc; xp[4 * g + 2] = xb[g].z * xsc; xp[4 * g + 3] = xb[g].w * xsc;
    }
    const float dv = ydh ? ydh[(int64_t)tokc * yden.stride] : 1.0f;
    dense::load_own_frags<D, float, M>(Yh, tok, n, D, hh, 1.0f / dv, yf);
  }
  const float c_own = (DQ && live) ? c_ld : 0.f;
  const float yx = hh == 0 ? (DQ ? -c_own : (live ? -1.0f : 0.f)) : 0.f;

  f16v out[2] = {dense::kZero16, dense::kZero16}, outx[2] = {dense::kZero16, dense::kZero16};
  slab_store(0);
  __syncthreads();
  static_for<NSLAB>([&](auto stag) __attribute__((always_inline)) {
    constexpr int S = decltype(stag)::value, BUF = S & 1;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (S + 1 < NSLAB) slab_load(S + 1);
    static_for<2>([&](auto atag) __attribute__((always_inline)) {
      constexpr int AB = decltype(atag)::value;
      const uint16_t* r0 = Pl + (BUF * D + AB * 32 + i) * GP + 8 * hh;
      f16v t = dense::kZero16;   // (the extra column nearly cancels the value columns: smallest products first)
#pragma unroll
      for (int m = 0; m < 4; ++m) t = M::mma_small(M::load(r0 + 16 * m, D), yf[m], t);
#pragma unroll
      for (int m = 0; m < 4; ++m) t = M::mma1(M::load_first(r0 + 16 * m), yf[m].p[0], t);
      t = FM_MFMA(Ex[BUF * D + AB * 32 + i], yx, t);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (S == NS && AB == 0) {   // order 2 is complete: f'(s) contributes 2 a2
#pragma unroll
        for (int ab = 0; ab < 2; ++ab)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            out[ab][r] *= 2.0f * a2;
            outx[ab][r] *= 2.0f * a2;
          }
      }
      credit_tile<D, S, AB, false>(t, out, outx, xo, xp, a1);
      asm volatile("" : "+v"(out[0]), "+v"(out[1]), "+v"(outx[0]), "+v"(outx[1]));   // (as in grad_kernel)
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (S + 1 < NSLAB) {
      slab_store(BUF ^ 1);
      __syncthreads();
    }
    __builtin_amdgcn_sched_barrier(0);
  });
  exchange_halves<D>(out, outx, hh);

  double rs = 0;
  if (!masked) {
#pragma unroll
    for (int ab = 0; ab < 2; ++ab)
#pragma unroll
      for (int r = 0; r < 16; ++r) rs += (double)out[ab][r] * (double)xo[16 * ab + r];
  }
  if (live) {
    float* orow = OUT.head(head).row(tok) + 4 * hh;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const f16v& o = out[g >> 2];
      const int r0 = 4 * (g & 3);
      *reinterpret_cast<float4*>(orow + 8 * g) = make_float4(o[r0] * xs, o[r0 + 1] * xs, o[r0 + 2] * xs, o[r0 + 3] * xs);
    }
  }
  if (!masked) {
    rs = dense::block_sum<8>(rs, red, tid);
    if (tid == 0) rpart[(int64_t)head * gridDim.x + bidx] = (float)rs;
  }
}

// ---------------------------------------------------------------------------------------
// State build: build_kernel (fm_forward.h, which explains the scan, the snapshots and the Gram wave) with the value
// rows cut on their way into LDS and the features cut per wave.  Per 16 tokens and row tile a wave forms and cuts
// eight features (~52 VALU instructions) for twelve bf16 instructions instead of sixteen fp32 ones.  Eight waves
// share the staged 64-token step, so a head takes three blocks (24 waves: 68 row tiles, three a wave, and the Gram
// wave, which stays on the fp32 instruction -- its twelve per eight tokens are less than the others' work -- and adds
// up the order-0 row from what it finds staged).
// grid = (3, heads, token splits).
// ---------------------------------------------------------------------------------------
constexpr int BTS = 64, BKP = BTS + 4, BVP = 3 * BTS + 8;   // tokens per step; pitches of the transposed X and Y tiles
constexpr int BUILD_LDS = 2 * ((D + 1) * BKP * 4 + D * BVP * 2 + BTS * 4);

__global__ __launch_bounds__(NT, 2) void cut_build_kernel(Rows<const float> X, Rows<const float> Y,
                                                          const float* __restrict__ xscale, RowScalars yden,
                                                          RowScalars ew, float* __restrict__ state, int n, int chunk,
                                                          int nslots, int masked, int reverse, int zlen) {
  constexpr int TS = BTS, RTW = 3, ROWS2 = Geo<D>::NS * D, RT2 = ROWS2 / 32, RT = RT2 + D / 32;
  static_assert(RT <= 23 * RTW, "the last wave of a head is free for the Gram tiles");
  extern __shared__ __attribute__((aligned(16))) unsigned char cut_smem[];
  float* Kl = reinterpret_cast<float*>(cut_smem);                              // [2][D + 1][BKP]; row D: 1 where a row exists
  uint16_t* Vl = reinterpret_cast<uint16_t*>(Kl + 2 * (D + 1) * BKP);          // [2][D][BVP]: a column's parts one after another
  float* El = reinterpret_cast<float*>(Vl + 2 * D * BVP);                      // [2][TS]

  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, i = l & 31, hh = l >> 5;
  const int lid = xcd_logical_id(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x * gridDim.y * gridDim.z);
  const int g = lid % gridDim.x, head = (lid / gridDim.x) % gridDim.y, zsplit = lid / (gridDim.x * gridDim.y);
  const int64_t SS = Geo<D>::state_floats(1);
  const int rt0 = (g * 8 + w) * RTW, nx = rt0 + RTW <= RT ? RTW : rt0 < RT ? RT - rt0 : 0;   // row tiles of this wave
  int ownoff[RTW], rotoff[RTW];
#pragma unroll
  for (int x = 0; x < RTW; ++x) {
    const int rt = rt0 + x, ab = rt & 1, s = rt >> 1;
    ownoff[x] = (ab * 32 + i) * BKP + 8 * hh;
    rotoff[x] = (rt < RT2 ? (ab * 32 + i + s) % D : D) * BKP + 8 * hh;   // (order 1: times one)
  }

  const HeadRows<const float> Xh = X.head(head), Yh = Y.head(head);
  const float* ydh = yden.head(head);
  const float* ewh = ew.head(head);
  const float xs = xscale[head];
  const int lo = Xh.lo;

  // staging: thread tid carries 16-byte pieces tid / 64 and tid / 64 + 8 of row tid % 64 of both tiles
  float4 xr[2], yr[2];
  float yd = 1.0f, ev = 1.0f;
  auto load = [&](int t0, int tend) __attribute__((always_inline)) {
    const int t = t0 + l, ps = max(t < tend ? t : tend - 1, lo);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      xr[u] = *reinterpret_cast<const float4*>(Xh.base + ((unsigned)ps * Xh.pitch + (unsigned)(4 * (w + 8 * u))));
      yr[u] = *reinterpret_cast<const float4*>(Yh.base + ((unsigned)ps * Yh.pitch + (unsigned)(4 * (w + 8 * u))));
    }
    if (ydh) yd = ydh[(int64_t)ps * yden.stride];
    if (ewh) ev = ewh[(int64_t)ps * ew.stride];
  };
  auto store = [&](int buf, int t0, int tend) __attribute__((always_inline)) {
    const bool live = t0 + l < tend && t0 + l >= lo;
    const float fx = live ? xs : 0.f, fy = live ? 1.0f / yd : 0.f;
    float* k0 = Kl + buf * (D + 1) * BKP + l;
    uint16_t* v0 = Vl + buf * D * BVP + l;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c0 = 4 * (w + 8 * u);
      k0[c0 * BKP] = live ? xr[u].x * fx : 0.f;
      k0[(c0 + 1) * BKP] = live ? xr[u].y * fx : 0.f;
      k0[(c0 + 2) * BKP] = live ? xr[u].z * fx : 0.f;
      k0[(c0 + 3) * BKP] = live ? xr[u].w * fx : 0.f;
      const float4 y = live ? make_float4(yr[u].x * fy, yr[u].y * fy, yr[u].z * fy, yr[u].w * fy) : make_float4(0.f, 0.f, 0.f, 0.f);
      M::put(nullptr, v0 + c0 * BVP, 0, BVP, TS,
             make_uint4(__float_as_uint(y.x), __float_as_uint(y.y), __float_as_uint(y.z), __float_as_uint(y.w)));
    }
    if (w == 0) {
      El[buf * TS + l] = live ? ev : 0.f;
      k0[D * BKP] = live ? 1.0f : 0.f;
    }
  };

  f16v acc[RTW][2];
#pragma unroll
  for (int x = 0; x < RTW; ++x) acc[x][0] = acc[x][1] = dense::kZero16;
  float k1[2] = {0.f, 0.f}, s0 = 0.f, es = 0.f;   // (Gram wave) order-1 extra column, order-0 row, sum of e

  auto compute = [&](int buf) __attribute__((always_inline)) {
    const float* kb = Kl + buf * (D + 1) * BKP;
    const uint16_t* vb = Vl + buf * D * BVP + i * BVP + 8 * hh;
#pragma unroll 1
    for (int gq = 0; gq < TS / 16; ++gq) {   // k-slots: tokens 16 gq + 8 hh .. + 7
      Frag b[2];
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) b[cb] = M::load(vb + cb * 32 * BVP + 16 * gq, TS);
#pragma unroll
      for (int x = 0; x < RTW; ++x) {
        if (x < nx) {
          const float4 o0 = *reinterpret_cast<const float4*>(kb + ownoff[x] + 16 * gq), o1 = *reinterpret_cast<const float4*>(kb + ownoff[x] + 16 * gq + 4);
          const float4 r0 = *reinterpret_cast<const float4*>(kb + rotoff[x] + 16 * gq), r1 = *reinterpret_cast<const float4*>(kb + rotoff[x] + 16 * gq + 4);
          const float f[8] = {o0.x * r0.x, o0.y * r0.y, o0.z * r0.z, o0.w * r0.w, o1.x * r1.x, o1.y * r1.y, o1.z * r1.z, o1.w * r1.w};
          const Frag a = M::make_own(f);
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) acc[x][cb] = M::mma(a, b[cb], acc[x][cb]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);   // (register pressure)
    }
  };
  // tiles (0,0), (0,1), (1,1) of G in acc[0][0], acc[0][1], acc[1][0]; sums of the staged value columns and of e
  auto compute_gram = [&](int buf) __attribute__((always_inline)) {
    const float* kb = Kl + buf * (D + 1) * BKP;
    const float* eb = El + buf * TS;
    const int r0 = i * BKP + 4 * hh, r1 = (32 + i) * BKP + 4 * hh;
#pragma unroll 1
    for (int gq = 0; gq < TS / 8; ++gq) {
      const float4 x0 = *reinterpret_cast<const float4*>(kb + r0 + 8 * gq);
      const float4 x1 = *reinterpret_cast<const float4*>(kb + r1 + 8 * gq);
      const float4 e4 = *reinterpret_cast<const float4*>(eb + 8 * gq + 4 * hh);
      const float xa[4] = {x0.x, x0.y, x0.z, x0.w}, xb[4] = {x1.x, x1.y, x1.z, x1.w}, e[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float ya = xa[u] * e[u], yb = xb[u] * e[u];
        acc[0][0] = FM_MFMA(xa[u], ya, acc[0][0]);
        acc[0][1] = FM_MFMA(xa[u], yb, acc[0][1]);
        acc[1][0] = FM_MFMA(xb[u], yb, acc[1][0]);
        k1[0] += ya;
        k1[1] += yb;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    es += eb[l];
    const uint16_t* v0 = Vl + buf * D * BVP + l * BVP;   // lane l: value column l
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < TS; t += 8) {
      float y[8];
      M::values(M::load(v0 + t, TS), y);
      s += ((y[0] + y[1]) + (y[2] + y[3])) + ((y[4] + y[5]) + (y[6] + y[7]));
    }
    s0 += s;
  };
  auto emit = [&](int slot, auto gtag) __attribute__((always_inline)) {
    float* st = state + ((int64_t)head * nslots + slot) * SS;
    if constexpr (!decltype(gtag)::value) {
#pragma unroll
      for (int x = 0; x < RTW; ++x)
        if (x < nx) {
          float* sx = st + (unsigned)((rt0 + x) * 32 * LD);   // (tile rt: rows 32 rt .. + 31)
#pragma unroll
          for (int r = 0; r < 16; ++r)
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) sx[(unsigned)(trow(r, hh) * LD + cb * 32 + i)] = acc[x][cb][r];
        }
    } else {
      // element (a, b) of G is the extra column of row (s, a), s = (b - a) mod D <= D/2, else of row (D - s, b); a
      // diagonal tile holds every pair twice, s = D/2 lists every pair from both sides
      int li = i, lh = hh;
      asm volatile("" : "+v"(li), "+v"(lh));   // (the offsets are formed here, not kept across the scan)
      auto put = [&](const f16v& gacc, int ra, int cb) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int a = ra * 32 + trow(r, lh), b = cb * 32 + li, sft = (b - a) & (D - 1);
          if (sft <= D / 2) {
            st[(unsigned)((sft * D + a) * LD + D)] = gacc[r];
            if (sft == D / 2) st[(unsigned)((sft * D + b) * LD + D)] = gacc[r];
          } else if (ra != cb) {
            st[(unsigned)(((D - sft) * D + b) * LD + D)] = gacc[r];
          }
          if ((r & 3) == 3) __builtin_amdgcn_sched_barrier(0);
        }
      };
      put(acc[0][0], 0, 0);
      put(acc[0][1], 0, 1);
      put(acc[1][0], 1, 1);
      const float ka = k1[0] + __shfl_xor(k1[0], 32, 64), kb = k1[1] + __shfl_xor(k1[1], 32, 64);
      if (lh == 0) {
        st[(unsigned)((ROWS2 + li) * LD + D)] = ka;
        st[(unsigned)((ROWS2 + 32 + li) * LD + D)] = kb;
      }
      float et = es;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) et += __shfl_xor(et, off, 64);
      st[(unsigned)((ROWS2 + D) * LD + l)] = s0;
      if (l == 0) st[(unsigned)((ROWS2 + D) * LD + D)] = et;
    }
  };

  // the walk (steps, the slot written after each): as in build_kernel
  const int spc = chunk / TS, nc = (n + chunk - 1) / chunk;
  int nsteps, first_len = 0, tbase = 0, tend = n;
  if (masked) {
    if (reverse) {
      first_len = (n - (nc - 1) * chunk + TS - 1) / TS;
      const int cl = lo / chunk;
      nsteps = nc > 1 ? first_len + (nc - 1 - (cl > 1 ? cl : 1)) * spc : 0;
    } else {
      nsteps = (nc - 1) * spc;
    }
  } else {
    tbase = zsplit * zlen;
    tend = tbase + zlen < n ? tbase + zlen : n;
    nsteps = tend > tbase ? (tend - tbase + TS - 1) / TS : 0;
  }
  auto step_tok = [&](int p) {
    if (!masked) return tbase + p * TS;
    if (!reverse) return p * TS;
    if (p < first_len) return (nc - 1) * chunk + p * TS;
    const int q = p - first_len;
    return (nc - 2 - q / spc) * chunk + (q % spc) * TS;
  };
  auto step_slot = [&](int p) {
    if (!masked) return p + 1 == nsteps ? zsplit : -1;
    if (!reverse) return (p + 1) % spc == 0 ? (p + 1) / spc : -1;
    if (p < first_len) return p + 1 == first_len ? nc - 2 : -1;
    const int q = p - first_len;
    return (q + 1) % spc == 0 ? nc - 3 - q / spc : -1;
  };
  auto scan = [&](auto gtag) __attribute__((always_inline)) {
    if (nsteps > 0) {
      load(step_tok(0), tend);
      store(0, step_tok(0), tend);
    }
    __syncthreads();
    for (int p = 0; p < nsteps; ++p) {
      const bool more = p + 1 < nsteps;
      const int tnext = step_tok(more ? p + 1 : p);
      if (more) load(tnext, tend);
      if constexpr (decltype(gtag)::value) compute_gram(p & 1);
      else compute(p & 1);
      if (more) store((p + 1) & 1, tnext, tend);
      const int slot = step_slot(p);   // (after the loads have arrived: one in-order counter covers loads and stores)
      if (slot >= 0) emit(slot, gtag);
      __syncthreads();
    }
    if (!masked && nsteps == 0) emit(zsplit, gtag);   // (an empty token split still owns its slot)
    if (masked && reverse && nsteps > 0)
      for (int slot = lo / chunk - 2; slot >= 0; --slot) emit(slot, gtag);   // (chunks below the one that holds lo)
  };
  if (nx == 0) scan(std::true_type{});   // (the Gram wave; every wave stages tiles and meets the barriers alike)
  else scan(std::false_type{});
}

}  // namespace cut
