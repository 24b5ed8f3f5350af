// Quantized GEMM on small tiles for gfx950: Y[M,N] = X[M,K] deq(W)[N,K]^T for W4/W8
// weights where 128 x 256 tiles (linear_pingpong.hip) leave most of the chip idle: a
// prompt's rows, a 512-pixel image's tokens, the context projections.
//
//   * Tile TM x TN = (32 MT) x (32 WN), computed as C^T = W X^T on v_mfma_f32_32x32x16_f16
//     by 16 waves: WN column tiles x WK of the quantisation groups (64 of K) that a K block
//     holds.  Wave (wn, wk) multiplies groups wk, wk + WK, ... of its 32 columns for all TM
//     rows, so no weight is dequantised twice in a workgroup; the WK partial tiles are
//     added in order in LDS.  16 waves because a single wave issues a vector instruction
//     every 6-8 cycles: 4 waves on 32 x 64 tiles took 11.8 us where 16 take 10.0 (W8, M=77
//     N=2048 K=2048).
//   * X and the packed weights of a block are loaded as whole row pieces two blocks ahead in
//     registers, and go through double-buffered LDS rows padded by 16 B (16 consecutive
//     rows on distinct banks).  Loading a wave's weights straight into its fragments
//     touches 32 rows with 16-32 bytes each, a quarter of the bytes per cycle.
//   * Two phases per block, a barrier after each: MFMAs (with the LDS and global copies
//     between them) and dequantisation.  Waves 8-15 run one phase behind, so the matrix
//     and the vector pipe of a SIMD work at once.
//   * Dequantisation is the bit-exact one of dequant.hpp: one rounding in packed fp16,
//     redone with the fp32 FMA when a lane's pair needs two roundings.
//   * Loads past M, N or the last block read zeros from bounded or empty descriptors; all
//     loads of a step are unconditional, so the compiler's wait counts stay exact.
//
// What bounds it: at M=1024 N=2048 K=8192 a block of 64 x 128 x 256 takes 1.4 us (1.0 on an
// otherwise idle chip) for 0.45 us of MFMAs; timing builds without the loads 1.0, without
// the copies into LDS 1.2, without the MFMAs 1.1, without any copy 0.8: the copies (48-64 KB
// per block and CU through one vector memory path and LDS port) and the two barriers.
// Before -> after, back to back with the weights in HBM (W8): M=77 N=3072 K=1024 18.9 -> 7.7
// us, M=77 N=2048 K=2048 22.9 -> 10.0, M=512 N=2048 K=2048 27.8 -> 15.3, M=1024 N=2048
// K=2048 29.4 -> 17.3 (500 TFLOP/s), M=1024 N=1024 K=4096 -> 23.3.
#include <type_traits>

#include "dequant.hpp"
#include "gemm_output.hpp"

namespace anima {

// Quantisation groups of one of ks K splits: whole 16-byte pieces of scales, so that every
// split starts on a block of either tile shape.
__host__ __device__ constexpr int split_groups(int groups, int ks) {
  return ks > 1 ? ((groups + ks - 1) / ks + 7) / 8 * 8 : groups;
}

constexpr int TG_GM = 8;        // M tiles per group of the tile order
constexpr int TG_AHEAD = 2;     // X fragments read ahead of their MFMAs

template <int STORAGE, int MT, int WN, int WK>
struct TileShape {
  static constexpr bool W4 = STORAGE == ANIMA_STORAGE_W4;
  static constexpr int TM = 32 * MT, TN = 32 * WN, BK = 64 * WK;
  static constexpr int THREADS = 64 * WN * WK;
  static constexpr int WROW = W4 ? BK / 2 : BK;               // packed bytes per row and block
  static constexpr int XPITCH = 2 * BK + 16, WPITCH = WROW + 16;
  static constexpr int XPIECES = BK / 8, WPIECES = WROW / 16; // 16-byte pieces per row and block
  static constexpr int XCH = TM * XPIECES / THREADS;          // pieces per thread and block
  static constexpr int WCH = TN * WPIECES / THREADS;
  static constexpr int SROW = 2 * WK;                         // scale (or zero) bytes per row and block
  static constexpr int XS = 0, WS = XS + 2 * TM * XPITCH, SZ = WS + 2 * TN * WPITCH;
  static constexpr int SZBUF = 2 * TN * SROW;
  static constexpr int LOOP_BYTES = SZ + 2 * SZBUF;
  static constexpr int OPITCH = TN + 4;                       // partial-sum tile row (floats)
  static constexpr int PIECES = TM * TN / 8, OUT_THREADS = PIECES < THREADS ? PIECES : THREADS;   // output stage
  static constexpr int END_BYTES = WK * TM * OPITCH * 4;
  static constexpr int SMEM = LOOP_BYTES > END_BYTES ? LOOP_BYTES : END_BYTES;
  static_assert(TM * XPIECES % THREADS == 0 && TN * WPIECES % THREADS == 0 && 2 * TN <= THREADS, "whole copies per thread");
  static_assert(WK == 4 || WK == 8, "scale pieces are 8 or 16 bytes");
};

// SWIN: the scale/zero rows are aligned runs of WK groups (one load per row and block).
// PAIR: the gated MLP's two linears at once (gp.p[0] the gate, gp.p[1] the up projection, of
// one shape and row stride): the tile's weight rows are TN / 2 rows of each, and the output
// stage writes half(silu(half(gate)) * half(up)) for TN / 2 columns.
template <int STORAGE, bool SWIN, bool PAIR, int MT, int WN, int WK>
__global__ __launch_bounds__(64 * WN * WK, 1) __attribute__((amdgpu_waves_per_eu(4, 4)))
void tile_gemm_kernel(GemmGroup gp) {
  using S = TileShape<STORAGE, MT, WN, WK>;
  constexpr bool W4 = S::W4;
  constexpr int QBITS = W4 ? 4 : 8;
  constexpr int RCH = W4 ? 1 : 2;           // 16-byte pieces of a lane's row and group
  constexpr int SDW = WK / 2;               // dwords of a row's scales per block
  __shared__ __attribute__((aligned(1024))) char smem[S::SMEM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave % WK, wn = wave / WK, group = wave / (WN * WK / 2);
  const int c32 = lane & 31, hh = lane >> 5;
  // Problem, K split and tile of this workgroup.  Tiles go in groups of TG_GM M tiles x all
  // N tiles, M varying fastest, so the 32 workgroups an XCD runs at once share 8 row and 4
  // column tiles in its L2 (M=2048 N=2048 K=2048: 35.2 us with all M tiles in one group,
  // 30.0 with 8, 30.6 with 4).
  const int lbg = xcd_logical_block(blockIdx.x, gridDim.x);
  int pi = 0;
  if constexpr (!PAIR) {
#pragma unroll
    for (int i = 1; i < PG_GROUP; ++i)
      if (i < gp.count && lbg >= gp.first_tile[i]) pi = i;
  }
  const GemmParams& p = gp.p[pi];
  constexpr int HR = PAIR ? S::TN / 2 : S::TN;   // weight rows (and output columns) per member
  const int vec_store = gp.vec[pi];
  const int ks = p.ksplit > 1 ? p.ksplit : 1;
  const int lb = lbg - gp.first_tile[pi], split = lb % ks, lt = lb / ks;
  const int ntm = (p.M + S::TM - 1) / S::TM;
  const int ntn = (p.N + HR - 1) / HR;
  const int gfirst = lt / (TG_GM * ntn) * TG_GM, gm = ntm - gfirst < TG_GM ? ntm - gfirst : TG_GM;
  const int gr = lt % (TG_GM * ntn);
  const int m0 = (gfirst + gr % gm) * S::TM, n0 = gr / gm * HR;
  // A split takes split_groups groups, the last one what is left of them.
  const int sg = split_groups(p.groups, ks), gbeg = split * sg;
  const int groups = p.groups - gbeg < sg ? p.groups - gbeg : sg;
  const int nblk = (groups + WK - 1) / WK;
  const int nown = (groups + WK - 1 - wk) / WK;   // groups wk, wk + WK, ... of this wave: nblk or nblk - 1

  const half_t* xb = p.x + (int64_t)m0 * p.K + 64 * gbeg;
  const int xbytes = ((p.M - m0) * p.K - 64 * gbeg) * 2;
  const int64_t woff = (int64_t)n0 * p.row_stride + (W4 ? 32 : 64) * gbeg;
  const uint8_t* wb[S::WCH];   // per copy: with PAIR its rows' member (one for the whole wave)
  const int wbytes = (int)((int64_t)(p.N - n0) * p.row_stride) - (W4 ? 32 : 64) * gbeg;
  const int sbytes = ((p.N - n0) * p.groups - gbeg) * 2;

  // Copies: piece tid + THREADS r of a block.
  uint32_t goff_x[S::XCH], goff_w[S::WCH];
  int loff_x[S::XCH], loff_w[S::WCH];
#pragma unroll
  for (int r = 0; r < S::XCH; ++r) {
    const int id = tid + S::THREADS * r, row = id / S::XPIECES, ch = id % S::XPIECES;
    goff_x[r] = (uint32_t)row * (uint32_t)p.K * 2u + 16u * ch;
    loff_x[r] = S::XS + row * S::XPITCH + 16 * ch;
  }
#pragma unroll
  for (int r = 0; r < S::WCH; ++r) {
    const int id = tid + S::THREADS * r, row = id / S::WPIECES, ch = id % S::WPIECES;
    wb[r] = (PAIR && (64 * wave + S::THREADS * r) / S::WPIECES >= HR ? gp.p[1].w : p.w) + woff;
    goff_w[r] = (uint32_t)(row % HR) * (uint32_t)p.row_stride + 16u * ch;
    loff_w[r] = S::WS + row * S::WPITCH + 16 * ch;
  }
  // Scales: waves 0 .. TN/64-1 take the scales of row tid, the next as many the zeros.  With
  // PAIR waves 0 to 3 take the gate's scales, the up's, the gate's zeros and the up's.
  static_assert(!PAIR || HR <= 64, "one wave per member's scales");
  const bool sz_wave = PAIR ? wave < 4 : 64 * wave < 2 * S::TN;
  const half_t* szb = (PAIR ? (wave == 0 ? p.scale : wave == 1 ? gp.p[1].scale : wave == 2 ? p.zero : gp.p[1].zero)
                            : (64 * wave < S::TN ? p.scale : p.zero)) +
                      (int64_t)n0 * p.groups + gbeg;
  const uint32_t goff_sz = (uint32_t)(PAIR ? lane % HR : tid % S::TN) * (uint32_t)p.groups * 2u;
  const int sz_slot = PAIR ? HR * wave + lane : tid;
  const bool sz_lane = sz_wave && (!PAIR || lane < HR);

  struct Sz { uint32_t d[SDW]; };
  auto load_x = [&](int kb, u32x4 (&v)[S::XCH]) __attribute__((always_inline)) {
    const int n = kb < nblk ? xbytes : 0;
#pragma unroll
    for (int r = 0; r < S::XCH; ++r) v[r] = load16_bounded(xb, n, goff_x[r], kb * S::BK * 2);
  };
  auto load_w = [&](int kb, u32x4 (&v)[S::WCH], Sz& z) __attribute__((always_inline)) {
    const int n = kb < nblk ? wbytes : 0, ns = kb < nblk && sz_wave ? sbytes : 0;
    if constexpr (SWIN && WK == 8) {
      const u32x4 q = load16_bounded(szb, ns, goff_sz, kb * S::SROW);
#pragma unroll
      for (int i = 0; i < SDW; ++i) z.d[i] = q[i];
    } else if constexpr (SWIN) {
      const u32x2 q = load8_bounded(szb, ns, goff_sz, kb * S::SROW);
#pragma unroll
      for (int i = 0; i < SDW; ++i) z.d[i] = q[i];
    } else {
#pragma unroll
      for (int i = 0; i < SDW; ++i)
        z.d[i] = load2_bounded(szb, ns, goff_sz, kb * S::SROW + 4 * i) |
                 load2_bounded(szb, ns, goff_sz, kb * S::SROW + 4 * i + 2) << 16;
    }
#pragma unroll
    for (int r = 0; r < S::WCH; ++r) v[r] = load16_bounded(wb[r], n, goff_w[r], kb * S::WROW);
  };
  auto store_x = [&](int buf, int r, const u32x4 (&v)[S::XCH]) __attribute__((always_inline)) {
    *reinterpret_cast<u32x4*>(smem + loff_x[r] + buf * S::TM * S::XPITCH) = W4 ? interleave_w4_order(v[r]) : v[r];
  };
  auto store_w = [&](int buf, int r, const u32x4 (&v)[S::WCH]) __attribute__((always_inline)) {
    *reinterpret_cast<u32x4*>(smem + loff_w[r] + buf * S::TN * S::WPITCH) = v[r];
  };
  auto store_sz = [&](int buf, const Sz& z) __attribute__((always_inline)) {
    if (sz_lane) *reinterpret_cast<Sz*>(smem + S::SZ + buf * S::SZBUF + sz_slot * S::SROW) = z;
  };
  // The lane's packed weights and scale/zero of its group of the block in stage buf: row
  // 32 wn + c32, k = 32 hh .. 32 hh + 31 of the group.
  u32x4 raw[RCH];
  half_t sh, zh;
  const int lrow = 32 * wn + c32;
  auto fetch_raw = [&](int buf) __attribute__((always_inline)) {
    const half_t* w = reinterpret_cast<const half_t*>(smem + S::SZ + buf * S::SZBUF);
    sh = w[lrow * WK + wk];
    zh = w[S::TN * WK + lrow * WK + wk];
#pragma unroll
    for (int c = 0; c < RCH; ++c)
      raw[c] = *reinterpret_cast<const u32x4*>(smem + S::WS + buf * S::TN * S::WPITCH + lrow * S::WPITCH +
                                               16 * (2 * RCH * wk + RCH * hh + c));
  };
  uint32_t w4k[3] = {0x000F000Fu, 0x00F000F0u, 0x64006400u};
#pragma unroll
  for (int i = 0; i < 3; ++i) asm volatile("" : "+v"(w4k[i]));

  half8v wf[4];         // dequantised fragments, one per k step of 16
  auto dq_half = [&](int s, int part) __attribute__((always_inline)) {
    const half2v s2 = {sh, sh}, z2 = {zh, zh};
    half4v h;
    if constexpr (W4) {
      const uint32_t x = raw[0][s];
      h = w4_half_one_rounding(part ? x >> 8 : x, s2, z2, w4k);
    } else {
      h = w8_half_one_rounding(raw[s >> 1][2 * (s & 1) + part], s2, z2);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) wf[s][4 * part + e] = h[e];
    asm volatile("" : "+v"(wf[s]));   // keeps it here, not in the redo's other branch
  };
  auto redo_exact = [&]() __attribute__((always_inline)) {
    const float sf = (float)sh, zf = (float)zh;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if constexpr (W4)
        wf[s] = w4_frag_exact(raw[0][s], sf, zf);
      else
        wf[s] = w8_frag_exact(raw[s >> 1][2 * (s & 1)], raw[s >> 1][2 * (s & 1) + 1], sf, zf);
    }
  };
  auto barrier = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  floatx16 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = floatx16{};

  // X(j) in xr[j & 1], W(j) in wr[j & 1]; blocks 0 (X) and 0, 1 (W) go straight to LDS.
  u32x4 xr[2][S::XCH], wr[2][S::WCH];
  Sz zr[2];
  {
    u32x4 x0[S::XCH], w0[S::WCH], w1[S::WCH];
    Sz z0, z1;
    load_w(0, w0, z0);
    load_x(0, x0);
    load_w(1, w1, z1);
    load_x(1, xr[1]);
    load_w(2, wr[0], zr[0]);
    load_x(2, xr[0]);
    load_w(3, wr[1], zr[1]);
    store_sz(0, z0);
    store_sz(1, z1);
#pragma unroll
    for (int r = 0; r < S::WCH; ++r) store_w(0, r, w0);
#pragma unroll
    for (int r = 0; r < S::XCH; ++r) store_x(0, r, x0);
#pragma unroll
    for (int r = 0; r < S::WCH; ++r) store_w(1, r, w1);
  }
  barrier();
  fetch_raw(0);
  barrier();   // block 0's weights are out of LDS before group 0's first step writes W(2) there
  auto dequant = [&]() __attribute__((always_inline)) {
    const bool fast = (bool)__all(one_rounding_exact<QBITS>(sh, zh));
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      dq_half(s, 0);
      dq_half(s, 1);
    }
    if (!fast) redo_exact();
  };
  dequant();
  if (group == 1) barrier();   // group 1 runs one phase behind

  // Block kb (parity CUR).  Multiply phase: its MFMAs (X stage CUR, fragments wf), the
  // weights and scales of block kb + 1 out of LDS, X(kb + 1) and W(kb + 2) into LDS, the
  // loads of X(kb + 3) and W(kb + 4).  Dequantisation phase: the fragments of kb + 1.
  // Group 0 multiplies block kb in interval 2 kb, group 1 in interval 2 kb + 1; a stage is
  // written there after its last read (X(kb - 1), W(kb): intervals 2 kb - 2 and 2 kb - 1, for
  // W(0) the prologue's, which its own barrier ends) and before its next (2 kb + 2).
  auto step = [&](int kb, auto cur_c) __attribute__((always_inline)) {
    constexpr int CUR = decltype(cur_c)::value, NXT = CUR ^ 1;
    constexpr int NOPS = 4 * MT, AHEAD = TG_AHEAD, RING = AHEAD + 1, COPIES = S::XCH + S::WCH;
    __builtin_amdgcn_s_setprio(1);
    const char* xs = smem + S::XS + CUR * S::TM * S::XPITCH + c32 * S::XPITCH + 128 * wk + 64 * hh;
    auto read_op = [&](int i) __attribute__((always_inline)) -> half8v {
      return *reinterpret_cast<const half8v*>(xs + (i % MT) * 32 * S::XPITCH + (i / MT) * 16);
    };
    half8v ring[RING];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) ring[i] = read_op(i);
#pragma unroll
    for (int i = 0; i < NOPS; ++i) {
      if (i + AHEAD < NOPS) ring[(i + AHEAD) % RING] = read_op(i + AHEAD);
      acc[i % MT] = mfma32(wf[i / MT], ring[i % RING], acc[i % MT]);
      if (i == NOPS - 2) fetch_raw(NXT);
#pragma unroll
      for (int c = i * COPIES / NOPS; c < (i + 1) * COPIES / NOPS; ++c) {
        if (c < S::XCH)
          store_x(NXT, c, xr[NXT]);
        else
          store_w(CUR, c - S::XCH, wr[CUR]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    store_sz(CUR, zr[CUR]);
    load_x(kb + 3, xr[NXT]);
    load_w(kb + 4, wr[CUR], zr[CUR]);
    __builtin_amdgcn_s_setprio(0);
    barrier();
    dequant();
    barrier();
  };
  // Whole blocks in pairs, with no branch between the loads; then the last one or two, of
  // which the last may end before this wave's group.
  const int pairs = groups / (2 * WK) * 2;
  for (int kb = 0; kb < pairs; kb += 2) {
    step(kb, std::integral_constant<int, 0>{});
    step(kb + 1, std::integral_constant<int, 1>{});
  }
  auto idle = [&]() __attribute__((always_inline)) {
    barrier();
    barrier();
  };
  if (pairs < nblk) {
    if (pairs < nown)
      step(pairs, std::integral_constant<int, 0>{});
    else
      idle();
  }
  if (pairs + 1 < nblk) {
    if (pairs + 1 < nown)
      step(pairs + 1, std::integral_constant<int, 1>{});
    else
      idle();
  }
  if (group == 0) barrier();
  // Every stage read done, every store landed: LDS is free.

  // Every wave's sums go to its partial tile; the output stage adds the WK tiles in order.
  float* part = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<floatx4*>(part + (wk * S::TM + 32 * m + c32) * S::OPITCH + 32 * wn + 8 * q + 4 * hh) =
          floatx4{acc[m][4 * q], acc[m][4 * q + 1], acc[m][4 * q + 2], acc[m][4 * q + 3]};
  barrier();
  constexpr int OUT_THREADS = PAIR && S::PIECES / 2 < S::THREADS ? S::PIECES / 2 : S::OUT_THREADS;
  if (tid >= OUT_THREADS) return;
  auto sum8 = [&](int r, int c, floatx4& a, floatx4& b) __attribute__((always_inline)) {
    const float* src = part + r * S::OPITCH + 8 * c;
    a = *reinterpret_cast<const floatx4*>(src);
    b = *reinterpret_cast<const floatx4*>(src + 4);
#pragma unroll
    for (int k = 1; k < WK; ++k) {
      a += *reinterpret_cast<const floatx4*>(src + k * S::TM * S::OPITCH);
      b += *reinterpret_cast<const floatx4*>(src + k * S::TM * S::OPITCH + 4);
    }
  };
  if constexpr (PAIR) {
    auto half8 = [&](int r, int c) __attribute__((always_inline)) {
      floatx4 a, b;
      sum8(r, c, a, b);
      return half8v{(half_t)a[0], (half_t)a[1], (half_t)a[2], (half_t)a[3],
                    (half_t)b[0], (half_t)b[1], (half_t)b[2], (half_t)b[3]};
    };
    store_tile_rows<GEMM_STORE, S::TM, HR, OUT_THREADS>(
        p, [&](int r, int c) { return gated_silu8(half8(r, c), half8(r, c + HR / 8)); }, m0, n0, vec_store, tid);
    return;
  }
  if (ks > 1) {
    // The fp32 sums of this K range; splitk_reduce_kernel finishes.
    constexpr int CHUNKS = S::TN / 8, STEP = S::OUT_THREADS / CHUNKS;
    const int c = tid % CHUNKS, n = n0 + 8 * c;
#pragma unroll
    for (int i = 0; i < S::TM / STEP; ++i) {
      const int r = tid / CHUNKS + STEP * i, m = m0 + r;
      floatx4 a, b;
      sum8(r, c, a, b);
      if (m >= p.M) continue;
      float* prow = p.part + ((int64_t)split * p.M + m) * p.N;
      if ((p.N & 3) == 0 && n + 8 <= p.N) {
        *reinterpret_cast<floatx4*>(prow + n) = a;
        *reinterpret_cast<floatx4*>(prow + n + 4) = b;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e < p.N) prow[n + e] = a[e];
          if (n + 4 + e < p.N) prow[n + 4 + e] = b[e];
        }
      }
    }
    return;
  }
  store_tile_epilogue<S::TM, S::TN, S::OUT_THREADS>(
      p,
      [&](int r, int c) {
        floatx4 a, b;
        sum8(r, c, a, b);
        return half8v{(half_t)a[0], (half_t)a[1], (half_t)a[2], (half_t)a[3],
                      (half_t)b[0], (half_t)b[1], (half_t)b[2], (half_t)b[3]};
      },
      m0, n0, vec_store, tid);
}

// Shape 0: 64 x 128, 4 waves per column tile along K; shape 1: 32 x 64, 8 along K.  The
// wide tile moves half the bytes per output; the small one gives four times the tiles and
// half the steps along K.  One round of small tiles wins (us, small / wide, W8): M=77 N=2048
// K=2048 10.0 / 14.9, M=300 N=1024 K=2048 10.4 / 15.2, M=512 N=1024 K=2048 (256 tiles) 10.6
// / 15.2; a second round loses: M=300 N=2048 K=2048 (320 tiles) 18.6 / 15.3.
constexpr int TG_TM[2] = {64, 32}, TG_TN[2] = {128, 64}, TG_WK[2] = {4, 8};

static int64_t tile_count(const GemmParams& p, int shape) {
  return (int64_t)((p.M + TG_TM[shape] - 1) / TG_TM[shape]) * ((p.N + TG_TN[shape] - 1) / TG_TN[shape]);
}

// One round of 64 x 128 tiles (a quarter of a chip of 128 x 256 ones) takes 1/1.5 to 1/3.4 of
// the ping-pong kernel's time: M=1024 N=2048 K=2048, 256 tiles, 17.3 / 29.4 us.  Two rounds,
// below half a chip of the other's tiles, only at K = 512 and 1280 to 2048 in whole K blocks
// (ping-pong / this over 288 to 512 tiles: plain 0.96-1.04 at 512, 1.03-1.11 at 1536, 0.94-1.07
// at 2048; GELU 1.12-1.19, 1.06-1.19, 1.04-1.11; gate-add 1.04-1.10, 1.00-1.17, 0.94-1.10).
// At 768 and 1024 the ping-pong kernel's halves of K are one window each (plain 0.91-1.00), at
// 256 a block cannot hide the loads (0.86-0.93), a last block of one group costs a whole one
// (320 0.70-0.74, 1088 0.74-0.77), and past 2048 the ping-pong kernel splits K (4096 0.83-0.96).
bool tile_preferred(const GemmParams& p, int storage) {
  if (!pingpong_supported(p, storage) || single_tile_over_input(p)) return false;
  const bool two_rounds = p.K % 256 == 0 && (p.K == 512 || (p.K > 1024 && p.K <= 2048));
  return tile_count(p, 0) <= 256 || (two_rounds && pingpong_tiles(p) < 128);
}

// One launch of several plain linears: where one round of tiles holds them.
bool tile_group_preferred(const GemmParams* ps, int count) {
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i) tiles += tile_count(ps[i], 0);
  return tiles <= 256;
}

int tile_group_shape(const GemmParams* ps, int count) {
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i) tiles += tile_count(ps[i], 1);
  return tiles <= 256 ? 1 : 0;
}

int tile_shape(const GemmParams& p) { return tile_group_shape(&p, 1); }

bool tile_takes_norm(const GemmParams& p) { return TG_TN[tile_shape(p)] % 128 == 0; }

// Splits that still fit one round, each (but the last, which takes what is left) of at least
// 4 (small tiles) or 8 blocks and of whole scale pieces: the saved steps then outweigh the
// fp32 rows and the second launch.  W8, us, unsplit / split in two: M=77 N=2048 K=8192 25.1 /
// 19.7, M=300 50.8 / 34.7, M=512 51.8 / 38.4, M=1024 N=1024 K=4096 25.7 / 23.3; with shorter
// splits M=77 N=2048 K=2048 10.0 / 11.0.  Uneven splits against the nearest even count (or
// none): W4 M=109 N=128 K=5696 26.4 -> 16.9, W8 M=191 N=752 K=6016 28.2 -> 18.6, W4 M=3153
// N=160 K=7232 50.4 -> 35.7, W8 M=1451 N=1200 K=4672 87 (before this kernel) -> 38.9.
int tile_ksplit(const GemmParams& p) {
  const int shape = tile_shape(p), min_blocks = shape ? 4 : 8;
  const int64_t tiles = tile_count(p, shape);
  for (int k = 8; k > 1; --k) {
    const int each = split_groups(p.groups, k), used = (p.groups + each - 1) / each;
    if (used > 1 && split_groups(p.groups, used) == each && each >= min_blocks * TG_WK[shape] && tiles * used <= 256)
      return used;
  }
  return 1;
}

template <int STORAGE, bool SWIN, bool PAIR>
static void launch_tile_s(const GemmGroup& g, int shape, unsigned tiles, hipStream_t stream) {
  if (shape == 0)
    hipLaunchKernelGGL((tile_gemm_kernel<STORAGE, SWIN, PAIR, 2, 4, 4>), dim3(tiles), dim3(1024), 0, stream, g);
  else
    hipLaunchKernelGGL((tile_gemm_kernel<STORAGE, SWIN, PAIR, 1, 2, 8>), dim3(tiles), dim3(1024), 0, stream, g);
}

template <bool PAIR>
static void launch_tile_t(const GemmGroup& g, int storage, bool swin, int shape, unsigned tiles, hipStream_t stream) {
  if (storage == ANIMA_STORAGE_W4) {
    if (swin)
      launch_tile_s<ANIMA_STORAGE_W4, true, PAIR>(g, shape, tiles, stream);
    else
      launch_tile_s<ANIMA_STORAGE_W4, false, PAIR>(g, shape, tiles, stream);
  } else {
    if (swin)
      launch_tile_s<ANIMA_STORAGE_W8, true, PAIR>(g, shape, tiles, stream);
    else
      launch_tile_s<ANIMA_STORAGE_W8, false, PAIR>(g, shape, tiles, stream);
  }
  ANIMA_HIP(hipGetLastError());
}

// Scale and zero rows that are aligned runs of a block's groups.
static bool tile_swin(const GemmParams& p, int shape) {
  const int piece = 2 * TG_WK[shape];   // scale bytes per row and block
  return p.groups % TG_WK[shape] == 0 && (reinterpret_cast<uintptr_t>(p.scale) & (piece - 1)) == 0 &&
         (reinterpret_cast<uintptr_t>(p.zero) & (piece - 1)) == 0;
}

void launch_tile_group(const GemmParams* ps, int count, int storage, int shape, hipStream_t stream) {
  if (count < 1 || count > PG_GROUP) fail(ANIMA_E_INVALID_ARGUMENT, "tiled GEMM group holds 1 to 3 problems");
  GemmGroup g{};
  bool swin = true;
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i) {
    const GemmParams& p = ps[i];
    if (!pingpong_supported(p, storage)) fail(ANIMA_E_INVALID_SHAPE, "tiled GEMM: unsupported shape or alignment");
    if (p.K != ps[0].K) fail(ANIMA_E_INVALID_SHAPE, "tiled GEMM group: problems must share K");
    check_gemm_epilogue(p);
    if (p.epilogue == GEMM_QK_NORM && TG_TN[shape] % 128 != 0)
      fail(ANIMA_E_INVALID_ARGUMENT, "GEMM Q/K-norm epilogue needs whole heads in a tile");
    if (p.ksplit > 1 && (count != 1 || !p.part || shape != tile_shape(p) || p.ksplit != tile_ksplit(p)))
      fail(ANIMA_E_INVALID_ARGUMENT, "tiled GEMM: split K needs a single GEMM and its partial buffer");
    swin = swin && tile_swin(p, shape);
    g.p[i] = p;
    g.first_tile[i] = (int)tiles;
    g.vec[i] = gemm_vec_output(p);
    tiles += tile_count(p, shape) * (p.ksplit > 1 ? p.ksplit : 1);
    if (tiles > 0x7fffffff) fail(ANIMA_E_INVALID_SHAPE, "GEMM grid too large");
  }
  for (int i = count; i < PG_GROUP; ++i) g.first_tile[i] = (int)tiles;
  g.count = count;
  launch_tile_t<false>(g, storage, swin, shape, (unsigned)tiles, stream);
  if (ps[0].ksplit > 1) launch_splitk_epilogue(ps[0], stream);
}

bool gated_pair_supported(const GemmParams* ps, int storage) {
  return pingpong_supported(ps[0], storage) && pingpong_supported(ps[1], storage) && ps[0].M == ps[1].M &&
         ps[0].N == ps[1].N && ps[0].K == ps[1].K && ps[0].row_stride == ps[1].row_stride && ps[0].x == ps[1].x &&
         ps[0].N <= 0x7fffffff - 256;
}

// The ping-pong kernel from half a chip of its 128-row tiles (128 columns of each member);
// below it 32-row tiles where one round holds them, else 64-row ones
// (two rounds of 32-row tiles cost a layer of 77 tokens 63.7 us against 60.0, of 250 84.3
// against 73.9).  Gate, up and product against two launches, encoder layer, us: 77 tokens 63.7
// -> 59.7, 4 x 512 166.1 -> 161.7, 344 x 2 120.1 -> 117.4, with a cheaper SiLU than gated_silu8's,
// which is 0.2 us of the first and 1.9 of the second.
void launch_gated_pair(const GemmParams* ps, int storage, hipStream_t stream) {
  if (!gated_pair_supported(ps, storage)) fail(ANIMA_E_INVALID_SHAPE, "gated pair: unsupported shapes or alignment");
  if (ps[0].epilogue != GEMM_STORE || ps[0].ksplit > 1)
    fail(ANIMA_E_INVALID_ARGUMENT, "gated pair: no other output stage and no split K");
  const GemmParams& p = ps[0];
  auto count = [&](int tm, int tn) { return (int64_t)((p.M + tm - 1) / tm) * ((p.N + tn - 1) / tn); };
  if (count(128, 128) >= 128) {
    launch_pingpong_pair(ps, storage, stream);
    return;
  }
  const int shape = count(TG_TM[1], TG_TN[1] / 2) <= 256 ? 1 : 0;
  GemmGroup g{};
  g.p[0] = ps[0];
  g.p[1] = ps[1];
  g.vec[0] = gemm_vec_output(p);
  g.count = 1;
  launch_tile_t<true>(g, storage, tile_swin(ps[0], shape) && tile_swin(ps[1], shape), shape,
                      (unsigned)count(TG_TM[shape], TG_TN[shape] / 2), stream);
}

void launch_tiled(const GemmParams& p, int storage, hipStream_t stream) {
  if (tile_preferred(p, storage))
    launch_tile_group(&p, 1, storage, tile_shape(p), stream);
  else
    launch_pingpong(p, storage, stream);
}

}  // namespace anima
