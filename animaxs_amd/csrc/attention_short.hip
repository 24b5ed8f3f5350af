// Flash attention for short sequences (gfx950): a prompt's self-attention, the adapter.
//
// A few hundred tokens give the 256-row kernel one workgroup per head, most of whose rows
// and time go to its prologue and its two-phase pipeline's fill and drain, behind a launch
// that normalises K.  Here a launch is latency: everything a workgroup needs goes out in one
// round of loads, K is normalised where it is used, and no launch comes before.
//
//   * One workgroup is 32 query rows of one (batch, head): 8 waves, keys in chunks of 128.
//     32 rows and not more, because the number of workgroups is what such launches lack.
//   * Q and K rows are normalised (per-head RMSNorm, split-half RoPE) by eight lanes a row,
//     every row once per workgroup, and go to LDS as fp16 (the Q rows with scale * log2 e
//     folded in before their one rounding).  Workgroups of one head repeat the K rows' work,
//     which is why more workgroups keep the prologue launch (flash_short_preferred).
//   * S^T = K Q^T on v_mfma_f32_16x16x32_f16, wave w on keys 16 w .. 16 w + 15 of the chunk;
//     row maxima and fp32 row sums of the eight waves meet in LDS; fp16 P goes to LDS and
//     O^T += V^T P^T runs with the waves split over the columns of O (and over the two
//     16-query halves at head_dim 64), so no partial O is ever merged.
//   * V^T fragments come from the row-major V rows with ds_read_b64_tr_b16: the 16 lanes of
//     group g take keys 4 g .. 4 g + 3 and 16 + 4 g .. of each 32, sixteen consecutive LDS
//     rows per read, whose pitch (D + 16 halfs) puts every eight of them on distinct banks.
//   * The next chunk's rows load into registers while the current one is multiplied.
//
// What bounds it: the chain launch, loads, norm, three barriers, store; 77 tokens (causal,
// 16 heads on 8 KV heads, head_dim 128) take 7.3 us in place of 18.1 for the prologue and
// the 256-row kernel.  A chunk's 128 KB of RoPE table rows alone are 0.9 us of the CU's
// load path.  Steps on the way: norms through shuffles 8.2, table rows not as whole lines 10.2.
#include <algorithm>

#include "flash_common.hpp"

namespace anima {

constexpr int FS_WAVES = 8;
constexpr int FS_NT = 64 * FS_WAVES;
constexpr int FS_BK = 128;   // keys per chunk
static_assert(FS_BK == 16 * FS_WAVES, "one 16-key block per wave");

// f32_to_f16 without its volatile asm, so that independent rows interleave.
__device__ __forceinline__ half_t round_half(float v) {
  asm("" : "+v"(v));
  return (half_t)v;
}
// Sum over the 8 lanes 8 i .. 8 i + 7: quad swaps and the half-row mirror, no LDS round trips.
__device__ __forceinline__ float sum8_lanes(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));    // lanes 1 0 3 2
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));    // lanes 2 3 0 1
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));   // lane 7 - i of 8
  return v;
}
// Maximum and sum over lanes l % 16 + {0, 16, 32, 48}.
__device__ __forceinline__ float max_groups(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return xlane32_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float sum_groups(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return xlane32_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

template <int D>
__global__ __launch_bounds__(FS_NT, 1) __attribute__((amdgpu_waves_per_eu(2, 2)))
void flash_attention_short_kernel(FlashParams p) {
  constexpr int BQ = FLASH_SHORT_ROWS;
  constexpr int LPR = 8, RPP = 64 / LPR;           // lanes per normalised row, rows per wave and pass
  constexpr int NP = D / 2 / LPR, XP = D / 8 / LPR;   // pairs and 16-byte pieces per lane of a row
  constexpr int KP = FS_BK / (FS_WAVES * RPP);     // K passes per chunk
  constexpr int VCH = D / 8;                       // 16-byte pieces of a V row
  constexpr int VP = FS_BK * VCH / FS_NT;          // V pieces per thread and chunk
  constexpr int KROW = D + 8, VROW = D + 16, PROW = FS_BK + 8;
  constexpr int QH = D == 128 ? 2 : 1;             // 16-query halves per wave in P V
  __shared__ __attribute__((aligned(16))) half_t Qs[BQ * KROW], Ks[FS_BK * KROW], Vs[FS_BK * VROW], Ps[BQ * PROW];
  __shared__ __attribute__((aligned(16))) half_t NW[2 * D];   // norm weights of Q, then K
  __shared__ float red_max[FS_WAVES * BQ], red_sum[FS_WAVES * BQ];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j16 = lane & 15, g = lane >> 4;
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int qt = lb % p.q_tiles, head = lb / p.q_tiles % p.H, b = lb / p.q_tiles / p.H;
  const int kvh = head / p.group, q0 = qt * BQ;
  int kv_len = p.Sk;
  if (p.key_lengths_dev) {
    const int L = p.key_lengths_dev[b];
    kv_len = L < 1 ? 1 : (L > p.Sk ? p.Sk : L);
  } else if (p.use_host_lengths) {
    kv_len = p.host_lengths[b];
  }
  const int kend = p.causal ? min(kv_len, q0 + BQ) : kv_len;
  const int nchunk = (kend + FS_BK - 1) / FS_BK;

  // s_barrier after lgkmcnt(0): __syncthreads would also wait for the next chunk's loads.
  auto barrier = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  // Eight lanes a row.  The row's bytes and its table row load as whole 128-byte lines (lane
  // sub the pieces sub, sub + 8, ...: with eight consecutive blocks per lane every table load
  // would touch 64 lines, 8 times the cycles); the row goes to LDS as it is and the lane
  // takes the pairs (8 i + sub, D/2 + 8 i + sub) back, the columns of its table blocks.
  struct Row {
    u32x4 x[XP];
    floatx4 r[NP];
  };
  const int sub = lane % LPR, prow = lane / LPR;
  auto load_row = [&](const half_t* base, int nbytes, int64_t tok, int r, const float* rope, int64_t trow, Row& x)
      __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XP; ++i)
      x.x[i] = load16_bounded(base, nbytes, (uint32_t)r * (uint32_t)tok * 2u + 16u * (uint32_t)(sub + LPR * i));
    if (rope) {
      const floatx4* t = reinterpret_cast<const floatx4*>(rope + trow * (2 * D)) + 2 * sub;
#pragma unroll
      for (int i = 0; i < NP; ++i) x.r[i] = t[2 * LPR * (i >> 1) + (i & 1)];
    }
  };
  auto put_row = [&](const Row& x, half_t* dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XP; ++i) *reinterpret_cast<u32x4*>(dst + 8 * (sub + LPR * i)) = x.x[i];
  };
  // Norm and RoPE in fp32, times mul, one rounding, in LDS row dst, which other lanes of the
  // row put there (wave_lds_exchange between).  The lower table row is
  // [sin, cos] for K and taken as [-(-sin), cos] for Q, as the Q prologue of the other flash
  // kernels and the K prologue kernel read it.
  auto norm_row = [&](const Row& x, const half_t* w, const float* rope, bool q, float mul, half_t* dst)
      __attribute__((always_inline)) {
    if (!w && !rope && !q) return;
    float a[NP], c[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const half2v pa = *reinterpret_cast<const half2v*>(dst + 2 * LPR * (i >> 1) + 2 * sub);
      const half2v pc = *reinterpret_cast<const half2v*>(dst + D / 2 + 2 * LPR * (i >> 1) + 2 * sub);
      a[i] = (float)pa[i & 1];
      c[i] = (float)pc[i & 1];
    }
    if (w) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < NP; ++i) ss = fmaf(a[i], a[i], fmaf(c[i], c[i], ss));
      const float inv = rsqrtf(sum8_lanes(ss) / (float)D + p.eps);
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const half2v pa = *reinterpret_cast<const half2v*>(w + 2 * LPR * (i >> 1) + 2 * sub);
        const half2v pc = *reinterpret_cast<const half2v*>(w + D / 2 + 2 * LPR * (i >> 1) + 2 * sub);
        a[i] = a[i] * inv * (float)pa[i & 1];
        c[i] = c[i] * inv * (float)pc[i & 1];
      }
    }
    if (rope) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const floatx4 r = x.r[i];
        const float sn = q ? -r[1] : r[2];
        const float ra = r[0] * a[i] + r[1] * c[i];
        const float rc = sn * a[i] + r[0] * c[i];
        a[i] = ra;
        c[i] = rc;
      }
    }
#pragma unroll
    for (int i = 0; i < NP; i += 2) {
      *reinterpret_cast<half2v*>(dst + LPR * i + 2 * sub) = half2v{round_half(a[i] * mul), round_half(a[i + 1] * mul)};
      *reinterpret_cast<half2v*>(dst + D / 2 + LPR * i + 2 * sub) = half2v{round_half(c[i] * mul), round_half(c[i + 1] * mul)};
    }
  };

  // Chunk loads, through descriptors that end at the last key row in use: rows past it are
  // zeros (their scores are masked, and 0 * V must stay 0).
  const half_t* kb = p.k + (int64_t)b * p.k_batch + (int64_t)kvh * p.k_head;
  const half_t* vb = p.v + (int64_t)b * p.v_batch + (int64_t)kvh * p.v_head;
  Row kr[KP];
  u32x4 vr[VP];
  auto load_chunk = [&](int ch) __attribute__((always_inline)) {
    const int k0 = ch * FS_BK, rows = min(kend - k0, FS_BK);
    const half_t* kc = kb + (int64_t)k0 * p.k_tok;
    const half_t* vc = vb + (int64_t)k0 * p.v_tok;
    const int kn = (rows - 1) * (int)p.k_tok * 2 + 2 * D, vn = (rows - 1) * (int)p.v_tok * 2 + 2 * D;
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int r = RPP * (FS_WAVES * i + wave) + prow;
      load_row(kc, kn, p.k_tok, r, p.k_rope, min(k0 + r, kend - 1), kr[i]);
    }
#pragma unroll
    for (int i = 0; i < VP; ++i)
      vr[i] = load16_bounded(vc, vn, (uint32_t)(tid / VCH + FS_NT / VCH * i) * (uint32_t)p.v_tok * 2u +
                                         16u * (uint32_t)(tid % VCH));
  };
  // rows: key rows of the chunk in use.  K rows past them are never multiplied into a score
  // that is kept, V rows must read as zeros up to the next multiple of 32.
  auto put_chunk = [&](int rows) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < KP; ++i)
      if (RPP * (FS_WAVES * i + wave) < rows) put_row(kr[i], Ks + (RPP * (FS_WAVES * i + wave) + prow) * KROW);
#pragma unroll
    for (int i = 0; i < VP; ++i)
      *reinterpret_cast<u32x4*>(Vs + (tid / VCH + FS_NT / VCH * i) * VROW + 8 * (tid % VCH)) = vr[i];
  };
  auto norm_chunk = [&](int rows) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < KP; ++i)
      if (RPP * (FS_WAVES * i + wave) < rows) norm_row(kr[i], p.k_norm_w ? NW + D : nullptr, p.k_rope, false, 1.f,
                Ks + (RPP * (FS_WAVES * i + wave) + prow) * KROW);
  };

  {
    const bool q_wave = RPP * wave < BQ;
    Row qr{};
    if (q_wave) {
      const half_t* qb = p.q + (int64_t)b * p.q_batch + (int64_t)head * p.q_head + (int64_t)q0 * p.q_tok;
      const int rows = min(p.Sq - q0, BQ), r = RPP * wave + prow;
      load_row(qb, (rows - 1) * (int)p.q_tok * 2 + 2 * D, p.q_tok, r, p.rope, min(q0 + r, p.Sq - 1), qr);
    }
    // Wave 0 brings the norm weights to LDS, Q's through lanes 0 .. D/8 - 1 and K's behind.
    const int wl = lane % (D / 8);
    const half_t* nw = wave == 0 && lane < D / 4 ? (lane < D / 8 ? p.q_norm_w : p.k_norm_w) : nullptr;
    half8v nv{};
    if (nw) nv = *reinterpret_cast<const half8v*>(nw + 8 * wl);
    load_chunk(0);
    if (nw) *reinterpret_cast<half8v*>(NW + 8 * lane) = nv;
    barrier();
    half_t* const q_row = Qs + (RPP * wave + prow) * KROW;
    if (q_wave) put_row(qr, q_row);
    put_chunk(kend);
    wave_lds_exchange();
    if (q_wave) norm_row(qr, p.q_norm_w ? NW : nullptr, p.rope, true, p.scale_log2, q_row);
    norm_chunk(kend);
  }
  barrier();

  half8v qf[2][D / 32];   // query 16 h + j16, columns 32 s + 8 g .. + 7
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int s = 0; s < D / 32; ++s)
      qf[h][s] = *reinterpret_cast<const half8v*>(Qs + (16 * h + j16) * KROW + 32 * s + 8 * g);

  typedef __attribute__((address_space(3))) short4v lds_short4v;
  const int d0 = D == 128 ? 16 * wave : 16 * (wave & 3);   // columns of O of this wave
  const int hq = D == 128 ? 0 : wave >> 2;                 // its first query half
  floatx4 acc[QH];
#pragma unroll
  for (int h = 0; h < QH; ++h) acc[h] = floatx4{};
  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};   // of query 16 h + j16

  for (int ch = 0; ch < nchunk; ++ch) {
    const int k0 = ch * FS_BK, left = kend - k0;   // keys from this chunk's first to the last in use
    if (ch + 1 < nchunk) load_chunk(ch + 1);
    floatx4 S[2];
    if (16 * wave < left) {
      S[0] = S[1] = floatx4{};
#pragma unroll
      for (int s = 0; s < D / 32; ++s) {
        const half8v kf = *reinterpret_cast<const half8v*>(Ks + (16 * wave + j16) * KROW + 32 * s + 8 * g);
#pragma unroll
        for (int h = 0; h < 2; ++h) S[h] = mfma16(kf, qf[h][s], S[h]);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = k0 + 16 * wave + 4 * g + e;
          if (key >= kv_len || (p.causal && key > q0 + 16 * h + j16)) S[h][e] = -INFINITY;
        }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) S[h] = floatx4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float m = fmaxf(fmaxf(S[h][0], S[h][1]), fmaxf(S[h][2], S[h][3]));
      m = max_groups(m);
      if (g == 0) red_max[wave * BQ + 16 * h + j16] = m;
    }
    barrier();
    float alpha[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float m = m_run[h];
#pragma unroll
      for (int w = 0; w < FS_WAVES; ++w) m = fmaxf(m, red_max[w * BQ + 16 * h + j16]);
      const float ms = m == -INFINITY ? 0.f : m;
      alpha[h] = m_run[h] == -INFINITY ? 1.f : fast_exp2(m_run[h] - ms);
      m_run[h] = m;
      half4v ph;
      float ls = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pe = fast_exp2(S[h][e] - ms);
        ph[e] = (half_t)pe;
        ls += pe;
      }
      ls = sum_groups(ls);
      if (g == 0) red_sum[wave * BQ + 16 * h + j16] = ls;
      *reinterpret_cast<half4v*>(Ps + (16 * h + j16) * PROW + 16 * wave + 4 * g) = ph;
    }
    barrier();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float ls = 0.f;
#pragma unroll
      for (int w = 0; w < FS_WAVES; ++w) ls += red_sum[w * BQ + 16 * h + j16];
      l_run[h] = fmaf(l_run[h], alpha[h], ls);
    }
#pragma unroll
    for (int h = 0; h < QH; ++h) acc[h] *= D == 128 ? alpha[h] : (hq ? alpha[1] : alpha[0]);
    lds_short4v* vs = (lds_short4v*)(Vs + (4 * g + (j16 >> 2)) * VROW + d0 + 4 * (j16 & 3));
    for (int ks = 0; ks < (min(left, FS_BK) + 31) / 32; ++ks) {
      const half4v lo = __builtin_bit_cast(half4v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(vs + ks * 32 * VROW / 4));
      const half4v hi =
          __builtin_bit_cast(half4v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(vs + (ks * 32 + 16) * VROW / 4));
      const half8v vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
      for (int h = 0; h < QH; ++h) {
        const half_t* pr = Ps + (16 * (hq + h) + j16) * PROW + 32 * ks + 4 * g;
        const half4v p0 = *reinterpret_cast<const half4v*>(pr), p1 = *reinterpret_cast<const half4v*>(pr + 16);
        acc[h] = mfma16(vf, half8v{p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]}, acc[h]);
      }
    }
    if (ch + 1 < nchunk) {
      barrier();   // every read of this chunk's K and V rows done
      put_chunk(left - FS_BK);
      wave_lds_exchange();
      norm_chunk(left - FS_BK);
      barrier();
    }
  }

#pragma unroll
  for (int h = 0; h < QH; ++h) {
    const int qi = q0 + 16 * (hq + h) + j16;
    const float l = D == 128 ? l_run[h] : (hq ? l_run[1] : l_run[0]);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const half4v o = {(half_t)(acc[h][0] * inv), (half_t)(acc[h][1] * inv), (half_t)(acc[h][2] * inv),
                      (half_t)(acc[h][3] * inv)};
    if (qi < p.Sq)
      *reinterpret_cast<half4v*>(p.o + (int64_t)b * p.o_batch + (int64_t)head * p.o_head + (int64_t)qi * p.o_tok + d0 +
                                 4 * g) = o;
  }
}

// One round of workgroups (they fill a CU's LDS), each paying about 2.5 us and 4.5 us per
// chunk, against 16 to 27 us of the K prologue and the 256-row kernel; two rounds only of
// one chunk.  us, this / those, launches back to back in a graph:
//   causal, 16 heads on 8, norm and RoPE: 77 tokens 7.3 / 18.1, 256 12.2 / 22.1, 512 (256
//   workgroups) 21.0 / 26.6, 4 x 128 8.3 / 18.6, 4 x 256 (512) 23.1 / 23.1, 2 x 512 37 / 27;
//   head_dim 64: 77 x 64 5.4 / 11.0, 512 x 512 (256) 16.0 / 18.8; no RoPE: 512 x 512 (256)
//   16.8 / 22.2, 1024 x 128 (512) 12.6 / 13.9, 1024 x 512 (512) 29 / 21, 4096 x 64 (2048) 38 / 18.
bool flash_short_preferred(const FlashParams& p, int D, int batch) {
  if (D != 64 && D != 128) return false;
  if (p.Sq < 1 || p.Sk < 1 || batch < 1) return false;
  // Rows of a chunk and of a query tile are addressed with 32-bit byte offsets.
  if (FS_BK * std::max(p.q_tok, std::max(p.k_tok, p.v_tok)) * (int64_t)sizeof(half_t) >= ((int64_t)1 << 31)) return false;
  const int64_t blocks = (int64_t)((p.Sq + FLASH_SHORT_ROWS - 1) / FLASH_SHORT_ROWS) * p.H * batch;
  return p.Sk <= 4 * FS_BK && (blocks <= 256 || (blocks <= 512 && p.Sk <= FS_BK));
}

void launch_flash_short(FlashParams p, int D, int batch, hipStream_t stream) {
  if (!flash_short_preferred(p, D, batch)) fail(ANIMA_E_INVALID_SHAPE, "short flash attention: unsupported shape");
  p.nbatch = batch;
  p.kv_splits = 0;
  p.q_tiles = (p.Sq + FLASH_SHORT_ROWS - 1) / FLASH_SHORT_ROWS;
  const dim3 grid((unsigned)((int64_t)p.q_tiles * p.H * batch));
  if (D == 128)
    hipLaunchKernelGGL(flash_attention_short_kernel<128>, grid, dim3(FS_NT), 0, stream, p);
  else
    hipLaunchKernelGGL(flash_attention_short_kernel<64>, grid, dim3(FS_NT), 0, stream, p);
  ANIMA_HIP(hipGetLastError());
}

}  // namespace anima
