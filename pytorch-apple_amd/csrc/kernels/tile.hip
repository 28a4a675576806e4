// MFMA GEMM on wide workgroups: out[m, n] = epi(sum_k x[m, k] w[n, k]) for activations [M, K] and
// weights [N, K] as the model stores them, K % 64 == 0. One workgroup of WR x WC waves (8, 10 or 12)
// per BM x BN output tile, and per CU (two with 64 x 64 tiles).
//
// What bounds a GEMM of these shapes (M = 128 .. 4096 against 1536- to 151936-row weights) is how
// many operand bytes a CU has in flight and takes in per MFMA, not the MFMA rate itself. So:
//   * the LDS of the whole CU (up to 160 KB) holds one workgroup's ring of ST stages of 64 of K,
//     filled by global_load_lds_dwordx4 (128-byte rows, whole cache lines; 64-byte rows, twice as
//     many stages of half the depth, were 10-15% slower: each line is then fetched twice);
//   * tiles are as large as the shape allows while the grid still fills the 256 CUs in whole
//     rounds (the host's tile_plan): 256 x 144 of both SiLU weights is 252 workgroups at M = 1000,
//     192 x 144 is 252 at 768 (45 us; 128 x 144 48), 128 x 80 224 at 256 (24 us; 128 x 144 33);
//   * 64 x 64 tiles take half the LDS (rings of 4 stages, 3 with two weights), so that two workgroups
//     share a CU and 257 to 512 of them are one round: o_proj (N = K = 1536) at M = 1025 14.2 us on
//     128 x 96 tiles, 18.0 on 64 x 64 with the whole LDS, 12.0 now; no slower where one has a CU to itself;
//   * each operand address is a scalar base plus a 32-bit lane offset (one SALU add per load);
//   * 12 waves (three per SIMD) on the tiles of width 3 x 48, 10 on those of 5 x 16, 8 on the others; the
//     16-byte chunks of a row sit in slot c ^ ((row >> 1) & 7), which the 16 x 4 fragment reads of
//     v_mfma_f32_16x16x32 cross without a bank conflict (237 bytes per clock and CU measured; 63 with
//     the chunks in order).
// The MFMA computes the transposed tile (weights as operand A), so that a lane holds 4 consecutive
// columns of one row: 8-byte LDS writes in the epilogue, 16-byte rows out of it, and float4 partials.
//
// Measured on MI355X (bf16, calls of one launch or of one and its reduce, as many copies of the weights as
// come from HBM), against the 4-wave kernels of gemm.hip that ran these before: gate/up with SiLU (N = 8960,
// K = 1536) at M = 192 / 512 / 1000 / 2000 27 / 46 / 75 / 133 -> 23 / 35 / 53 / 103 us; lm_head
// (N = 151936, K = 1536) at M = 513 373 -> 321 us; down_proj (N = 1536, K = 8960) at M = 512 / 1000 / 2000
// 35 / 75 / 99 -> 28 / 42 / 68 us. The slowest rounds left: gate/up at M = 1090 .. 1152, 378 tiles of 192 x 144
// in two rounds, is where the 4-wave kernels' 846 tiles were (83-84 us both). A steady K step of
// 256 x 256 takes 1.56 us (1,376 TFLOP/s over 256 CUs); a launch spends the rest (8-11 us) on its first
// stage's latency and its epilogue.
//
// Epilogues (fp32 accumulator, ATen's rounding points), rows past M and columns past N clamped when
// read and not stored:
//   BIAS  out = round(acc + b)
//   RESID out = round(r + round(acc + b))
//   SILU  out = round(round(silu(round(acc_g + b_g))) * round(acc_u + b_u))   (NW = 2)
//   CONV  round(acc + b), batch norm, residual and ReLU as gemm.hip's conv epilogue
// ksplit > 1 (NW = 1): grid.z workgroups take kchunk of K each and store fp32 partials [z, M, N]; a
// k_gemm_reduce_* kernel (gemm.hip) sums them in order and applies the epilogue.
// CV: x rows are gathered from an NHWC image, one tap and 64 channels per stage (K = (kh, kw, ci),
// cCin % 64 == 0), taps outside it from a.zero. ResNet-50's 3 x 3 convs at batch 32 with 128 / 256 / 512
// channels: 23.0 / 26.8 / 26.4 -> 20.3 / 24.1 / 19.6 us against the 4-wave kernels; they take in 45-60 GB/s
// per CU from the L2, which bounds them.
// GRP: output columns [0, n1), [n1, n2), [n2, N) come from three weights and biases (n1, n2
// multiples of BN), e.g. q | k | v of one activation.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 tg_bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 tg_f16x8;
typedef __attribute__((ext_vector_type(4))) float tg_f32x4;

template <int DT>
__device__ __forceinline__ tg_f32x4 tg_mfma(const uint4 a, const uint4 b, tg_f32x4 c) {
  if constexpr (DT == HS_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(tg_bf16x8, a), __builtin_bit_cast(tg_bf16x8, b),
                                                   c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(tg_f16x8, a), __builtin_bit_cast(tg_f16x8, b),
                                                  c, 0, 0, 0);
}

// the same from a 64-bit address per lane
__device__ __forceinline__ void tg_dma16v(const void* p, unsigned lds) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(p), "s"(lds) : "memory", "m0");
}

template <int DT, int EPI, int NW, int BM, int BN, int WR, int WC, int ST, bool GRP = false, bool CV = false>
__device__ __forceinline__ void tile_body(const GemmArgs& a) {
  constexpr int NWV = WR * WC, NTH = 64 * NWV, BNT = BN * NW;
  constexpr int WM = BM / WR, WN = BN / WC, TI = WM / 16, TJ = WN / 16;   // wave tile, in 16 x 16 MFMA tiles
  static_assert(WM % 16 == 0 && WN % 16 == 0 && BM % 16 == 0 && BN % 16 == 0, "wave tile");
  constexpr int RB = 128, ROWS = BM + BNT, SB = ROWS * RB;   // bytes per staged row and per stage
  constexpr int INS = ROWS / 8, NI = (INS + NWV - 1) / NWV;  // loads (8 rows each) per stage, per wave and stage
  constexpr int TLD = BN + 8;                                // epilogue tile row (elements)
  static_assert(ST * SB >= BM * TLD * 2 || ST == 2, "epilogue tile");
  constexpr int LDSB = ST * SB > BM * TLD * 2 ? ST * SB : BM * TLD * 2;
  __shared__ __attribute__((aligned(16))) char Ls[LDSB];
  __shared__ __attribute__((aligned(16))) float Fb[(EPI == GE_CONV ? 3 : NW) * BN];   // bias per weight; conv: bias, al, be
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WC, wc = wave % WC;
  const TilePos at = tile_order(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), gridDim.x, gridDim.y,
                                gridDim.z, (unsigned)max(a.gn, 1));
  const unsigned kz = at.kz;
  const int m_base = (int)at.row * BM, n_base = (int)at.col * BN;
  const int M = (int)a.M, N = a.N;
  const int kbeg = (int)kz * a.kchunk, nsteps = min(a.kchunk, a.K - kbeg) / 64;
  int g_lo = 0, g_hi = N;   // GRP: the columns of this tile's group
  const void *W0 = a.w, *B0 = a.bias;
  if constexpr (GRP) {
    const int g = (n_base >= a.n1) + (n_base >= a.n2);
    g_lo = g == 0 ? 0 : (g == 1 ? a.n1 : a.n2);
    g_hi = g == 0 ? a.n1 : (g == 1 ? a.n2 : N);
    W0 = g == 0 ? a.w : (g == 1 ? a.w2 : a.w3);
    B0 = g == 0 ? a.bias : (g == 1 ? a.bias2 : a.bias3);
  }
  // staging: load i of this wave fills rows 8q .. 8q + 7 of a stage (x rows, then each weight's); lane ->
  // row 8q + lane / 8, slot lane % 8. The loads past INS repeat the last one (same bytes, same place)
  unsigned voff[NI];
  const char* gb[NI];
  unsigned ldst[NI];
  // CV: the row's image, its pixel's first input row and column (padding: < 0), and the lane's chunk
  int gim[CV ? NI : 1], ghi[CV ? NI : 1], gwi[CV ? NI : 1];
  unsigned gch[CV ? NI : 1];
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void*)&Ls[0];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int q = min(wave + i * NWV, INS - 1), r = 8 * q + (lane >> 3);
    const unsigned chunk = (unsigned)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    ldst[i] = lds0 + (unsigned)q * 1024u;
    if (CV && 8 * q < BM) {   // lane pointer offsets are made per step (the taps)
      const int HoWo = a.cHo * a.cWo, m = min(m_base + r, M - 1), n = m / HoWo, p = m - n * HoWo, ho = p / a.cWo;
      ghi[i] = ho * a.csh - a.cph;
      gwi[i] = (p - ho * a.cWo) * a.csw - a.cpw;
      gim[i] = n;
      gch[i] = chunk;
      voff[i] = 0;
      gb[i] = (const char*)a.x;
    } else if (8 * q < BM) {
      gb[i] = (const char*)a.x + ((long long)m_base * a.ldx + kbeg) * 2;
      voff[i] = (unsigned)(min(m_base + r, M - 1) - m_base) * (unsigned)(a.ldx * 2) + chunk;
    } else {
      const int u = (8 * q - BM) / BN, rr = r - BM - u * BN;
      gb[i] = (const char*)(u == 0 ? W0 : a.w2) + ((long long)(n_base - g_lo) * a.ldw + kbeg) * 2;
      voff[i] = (unsigned)(min(n_base + rr, g_hi - 1) - n_base) * (unsigned)(a.ldw * 2) + chunk;
    }
  }
  // the tile's bias columns, loaded ahead of the operands, kept in a register until the epilogue
  float bv[NW];
#pragma unroll
  for (int u = 0; u < NW; ++u) bv[u] = 0.f;
  if (tid < BN && a.ksplit == 1) {
    const int n = min(n_base + tid, g_hi - 1) - g_lo;
    if (a.flags & 1) bv[0] = gm_ld<DT>(B0, n);
    if constexpr (NW == 2)
      if (a.flags & 2) bv[1] = gm_ld<DT>(a.bias2, n);
  }
  int ib = 0, is = 0;   // the next stage to load, and its buffer
  int c0 = 0, kh = 0, kw = 0;   // CV: its channels and tap (64 channels of one tap per stage)
  if constexpr (CV) {
    const int tap = kbeg / a.cCin;
    c0 = kbeg - tap * a.cCin;
    kh = tap / a.cKW;
    kw = tap - kh * a.cKW;
  }
  auto issue = [&]() {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const unsigned dst = ldst[i] + (unsigned)(ib * SB);
      if (CV && 8 * min(wave + i * NWV, INS - 1) < BM) {   // uniform; taps outside the image read a.zero
        const int hi = ghi[i] + kh, wi = gwi[i] + kw;
        const bool ok = (unsigned)hi < (unsigned)a.cH && (unsigned)wi < (unsigned)a.cW;
        const long long e = (((long long)gim[i] * a.cH + hi) * a.cW + wi) * a.cCin + c0;
        tg_dma16v(ok ? (const char*)a.x + 2 * e + gch[i] : (const char*)a.zero, dst);
      } else {
        gm_dma16s(gb[i] + (long long)is * RB, voff[i], dst);
      }
    }
    if constexpr (CV) {
      c0 += 64;
      if (c0 == a.cCin) {
        c0 = 0;
        if (++kw == a.cKW) {
          kw = 0;
          ++kh;
        }
      }
    }
    ++is;
    ib = ib + 1 == ST ? 0 : ib + 1;
  };
  tg_f32x4 acc[NW][TJ][TI];
#pragma unroll
  for (int u = 0; u < NW; ++u)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int i = 0; i < TI; ++i) acc[u][j][i] = tg_f32x4{0.f, 0.f, 0.f, 0.f};
  // fragments: lane -> row lane % 16, chunk lane / 16 (+ 4 for the second half of a stage); a
  // multiple of 16 rows leaves the slot permutation unchanged, so it is one offset per lane
  const int fr = lane & 15, fc = lane >> 4;
  const int fo[2] = {fr * RB + ((fc ^ ((fr >> 1) & 7)) * 16), fr * RB + (((fc + 4) ^ ((fr >> 1) & 7)) * 16)};
#pragma unroll
  for (int st = 0; st < ST - 1; ++st)
    if (st < nsteps) issue();
  int cb = 0;
  for (int s = 0; s < nsteps; ++s) {
    // stage s has landed when at most the stages issued after it are outstanding
    gm_vmcnt_after<NI, ST - 2>(min(nsteps - 1 - s, ST - 2));
    __syncthreads();                      // every wave's part of stage s is there, and every wave is done with s - 1
    if (s + ST - 1 < nsteps) issue();     // into the buffer stage s - 1 used
    const char* xs = Ls + cb * SB + wr * WM * RB;
    const char* ws = Ls + cb * SB + (BM + wc * WN) * RB;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      uint4 fx[TI], fw[NW][TJ];
#pragma unroll
      for (int i = 0; i < TI; ++i) fx[i] = *(const uint4*)(xs + fo[k] + i * 16 * RB);
#pragma unroll
      for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int j = 0; j < TJ; ++j) fw[u][j] = *(const uint4*)(ws + fo[k] + (u * BN + j * 16) * RB);
      __builtin_amdgcn_s_setprio(1);   // a wave with its fragments goes ahead of one still reading (1-3%)
#pragma unroll
      for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
          for (int i = 0; i < TI; ++i) acc[u][j][i] = tg_mfma<DT>(fw[u][j], fx[i], acc[u][j][i]);
      __builtin_amdgcn_s_setprio(0);
    }
    cb = cb + 1 == ST ? 0 : cb + 1;
  }

  // this lane's part of a 16 x 16 tile: row fr, columns cn .. cn + 3
  const int cn = 4 * fc;
  if (NW == 1 && a.ksplit > 1) {
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const int m = m_base + wr * WM + i * 16 + fr;
      if (m >= M) continue;
      float* p = a.part + ((long long)kz * a.M + m) * N;
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int n = n_base + wc * WN + j * 16 + cn;
        if ((N & 3) == 0) {
          if (n < N) *(tg_f32x4*)(p + n) = acc[0][j][i];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) p[n + e] = acc[0][j][i][e];
        }
      }
    }
    return;
  }
  // epilogue: the rounded tile through LDS (round(acc + bias) is the first rounding point, so a
  // 16-bit value holds it), then 16-byte row chunks; the residual's chunks are loaded first
  uint16_t* T = (uint16_t*)Ls;
  constexpr int CPR = BN / 8, CH = (BM * CPR + NTH - 1) / NTH;   // chunks per row, chunks per thread
  const bool vec = (N & 7) == 0 && (a.ldo & 7) == 0 && ((size_t)a.out & 15) == 0 &&
                   (!(EPI == GE_RESID || (EPI == GE_CONV && (a.flags & 4))) || ((a.ldr & 7) == 0 && ((size_t)a.resid & 15) == 0));
  constexpr bool HAS_R = EPI == GE_RESID || EPI == GE_CONV;
  uint4 rv[HAS_R ? CH : 1];
  if constexpr (HAS_R) {
    if (vec && (EPI == GE_RESID || (a.flags & 4))) {
#pragma unroll
      for (int k = 0; k < CH; ++k) {
        const int idx = min(tid + NTH * k, BM * CPR - 1), r = idx / CPR, q = idx - r * CPR;
        rv[k] = *(const uint4*)((const uint16_t*)a.resid + (long long)min(m_base + r, M - 1) * a.ldr +
                                min(n_base + q * 8, N - 8));
      }
    }
  }
  if (tid < BN) {
#pragma unroll
    for (int u = 0; u < NW; ++u) Fb[u * BN + tid] = bv[u];
    if constexpr (EPI == GE_CONV) {
      float al = 1.f, be = 0.f;
      if (a.flags & 2) gm_bn_factors<DT>(a, min(n_base + tid, N - 1), al, be);
      Fb[BN + tid] = al;
      Fb[2 * BN + tid] = be;
    }
  }
  __syncthreads();   // every wave is done with the operand buffers
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int nl = wc * WN + j * 16 + cn;
    const tg_f32x4 b0 = *(const tg_f32x4*)&Fb[nl];
    tg_f32x4 b1{};
    if constexpr (NW == 2) b1 = *(const tg_f32x4*)&Fb[BN + nl];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const tg_f32x4 v = acc[0][j][i] + b0;
      uint2 h = make_uint2(gm_pack2<DT>(v[0], v[1]), gm_pack2<DT>(v[2], v[3]));
      if constexpr (EPI == GE_SILU) {
        const tg_f32x4 w = acc[NW - 1][j][i] + b1;
        const uint2 up = make_uint2(gm_pack2<DT>(w[0], w[1]), gm_pack2<DT>(w[2], w[3]));
        const uint2 sg = make_uint2(gm_pack2<DT>(gm_silu(gm_lo<DT>(h.x)), gm_silu(gm_hi<DT>(h.x))),
                                    gm_pack2<DT>(gm_silu(gm_lo<DT>(h.y)), gm_silu(gm_hi<DT>(h.y))));
        h = make_uint2(gm_pack2<DT>(gm_lo<DT>(sg.x) * gm_lo<DT>(up.x), gm_hi<DT>(sg.x) * gm_hi<DT>(up.x)),
                       gm_pack2<DT>(gm_lo<DT>(sg.y) * gm_lo<DT>(up.y), gm_hi<DT>(sg.y) * gm_hi<DT>(up.y)));
      }
      *(uint2*)&T[(wr * WM + i * 16 + fr) * TLD + nl] = h;
    }
  }
  __syncthreads();
  uint16_t* OUT = (uint16_t*)a.out;
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    const int idx = tid + NTH * k, r = idx / CPR, q = idx - r * CPR;
    const int m = m_base + r, n0 = n_base + q * 8;
    if (idx >= BM * CPR || m >= M || n0 >= N) continue;
    const uint4 tv = *(const uint4*)&T[r * TLD + q * 8];
    uint32_t tw[4] = {tv.x, tv.y, tv.z, tv.w};
    if (vec) {
      if constexpr (EPI == GE_RESID) {
        const uint32_t rw[4] = {rv[k].x, rv[k].y, rv[k].z, rv[k].w};
#pragma unroll
        for (int c = 0; c < 4; ++c)
          tw[c] = gm_pack2<DT>(gm_lo<DT>(rw[c]) + gm_lo<DT>(tw[c]), gm_hi<DT>(rw[c]) + gm_hi<DT>(tw[c]));
      }
      if constexpr (EPI == GE_CONV) {
        const uint32_t rw[4] = {rv[k].x, rv[k].y, rv[k].z, rv[k].w};
        const float* f = &Fb[BN + q * 8];
#pragma unroll
        for (int c = 0; c < 4; ++c)
          tw[c] = gm_pack2<DT>(gm_conv_tail_f<DT>(a, gm_lo<DT>(tw[c]), f[2 * c], f[BN + 2 * c], gm_lo<DT>(rw[c])),
                               gm_conv_tail_f<DT>(a, gm_hi<DT>(tw[c]), f[2 * c + 1], f[BN + 2 * c + 1], gm_hi<DT>(rw[c])));
      }
      *(uint4*)(OUT + (long long)m * a.ldo + n0) = make_uint4(tw[0], tw[1], tw[2], tw[3]);
    } else {   // rows that are no multiple of 16 bytes, or unaligned: one value at a time
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (n0 + e >= N) continue;
        float v = (e & 1) ? gm_hi<DT>(tw[e >> 1]) : gm_lo<DT>(tw[e >> 1]);
        if constexpr (EPI == GE_RESID) v = gm_ld<DT>(a.resid, (long long)m * a.ldr + n0 + e) + v;
        if constexpr (EPI == GE_CONV)
          v = gm_conv_tail_f<DT>(a, v, Fb[BN + q * 8 + e], Fb[2 * BN + q * 8 + e],
                                 (a.flags & 4) ? gm_ld<DT>(a.resid, (long long)m * a.ldr + n0 + e) : 0.f);
        OUT[(long long)m * a.ldo + n0 + e] = gm_pack<DT>(v);
      }
    }
  }
}

// k_gemm_<dtype>_<epilogue>_m<BM>n<BN>_w<waves>_k64d (BN columns per weight); the grouped kernels keep
// the names of the tiles they are
#define TILE_KERNEL(NAME, DT, EPI, NW, BM, BN, WR, WC, ST)                                        \
  extern "C" __global__ void __launch_bounds__(64 * WR * WC) NAME(const GemmArgs a) {             \
    tile_body<DT, EPI, NW, BM, BN, WR, WC, ST>(a);                                                \
  }
#define TILE_GRP(NAME, DT, BM, BN, WR, WC, ST)                                                    \
  extern "C" __global__ void __launch_bounds__(64 * WR * WC) NAME(const GemmArgs a) {             \
    tile_body<DT, GE_BIAS, 1, BM, BN, WR, WC, ST, true>(a);                                       \
  }
#define TILE_BIAS(DTN, DT)                                                                        \
  TILE_KERNEL(k_gemm_##DTN##_bias_m64n64_w8_k64d, DT, GE_BIAS, 1, 64, 64, 4, 2, 4)                \
  TILE_KERNEL(k_gemm_##DTN##_bias_m64n96_w8_k64d, DT, GE_BIAS, 1, 64, 96, 4, 2, 6)                \
  TILE_KERNEL(k_gemm_##DTN##_bias_m128n96_w8_k64d, DT, GE_BIAS, 1, 128, 96, 4, 2, 5)              \
  TILE_KERNEL(k_gemm_##DTN##_bias_m128n128_w8_k64d, DT, GE_BIAS, 1, 128, 128, 2, 4, 4)            \
  TILE_KERNEL(k_gemm_##DTN##_bias_m256n128_w8_k64d, DT, GE_BIAS, 1, 256, 128, 4, 2, 3)            \
  TILE_KERNEL(k_gemm_##DTN##_bias_m256n256_w8_k64d, DT, GE_BIAS, 1, 256, 256, 2, 4, 2)
TILE_BIAS(bf16, HS_BF16)
TILE_BIAS(f16, HS_F16)
TILE_KERNEL(k_gemm_bf16_resid_m64n64_w8_k64d, HS_BF16, GE_RESID, 1, 64, 64, 4, 2, 4)
TILE_KERNEL(k_gemm_bf16_resid_m64n96_w8_k64d, HS_BF16, GE_RESID, 1, 64, 96, 4, 2, 6)
TILE_KERNEL(k_gemm_bf16_resid_m128n96_w8_k64d, HS_BF16, GE_RESID, 1, 128, 96, 4, 2, 5)
TILE_KERNEL(k_gemm_bf16_resid_m128n128_w8_k64d, HS_BF16, GE_RESID, 1, 128, 128, 2, 4, 4)
TILE_KERNEL(k_gemm_bf16_resid_m256n128_w8_k64d, HS_BF16, GE_RESID, 1, 256, 128, 4, 2, 3)
TILE_KERNEL(k_gemm_bf16_resid_m256n256_w8_k64d, HS_BF16, GE_RESID, 1, 256, 256, 2, 4, 2)
TILE_KERNEL(k_gemm_bf16_silu_m64n64_w8_k64d, HS_BF16, GE_SILU, 2, 64, 64, 2, 4, 3)
TILE_KERNEL(k_gemm_bf16_silu_m128n80_w10_k64d, HS_BF16, GE_SILU, 2, 128, 80, 2, 5, 4)
TILE_KERNEL(k_gemm_bf16_silu_m128n144_w12_k64d, HS_BF16, GE_SILU, 2, 128, 144, 4, 3, 3)
TILE_KERNEL(k_gemm_bf16_silu_m192n144_w12_k64d, HS_BF16, GE_SILU, 2, 192, 144, 4, 3, 2)
TILE_KERNEL(k_gemm_bf16_silu_m256n144_w12_k64d, HS_BF16, GE_SILU, 2, 256, 144, 4, 3, 2)
TILE_GRP(k_gemm_bf16_grp_m64n64_k64d, HS_BF16, 64, 64, 4, 2, 4)
TILE_GRP(k_gemm_bf16_grp_m64n128_k64d, HS_BF16, 64, 128, 2, 4, 6)
TILE_GRP(k_gemm_bf16_grp_m128n128_k64d, HS_BF16, 128, 128, 2, 4, 4)
// convolutions on channels-last activations with K > 1024 over many tiles (conv epilogue of gemm.hip): _conv reads the
// [pixels, Cin] rows of the image (1 x 1, stride 1), _convg gathers 64 channels of one tap per stage
#define TILE_CONV(DTN, DT, BM, BN, WR, WC, ST)                                                                          \
  TILE_KERNEL(k_gemm_##DTN##_conv_m##BM##n##BN##_w8_k64d, DT, GE_CONV, 1, BM, BN, WR, WC, ST)                           \
  extern "C" __global__ void __launch_bounds__(512) k_gemm_##DTN##_convg_m##BM##n##BN##_w8_k64d(const GemmArgs a) {     \
    tile_body<DT, GE_CONV, 1, BM, BN, WR, WC, ST, false, true>(a);                                                      \
  }
TILE_CONV(f16, HS_F16, 64, 64, 4, 2, 4)
TILE_CONV(f16, HS_F16, 64, 128, 2, 4, 6)
TILE_CONV(f16, HS_F16, 128, 128, 2, 4, 4)
TILE_CONV(bf16, HS_BF16, 64, 64, 4, 2, 4)
TILE_CONV(bf16, HS_BF16, 64, 128, 2, 4, 6)
TILE_CONV(bf16, HS_BF16, 128, 128, 2, 4, 4)
