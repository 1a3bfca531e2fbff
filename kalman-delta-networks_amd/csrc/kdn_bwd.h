// Chunk-parallel backward of the KDN memory scan on bf16x3 MFMA (one kernel per chunk).
//
// Per chunk of C = 64 tokens (h = state entering the chunk, dh = gradient of the state leaving it,
// delta = A X of the forward pass with X = V - Kg h and A = (I + N)^{-1}, dX = A^T d delta of the reverse pass):
//   products                 dV = dX,  dQg = dO h^T,  dKg = -dX h^T,  dKf = delta dh^T,
//                            dM = lower(dO delta^T),  dgl_i = 2^{G_last,i} sum_v h_iv dh_iv,
//                            dN = -strict_lower(A^T (d delta X^T) A^T) = -strict_lower(dX delta^T)
//   gradients                with block anchors m (below): e = 2^{G_c - m}, Lk = k e, Lq = q e,
//                            R = kappa / e, eg = 2^{G_c}, f = 2^{G_last - G_c}
//                            dLk = dN R,  dLq = scale dM R,  dR = dN^T Lk + scale dM^T Lq
//                            dk = dLk e + dKg eg,  dq = dLq e + scale dQg eg,  dkappa = dR / e + dKf f
//                            dg = Lk dLk + Lq dLq - R dR + k eg dKg + scale q eg dQg - kappa f dKf
//                            dg[last row] += sum_c kappa f dKf + dgl;  iso: dbeta = sum_i dkappa k,
//                            dk += beta dkappa
// dg is in natural-log coordinates.  Each output row block tl uses the forward's anchor of that block,
// m = (G_{16tl} + G_{16tl+15}) / 2 per channel (rows clamped to the chunk), for every factor it
// contracts with, so each factor is <= 2^{span/2} on the diagonal block and <= 1 off it; the anchor
// terms cancel exactly (N and M do not depend on the anchors) and are omitted.
//
// Bound by the CU's load path: per token-head (d = 128) h and dh 512 B each isotropic (1,024 diagonal), delta and
// dX 512 each, dO, q, k 256 each and G 512.  A task's LDS (~140 KB) leaves one workgroup per CU, so nothing else
// hides its loads.  Forming U, W, the solves' transposes and dX here as well (A^T, U, W read: 1,280 B more) it took
// 609 us isotropic / 617 us diagonal at B4 T4096 H18, against 446 / 480.
#pragma once
#include "kdn_common.h"
#include "kdn_intra.h"
#include "kdn_state.h"

namespace kdn_bwd {

using kdn_intra::ld8;
using kdn_intra::split8;
using kdn_intra::unpack8;
using kdn_state::C;
using kdn_state::mfma;
using kdn_state::mma3;
using kdn_state::zero4;
using kdn_state::afrag;
using kdn_state::TILE;

// a*b where each operand is split (hi + lo, AL / BL) or exact in bf16 (hi only): hi*hi, hi*lo, lo*hi
// in the order of mma3, dropping the terms of an absent lo half.
template <bool AL, bool BL>
__device__ __forceinline__ f32x4 mmx(uint4 ah, uint4 al, uint4 bh, uint4 bl, f32x4 c) {
  c = mfma(ah, bh, c);
  if constexpr (BL) c = mfma(ah, bl, c);
  if constexpr (AL) c = mfma(al, bh, c);
  return c;
}
// a staged fragment; without LO the tensor was staged as its bf16 values alone (lo = 0)
template <bool LO>
__device__ __forceinline__ void afragx(const bf16_t* buf, int tile, int lane, uint4& hi, uint4& lo) {
  hi = *reinterpret_cast<const uint4*>(buf + tile * TILE + lane * 8);
  if constexpr (LO) lo = *reinterpret_cast<const uint4*>(buf + tile * TILE + 512 + lane * 8);
  else lo = uint4{0u, 0u, 0u, 0u};
}

// Lower 16x16 tiles (I, J), J <= I, 2-bit packed: 0:(0,0) 1:(1,1) 2:(2,2) 3:(3,3) 4:(1,0)
// 5:(2,1) 6:(3,2) 7:(2,0) 8:(3,1) 9:(3,0); upper tiles (0,1) (0,2) (0,3) (1,2) (1,3) (2,3).
__device__ __forceinline__ void lower_tile(int t, int& I, int& J) {
  I = (0xfb9e4u >> (2 * t)) & 3;
  J = (0x124e4u >> (2 * t)) & 3;
}
__device__ __forceinline__ void upper_tile(int t, int& I, int& J) {
  I = (0x940u >> (2 * t)) & 3;
  J = (0xfb9u >> (2 * t)) & 3;
}

// ---------------------------------------------------------------------------------------------
// The whole chunk-parallel backward of one chunk in one kernel: the products with h, dh and dX and the
// gradients.  dQg, dKf, dM, dKg, dN and the g_last dots never go to HBM: each is produced in the register or
// LDS layout its consumer takes.
// One chunk-head task of the order task = (NT - 1 - n) * B*H + bh (last chunks first, the order in
// which the reverse state pass finishes them); block 512 (8 waves), one workgroup per CU (LDS 141 KB).
//  * Staging.  The chunk rows of dO, delta and dX are split into LDS fragments (rows c, k = v, natural
//    order), all 64 rows at once; delta and dX come as the state passes' accumulator tiles
//    (kdn_state::st_tiles) and turn from columns to rows by a quad transpose, dX leaving as dv on the way.
//  * Wave w owns channel tile it = w (16 channels of K).  It loads its 16 rows of h and of dh straight into
//    split fragments (A operand, rows i, k = v) and forms
//      dQg^T = h dO^T,  dKg^T = -h dX^T,  dKf^T = dh delta^T    (D tile: lane -> chunk row, 4 consecutive
//                                              channels: the layout of the gradient phase's elementwise terms)
//      dgl_i = 2^{G_last,i} sum_v h_iv dh_iv,  and dM = lower(dO delta^T), dN = -strict_lower(dX delta^T)
//    for lower tiles w, w + 8.  dX carries everything the inverse's gradient needs: with
//    dN = -strict_lower(dV U^T + dKg W^T) the kernel read U, W and A^T (1,280 B more per token-head) and summed
//    eight waves' dN shares through LDS.
//  * Gradients.  dN, dM and their transposes are split once into LDS fragments (permuted k order:
//    slot 4h + j of lane group g <-> k = 32 kb + 16 h + 4 g + j).  Per channel tile the factors R,
//    Lk, Lq are built per lane for one channel and 16 chunk rows (rows outside the contraction's
//    nonzero range zeroed) and enter the time contractions as the A operand, with the dN / dM
//    fragments as B: the D tiles give each lane 4 consecutive channels of one chunk row, the layout
//    of dQg, dKf and dKg, so the elementwise inputs and outputs move as 16-byte (fp32) and 8-byte
//    (bf16) vectors.
// Chunks flagged by the forward store the products (dQg, dKg, dKf, dM, dN, dgl) for the exact kernel and
// stop after them.
// ---------------------------------------------------------------------------------------------
template <int K, int V, bool ISO, typename TDO, int HM>
__device__ __forceinline__ void chunk_bwd_task(
    int task, const void* __restrict__ hbuf, const void* __restrict__ dhbuf, const float* __restrict__ Dl,
    const float* __restrict__ dXl, const TDO* __restrict__ dO, const int* __restrict__ flags,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const float* __restrict__ kap,
    const float* __restrict__ gc, const float* __restrict__ q_rstd, const float* __restrict__ k_rstd, int T, int H,
    int NT, int BH, float scale, bf16_t* __restrict__ dv, bf16_t* __restrict__ dq, bf16_t* __restrict__ dk,
    float* __restrict__ dkap, float* __restrict__ dbeta, float* __restrict__ dg, float* __restrict__ xQg,
    float* __restrict__ xKg, float* __restrict__ xKf, float* __restrict__ xM, float* __restrict__ xN,
    float* __restrict__ xgl) {
  constexpr bool DO_BF16 = sizeof(TDO) == 2;
  // HM: which of h, dh were stored in bf16 (kdn_state::HB_*; the recurrences ran in fp32 and rounded
  // those copies once).  A bf16 operand enters a product without a lo half: one MFMA against another
  // bf16 operand, two against a split fp32 one.
  constexpr bool LH = !(HM & kdn_state::HB_H), LDH = !(HM & kdn_state::HB_DH);  // fp32 (split) copies
  constexpr bool LO_ = !DO_BF16;
  constexpr int EH = LH ? 4 : 2, EDH = LDH ? 4 : 2;  // bytes per element
  constexpr int NW = 8;
  constexpr int VB = V / 32;        // k-blocks of the V contraction
  constexpr int NIT = K / 16;       // channel tiles (waves 0 .. NIT-1 own one each)
  constexpr int RB = VB * TILE;     // one 16-row block of a [rows][V] operand as fragments
  constexpr int FR = 8 * TILE;      // one 64 x 64 operand as (4 row tiles x 2 k-blocks) fragments
  constexpr int STAGE_BYTES = 3 * 4 * RB * 2;
  constexpr int CONTRIB_BYTES = 4 * FR * 2;
  constexpr int LDS_BYTES = STAGE_BYTES > CONTRIB_BYTES ? STAGE_BYTES : CONTRIB_BYTES;
  constexpr int SU = C * V / 8 / 512;  // staging units (8 consecutive v of one row) per thread per operand
  static_assert(SU >= 1 && (C * V / 8) % 512 == 0, "staging units per thread");
  constexpr int TU = C * V / 4 / 512;  // tile units (4 rows of one column) of delta and of dX per thread
  static_assert(NIT <= NW, "K <= 128");
  __shared__ __attribute__((aligned(16))) unsigned char smem[LDS_BYTES];
  __shared__ float sDgl[K];
  __shared__ float sBeta[NW * C];
  __shared__ float sDot[2][NW][C];  // in-op L2 norm: per-wave partial row dots y . dy of q and k
  __shared__ float sRs[2][C];       // ... and the rows' rstd of q and k (their raw values in memory)
  __shared__ float sBt[ISO ? C : 1];  // iso: the rows' beta (0 past L), for the gradient phase
  bf16_t* sO = reinterpret_cast<bf16_t*>(smem);  // dO, delta, dX row fragments
  bf16_t* sD = sO + 4 * RB;
  bf16_t* sX = sD + 4 * RB;
  bf16_t* sF = reinterpret_cast<bf16_t*>(smem);  // gradients: dN, dM, dN^T, dM^T fragments
  const int n = NT - 1 - task / BH, bh = task % BH, b = bh / H, h = bh % H;
  const int t0 = n * C, L = min(C, T - t0);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r16 = lane & 15, g4 = lane >> 4;
  const int64_t chunk = (int64_t)bh * NT + n;
  const bool flagged = flags[chunk] != 0;
  const bool own_k = w < NIT;
  const int it = w;  // this wave's channel tile (when own_k)
  const int i0 = 16 * it + 4 * g4;
  if (q_rstd && tid < 2 * C) {  // read in the gradient phase, after phase 1's barriers
    const int c = tid & 63;
    sRs[tid >> 6][c] = c < L ? ((tid >> 6) ? k_rstd : q_rstd)[((int64_t)b * T + t0 + c) * H + h] : 0.f;
  }
  if (ISO && tid >= 2 * C && tid < 3 * C) {  // read in the gradient phase, after phase 1's barriers
    const int c = tid - 2 * C;
    sBt[ISO ? c : 0] = c < L ? kap[((int64_t)b * T + t0 + c) * H + h] : 0.f;
  }

  // ================================ loads ================================
  const bufrsrc rO = make_buf(dO + (((int64_t)b * T + t0) * H + h) * V, ((L - 1) * H + 1) * V * sizeof(TDO));
  // delta and dX: unit e = lane e % 64 of accumulator tile e / 64 (rows past L hold 0)
  float4 td[TU], tx[TU];
#pragma unroll
  for (int u = 0; u < TU; ++u) {
    td[u] = reinterpret_cast<const float4*>(Dl + chunk * C * V)[tid + 512 * u];
    tx[u] = reinterpret_cast<const float4*>(dXl + chunk * C * V)[tid + 512 * u];
  }
  u32x4 sr_O[SU][DO_BF16 ? 1 : 2];
#pragma unroll
  for (int u = 0; u < SU; ++u) {  // unit e: 16-row block, k-block, fragment lane
    const int e = tid + 512 * u, blk = e / (VB * 64), kb = (e / 64) % VB, sl = e & 63;
    const uint32_t c = (uint32_t)(16 * blk + (sl & 15)), v0 = (uint32_t)(32 * kb + 8 * (sl >> 4));
    if constexpr (DO_BF16) {
      sr_O[u][0] = __builtin_amdgcn_raw_buffer_load_b128(rO, (c * H * V + v0) * 2, 0, 0);
    } else {
      sr_O[u][0] = __builtin_amdgcn_raw_buffer_load_b128(rO, (c * H * V + v0) * 4, 0, 0);
      sr_O[u][1] = __builtin_amdgcn_raw_buffer_load_b128(rO, (c * H * V + v0) * 4 + 16, 0, 0);
    }
  }
  // this wave's rows of h and dh (row i = 16 it + r16, v = 32 kb + 8 g4 .. + 7) and the g_last factor
  const bufrsrc rh = make_buf(reinterpret_cast<const char*>(hbuf) + chunk * K * V * EH, K * V * EH);
  const bufrsrc rdh = make_buf(reinterpret_cast<const char*>(dhbuf) + chunk * K * V * EDH, K * V * EDH);
  float hv[VB][8], dhv[VB][8];
  u32x4 hr[VB], dhr[VB];  // bf16 copies: the rows are the MFMA fragments themselves
  float gl_i = 0.f;
  if (own_k) {
    const int i = 16 * it + r16;
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {
      // the state passes' tiled layout (kdn_state::hb_off): 8 consecutive columns are contiguous
      const uint32_t et = kdn_state::hb_off<K>(i, 32 * kb + 8 * g4);
      if constexpr (LH) kdn_intra::ld8(rh, et * 4, hv[kb]);
      else hr[kb] = __builtin_amdgcn_raw_buffer_load_b128(rh, et * 2, 0, 0);
      if constexpr (LDH) kdn_intra::ld8(rdh, et * 4, dhv[kb]);
      else dhr[kb] = __builtin_amdgcn_raw_buffer_load_b128(rdh, et * 2, 0, 0);
    }
    gl_i = buf_ld(make_buf(gc + (((int64_t)b * T + t0 + L - 1) * H + h) * K, K * 4), i * 4);
  }
  // Diagonal variant, K = 128: the chunk's k and q rows for the gradient phase go straight from memory
  // into LDS (buffer loads with the LDS flag: no registers held), issued once phase 1's operands have
  // arrived, so they land during phase 1 instead of as per-channel gathers in the gradient
  // phase (diag step -30 us; the isotropic variant, whose gradient phase loads less, measured 7 us
  // slower with it and keeps the gathers).
  // One instruction moves 64 lanes x 16 B = 4 rows of 256 B; row c of tensor x sits at
  // x * QK_T + (c / 4) * QK_S + (c % 4) * 256 bytes.  The 64-byte gap after each 4-row group puts the
  // rows 4 apart, which one gradient-phase read gathers, on different banks.  Rows past L read 0.
  constexpr bool QK_LDS = K == 128 && !ISO;
  constexpr int QK_S = 4 * K * 2 + 64, QK_T = (C / 4) * QK_S;
  __shared__ __attribute__((aligned(16))) unsigned char sQK[QK_LDS ? 2 * QK_T : 16];
  const int64_t in_row0 = ((int64_t)b * T + t0) * H + h;
  const uint32_t rows_in = (uint32_t)((L - 1) * H + 1);
  auto issue_qk = [&]() {
    if constexpr (QK_LDS) {
      if (!flagged) {
        const bufrsrc rkq[2] = {make_buf(k + in_row0 * K, rows_in * K * 2),
                                make_buf(q + in_row0 * K, rows_in * K * 2)};
        const int wu = __builtin_amdgcn_readfirstlane(w);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int gi = 0; gi < C / 4 / NW; ++gi) {  // wave w: 4-row groups NW gi + w
            const int grp = NW * gi + wu, c = 4 * grp + (lane >> 4);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rkq[x], (__attribute__((address_space(3))) void*)(sQK + x * QK_T + grp * QK_S), 16,
                (uint32_t)((c * H * K + 8 * (lane & 15)) * 2), 0, 0, 0);
          }
      }
    }
  };
  auto qk_lds = [&](int x, int c, int ch) -> const unsigned char* {
    return sQK + x * QK_T + (c >> 2) * QK_S + (c & 3) * (K * 2) + ch * 2;
  };
  // Isotropic variant, K = 128: the chunk's gate rows G (fp32) for the gradient phase go to LDS the same way,
  // issued with the k, q rows' slot: one instruction moves 64 lanes x 16 B = 2 rows of 512 B, and row c sits at
  // (c / 2) * G_S + (c % 2) * 512 bytes.  The 32-byte gap after each pair puts the rows 4 apart, which one
  // gradient-phase read gathers, on different banks.  Rows past L read 0; the reads clamp to row L - 1.
  constexpr bool G_LDS = K == 128 && ISO;
  constexpr int G_S = 2 * K * 4 + 32, G_T = (C / 2) * G_S;
  __shared__ __attribute__((aligned(16))) unsigned char sGr[G_LDS ? G_T : 16];
  auto issue_g = [&]() {
    if constexpr (G_LDS) {
      if (!flagged) {
        const bufrsrc rg = make_buf(gc + in_row0 * K, rows_in * K * 4);
        const int wu = __builtin_amdgcn_readfirstlane(w);
#pragma unroll
        for (int gi = 0; gi < C / 2 / NW; ++gi) {  // wave w: row pairs NW gi + w
          const int pr = NW * gi + wu, c = 2 * pr + (lane >> 5);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rg, (__attribute__((address_space(3))) void*)(sGr + pr * G_S), 16,
                                                   (uint32_t)((c * H * K + 4 * (lane & 31)) * 4), 0, 0, 0);
        }
      }
    }
  };
  auto g_lds = [&](int c, int ch) -> const float* {
    return reinterpret_cast<const float*>(sGr + (c >> 1) * G_S + (c & 1) * (K * 4) + ch * 4);
  };

  // ---- phase-1 fragments into LDS
#pragma unroll
  for (int u = 0; u < SU; ++u) {
    const int e = tid + 512 * u, blk = e / (VB * 64), kb = (e / 64) % VB, sl = e & 63;
    const int off = blk * RB + kb * TILE + sl * 8;
    if constexpr (DO_BF16) {  // exact in bf16: the lo half stays unused
      *reinterpret_cast<uint4*>(sO + off) = uint4{sr_O[u][0].x, sr_O[u][0].y, sr_O[u][0].z, sr_O[u][0].w};
    } else {
      const float4 x0 = __builtin_bit_cast(float4, sr_O[u][0]), x1 = __builtin_bit_cast(float4, sr_O[u][1]);
      const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
      uint4 hi, lo;
      split8(x, hi, lo);
      *reinterpret_cast<uint4*>(sO + off) = hi;
      *reinterpret_cast<uint4*>(sO + off + 512) = lo;
    }
  }
  {
    const bufrsrc rdv = make_buf(dv + (((int64_t)b * T + t0) * H + h) * V, ((L - 1) * H + 1) * V * 2);
#pragma unroll
    for (int u = 0; u < TU; ++u) {  // after the transpose: row c, columns v0 .. v0 + 3
      const int e = tid + 512 * u, tile = e >> 6, ln = e & 63;
      const int c = 16 * (tile & 3) + 4 * (ln >> 4) + (ln & 3), v0 = 16 * (tile >> 2) + 4 * ((ln & 15) >> 2);
      const int off = (c >> 4) * RB + (v0 >> 5) * TILE + ((c & 15) + 16 * ((v0 & 31) >> 3)) * 8 + (v0 & 7);
      const float4 d4 = kdn_state::quad_transpose(td[u], ln & 3), x4 = kdn_state::quad_transpose(tx[u], ln & 3);
      kdn_state::put_unit(sD, off, d4.x, d4.y, d4.z, d4.w);
      kdn_state::put_unit(sX, off, x4.x, x4.y, x4.z, x4.w);
      __builtin_amdgcn_raw_buffer_store_b64(u32x2{(uint32_t)f2bf(x4.x) | ((uint32_t)f2bf(x4.y) << 16),
                                                  (uint32_t)f2bf(x4.z) | ((uint32_t)f2bf(x4.w) << 16)},
                                            rdv, ((uint32_t)(c * H) * V + v0) * 2, 0, 0);
    }
  }
  __syncthreads();

  // ================================ phase 1: products with h, dh, dX ================================
  issue_qk();  // after phase 1's operands
  issue_g();
  f32x4 aQ[4], aK[4], kg[4];  // dQg^T, dKf^T, dKg^T (rows i, cols c): lane -> chunk row 16 J + r16, channels i0 ..
#pragma unroll
  for (int tl = 0; tl < 4; ++tl) aQ[tl] = aK[tl] = kg[tl] = zero4();
  if (own_k) {
    uint4 fh[VB], fl[VB];  // h (split, or its bf16 values), then dh
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {
      if constexpr (LH) split8(hv[kb], fh[kb], fl[kb]);
      else fh[kb] = __builtin_bit_cast(uint4, hr[kb]), fl[kb] = uint4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int kb = 0; kb < VB; ++kb)
#pragma unroll
      for (int tl = 0; tl < 4; ++tl) {
        uint4 oh, ol;
        afragx<LO_>(sO + tl * RB, kb, lane, oh, ol);
        aQ[tl] = mmx<LH, LO_>(fh[kb], fl[kb], oh, ol, aQ[tl]);
        uint4 xh, xl;
        afrag(sX + tl * RB, kb, lane, xh, xl);
        kg[tl] = mmx<LH, true>(fh[kb], fl[kb], xh, xl, kg[tl]);
      }
#pragma unroll
    for (int tl = 0; tl < 4; ++tl) kg[tl] = -kg[tl];
    float dot = 0.f;
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {
      float hf[8], df[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) hf[j] = hv[kb][j], df[j] = dhv[kb][j];
      if constexpr (!LH) kdn_intra::unpack8(hr[kb], hf);
      if constexpr (!LDH) kdn_intra::unpack8(dhr[kb], df);
#pragma unroll
      for (int j = 0; j < 8; ++j) dot += hf[j] * df[j];
      if constexpr (LDH) split8(dhv[kb], fh[kb], fl[kb]);
      else fh[kb] = __builtin_bit_cast(uint4, dhr[kb]), fl[kb] = uint4{0u, 0u, 0u, 0u};
    }
    dot += __shfl_xor(dot, 16, 64);
    dot += __shfl_xor(dot, 32, 64);
    if (g4 == 0) sDgl[16 * it + r16] = dot * fexp2(gl_i);
#pragma unroll
    for (int kb = 0; kb < VB; ++kb)
#pragma unroll
      for (int tl = 0; tl < 4; ++tl) {
        uint4 xh, xl;
        afrag(sD + tl * RB, kb, lane, xh, xl);
        aK[tl] = mmx<LDH, true>(fh[kb], fl[kb], xh, xl, aK[tl]);
      }
  }
  // dM = lower(dO delta^T) and dN = -strict_lower(dX delta^T), lower tiles (c-block I, s-block J) w and w + 8:
  // mt, nt lane -> column s = 16 J + r16, rows c = 16 I + 4 g4 + j; mtT, ntT the same tiles transposed, lane ->
  // row c = 16 I + r16, columns s = 16 J + 4 g4 + j.  Each gives one of the gradient phase's fragment forms.
  f32x4 mt[2], mtT[2], nt[2], ntT[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    mt[x] = mtT[x] = nt[x] = ntT[x] = zero4();
    const int t = w + NW * x;
    if (t >= 10) continue;
    int I, J;
    lower_tile(t, I, J);
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {
      uint4 xh, xl, oh, ol, yh, yl;
      afrag(sD + J * RB, kb, lane, xh, xl);
      afragx<LO_>(sO + I * RB, kb, lane, oh, ol);
      mt[x] = mmx<LO_, true>(oh, ol, xh, xl, mt[x]);
      mtT[x] = mmx<true, LO_>(xh, xl, oh, ol, mtT[x]);
      afrag(sX + I * RB, kb, lane, yh, yl);
      nt[x] = mma3(yh, yl, xh, xl, nt[x]);
      ntT[x] = mma3(xh, xl, yh, yl, ntT[x]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = 4 * g4 + j;
      if (I == J && r16 > c) mt[x][j] = 0.f;
      if (I == J && c > r16) mtT[x][j] = 0.f;
      nt[x][j] = I == J && r16 >= c ? 0.f : -nt[x][j];
      ntT[x][j] = I == J && c >= r16 ? 0.f : -ntT[x][j];
    }
  }

  if (flagged) {  // the exact kernel takes it from here: store the products in its layouts
    __syncthreads();  // sDgl
    if (own_k) {
      const bufrsrc rQ = make_buf(xQg + ((int64_t)bh * T + t0) * K, L * K * 4);
      const bufrsrc rKg = make_buf(xKg + ((int64_t)bh * T + t0) * K, L * K * 4);
      const bufrsrc rKf = make_buf(xKf + ((int64_t)bh * T + t0) * K, L * K * 4);
#pragma unroll
      for (int tl = 0; tl < 4; ++tl) {
        const uint32_t o = ((uint32_t)(16 * tl + r16) * K + i0) * 4;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, aQ[tl]), rQ, o, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, kg[tl]), rKg, o, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, aK[tl]), rKf, o, 0, 0);
      }
      if (g4 == 0) xgl[chunk * K + 16 * it + r16] = sDgl[16 * it + r16];
    }
    float *Mn = xM + chunk * C * C, *Nn = xN + chunk * C * C;
#pragma unroll
    for (int x = 0; x < 2; ++x) {  // tiles 10 .. 15: the upper ones, zero
      const int t = w + NW * x;
      int I, J;
      if (t < 10) lower_tile(t, I, J);
      else upper_tile(t - 10, I, J);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        Mn[(16 * I + 4 * g4 + j) * C + 16 * J + r16] = mt[x][j];
        Nn[(16 * I + 4 * g4 + j) * C + 16 * J + r16] = nt[x][j];
      }
    }
    return;
  }
  __syncthreads();  // every fragment read: the gradient phase's fragments may overwrite them

  // ======================= dN, dM staging (the gradient phase's fragments) =======================
  // fragment offset of 4 consecutive k = k0 .. k0 + 3 (k0 % 4 == 0) of one row: permuted k order, slot
  // 4 hh + j of lane group gg <-> k = 32 kb + 16 hh + 4 gg + j
  auto foff = [](int row, int k0) {
    return ((row >> 4) * 2 + (k0 >> 5)) * TILE + ((row & 15) + 16 * ((k0 & 15) >> 2)) * 8 + 4 * ((k0 >> 4) & 1);
  };
#pragma unroll
  for (int x = 0; x < 2; ++x) {  // rows form (row c, k = s) from the T tiles, transposed form (row s, k = c)
    const int t = w + NW * x;
    int I, J;  // tiles 10 .. 15: I < J, zero in both forms
    if (t < 10) lower_tile(t, I, J);
    else upper_tile(t - 10, I, J);
    const int fr = foff(16 * I + r16, 16 * J + 4 * g4), ft = foff(16 * J + r16, 16 * I + 4 * g4);
    kdn_state::put_unit(sF, fr, ntT[x][0], ntT[x][1], ntT[x][2], ntT[x][3]);
    kdn_state::put_unit(sF + FR, fr, mtT[x][0], mtT[x][1], mtT[x][2], mtT[x][3]);
    kdn_state::put_unit(sF + 2 * FR, ft, nt[x][0], nt[x][1], nt[x][2], nt[x][3]);
    kdn_state::put_unit(sF + 3 * FR, ft, mt[x][0], mt[x][1], mt[x][2], mt[x][3]);
  }
  if constexpr (QK_LDS || G_LDS) __builtin_amdgcn_s_waitcnt(0);  // this wave's k, q or G rows have reached LDS
  __syncthreads();

  // ================================ gradient phase ================================
  // With the in-op L2 norm (q_rstd, k_rstd [B,T,H] given) q and k are the raw inputs x, the operand is
  // y = bf16(x rstd) (the forward's), and dq, dk are returned for x: dx = rstd (dy - y (y . dy)), the
  // row dot summed over the waves.
  const bool qk_norm = q_rstd != nullptr;
  float bpart[4] = {0.f, 0.f, 0.f, 0.f};  // iso: dbeta partials of rows 16 tl + r16
  float dqs[4][4], dks[4][4];             // in-op norm: dy of q, k (rows 16 tl + r16, channels i0 ..)
  u32x2 yq2[4], yk2[4];                   // ... and y (bf16 pairs)
  if (own_k) {
    const bufrsrc rG = make_buf(gc + in_row0 * K, rows_in * K * 4);
    const bufrsrc rk = make_buf(k + in_row0 * K, rows_in * K * 2);
    const bufrsrc rq = make_buf(q + in_row0 * K, rows_in * K * 2);
    const bufrsrc rkap = ISO ? make_buf(kap + in_row0, rows_in * 4) : make_buf(kap + in_row0 * K, rows_in * K * 4);
    const bufrsrc rdq = make_buf(dq + in_row0 * K, rows_in * K * 2);
    const bufrsrc rdk = make_buf(dk + in_row0 * K, rows_in * K * 2);
    const bufrsrc rdkap = ISO ? make_buf(dkap, 0) : make_buf(dkap + in_row0 * K, rows_in * K * 4);
    const bufrsrc rdg = make_buf(dg + in_row0 * K, rows_in * K * 4);
    const int i = 16 * it + r16;
    // ---- factor loads, one channel per lane: rows c = 16 tl + 4 g4 + j, slot p = 4 tl + j; the gate
    // of rows past L repeats row L-1 (their k, q, kappa read zero)
    float av[16], Gv[16];
    uint16_t kraw[16], qraw[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) {
      const int c = 16 * (p >> 2) + 4 * g4 + (p & 3);
      const uint32_t crow = (uint32_t)(c * H), o = crow * K + i;
      if constexpr (QK_LDS) {
        kraw[p] = *reinterpret_cast<const uint16_t*>(qk_lds(0, c, i));
        qraw[p] = *reinterpret_cast<const uint16_t*>(qk_lds(1, c, i));
      } else {
        kraw[p] = __builtin_amdgcn_raw_buffer_load_b16(rk, o * 2, 0, 0);
        qraw[p] = __builtin_amdgcn_raw_buffer_load_b16(rq, o * 2, 0, 0);
      }
      av[p] = ISO ? sBt[ISO ? c : 0] : buf_ld(rkap, o * 4);
      if constexpr (G_LDS) Gv[p] = *g_lds(min(c, L - 1), i);
      else Gv[p] = buf_ld(rG, ((uint32_t)(min(c, L - 1) * H) * K + i) * 4);
    }
    __builtin_amdgcn_sched_barrier(0);
    float mA[4];  // block anchors m_J = (G_{16J} + G_{16J+15}) / 2 of this lane's channel
#pragma unroll
    for (int J = 0; J < 4; ++J) mA[J] = 0.5f * (__shfl(Gv[4 * J], r16, 64) + __shfl(Gv[4 * J + 3], 48 + r16, 64));
    float Rown[16], Kown[16], Qown[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) {
      const int c = 16 * (p >> 2) + 4 * g4 + (p & 3);
      float kvp = bf2f(kraw[p]), qvp = bf2f(qraw[p]);
      if (qk_norm) {
        kvp = l2n(kvp, sRs[1][c]);
        qvp = l2n(qvp, sRs[0][c]);
      }
      const float e = fexp2(Gv[p] - mA[p >> 2]);
      Kown[p] = kvp * e;
      Qown[p] = scale * qvp * e;
      Rown[p] = (ISO ? av[p] * kvp : av[p]) * frcp(e);
    }
    const float4 glv = G_LDS ? *reinterpret_cast<const float4*>(g_lds(L - 1, i0))
                             : buf_ld4(rG, ((uint32_t)((L - 1) * H) * K + i0) * 4);
    u32x2 kq4[4], qq4[4];
    float4 kap4[4], G4[4];
#pragma unroll
    for (int tl = 0; tl < 4; ++tl) {
      const uint32_t c = (uint32_t)(16 * tl + r16), o = c * H * K + i0;
      if constexpr (QK_LDS) {
        kq4[tl] = *reinterpret_cast<const u32x2*>(qk_lds(0, (int)c, i0));
        qq4[tl] = *reinterpret_cast<const u32x2*>(qk_lds(1, (int)c, i0));
      } else {
        kq4[tl] = __builtin_amdgcn_raw_buffer_load_b64(rk, o * 2, 0, 0);
        qq4[tl] = __builtin_amdgcn_raw_buffer_load_b64(rq, o * 2, 0, 0);
      }
      if (ISO) {
        const float be = sBt[ISO ? c : 0];
        kap4[tl] = float4{be, be, be, be};
      } else {
        kap4[tl] = buf_ld4(rkap, o * 4);
      }
      G4[tl] = G_LDS ? *reinterpret_cast<const float4*>(g_lds(min(16 * tl + r16, L - 1), i0))
                     : buf_ld4(rG, ((uint32_t)(min(16 * tl + r16, L - 1) * H) * K + i0) * 4);
    }
    float colpart[4] = {0.f, 0.f, 0.f, 0.f};
    float4 dg_last = float4{0.f, 0.f, 0.f, 0.f};
    bool has_last = false;
    const float gla[4] = {glv.x, glv.y, glv.z, glv.w};
#pragma unroll
    for (int tl = 0; tl < 4; ++tl) {
      f32x4 dLk = zero4(), dLq = zero4(), dR = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        uint4 ah, al;
        if (kb <= tl / 2) {
          const float s0 = 2 * kb <= tl ? fexp2(mA[tl] - mA[2 * kb]) : 0.f;
          const float s1 = 2 * kb + 1 <= tl ? fexp2(mA[tl] - mA[2 * kb + 1]) : 0.f;
          float rv[8];
#pragma unroll
          for (int sl = 0; sl < 8; ++sl) rv[sl] = Rown[8 * kb + sl] * (sl < 4 ? s0 : s1);
          uint4 Rh, Rl;
          split8(rv, Rh, Rl);
          afrag(sF, tl * 2 + kb, lane, ah, al);
          dLk = mma3(Rh, Rl, ah, al, dLk);
          afrag(sF + FR, tl * 2 + kb, lane, ah, al);
          dLq = mma3(Rh, Rl, ah, al, dLq);
        }
        if (2 * kb + 1 >= tl) {
          const float s0 = 2 * kb >= tl ? fexp2(mA[2 * kb] - mA[tl]) : 0.f;
          const float s1 = 2 * kb + 1 >= tl ? fexp2(mA[2 * kb + 1] - mA[tl]) : 0.f;
          float lk[8], lq[8];
#pragma unroll
          for (int sl = 0; sl < 8; ++sl) {
            const float sc = sl < 4 ? s0 : s1;
            lk[sl] = Kown[8 * kb + sl] * sc;
            lq[sl] = Qown[8 * kb + sl] * sc;
          }
          uint4 Kh, Kl, Qh, Ql;
          split8(lk, Kh, Kl);
          split8(lq, Qh, Ql);
          afrag(sF + 2 * FR, tl * 2 + kb, lane, ah, al);
          dR = mma3(Kh, Kl, ah, al, dR);
          afrag(sF + 3 * FR, tl * 2 + kb, lane, ah, al);
          dR = mma3(Qh, Ql, ah, al, dR);
        }
      }
      const uint32_t c = (uint32_t)(16 * tl + r16), o = c * H * K + i0;
      float kv4[4] = {__uint_as_float(kq4[tl].x << 16), __uint_as_float(kq4[tl].x & 0xffff0000u),
                      __uint_as_float(kq4[tl].y << 16), __uint_as_float(kq4[tl].y & 0xffff0000u)};
      float qv4[4] = {__uint_as_float(qq4[tl].x << 16), __uint_as_float(qq4[tl].x & 0xffff0000u),
                      __uint_as_float(qq4[tl].y << 16), __uint_as_float(qq4[tl].y & 0xffff0000u)};
      if (qk_norm) {
        const float rk_ = sRs[1][c], rq_ = sRs[0][c];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          kv4[j] = l2n(kv4[j], rk_);
          qv4[j] = l2n(qv4[j], rq_);
        }
        yk2[tl] = u32x2{(uint32_t)f2bf(kv4[0]) | ((uint32_t)f2bf(kv4[1]) << 16),
                        (uint32_t)f2bf(kv4[2]) | ((uint32_t)f2bf(kv4[3]) << 16)};  // exact: already bf16
        yq2[tl] = u32x2{(uint32_t)f2bf(qv4[0]) | ((uint32_t)f2bf(qv4[1]) << 16),
                        (uint32_t)f2bf(qv4[2]) | ((uint32_t)f2bf(qv4[3]) << 16)};
      }
      const float a4[4] = {kap4[tl].x, kap4[tl].y, kap4[tl].z, kap4[tl].w};
      const float gv[4] = {G4[tl].x, G4[tl].y, G4[tl].z, G4[tl].w};
      const float mz[4] = {__shfl(mA[tl], 4 * g4, 64), __shfl(mA[tl], 4 * g4 + 1, 64), __shfl(mA[tl], 4 * g4 + 2, 64),
                           __shfl(mA[tl], 4 * g4 + 3, 64)};
      float dkv[4], dqv[4], dav[4], dgv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float beta = ISO ? a4[j] : 0.f;
        const float kap_p = ISO ? beta * kv4[j] : a4[j];
        const float e = fexp2(gv[j] - mz[j]), er = frcp(e);
        const float eg = fexp2(gv[j]), f = fexp2(gla[j] - gv[j]);
        const float a_lk = dLk[j], a_lq = dLq[j] * scale, a_r = dR[j];
        const float dkgv = kg[tl][j], dqgv = aQ[tl][j], dkfv = aK[tl][j];
        dkv[j] = a_lk * e + dkgv * eg;
        dqv[j] = a_lq * e + scale * dqgv * eg;
        dav[j] = a_r * er + dkfv * f;
        dgv[j] = kv4[j] * e * a_lk + qv4[j] * e * a_lq - kap_p * er * a_r + kv4[j] * eg * dkgv +
                 scale * qv4[j] * eg * dqgv - kap_p * f * dkfv;
        if ((int)c < L) colpart[j] += kap_p * f * dkfv;
        if (ISO) {
          dkv[j] += beta * dav[j];
          bpart[tl] += dav[j] * kv4[j];
        }
      }
      if (!ISO)
        __builtin_amdgcn_raw_buffer_store_b128(
            u32x4{__float_as_uint(dav[0]), __float_as_uint(dav[1]), __float_as_uint(dav[2]), __float_as_uint(dav[3])},
            rdkap, o * 4, 0, 0);
      if (qk_norm) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          dqs[tl][j] = dqv[j];
          dks[tl][j] = dkv[j];
        }
      } else {
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{(uint32_t)f2bf(dqv[0]) | ((uint32_t)f2bf(dqv[1]) << 16),
                                                    (uint32_t)f2bf(dqv[2]) | ((uint32_t)f2bf(dqv[3]) << 16)},
                                              rdq, o * 2, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{(uint32_t)f2bf(dkv[0]) | ((uint32_t)f2bf(dkv[1]) << 16),
                                                    (uint32_t)f2bf(dkv[2]) | ((uint32_t)f2bf(dkv[3]) << 16)},
                                              rdk, o * 2, 0, 0);
      }
      if ((int)c == L - 1) {
        dg_last = float4{dgv[0], dgv[1], dgv[2], dgv[3]};
        has_last = true;
      } else {
        __builtin_amdgcn_raw_buffer_store_b128(
            u32x4{__float_as_uint(dgv[0]), __float_as_uint(dgv[1]), __float_as_uint(dgv[2]), __float_as_uint(dgv[3])},
            rdg, o * 4, 0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) colpart[j] = row16_sum(colpart[j]);
    if (has_last) {
      const float4 gl4 = *reinterpret_cast<const float4*>(sDgl + i0);
      const float4 v = float4{dg_last.x + colpart[0] + gl4.x, dg_last.y + colpart[1] + gl4.y,
                              dg_last.z + colpart[2] + gl4.z, dg_last.w + colpart[3] + gl4.w};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rdg,
                                             ((uint32_t)((L - 1) * H) * K + i0) * 4, 0, 0);
    }
  }
  if (!ISO && !qk_norm) return;
  auto unpack4 = [](u32x2 v, float* f) {
    f[0] = __uint_as_float(v.x << 16), f[1] = __uint_as_float(v.x & 0xffff0000u);
    f[2] = __uint_as_float(v.y << 16), f[3] = __uint_as_float(v.y & 0xffff0000u);
  };
  if (own_k) {  // per-wave partials over this wave's 16 channels of rows 16 tl + r16
#pragma unroll
    for (int tl = 0; tl < 4; ++tl) {
      float v = bpart[tl], pq = 0.f, pk = 0.f;
      if (qk_norm) {
        float yq[4], yk[4];
        unpack4(yq2[tl], yq);
        unpack4(yk2[tl], yk);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          pq += yq[j] * dqs[tl][j];
          pk += yk[j] * dks[tl][j];
        }
      }
      v = swz16_add(v);
      pq = swz16_add(pq);
      pk = swz16_add(pk);
      v += __shfl_xor(v, 32, 64);
      pq += __shfl_xor(pq, 32, 64);
      pk += __shfl_xor(pk, 32, 64);
      if (g4 == 0) {
        sBeta[w * C + 16 * tl + r16] = v;
        sDot[0][w][16 * tl + r16] = pq;
        sDot[1][w][16 * tl + r16] = pk;
      }
    }
  }
  __syncthreads();
  if (ISO && tid < L) {
    float s = 0.f;
#pragma unroll
    for (int ww = 0; ww < NIT; ++ww) s += sBeta[ww * C + tid];
    dbeta[((int64_t)b * T + t0 + tid) * H + h] = s;
  }
  if (!qk_norm) return;
  if (tid < 2 * C) {  // the row dots: sum of the waves' partials, into slot 0
    const int tq = tid >> 6, c = tid & 63;
    float dsum = 0.f;
#pragma unroll
    for (int ww = 0; ww < NIT; ++ww) dsum += sDot[tq][ww][c];
    sDot[tq][NW - 1][c] = dsum;  // each (tensor, row) is read and overwritten by this one thread
  }
  __syncthreads();
  // dx = rstd (dy - y (y . dy)) for the raw q, k, regrouped through LDS (the gradient phase's fragments are
  // dead) so that a store writes whole rows: straight from the lanes it covered 16 rows in 32-byte pieces, at the
  // end of the workgroup's life (chunk backward 462 -> 446 us isotropic at B4 T4096 H18).  Stores in
  // mid-kernel overlap the arithmetic as they are: dg and the diagonal dq, dk gathered the same way lost 10 to 20 us
  constexpr int XR = K + 8;  // row stride, bf16
  bf16_t* sOut = reinterpret_cast<bf16_t*>(smem);  // [q, k][row][XR]
  static_assert(2 * C * XR * 2 <= LDS_BYTES, "dq, dk rows");
  if (own_k) {
#pragma unroll
    for (int tl = 0; tl < 4; ++tl) {
      const int c = 16 * tl + r16;
      const float dotq = sDot[0][NW - 1][c], dotk = sDot[1][NW - 1][c];
      const float rq_ = sRs[0][c], rk_ = sRs[1][c];
      float yq[4], yk[4], xq[4], xk[4];
      unpack4(yq2[tl], yq);
      unpack4(yk2[tl], yk);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        xq[j] = rq_ * (dqs[tl][j] - yq[j] * dotq);
        xk[j] = rk_ * (dks[tl][j] - yk[j] * dotk);
      }
      *reinterpret_cast<uint2*>(sOut + c * XR + i0) =
          uint2{(uint32_t)f2bf(xq[0]) | ((uint32_t)f2bf(xq[1]) << 16), (uint32_t)f2bf(xq[2]) | ((uint32_t)f2bf(xq[3]) << 16)};
      *reinterpret_cast<uint2*>(sOut + (C + c) * XR + i0) =
          uint2{(uint32_t)f2bf(xk[0]) | ((uint32_t)f2bf(xk[1]) << 16), (uint32_t)f2bf(xk[2]) | ((uint32_t)f2bf(xk[3]) << 16)};
    }
  }
  __syncthreads();
  const bufrsrc rdq = make_buf(dq + in_row0 * K, rows_in * K * 2), rdk = make_buf(dk + in_row0 * K, rows_in * K * 2);
  constexpr int CH = K / 8;  // 16-byte pieces of a row
#pragma unroll
  for (int u = 0; u < C * CH / 512; ++u) {
    const int e = tid + 512 * u, c = e / CH, i8 = 8 * (e % CH);
    const uint32_t o = ((uint32_t)(c * H) * K + i8) * 2;  // rows past L dropped
    __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(sOut + c * XR + i8), rdq, o, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(sOut + (C + c) * XR + i8), rdk, o, 0, 0);
  }
}

// One workgroup per task: tasks task0 .. task0 + gridDim.x - 1.
template <int K, int V, bool ISO, typename TDO, int HM>
__global__ __launch_bounds__(512, 1) void chunk_bwd_kernel(
    const void* __restrict__ hbuf, const void* __restrict__ dhbuf, const float* __restrict__ Dl,
    const float* __restrict__ dXl, const TDO* __restrict__ dO, const int* __restrict__ flags,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const float* __restrict__ kap,
    const float* __restrict__ gc, const float* __restrict__ q_rstd, const float* __restrict__ k_rstd, int T, int H,
    int NT, int BH, int task0, float scale, bf16_t* __restrict__ dv, bf16_t* __restrict__ dq, bf16_t* __restrict__ dk,
    float* __restrict__ dkap, float* __restrict__ dbeta, float* __restrict__ dg, float* __restrict__ xQg,
    float* __restrict__ xKg, float* __restrict__ xKf, float* __restrict__ xM, float* __restrict__ xN,
    float* __restrict__ xgl) {
  chunk_bwd_task<K, V, ISO, TDO, HM>(task0 + (int)blockIdx.x, hbuf, dhbuf, Dl, dXl, dO, flags, q, k, kap, gc, q_rstd,
                                 k_rstd, T, H, NT, BH, scale, dv, dq, dk, dkap, dbeta, dg, xQg, xKg, xKf, xM, xN, xgl);
}

}  // namespace kdn_bwd
