// One token through a block (decoding with a carried state): the skinny projections with what surrounds
// them, and the whole mixer between its input and output projections.
//
// A decode step is a chain of small dependent launches, and a launch that depends on the one before it
// costs 3-4 us however little it does, so the step is bound by their number and by the weight stream.
// Per block there are five here (input projection with its RMS norm, mixer, output projection with the
// residual, SwiGLU gate with its norm, down projection with the residual) in place of 16 to 25.
// The reference has no decoding path (lit_gpt/model.py:104,184 refuse caching); the arithmetic is that
// of the layers' one-token forward.
#include "kdn_common.h"
#include "kdn_state.h"
#include "../../include/kdn.h"

namespace {

using kdn_state::mfma;

__device__ __forceinline__ void unpack8(uint4 v, float* f) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) f[2 * q] = __uint_as_float(w[q] << 16), f[2 * q + 1] = __uint_as_float(w[q] & 0xffff0000u);
}
__device__ __forceinline__ uint4 pack8(const float* f) {
  uint32_t w[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) w[q] = (uint32_t)f2bf(f[2 * q]) | ((uint32_t)f2bf(f[2 * q + 1]) << 16);
  return uint4{w[0], w[1], w[2], w[3]};
}

// ---------------------------------------------------------------------------------------------
// y[m, n] = epilogue(sum_k xn[m, k] W[n, k]) for M <= 64 rows, bf16 W [N, K], fp32 accumulation.
// xn = x, or with NORM the RMS-normed row x rsqrt(mean x^2 + eps) nw: x nw goes to the matrix cores in bf16
// (for M <= 16 as hi + lo, the norm's rounding left out) and the row's rsqrt multiplies the sum.
// Epilogue: + bias; GATED (W = [W1; W2]): silu(W1 x + b1) (W2 x + b2); + res[m, n], all in fp32 before the
// one rounding.
//
// Bound by the weight stream.  A workgroup's waves split K and its partial sums meet in LDS; the tokens are
// the other operand of the 16x16x32 products (MT tiles of 16, the columns past M unused: the matrix cores
// are idle anyway).  K % 8 == 0: an 8-element segment past K is zero.
//   resident (K <= 2304 = 8 waves x 9 steps of 32): a wave keeps its share of x in registers and the
//     workgroup walks tiles of up to 16 rows of W (GATED: of each half), a tile's loads all in flight at
//     once, the next tile's issued before the current one's sums meet.  Streaming x beside W instead halved
//     the weight bytes in flight and read x once per tile from L2: M 1 / 32, N 32000 K 2304 took
//     39.7 / 84.0 us, now 27.8 / 36.5 (5.3 / 4.0 TB/s); [2 x 6912, 2304] gated 21.0 / 27.2, now 17.3 / 22.5.
//   streaming (longer K, and more than 32 rows with the norm or the gate): 16 waves, one tile per workgroup, x beside
//     W and so read once per tile.  Up to 8 rows that is little; beyond, x is the larger stream (M 64, N 32000 K 2304:
//     590 MB of it for 147 MB of W, 152 us), and a caller with a choice takes the norm and the product apart.
// ---------------------------------------------------------------------------------------------
struct ProjArgs {
  const bf16_t* x;
  int64_t xs;
  const bf16_t* nw;
  float eps;
  const bf16_t *W, *bias, *res;
  int64_t rs;
  int M, N, K;
  bf16_t* y;
  int64_t ys;
  float* part;  // split: the partial products [split][M][N]
  int tr;       // rows of W per tile, at most 16 (the 16-row operand repeats the last one)
};
constexpr int kResWaves = 8, kResSteps = 9, kStrWaves = 16;

// the workgroup's NW partial tiles (float4 per lane, as accumulated) -> y
template <int MT, int NA, int NW, bool NORM>
__device__ __forceinline__ void proj_epilogue(const ProjArgs& A, const float (*acc)[NA * MT][256],
                                              const float (*ss)[MT * 16], int n0) {
  for (int e = threadIdx.x; e < MT * 256; e += 64 * NW) {
    const int mt = e >> 8, l = (e >> 2) & 63, m = 16 * mt + (l & 15), nl = 4 * (l >> 4) + (e & 3), n = n0 + nl;
    if (m >= A.M || nl >= A.tr || n >= A.N) continue;
    float v[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      v[a] = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v[a] += acc[w][a * MT + mt][e & 255];
    }
    if (NA == 1 && !NORM && A.part) {
      A.part[((int64_t)blockIdx.y * A.M + m) * A.N + n] = v[0];
      continue;
    }
    float rs = 1.f;
    if constexpr (NORM) {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) sum += ss[w][m];
      rs = rsqrtf(sum / (float)A.K + A.eps);
    }
    float o = v[0] * rs + (A.bias ? bf2f(A.bias[n]) : 0.f);
    if constexpr (NA == 2) {
      const float o2 = v[1] * rs + (A.bias ? bf2f(A.bias[A.N + n]) : 0.f);
      o = o / (1.f + __expf(-o)) * o2;  // silu(o) o2; e^-o = inf for very negative o gives -0
    }
    if (A.res) o += bf2f(A.res[(int64_t)m * A.rs + n]);
    A.y[(int64_t)m * A.ys + n] = f2bf(o);
  }
}
// x nw of 8 elements (sum of squares of x added to ss); LO: the rounding's remainder in lo
template <bool LO>
__device__ __forceinline__ void norm_frag(uint4& x, uint4& lo, uint4 nw, float& ss) {
  float xv[8], nv[8];
  unpack8(x, xv), unpack8(nw, nv);
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = fmaf(xv[e], xv[e], ss), xv[e] *= nv[e];
  x = pack8(xv);
  if constexpr (LO) {
    unpack8(x, nv);
#pragma unroll
    for (int e = 0; e < 8; ++e) xv[e] -= nv[e];
    lo = pack8(xv);
  }
}

template <int MT, int NA, bool NORM, int SW>
__global__ __launch_bounds__(64 * kResWaves) void decode_proj_resident_kernel(const ProjArgs A) {
  constexpr int NW = kResWaves;
  constexpr bool LO = NORM && MT == 1;
  __shared__ float s_acc[2][NW][NA * MT][256];
  __shared__ float s_ss[NORM ? NW : 1][MT * 16];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kg = lane >> 4, K = A.K, N = A.N;
  const int S = (K + 31) / 32, y0 = S * blockIdx.y / gridDim.y, y1 = S * (blockIdx.y + 1) / gridDim.y;
  const int s0 = y0 + (y1 - y0) * wv / NW, s1 = y0 + (y1 - y0) * (wv + 1) / NW;  // at most SW steps, possibly none
  const int tr = A.tr, tiles = (N + tr - 1) / tr;
  uint4 wf[SW][NA], xf[SW][MT], xl[LO ? SW : 1];
  // buffer loads: one offset per row and an immediate per step in place of 64-bit addresses.  A step past the
  // wave's share is loaded but not used; past the tensor's end the load returns 0.
  const bufrsrc rx = make_buf(A.x, (uint32_t)(((int64_t)(A.M - 1) * A.xs + K) * 2)), rn = make_buf(A.nw, (uint32_t)K * 2);
  bufrsrc rw[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) rw[a] = make_buf(A.W + (int64_t)a * N * K, (uint32_t)N * K * 2);
  auto ld = [](bufrsrc b, uint32_t v) { return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(b, v, 0, 0)); };
  const uint32_t vk = (uint32_t)s0 * 64 + 16 * kg;  // bytes into a row
  auto load_w = [&](int tile) {
    const uint32_t vw = (uint32_t)min(tr * tile + min(r, tr - 1), N - 1) * (uint32_t)K * 2 + vk;
#pragma unroll
    for (int u = 0; u < SW; ++u)
#pragma unroll
      for (int a = 0; a < NA; ++a) wf[u][a] = ld(rw[a], vw + 64 * u);
  };
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const uint32_t vx = (uint32_t)min(16 * mt + r, A.M - 1) * (uint32_t)A.xs * 2 + vk;
#pragma unroll
    for (int u = 0; u < SW; ++u) xf[u][mt] = ld(rx, vx + 64 * u);
  }
  if constexpr (MT == 1) load_w(blockIdx.x);  // (wider: the norm weights and both would not fit the registers)
  // x's share: zero past the wave's steps and past K, normed in place
  float ss[MT] = {};
#pragma unroll
  for (int u = 0; u < SW; ++u) {
    // with several token tiles the norm weights come 3 steps at a time: all at once they would spill
    if (NORM && MT > 1 && u % 3 == 0) __builtin_amdgcn_sched_barrier(0);
    const bool in = s0 + u < s1 && 32 * (s0 + u) + 8 * kg < K;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (!in) xf[u][mt] = uint4{0u, 0u, 0u, 0u};
      if constexpr (NORM)
        norm_frag<LO>(xf[u][mt], xl[LO ? u : 0], ld(rn, vk + 64 * u), ss[mt]);
    }
  }
  if (NORM && MT > 1) __builtin_amdgcn_sched_barrier(0);
  if constexpr (MT != 1) load_w(blockIdx.x);
  if constexpr (NORM) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      ss[mt] += __shfl_xor(ss[mt], 16, 64);
      ss[mt] += __shfl_xor(ss[mt], 32, 64);
      if (lane < 16) s_ss[wv][16 * mt + lane] = ss[mt];
    }
  }
  int buf = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, buf ^= 1) {
    f32x4 acc[NA][MT];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[a][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < SW; ++u) {
      if (s0 + u >= s1) break;  // uniform
      if (32 * (s0 + u) + 8 * kg >= K)  // only in the last step of a K that is not a multiple of 32
#pragma unroll
        for (int a = 0; a < NA; ++a) wf[u][a] = uint4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int a = 0; a < NA; ++a) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[a][mt] = mfma(wf[u][a], xf[u][mt], acc[a][mt]);
        if constexpr (LO) acc[a][0] = mfma(wf[u][a], xl[u], acc[a][0]);
      }
    }
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        *reinterpret_cast<f32x4*>(&s_acc[buf][wv][a * MT + mt][4 * lane]) = acc[a][mt];
    if (tile + (int)gridDim.x < tiles) load_w(tile + gridDim.x);
    __syncthreads();  // s_acc[buf] is written again two tiles on, after the next barrier
    proj_epilogue<MT, NA, NW, NORM>(A, s_acc[buf], s_ss, tr * tile);
  }
}

template <int MT, int NA, bool NORM>
__global__ __launch_bounds__(64 * kStrWaves) void decode_proj_stream_kernel(const ProjArgs A) {
  constexpr int NW = kStrWaves;
  constexpr int U = 20 / (NA + MT + (NORM ? 1 : 0));  // steps in flight: at most 80 registers of loads
  constexpr bool LO = NORM && MT == 1;
  __shared__ float s_acc[NW][NA * MT][256];
  __shared__ float s_ss[NORM ? NW : 1][MT * 16];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kg = lane >> 4, K = A.K, N = A.N;
  const int S = (K + 31) / 32, s1 = S * (wv + 1) / NW;
  const bf16_t* wr = A.W + (int64_t)min(A.tr * (int)blockIdx.x + min(r, A.tr - 1), N - 1) * K;
  const bf16_t* xr[MT];
  f32x4 acc[NA][MT];
  float ss[MT] = {};
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    xr[mt] = A.x + (int64_t)min(16 * mt + r, A.M - 1) * A.xs;
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int s = S * wv / NW; s < s1; s += U) {
    uint4 wf[U][NA], xf[U][MT], nf[NORM ? U : 1];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = min(32 * min(s + u, s1 - 1) + 8 * kg, K - 8);
#pragma unroll
      for (int a = 0; a < NA; ++a) wf[u][a] = *reinterpret_cast<const uint4*>(wr + (int64_t)a * N * K + kk);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xf[u][mt] = *reinterpret_cast<const uint4*>(xr[mt] + kk);
      if constexpr (NORM) nf[u] = *reinterpret_cast<const uint4*>(A.nw + kk);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u >= s1) break;  // uniform
      if (32 * (s + u) + 8 * kg >= K) {  // only in the last step of a K that is not a multiple of 32
#pragma unroll
        for (int a = 0; a < NA; ++a) wf[u][a] = uint4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[u][mt] = uint4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        uint4 xl = uint4{0u, 0u, 0u, 0u};
        if constexpr (NORM) norm_frag<LO>(xf[u][mt], xl, nf[u], ss[mt]);
#pragma unroll
        for (int a = 0; a < NA; ++a) {
          acc[a][mt] = mfma(wf[u][a], xf[u][mt], acc[a][mt]);
          if constexpr (LO) acc[a][mt] = mfma(wf[u][a], xl, acc[a][mt]);
        }
      }
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int a = 0; a < NA; ++a) *reinterpret_cast<f32x4*>(&s_acc[wv][a * MT + mt][4 * lane]) = acc[a][mt];
    if constexpr (NORM) {
      ss[mt] += __shfl_xor(ss[mt], 16, 64);
      ss[mt] += __shfl_xor(ss[mt], 32, 64);
      if (lane < 16) s_ss[wv][16 * mt + lane] = ss[mt];
    }
  }
  __syncthreads();
  proj_epilogue<MT, NA, NW, NORM>(A, s_acc, s_ss, A.tr * blockIdx.x);
}

// y = the splits' partial products in order, + bias, + res
__global__ __launch_bounds__(256) void decode_proj_sum_kernel(const ProjArgs A, int splits) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (int64_t)A.M * A.N) return;
  const int m = (int)(e / A.N), n = (int)(e % A.N);
  float o = A.bias ? bf2f(A.bias[n]) : 0.f, v = 0.f;
  for (int s = 0; s < splits; ++s) v += A.part[(int64_t)s * A.M * A.N + e];
  o += v;
  if (A.res) o += bf2f(A.res[(int64_t)m * A.rs + n]);
  A.y[(int64_t)m * A.ys + n] = f2bf(o);
}

// Splits of K for more than 8 rows past the resident form's K: with x streamed beside W by one workgroup per tile,
// the 144 workgroups of N 2304, K 6912 each loaded 442 KB of x and 221 KB of W at 32 rows (32.8 us); three
// splits keep x resident over two tiles (16.6 us with the sum; K 7208, four splits, M 9 / 16: 15.4 / 19.3 us streamed, 12.8 /
// 13.8 split).  At most 8 rows stream: x is small there and the sum's launch costs what it saves (K 4608, N 1536,
// M 8 / 9: 8.2 streamed, 8.0 split).
inline int proj_splits(int M, int N, int K, bool norm, bool gated) {
  const int S = (K + 31) / 32, one = kResWaves * kResSteps;
  if (M <= 8 || norm || gated || S <= one || (int64_t)N * K >= (1ll << 31)) return 1;
  return (S + one - 1) / one;
}

// Tile height and count for `splits` products of N rows on 256 CUs, one workgroup each: as few tiles per workgroup as
// 16-row tiles allow within a split's share of the CUs, then the rows spread evenly (N 2304: 256 tiles of 9 rows,
// where 144 of 16 left 112 CUs idle; N 6912: 494 of 14, two each, where 432 of 16 gave 216 workgroups 32 rows).
// M 1: N 2304 K 6912 15.1 -> 12.4 us, K 2304 5.9 -> 5.3.  Shares: N 2048 in 3 splits runs 3 x 79 workgroups, where rows
// spread over all the CUs alike gave 3 x 86, two too many (K 6144, M 17 / 64: 18.1 / 31.5 -> 13.7 / 20.3 us).
struct ProjShape {
  int tr, tiles, grid;
  ProjShape(int N, int splits) {
    const int cols = splits < 256 ? 256 / splits : 1;  // workgroups of one split, so that all splits run at once
    const int per = (int)(((int64_t)N + 16 * cols - 1) / (16 * cols));
    tr = (int)(((int64_t)N + (int64_t)cols * per - 1) / ((int64_t)cols * per));
    tiles = (N + tr - 1) / tr, grid = (tiles + per - 1) / per;
  }
};

template <int MT, int NA, bool NORM>
void launch_proj(ProjArgs A, hipStream_t stream) {
  const int S = (A.K + 31) / 32;
  // (x of 64 rows fits the registers only without the norm and beside one weight tile)
  if constexpr (MT < 4 || (NA == 1 && !NORM)) {
    // (buffer offsets are 32 bits)
    const bool fits = (int64_t)A.N * A.K < (1ll << 31) && A.xs >= 0 && 64 * A.xs + A.K < (1ll << 31);
    const int splits = proj_splits(A.M, A.N, A.K, NORM, NA == 2);
    if (splits > 1 && fits) {
      if constexpr (NA == 1 && !NORM) {
        const ProjShape p(A.N, splits);
        A.tr = p.tr;
        hipLaunchKernelGGL((decode_proj_resident_kernel<MT, NA, NORM, kResSteps>), dim3(p.grid, splits),
                           dim3(64 * kResWaves), 0, stream, A);
        hipLaunchKernelGGL(decode_proj_sum_kernel, dim3((unsigned)(((int64_t)A.M * A.N + 255) / 256)), dim3(256), 0, stream,
                           A, splits);
        return;
      }
    }
    if (S <= kResWaves * kResSteps && fits) {
      const ProjShape p(A.N, 1);
      A.tr = p.tr;
      const int grid = p.grid;
      if (S <= kResWaves * 4)
        hipLaunchKernelGGL((decode_proj_resident_kernel<MT, NA, NORM, 4>), dim3(grid), dim3(64 * kResWaves), 0, stream, A);
      else
        hipLaunchKernelGGL((decode_proj_resident_kernel<MT, NA, NORM, kResSteps>), dim3(grid), dim3(64 * kResWaves), 0,
                           stream, A);
      return;
    }
  }
  // (beyond 16 rows x is the larger stream, and a tile's rows share it)
  A.part = nullptr;
  A.tr = MT == 1 ? ProjShape(A.N, 1).tr : 16;
  hipLaunchKernelGGL((decode_proj_stream_kernel<MT, NA, NORM>), dim3((A.N + A.tr - 1) / A.tr), dim3(64 * kStrWaves), 0,
                     stream, A);
}
template <int MT>
void launch_proj_m(const ProjArgs& A, int gated, hipStream_t stream) {
  if (gated) {
    if (A.nw) launch_proj<MT, 2, true>(A, stream);
    else launch_proj<MT, 2, false>(A, stream);
  } else {
    if (A.nw) launch_proj<MT, 1, true>(A, stream);
    else launch_proj<MT, 1, false>(A, stream);
  }
}

// ---------------------------------------------------------------------------------------------
// The mixer of one token between its projections, one workgroup per (sequence, head): short convolution
// of q, k, v with the carried inputs (advanced in place), the low-rank second projections of the gates,
// the gate frontend, the Kalman gain (precision advanced in place), the memory update and read
// (memory advanced in place) and the sigmoid-gated RMS norm of the output.
//
// Loads that depend on no other (the state, the decay weights' rows of this head, the projection's slices,
// the carried inputs) are issued first, so the workgroup waits for memory about once; with the steps
// apart each launch waited for its own.  Nothing is rounded between the projections.  H 18, K 128: 9.5 us
// at B 1 (seven launches before), 25 at B 32 (75 MB of state read and written: 16 us at the copy rate; 576
// workgroups, two per CU).  4 D threads: thread t holds columns 4 (t % (D/4)) of the
// state rows t / (D/4) + 16 j, and row t / 4 of the gate weights, a quarter of it.
// ---------------------------------------------------------------------------------------------
struct MixerArgs {
  const bf16_t* p;  // the input projection's rows: q | k | v, then at the offsets below
  int64_t ps;
  int off_f, off_w, off_r, off_g;
  bf16_t* tail[3];
  const bf16_t* cw[3];
  int64_t tail_sb, tail_row;
  const bf16_t *Wf, *Wo, *bo, *Wg, *bg;
  const float *omega_bias, *r_bias, *A_log, *dt_bias;
  float omega_min, r_min, s, scale, eps;
  float *prec, *mem;
  const bf16_t* nw;
  bf16_t* y;
  int H;
};

template <int D>
__device__ __forceinline__ void load_wrow(const bf16_t* W, int64_t row, int part, uint4 (&w)[D / 32]) {
#pragma unroll
  for (int u = 0; u < D / 32; ++u) w[u] = *reinterpret_cast<const uint4*>(W + row * D + 32 * u + 8 * part);
}
// dot of the row with the hidden vector in LDS, the row's 4 threads' quarters added: valid in each
template <int D>
__device__ __forceinline__ float dot_wrow(const uint4 (&w)[D / 32], const float* hid, int part) {
  float a = 0.f;
#pragma unroll
  for (int u = 0; u < D / 32; ++u) {
    float wf[8];
    unpack8(w[u], wf);
#pragma unroll
    for (int e = 0; e < 8; ++e) a = fmaf(wf[e], hid[32 * u + 8 * part + e], a);
  }
  a += __shfl_xor(a, 1, 64);
  a += __shfl_xor(a, 2, 64);
  return a;
}

template <int D, bool ISO>
__global__ __launch_bounds__(4 * D) void decode_mixer_kernel(const MixerArgs A) {
  constexpr int C4 = D / 4, NW = D / 16, R = D / 16;  // column groups, waves, state rows per thread
  __shared__ float s_q[D], s_k[D], s_v[D], s_f[D], s_w[D], s_g[D], s_e[D], s_x[D], s_gate[D];
  __shared__ float4 s_red[2][NW][C4];
  const int b = blockIdx.x / A.H, h = blockIdx.x % A.H, t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t bh = blockIdx.x;
  const int c4 = t % C4, rg = t / C4, row = t >> 2, part = t & 3;
  const bf16_t* p = A.p + b * A.ps;
  // loads
  float* sp = A.mem + bh * D * D + 4 * c4;
  float4 S[R];
#pragma unroll
  for (int j = 0; j < R; ++j) S[j] = *reinterpret_cast<const float4*>(sp + (rg + 16 * j) * D);
  uint4 wf[D / 32], wg[D / 32], wo[ISO ? 1 : D / 32];
  const int64_t wrow = (int64_t)h * D + row;
  load_wrow<D>(A.Wf, wrow, part, wf);
  load_wrow<D>(A.Wg, wrow, part, wg);
  if constexpr (!ISO) load_wrow<D>(A.Wo, wrow, part, wo);
  if (t < 3 * D) {  // one channel of the short convolution
    const int sec = t / D, c = t % D;
    const int64_t ch = (int64_t)h * D + c;
    bf16_t* tl = A.tail[sec] + b * A.tail_sb + ch;
    const uint2 taps = *reinterpret_cast<const uint2*>(A.cw[sec] + 4 * ch);
    const bf16_t x0 = tl[0], x1 = tl[A.tail_row], x2 = tl[2 * A.tail_row];
    const bf16_t x3 = p[(int64_t)sec * A.H * D + ch];
    float a = __uint_as_float(taps.x << 16) * bf2f(x0);
    a += __uint_as_float(taps.x & 0xffff0000u) * bf2f(x1);
    a += __uint_as_float(taps.y << 16) * bf2f(x2);
    a += __uint_as_float(taps.y & 0xffff0000u) * bf2f(x3);
    const float yv = a * sigmoidf(a);
    (sec == 0 ? s_q : sec == 1 ? s_k : s_v)[c] = yv;
    tl[0] = x1, tl[A.tail_row] = x2, tl[2 * A.tail_row] = x3;
  } else {  // D threads: the hidden vectors of the gates
    const int c = t - 3 * D;
    s_f[c] = bf2f(p[A.off_f + c]);
    s_g[c] = bf2f(p[A.off_g + c]);
    if constexpr (!ISO) s_w[c] = bf2f(p[A.off_w + c]);
  }
  __syncthreads();
  const float dt = A.dt_bias[wrow], gb = A.bg ? bf2f(A.bg[wrow]) : 0.f, nwv = bf2f(A.nw[row]);
  const float rate = __expf(A.A_log[h]);
  const float pin = A.prec[ISO ? bh : bh * D + row];
  float r_raw = bf2f(p[A.off_r + (ISO ? A.H : 0) + h]), om_raw = 0.f;
  if constexpr (ISO) om_raw = bf2f(p[A.off_r + h]);
  else om_raw = A.bo ? bf2f(A.bo[wrow]) : 0.f;  // the bias of omega's second projection
  // squared norms of q and k, formed by every wave
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int i = lane; i < D; i += 64) sq = fmaf(s_q[i], s_q[i], sq), sk = fmaf(s_k[i], s_k[i], sk);
  sq = wave_sum(sq), sk = wave_sum(sk);
  float qs, ks;
  if constexpr (ISO) qs = 1.f / sqrtf(sq + 1e-6f), ks = 1.f / sqrtf(sk + 1e-6f);
  else qs = 1.f / fmaxf(sqrtf(sq), 1e-12f), ks = 1.f / fmaxf(sqrtf(sk), 1e-12f);
  // gate frontend of channel `row` (each of its 4 threads)
  const float g_raw = dot_wrow<D>(wf, s_f, part);
  const float gate = dot_wrow<D>(wg, s_g, part) + gb;
  const float r = A.r_min + softplusf(r_raw + (ISO ? A.r_bias[h] : 0.f));
  const float ell = -rate * softplusf(g_raw + dt);
  float ph = 0.f, kgn = 0.f, al = 0.f;
  if constexpr (!ISO) {
    al = expf(ell);
    const float om = softplusf(dot_wrow<D>(wo, s_w, part) + om_raw);
    ph = al * al / pin + om;
    kgn = s_k[row] * ks;
  }
  if (part == 0) {
    s_gate[row] = nwv * sigmoidf(gate);
    if constexpr (ISO) {
      s_e[row] = exp2f(ell * KDN_LOG2E);
      s_x[row] = __expf(2.f * ell);
    } else {
      // the memory path clamps alpha at 1e-6 (NaN propagates)
      s_e[row] = exp2f(((al >= 1e-6f || al != al) ? ell : -13.815510557964274f) * KDN_LOG2E);
      s_x[row] = ph * kgn * kgn;
    }
  }
  __syncthreads();
  float sx = 0.f;
#pragma unroll
  for (int i = lane; i < D; i += 64) sx += s_x[i];
  sx = wave_sum(sx);
  float beta = 0.f;
  if constexpr (ISO) {
    const float z = sx * (1.f / D) * (1.f / pin) + (A.omega_min + softplusf(om_raw + A.omega_bias[h]));
    beta = z / (r + z);
    if (t == 0) A.prec[bh] = (r + A.s * z) / (r * z);  // every thread read it before the last barrier
  } else {
    const float iD = 1.f / (r + sx);
    if (part == 0) {
      s_f[row] = ph * kgn * iD;  // kappa (s_f is free: read before the last barrier)
      A.prec[bh * D + row] = (1.f + A.s * kgn * kgn * (1.f / r) * ph) / ph;
    }
    __syncthreads();
  }
  float4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int i = rg + 16 * j;
    const float kr = s_k[i] * ks, e = s_e[i];
    S[j] = float4{e * S[j].x, e * S[j].y, e * S[j].z, e * S[j].w};
    acc = float4{fmaf(kr, S[j].x, acc.x), fmaf(kr, S[j].y, acc.y), fmaf(kr, S[j].z, acc.z), fmaf(kr, S[j].w, acc.w)};
  }
  // sum over the 16 row groups, valid in every thread
  auto rows_sum = [&](float4 a, int slot) {
#pragma unroll
    for (int o = C4; o < 64; o <<= 1)
      a.x += __shfl_xor(a.x, o, 64), a.y += __shfl_xor(a.y, o, 64), a.z += __shfl_xor(a.z, o, 64),
          a.w += __shfl_xor(a.w, o, 64);
    if (lane < C4) s_red[slot][wv][lane] = a;
    __syncthreads();
    float4 o = s_red[slot][0][c4];
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      const float4 q = s_red[slot][w][c4];
      o.x += q.x, o.y += q.y, o.z += q.z, o.w += q.w;
    }
    return o;
  };
  const float4 kS = rows_sum(acc, 0);
  const float4 v4 = *reinterpret_cast<const float4*>(s_v + 4 * c4);
  const float4 dl{v4.x - kS.x, v4.y - kS.y, v4.z - kS.z, v4.w - kS.w};
  acc = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int i = rg + 16 * j;
    const float kap = ISO ? beta * (s_k[i] * ks) : s_f[i], qr = s_q[i] * qs;
    S[j] = float4{fmaf(kap, dl.x, S[j].x), fmaf(kap, dl.y, S[j].y), fmaf(kap, dl.z, S[j].z), fmaf(kap, dl.w, S[j].w)};
    *reinterpret_cast<float4*>(sp + i * D) = S[j];
    acc = float4{fmaf(qr, S[j].x, acc.x), fmaf(qr, S[j].y, acc.y), fmaf(qr, S[j].z, acc.z), fmaf(qr, S[j].w, acc.w)};
  }
  const float4 ov = rows_sum(acc, 1);
  float o[4] = {ov.x * A.scale, ov.y * A.scale, ov.z * A.scale, ov.w * A.scale}, ss = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) ss = fmaf(o[i], o[i], ss);
#pragma unroll
  for (int x = 1; x < C4; x <<= 1) ss += __shfl_xor(ss, x, 64);
  const float rs = rsqrtf(ss / (float)D + A.eps);
  if (t < C4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] *= rs * s_gate[4 * c4 + i];
    const uint2 w{(uint32_t)f2bf(o[0]) | ((uint32_t)f2bf(o[1]) << 16), (uint32_t)f2bf(o[2]) | ((uint32_t)f2bf(o[3]) << 16)};
    *reinterpret_cast<uint2*>(A.y + bh * D + 4 * c4) = w;
  }
}

bool al(const void* p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

}  // namespace

extern "C" {

size_t kdn_decode_proj_workspace_size(int M, int N, int K, int norm, int gated) {
  if (M <= 0 || M > 64 || N <= 0 || K <= 0) return 0;
  const int splits = proj_splits(M, N, K, norm != 0, gated != 0);
  return splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
}

int kdn_decode_proj(const void* x, int64_t x_row_stride, const void* norm_weight, float eps, const void* W,
                    const void* bias, const void* res, int64_t res_row_stride, int M, int N, int K, int gated, void* y,
                    int64_t y_row_stride, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (M < 0 || M > 64 || N < 0 || K <= 0 || K % 8 || !x || !W || !y || !(eps >= 0.f)) return KDN_ERR_ARG;
  if (M == 0 || N == 0) return 0;
  if (!al(x, 16) || !al(W, 16) || (norm_weight && !al(norm_weight, 16)) || x_row_stride % 8) return KDN_ERR_ARG;
  const size_t need = kdn_decode_proj_workspace_size(M, N, K, norm_weight != nullptr, gated);
  if (need && (!workspace || workspace_bytes < need || !al(workspace, 4))) return KDN_ERR_ARG;
  const ProjArgs a{(const bf16_t*)x, x_row_stride, (const bf16_t*)norm_weight, eps, (const bf16_t*)W,
                   (const bf16_t*)bias, (const bf16_t*)res, res_row_stride, M, N, K, (bf16_t*)y, y_row_stride, need ? (float*)workspace : nullptr, 16};
  if (M <= 16) launch_proj_m<1>(a, gated, stream);
  else if (M <= 32) launch_proj_m<2>(a, gated, stream);
  else launch_proj_m<4>(a, gated, stream);
  KDN_CHECK_LAUNCH();
  return 0;
}

int kdn_decode_mixer(const void* p, int64_t p_row_stride, int off_f, int off_w, int off_r, int off_g, void* tail_q,
                     void* tail_k, void* tail_v, int64_t tail_stride_b, int64_t tail_row_stride, const void* conv_q,
                     const void* conv_k, const void* conv_v, const void* Wf, const void* Wo, const void* bo,
                     const void* Wg, const void* bg, const float* omega_bias, const float* r_bias, const float* A_log,
                     const float* dt_bias, float omega_min, float r_min, float info_scale, float scale,
                     float* precision, float* memory, const void* norm_weight, float eps, int iso, int B, int H, int K,
                     void* y, hipStream_t stream) {
  if (B < 0 || H <= 0 || (K != 64 && K != 128) || !(info_scale > 0.f) || !(eps >= 0.f)) return KDN_ERR_ARG;
  if (B == 0) return 0;
  if (!p || !tail_q || !tail_k || !tail_v || !conv_q || !conv_k || !conv_v || !Wf || !Wg || !A_log || !dt_bias ||
      !precision || !memory || !norm_weight || !y || (iso ? (!omega_bias || !r_bias) : !Wo))
    return KDN_ERR_ARG;
  if (!al(memory, 16) || !al(Wf, 16) || !al(Wg, 16) || (!iso && !al(Wo, 16)) || !al(conv_q, 8) || !al(conv_k, 8) ||
      !al(conv_v, 8) || !al(y, 8))
    return KDN_ERR_ARG;
  MixerArgs a;
  a.p = (const bf16_t*)p, a.ps = p_row_stride;
  a.off_f = off_f, a.off_w = off_w, a.off_r = off_r, a.off_g = off_g;
  a.tail[0] = (bf16_t*)tail_q, a.tail[1] = (bf16_t*)tail_k, a.tail[2] = (bf16_t*)tail_v;
  a.cw[0] = (const bf16_t*)conv_q, a.cw[1] = (const bf16_t*)conv_k, a.cw[2] = (const bf16_t*)conv_v;
  a.tail_sb = tail_stride_b, a.tail_row = tail_row_stride;
  a.Wf = (const bf16_t*)Wf, a.Wo = (const bf16_t*)Wo, a.bo = (const bf16_t*)bo;
  a.Wg = (const bf16_t*)Wg, a.bg = (const bf16_t*)bg;
  a.omega_bias = omega_bias, a.r_bias = r_bias, a.A_log = A_log, a.dt_bias = dt_bias;
  a.omega_min = omega_min, a.r_min = r_min, a.s = iso ? info_scale / (float)K : info_scale, a.scale = scale, a.eps = eps;
  a.prec = precision, a.mem = memory, a.nw = (const bf16_t*)norm_weight, a.y = (bf16_t*)y, a.H = H;
  const dim3 grid((unsigned)(B * H)), block(4 * K);
  if (K == 128) {
    if (iso) hipLaunchKernelGGL((decode_mixer_kernel<128, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((decode_mixer_kernel<128, false>), grid, block, 0, stream, a);
  } else {
    if (iso) hipLaunchKernelGGL((decode_mixer_kernel<64, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((decode_mixer_kernel<64, false>), grid, block, 0, stream, a);
  }
  KDN_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
