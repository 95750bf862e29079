// EGGROLL update path: fitness from the antithetic losses, the weighted sum of perturbation outer
// products (the gradient estimate), and Adam.
//
// Reference: Eggroll.step (train/val/eggroll.py:151-167) and torch.optim.AdamW(lr, betas=(0.5, 0.95),
// eps=1e-8, weight_decay=0) (:205). All fp32.
#include <algorithm>

#include "common.h"
#include "eggroll.h"

namespace {

// Z-score fitness in one workgroup (O(n) work): f_j = L[2j+1] - L[2j], divided by (unbiased std + 1e-8) with no
// centering (:151-152).
__global__ void __launch_bounds__(1024) zscore_fitness_kernel(const float* __restrict__ losses, int nf,
                                                              float* __restrict__ fit) {
  __shared__ float red[1024];
  __shared__ float stat;
  const int tid = threadIdx.x;
  for (int j = tid; j < nf; j += 1024) fit[j] = losses[2 * j + 1] - losses[2 * j];
  __syncthreads();
  {
    float s = 0.f;
    for (int j = tid; j < nf; j += 1024) s += fit[j];
    red[tid] = s;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
      if (tid < w) red[tid] += red[tid + w];
      __syncthreads();
    }
    const float mean = red[0] / (float)nf;
    __syncthreads();
    float q = 0.f;
    for (int j = tid; j < nf; j += 1024) {
      const float d = fit[j] - mean;
      q += d * d;
    }
    red[tid] = q;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
      if (tid < w) red[tid] += red[tid + w];
      __syncthreads();
    }
    if (tid == 0) stat = sqrtf(red[0] / (float)(nf - 1)) + 1e-8f;
    __syncthreads();
    const float den = stat;
    for (int j = tid; j < nf; j += 1024) fit[j] = fit[j] / den;
  }
}

// Rank fitness (config-4 option; no reference function), spread over the GPU: LANES threads own f_j and count
// #{i : f_i < f_j or (f_i == f_j and i < j)}, each over every LANES-th f_i, which the workgroup stages through LDS RTILE
// at a time (the groups of LANES threads read the same words: a broadcast). fit_j = rank / (n - 1) - 0.5, ties broken
// by index. One thread per j once its workgroups fill the GPU; 16 before that, where a few workgroups would each walk
// the whole population serially (1536 pairs, 6 workgroups: 45.6 us -> 9.6 with 96).
constexpr int RTILE = 2048;
template <int LANES>
__global__ void __launch_bounds__(256) rank_fitness_kernel(const float* __restrict__ losses, int nf,
                                                           float* __restrict__ fit) {
  __shared__ float tile[RTILE];
  const int j = blockIdx.x * (256 / LANES) + threadIdx.x / LANES, l = threadIdx.x % LANES;
  const float fj = j < nf ? losses[2 * j + 1] - losses[2 * j] : 0.f;
  int r = 0;
  for (int i0 = 0; i0 < nf; i0 += RTILE) {
    const int n = min(RTILE, nf - i0);
    __syncthreads();  // the previous tile has been read by every thread
    for (int i = threadIdx.x; i < n; i += 256) tile[i] = losses[2 * (i0 + i) + 1] - losses[2 * (i0 + i)];
    __syncthreads();
    const int lt = j - i0;  // tile entries i < lt have index i0 + i < j
    for (int i = l; i < n; i += LANES) {
      const float fi = tile[i];
      r += (fi < fj) || (fi == fj && i < lt);
    }
  }
#pragma unroll
  for (int o = 1; o < LANES; o <<= 1) r += __shfl_xor(r, o);
  if (j < nf && l == 0) fit[j] = nf > 1 ? (float)r / (float)(nf - 1) - 0.5f : 0.f;
}

// weight[d] = sum of fit_j over j = d mod pairs, in increasing j (:153-154): one thread per direction.
__global__ void __launch_bounds__(256) fold_fitness_kernel(const float* __restrict__ fit, int nf, int pairs,
                                                           float* __restrict__ weight) {
  const int d = blockIdx.x * 256 + threadIdx.x;
  if (d >= pairs) return;
  float s = 0.f;
  for (int j = d; j < nf; j += pairs) s += fit[j];
  weight[d] = s;
}

// G[o, i] = scale * sum_j (w_j a_j[o]) b_j[i] over ndir directions (a null: a_j[o] = 1, out = 1), for up
// to OUTER_MAX matrices in one launch, where they make fewer 128 x 128 tiles than CUs (outer_split_kernel otherwise). On
// the fp32 MFMA (v_mfma_f32_16x16x4_f32): a 64 x 64 output tile per workgroup of 4 waves (32 x 32 each); directions pass
// through a double-buffered LDS stage 32 at a time with w_j folded into the a rows, the next 32 loaded into registers
// while the current ones feed the MFMAs.
__global__ void __launch_bounds__(256) outer_update_kernel(const OuterBatchArgs g) {
  constexpr int TK = 32, LD = 64 + 4;
  __shared__ __attribute__((aligned(16))) float sa[2][TK][LD];
  __shared__ __attribute__((aligned(16))) float sb[2][TK][LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // this workgroup's matrix and tile (uniform scan over the prefix sums of tile counts)
  const int t = blockIdx.x;
  int mi = 0;
  while (mi + 1 < g.n && t >= g.m[mi].tile_end) ++mi;
  const OuterMat& M = g.m[mi];
  const int lt = t - (mi ? g.m[mi - 1].tile_end : 0);
  const int o0 = (lt / M.tiles_i) * 64, i0 = (lt % M.tiles_i) * 64;
  // loader: thread tid fills direction jj = tid / 8 (of 32), columns 8 (tid % 8) .. + 7 of a and of b
  const int ljj = tid >> 3, lc = 8 * (tid & 7);
  const bool a_full = M.a && o0 + 64 <= M.out && M.a_ld % 4 == 0, b_full = i0 + 64 <= M.in && M.b_ld % 4 == 0;
  float ra[8], rb[8];
  auto load = [&](int j0) {
    const int j = j0 + ljj;
    const bool live = j < g.ndir;
    const float wj = live ? g.w[j] : 0.f;
    if (live && a_full) {
      const float4 x0 = *reinterpret_cast<const float4*>(M.a + (long)j * M.a_ld + o0 + lc);
      const float4 x1 = *reinterpret_cast<const float4*>(M.a + (long)j * M.a_ld + o0 + lc + 4);
      ra[0] = x0.x, ra[1] = x0.y, ra[2] = x0.z, ra[3] = x0.w, ra[4] = x1.x, ra[5] = x1.y, ra[6] = x1.z, ra[7] = x1.w;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        ra[e] = live && o0 + lc + e < M.out ? (M.a ? M.a[(long)j * M.a_ld + o0 + lc + e] : 1.f) : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ra[e] *= wj;
    if (live && b_full) {
      const float4 x0 = *reinterpret_cast<const float4*>(M.b + (long)j * M.b_ld + i0 + lc);
      const float4 x1 = *reinterpret_cast<const float4*>(M.b + (long)j * M.b_ld + i0 + lc + 4);
      rb[0] = x0.x, rb[1] = x0.y, rb[2] = x0.z, rb[3] = x0.w, rb[4] = x1.x, rb[5] = x1.y, rb[6] = x1.z, rb[7] = x1.w;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) rb[e] = live && i0 + lc + e < M.in ? M.b[(long)j * M.b_ld + i0 + lc + e] : 0.f;
    }
  };
  auto stage = [&](int buf) {
    *reinterpret_cast<float4*>(&sa[buf][ljj][lc]) = make_float4(ra[0], ra[1], ra[2], ra[3]);
    *reinterpret_cast<float4*>(&sa[buf][ljj][lc + 4]) = make_float4(ra[4], ra[5], ra[6], ra[7]);
    *reinterpret_cast<float4*>(&sb[buf][ljj][lc]) = make_float4(rb[0], rb[1], rb[2], rb[3]);
    *reinterpret_cast<float4*>(&sb[buf][ljj][lc + 4]) = make_float4(rb[4], rb[5], rb[6], rb[7]);
  };
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  load(0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int j0 = 0; j0 < g.ndir; j0 += TK) {
    const bool more = j0 + TK < g.ndir;
    if (more) load(j0 + TK);  // in flight during this chunk's MFMAs
#pragma unroll
    for (int ks = 0; ks < TK / 4; ++ks) {
      const int jj = 4 * ks + (lane >> 4);
      float af[2], bf[2];
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        af[f] = sa[buf][jj][wm * 32 + 16 * f + (lane & 15)];
        bf[f] = sb[buf][jj][wn * 32 + 16 * f + (lane & 15)];
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[a], bf[b], acc[a][b], 0, 0, 0);
    }
    if (more) {
      // the other buffer was last read in the previous chunk, before the barrier that ended it
      stage(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }
  // lane holds C[row = 4 (lane / 16) + e][col = lane % 16] of each 16 x 16 block
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int o = o0 + wm * 32 + 16 * a + 4 * (lane >> 4) + e, i = i0 + wn * 32 + 16 * b + (lane & 15);
        if (o < M.out && i < M.in) M.grad[(long)o * M.in + i] = g.scale * acc[a][b][e];
      }
}

// The same sums on the bf16 MFMA, for updates that fill the GPU with 128 x 128 tiles. An fp32 value is
// the sum of three bf16 (8 significant bits each: a1 = bf16(a), a2 = bf16(a - a1), a3 = bf16(a - a1 - a2), both
// differences exact), and a b is a1 b1 + (a1 b2 + a2 b1) + (a1 b3 + a2 b2 + a3 b1) up to terms below 2^-25 |a b|, each
// product exact in the fp32 accumulation. Six bf16 MFMAs of 32 directions take 96 cycles where eight fp32 ones take 256,
// and the sum rounds 6 times per 32 directions instead of 8: its error against 64 bits is the smaller one at every
// population measured (relative, N(0, 1) rows: 16 directions 5.5e-8 against 8.5e-8 of the fp32 kernel, 256 2.4e-7 against
// 2.9e-7, 1536 6.1e-7 against 7.1e-7). The model's 37.7M weights: 1536 directions 1227 -> 656 us, 256 230 -> 129, 64
// 93 -> 57, 16 68 -> 48.
// A workgroup of 4 waves owns a 128 x 128 tile (64 x 64 per wave; half the operand traffic per product of 64 x 64 tiles,
// which held the fp32 kernel at half its peak); the tiles of an XCD are consecutive, so the tiles of a matrix share its
// a and b in that L2. A thread loads 4 directions x 4 columns of each operand, 32 directions ahead, splits them in
// registers and writes the planes transposed to rows of 32 directions. LDS row r of a plane sits in 64-byte slot (r % 4) ^
// (r / 16 % 4) of its group of four, 16-byte chunk c at c ^ (r / 4 % 4): a fragment's 16 rows fall in distinct banks, and
// a store's 64 lanes two to a bank.
// Infinities and NaN (and values beyond bf16's largest, which round to infinity) do not survive the split as they would
// an fp32 sum: a tile with a non-finite result is summed again in fp32.
constexpr int OS_TILE = 128, OS_TK = 32, OS_PLANE = OS_TILE * OS_TK;
__device__ __forceinline__ int os_row(int r) { return (r >> 2) * 128 + (((r & 3) ^ ((r >> 4) & 3)) << 5); }
__device__ __forceinline__ int os_at(int r, int c) { return os_row(r) + ((c ^ ((r >> 2) & 3)) << 3); }
__device__ __forceinline__ float bf16_hi(unsigned pair) { return __uint_as_float(pair & 0xffff0000u); }
__device__ __forceinline__ float bf16_lo(unsigned pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  bf16x2 p = {to_bf16(a), to_bf16(b)};
  return *reinterpret_cast<unsigned*>(&p);
}
__global__ void __launch_bounds__(256, 2) outer_split_kernel(const OuterBatchArgs g) {
  __shared__ __attribute__((aligned(16))) bf16 sp[2][3][OS_PLANE];  // operand (0: b rows i, 1: w a rows o), plane
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, grp = lane >> 4;
  const int wi = wave & 1, wo = wave >> 1;
  // XCD x takes a contiguous range of tiles
  const unsigned G = gridDim.x, bl = blockIdx.x, x = bl & 7, qg = G >> 3, rg = G & 7;
  const int t = (int)(x * qg + min(x, rg) + (bl >> 3));
  int mi = 0, hi = g.n - 1;
  while (mi < hi) {
    const int mid = (mi + hi) >> 1;
    if (t < g.m[mid].tile_end) hi = mid;
    else mi = mid + 1;
  }
  const OuterMat& M = g.m[mi];
  const int lt = t - (mi ? g.m[mi - 1].tile_end : 0);
  const int o0 = (lt / M.tiles_i) * OS_TILE, i0 = (lt % M.tiles_i) * OS_TILE;
  // loader: directions 4 jg .. 4 jg + 3 of the 32, columns 4 q .. 4 q + 3 of the 128
  const int q = tid & 31, jg = tid >> 5;
  // 16-byte loads only where every row starts at a 16-byte address
  const bool full = M.a && o0 + OS_TILE <= M.out && i0 + OS_TILE <= M.in && M.a_ld % 4 == 0 && M.b_ld % 4 == 0 &&
                    !(((uintptr_t)M.a | (uintptr_t)M.b) & 15);
  // the w factors stay apart until the rows are staged: a use here would wait for the loads
  float4 ra[4], rb[4];
  float rw[4];
  auto load = [&](int j0) {
    const int j = j0 + 4 * jg;
    if (full && j0 + OS_TK <= g.ndir) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        rw[d] = g.w[j + d];
        ra[d] = *reinterpret_cast<const float4*>(M.a + (long)(j + d) * M.a_ld + o0 + 4 * q);
        rb[d] = *reinterpret_cast<const float4*>(M.b + (long)(j + d) * M.b_ld + i0 + 4 * q);
      }
      return;
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const bool live = j + d < g.ndir;
      const int na = live ? M.out - o0 - 4 * q : 0, nb = live ? M.in - i0 - 4 * q : 0;
      const float* ap = M.a ? M.a + (long)(j + d) * M.a_ld + o0 + 4 * q : nullptr;
      const float* bp = M.b + (long)(j + d) * M.b_ld + i0 + 4 * q;
      float av[4], bv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        av[e] = e < na ? (ap ? ap[e] : 1.f) : 0.f;
        bv[e] = e < nb ? bp[e] : 0.f;
      }
      rw[d] = live ? g.w[j + d] : 0.f;
      ra[d] = make_float4(av[0], av[1], av[2], av[3]);
      rb[d] = make_float4(bv[0], bv[1], bv[2], bv[3]);
    }
  };
  // one column's four directions, split into the three planes: 8 bytes each
  auto put = [&](int op, int row, float v0, float v1, float v2, float v3) {
    bf16* p = &sp[op][0][os_at(row, jg >> 1) + 4 * (jg & 1)];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const unsigned lo = pack_bf16(v0, v1), hw = pack_bf16(v2, v3);
      *reinterpret_cast<uint2*>(p + k * OS_PLANE) = make_uint2(lo, hw);
      v0 -= bf16_lo(lo), v1 -= bf16_hi(lo), v2 -= bf16_lo(hw), v3 -= bf16_hi(hw);
    }
  };
  auto stage = [&]() {
    put(0, 4 * q, rb[0].x, rb[1].x, rb[2].x, rb[3].x);
    put(0, 4 * q + 1, rb[0].y, rb[1].y, rb[2].y, rb[3].y);
    put(0, 4 * q + 2, rb[0].z, rb[1].z, rb[2].z, rb[3].z);
    put(0, 4 * q + 3, rb[0].w, rb[1].w, rb[2].w, rb[3].w);
    put(1, 4 * q, ra[0].x * rw[0], ra[1].x * rw[1], ra[2].x * rw[2], ra[3].x * rw[3]);
    put(1, 4 * q + 1, ra[0].y * rw[0], ra[1].y * rw[1], ra[2].y * rw[2], ra[3].y * rw[3]);
    put(1, 4 * q + 2, ra[0].z * rw[0], ra[1].z * rw[1], ra[2].z * rw[2], ra[3].z * rw[3]);
    put(1, 4 * q + 3, ra[0].w * rw[0], ra[1].w * rw[1], ra[2].w * rw[2], ra[3].w * rw[3]);
  };
  f32x4 acc[4][4];  // [i block][o block]: lane holds i = 4 grp + e, o = lane % 16 of each 16 x 16 block
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  load(0);
  for (int j0 = 0; j0 < g.ndir; j0 += OS_TK) {
    if (j0) __syncthreads();  // the previous planes have been read
    stage();
    __syncthreads();
    if (j0 + OS_TK < g.ndir) load(j0 + OS_TK);  // in flight during this chunk's MFMAs
    bf16x8 fb[4][3];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        fb[a][k] = *reinterpret_cast<const bf16x8*>(&sp[0][k][os_at(64 * wi + 16 * a + (lane & 15), grp)]);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      bf16x8 fa[3];
#pragma unroll
      for (int k = 0; k < 3; ++k)
        fa[k] = *reinterpret_cast<const bf16x8*>(&sp[1][k][os_at(64 * wo + 16 * b + (lane & 15), grp)]);
      // the smallest terms first
#pragma unroll
      for (int s = 2; s >= 0; --s)
#pragma unroll
        for (int k = 0; k <= s; ++k)
#pragma unroll
          for (int a = 0; a < 4; ++a) acc[a][b] = mfma16x16x32(fb[a][k], fa[s - k], acc[a][b]);
    }
  }
  bool bad = false;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) bad |= !(fabsf(acc[a][b][e]) < INFINITY);
  bad = __syncthreads_or(bad);
  const bool vec = M.in % 4 == 0 && !((uintptr_t)M.grad & 15);
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int o = o0 + 64 * wo + 16 * b + (lane & 15), i = i0 + 64 * wi + 16 * a + 4 * grp;
      if (o >= M.out || i >= M.in) continue;
      float v[4] = {acc[a][b][0], acc[a][b][1], acc[a][b][2], acc[a][b][3]};
      if (bad) {
        const int n = min(4, M.in - i);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float sum = 0.f;
          for (int j = 0; j < g.ndir && e < n; ++j)
            sum = fmaf(g.w[j] * (M.a ? M.a[(long)j * M.a_ld + o] : 1.f), M.b[(long)j * M.b_ld + i + e], sum);
          v[e] = sum;
        }
      }
      float* out = M.grad + (long)o * M.in + i;
      if (vec) {
        *reinterpret_cast<float4*>(out) = make_float4(g.scale * v[0], g.scale * v[1], g.scale * v[2], g.scale * v[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i + e < M.in) out[e] = g.scale * v[e];
      }
    }
}

// torch.optim.AdamW (single-tensor path) with weight_decay = 0:
// m = lerp(m, g, 1 - b1); v = b2 v + (1 - b2) g^2; p -= (lr / bc1) m / (sqrt(v) / sqrt(bc2) + eps).
struct AdamConst {
  float step_size, bc2_sqrt, beta1, beta2, eps;
};
__device__ __forceinline__ void adam_element(float& param, float gr, float& m, float& v, const AdamConst& c) {
  // the fused operations are written out, so that the vector and the scalar path round alike
  const float w = 1.f - c.beta1, d = gr - m;
  m = w < 0.5f ? fmaf(w, d, m) : fmaf(-(1.f - w), d, gr);
  v = fmaf(gr, (1.f - c.beta2) * gr, c.beta2 * v);
  const float denom = sqrtf(v) / c.bc2_sqrt + c.eps;
  param = fmaf(-c.step_size, m / denom, param);
}
// Every tensor of an optimizer step in one launch: block b serves the tensor whose range of ADAM_BLOCK-element blocks
// holds it (a binary search over the running totals). Bound by HBM, 28 bytes per element. Four elements per thread and
// access where the tensor's four pointers allow 16-byte vectors, two of them in flight before any is used: 37.7M
// parameters 497 us (2.1 TB/s) with one element per thread -> 176 us
// (6.0 TB/s).
__global__ void __launch_bounds__(256) adam_batch_kernel(const AdamBatchArgs g) {
  const long b = blockIdx.x;
  int lo = 0, hi = g.n - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (b < g.t[mid].block_end) hi = mid;
    else lo = mid + 1;
  }
  const AdamTensor& t = g.t[lo];
  const AdamConst c{t.step_size, t.bc2_sqrt, g.beta1, g.beta2, g.eps};
  const long base = (b - (lo ? g.t[lo - 1].block_end : 0)) * ADAM_BLOCK;
  if (t.vec && base + ADAM_BLOCK <= t.n) {
    constexpr int V = ADAM_BLOCK / 1024;
    float4 p4[V], g4[V], m4[V], v4[V];
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const long i = base + 1024 * q + 4 * threadIdx.x;
      p4[q] = *reinterpret_cast<const float4*>(t.param + i);
      g4[q] = *reinterpret_cast<const float4*>(t.grad + i);
      m4[q] = *reinterpret_cast<const float4*>(t.m + i);
      v4[q] = *reinterpret_cast<const float4*>(t.v + i);
    }
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const long i = base + 1024 * q + 4 * threadIdx.x;
      adam_element(p4[q].x, g4[q].x, m4[q].x, v4[q].x, c);
      adam_element(p4[q].y, g4[q].y, m4[q].y, v4[q].y, c);
      adam_element(p4[q].z, g4[q].z, m4[q].z, v4[q].z, c);
      adam_element(p4[q].w, g4[q].w, m4[q].w, v4[q].w, c);
      *reinterpret_cast<float4*>(t.param + i) = p4[q];
      *reinterpret_cast<float4*>(t.m + i) = m4[q];
      *reinterpret_cast<float4*>(t.v + i) = v4[q];
    }
    return;
  }
  for (long i = base + threadIdx.x; i < min(base + ADAM_BLOCK, t.n); i += 256) {
    float p = t.param[i], m = t.m[i], v = t.v[i];
    adam_element(p, t.grad[i], m, v, c);
    t.param[i] = p;
    t.m[i] = m;
    t.v[i] = v;
  }
}

}  // namespace

int fitness_launch(const float* losses, int n, int pairs, int mode, float* fit, float* weight, hipStream_t s) {
  if (!losses || !fit || !weight || n < 4 || n % 2 || pairs <= 0 ||
      (mode != NOISE_FITNESS_ZSCORE && mode != NOISE_FITNESS_RANK))
    return NOISE_EINVAL;
  const int nf = n / 2;
  if (mode == NOISE_FITNESS_ZSCORE)
    hipLaunchKernelGGL(zscore_fitness_kernel, dim3(1), dim3(1024), 0, s, losses, nf, fit);
  else if ((nf + 255) / 256 < num_cus())
    hipLaunchKernelGGL(rank_fitness_kernel<16>, dim3((unsigned)((nf + 15) / 16)), dim3(256), 0, s, losses, nf, fit);
  else
    hipLaunchKernelGGL(rank_fitness_kernel<1>, dim3((unsigned)((nf + 255) / 256)), dim3(256), 0, s, losses, nf, fit);
  NOISE_CHECK_LAUNCH();
  hipLaunchKernelGGL(fold_fitness_kernel, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, s, fit, nf, pairs,
                     weight);
  NOISE_CHECK_LAUNCH();
  return NOISE_OK;
}

namespace {
// One workgroup per (direction j, parameter k): copies the out + in floats of the parameter's slice for pair
// directions[j]. A direction or offset outside its range writes NaN rows (never an out-of-bounds read).
__global__ void __launch_bounds__(256) gather_rows_kernel(const GatherArgs g) {
  const int j = blockIdx.x, k = blockIdx.y, tid = threadIdx.x;
  const GatherParam& q = g.p[k];
  const long d = g.directions[j];
  const long off = (d >= 0 && d < g.pairs) ? q.offsets[d] : -1;
  const bool ok = off >= 0 && off <= g.buffer_len - (long)(q.out + q.in);
  const float* src = g.buffer + (ok ? off : 0);
  for (int c = tid; c < q.out; c += 256) q.a[(long)j * q.out + c] = ok ? src[c] : __builtin_nanf("");
  for (int c = tid; c < q.in; c += 256) q.b[(long)j * q.in + c] = ok ? src[q.out + c] : __builtin_nanf("");
}
}  // namespace

int gather_rows_launch(const GatherParam* params, int n, const float* buffer, long buffer_len,
                       const int64_t* directions, int ndir, int pairs, hipStream_t s) {
  if (n <= 0 || !params || !buffer || buffer_len <= 0 || !directions || ndir <= 0 || pairs <= 0) return NOISE_EINVAL;
  if (ndir > 0x7fffffff) return NOISE_ENOTSUP;
  for (int base = 0; base < n; base += GATHER_MAX) {
    GatherArgs g{};
    g.n = std::min(GATHER_MAX, n - base);
    g.buffer = buffer;
    g.buffer_len = buffer_len;
    g.directions = directions;
    g.ndir = ndir;
    g.pairs = pairs;
    for (int k = 0; k < g.n; ++k) {
      const GatherParam& q = params[base + k];
      if (!q.offsets || !q.a || q.out <= 0 || q.in < 0 || (q.in > 0 && !q.b)) return NOISE_EINVAL;
      g.p[k] = q;
    }
    hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)ndir, (unsigned)g.n), dim3(256), 0, s, g);
    NOISE_CHECK_LAUNCH();
  }
  return NOISE_OK;
}

int outer_update_launch(const OuterUpdateArgs* mats, int n, const float* w, int ndir, float scale, hipStream_t s) {
  if (n <= 0 || !mats || !w || ndir <= 0) return NOISE_EINVAL;
  for (int base = 0; base < n; base += OUTER_MAX) {
    OuterBatchArgs g{};
    g.n = std::min(OUTER_MAX, n - base);
    g.w = w;
    g.ndir = ndir;
    g.scale = scale;
    auto tiles_of = [&](int tile) {
      long tiles = 0;
      for (int k = 0; k < g.n; ++k) {
        OuterMat& m = g.m[k];
        m.tiles_i = (m.in + tile - 1) / tile;
        tiles += (long)((m.out + tile - 1) / tile) * m.tiles_i;
        m.tile_end = (int)std::min(tiles, 0x7fffffffL);
      }
      return tiles;
    };
    for (int k = 0; k < g.n; ++k) {
      const OuterUpdateArgs& u = mats[base + k];
      if (!u.b || !u.grad || u.out <= 0 || u.in <= 0 || (!u.a && u.out != 1) || u.b_ld < u.in ||
          (u.a && u.a_ld < u.out))
        return NOISE_EINVAL;
      OuterMat& m = g.m[k];
      m.a = u.a, m.b = u.b, m.grad = u.grad, m.a_ld = u.a_ld, m.b_ld = u.b_ld, m.out = u.out, m.in = u.in;
    }
    long tiles = tiles_of(OS_TILE);
    // at least one 128 x 128 tile per CU: below that the smaller tiles of the fp32 kernel fill the GPU better (one
    // 512 x 512 matrix, 1536 directions: 67 us on 64 tiles against 89 on 16)
    const bool split = tiles >= num_cus();
    if (!split) tiles = tiles_of(64);
    if (tiles > 0x7fffffffL) return NOISE_ENOTSUP;
    if (split)
      hipLaunchKernelGGL(outer_split_kernel, dim3((unsigned)tiles), dim3(256), 0, s, g);
    else
      hipLaunchKernelGGL(outer_update_kernel, dim3((unsigned)tiles), dim3(256), 0, s, g);
    NOISE_CHECK_LAUNCH();
  }
  return NOISE_OK;
}

int adam_batch_launch(const AdamTensor* tensors, int n, float beta1, float beta2, float eps, hipStream_t s) {
  if (n <= 0 || !tensors) return NOISE_EINVAL;
  // every tensor and every chunk's block count is checked before the first launch: a rejected call updates nothing
  for (int base = 0; base < n; base += ADAM_MAX) {
    long blocks = 0;
    for (int k = base; k < std::min(n, base + ADAM_MAX); ++k) {
      const AdamTensor& t = tensors[k];
      if (!t.param || !t.grad || !t.m || !t.v || t.n <= 0 || !(t.bc2_sqrt > 0.f)) return NOISE_EINVAL;
      blocks += (t.n + ADAM_BLOCK - 1) / ADAM_BLOCK;
    }
    if (blocks > 0x7fffffffL) return NOISE_ENOTSUP;
  }
  for (int base = 0; base < n; base += ADAM_MAX) {
    AdamBatchArgs g{};
    g.n = std::min(ADAM_MAX, n - base);
    g.beta1 = beta1, g.beta2 = beta2, g.eps = eps;
    long blocks = 0;
    for (int k = 0; k < g.n; ++k) {
      AdamTensor& t = g.t[k] = tensors[base + k];
      t.vec = !(((uintptr_t)t.param | (uintptr_t)t.grad | (uintptr_t)t.m | (uintptr_t)t.v) & 15);
      blocks += (t.n + ADAM_BLOCK - 1) / ADAM_BLOCK;
      t.block_end = (int)blocks;
    }
    hipLaunchKernelGGL(adam_batch_kernel, dim3((unsigned)blocks), dim3(256), 0, s, g);
    NOISE_CHECK_LAUNCH();
  }
  return NOISE_OK;
}
