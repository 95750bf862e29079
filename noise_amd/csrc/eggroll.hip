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
// to OUTER_MAX matrices in one launch (every perturbed parameter of the model: ~9k 64 x 64 tiles fill the
// GPU, where one 512 x 512 matrix alone is 64 workgroups). On the fp32 MFMA (v_mfma_f32_16x16x4_f32): a
// 64 x 64 output tile per workgroup of 4 waves (32 x 32 each); directions pass through a double-buffered
// LDS stage 32 at a time with w_j folded into the a rows, the next 32 loaded into registers while the
// current ones feed the MFMAs. Every output adds its directions four at a time in increasing order, so a matrix's
// gradient is the same bits alone and beside any others, and infinities and NaN go where the fp32 sum takes them.
// Bound by the fp32 MFMA: the model's 37.7M weights and 1536 directions (116 GFLOP) take 1100 us, 105 TFLOP/s of 157.
// Before, one branch per operand row made each load wait for the last, and the w factors waited for the a rows: 1275 us.
// (128 x 128 tiles, half the operand traffic, measured the same, 1083, and lose where tiles are few or ragged. Three bf16
// planes per operand on the bf16 MFMA take 677, with a smaller error at these sizes, but hold fewer bits of operands
// below 2^-110 and give bits that depend on whether the launch fills the GPU.)
// LDS rows of 64 + 16 floats: the four directions of an MFMA operand fall in four different quarters of the banks.
__global__ void __launch_bounds__(256, 2) outer_update_kernel(const OuterBatchArgs g) {
  constexpr int TILE = OUTER_TILE, TK = 32, LD = TILE + 16, W = TILE / 2, F = W / 16, Q = TILE / 32;
  __shared__ __attribute__((aligned(16))) float sa[2][TK][LD];
  __shared__ __attribute__((aligned(16))) float sb[2][TK][LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, grp = lane >> 4;
  const int wi = wave & 1, wo = wave >> 1;
  // XCD x takes a contiguous range of tiles: the tiles of a matrix share its a and b in that L2
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
  const int o0 = (lt / M.tiles_i) * TILE, i0 = (lt % M.tiles_i) * TILE;
  // loader: thread tid fills direction jj = tid / 8 (of 32), columns 4 (tid % 8) + 32 q .. + 3 of a and of b; 16-byte
  // loads only where every row starts at a 16-byte address
  const int ljj = tid >> 3, lc = 4 * (tid & 7);
  const bool full = M.a && o0 + TILE <= M.out && i0 + TILE <= M.in && M.a_ld % 4 == 0 && M.b_ld % 4 == 0 &&
                    !(((uintptr_t)M.a | (uintptr_t)M.b) & 15);
  float4 ra[Q], rb[Q];
  float rw;  // apart from the a row until it is staged: a use here would wait for the loads
  auto load_row = [&](float4 (&r)[Q], const float* row, int cols) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = lc + 32 * q + e < cols ? (row ? row[lc + 32 * q + e] : 1.f) : 0.f;
      r[q] = make_float4(v[0], v[1], v[2], v[3]);
    }
  };
  auto load = [&](int j0) {
    const int j = j0 + ljj;
    const bool live = j < g.ndir;
    const float *ap = M.a ? M.a + (long)j * M.a_ld + o0 : nullptr, *bp = M.b + (long)j * M.b_ld + i0;
    rw = live ? g.w[j] : 0.f;
    // one branch for both rows: with one each, the second row's loads waited for the first's
    if (full && j0 + TK <= g.ndir) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        ra[q] = *reinterpret_cast<const float4*>(ap + lc + 32 * q);
        rb[q] = *reinterpret_cast<const float4*>(bp + lc + 32 * q);
      }
      return;
    }
    load_row(ra, ap, live ? M.out - o0 : 0);
    load_row(rb, bp, live ? M.in - i0 : 0);
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      *reinterpret_cast<float4*>(&sa[buf][ljj][lc + 32 * q]) =
          make_float4(ra[q].x * rw, ra[q].y * rw, ra[q].z * rw, ra[q].w * rw);
      *reinterpret_cast<float4*>(&sb[buf][ljj][lc + 32 * q]) = rb[q];
    }
  };
  f32x4 acc[F][F];  // [i block][o block]: lane holds i = 4 grp + e, o = lane % 16 of each 16 x 16 block
#pragma unroll
  for (int a = 0; a < F; ++a)
#pragma unroll
    for (int b = 0; b < F; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  load(0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int j0 = 0; j0 < g.ndir; j0 += TK) {
    const bool more = j0 + TK < g.ndir;
    if (more) load(j0 + TK);  // in flight during this chunk's MFMAs
#pragma unroll
    for (int ks = 0; ks < TK / 4; ++ks) {
      const int jj = 4 * ks + grp;
      float bf[F], af[F];
#pragma unroll
      for (int f = 0; f < F; ++f) {
        bf[f] = sb[buf][jj][wi * W + 16 * f + (lane & 15)];
        af[f] = sa[buf][jj][wo * W + 16 * f + (lane & 15)];
      }
#pragma unroll
      for (int a = 0; a < F; ++a)
#pragma unroll
        for (int b = 0; b < F; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[a], af[b], acc[a][b], 0, 0, 0);
    }
    if (more) {
      // the other buffer was last read in the previous chunk, before the barrier that ended it
      stage(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }
  const bool vec = M.in % 4 == 0 && !((uintptr_t)M.grad & 15);
#pragma unroll
  for (int a = 0; a < F; ++a)
#pragma unroll
    for (int b = 0; b < F; ++b) {
      const int o = o0 + wo * W + 16 * b + (lane & 15), i = i0 + wi * W + 16 * a + 4 * grp;
      if (o >= M.out || i >= M.in) continue;
      const f32x4 v = acc[a][b];
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
// m = lerp(m, g, 1 - b1); v = b2 v + (1 - b2) g^2; p -= (lr / bc1) m / (sqrt(v) / sqrt(bc2) + eps), the fused operations
// written out.
// Every tensor of an optimizer step in one launch: block b serves the tensor whose range of ADAM_BLOCK-element blocks
// holds it (a binary search over the running totals; a linear scan took 481 us for the model's tensors). Bound by HBM, 28
// bytes per element. Two elements per thread, every load before the first store: the model's 61 tensors 190 us (5.6 TB/s),
// 37.7M parameters in one tensor 181, off 16-byte addresses 187. (One element per thread 202, 173 and 187; blocks of 2048
// elements in 16-byte vectors 200, 198 and 228, and 5.4 against 4.5 for 100,000 elements.)
// MAX: tensors the arguments hold; one tensor's launch copies 64 bytes of them instead of 3.6 KiB.
template <int MAX>
__global__ void __launch_bounds__(256) adam_batch_kernel(const AdamBatchArgs<MAX> g) {
  constexpr int V = ADAM_BLOCK / 256;
  const long b = blockIdx.x;
  int lo = 0, hi = MAX > 1 ? g.n - 1 : 0;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (b < g.t[mid].block_end) hi = mid;
    else lo = mid + 1;
  }
  const AdamTensor& t = g.t[lo];
  const long i0 = (b - (lo ? g.t[lo - 1].block_end : 0)) * ADAM_BLOCK + threadIdx.x;
  const float w = 1.f - g.beta1;
  float p[V], gr[V], m[V], v[V];
#pragma unroll
  for (int q = 0; q < V; ++q) {
    const long i = i0 + 256 * q;
    if (i < t.n) p[q] = t.param[i], gr[q] = t.grad[i], m[q] = t.m[i], v[q] = t.v[i];
  }
#pragma unroll
  for (int q = 0; q < V; ++q) {
    const long i = i0 + 256 * q;
    if (i >= t.n) return;
    const float d = gr[q] - m[q];
    m[q] = w < 0.5f ? fmaf(w, d, m[q]) : fmaf(-(1.f - w), d, gr[q]);
    v[q] = fmaf(gr[q], (1.f - g.beta2) * gr[q], g.beta2 * v[q]);
    t.m[i] = m[q];
    t.v[i] = v[q];
    t.param[i] = fmaf(-t.step_size, m[q] / (sqrtf(v[q]) / t.bc2_sqrt + g.eps), p[q]);
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
    long tiles = 0;
    for (int k = 0; k < g.n; ++k) {
      const OuterUpdateArgs& u = mats[base + k];
      if (!u.b || !u.grad || u.out <= 0 || u.in <= 0 || (!u.a && u.out != 1) || u.b_ld < u.in ||
          (u.a && u.a_ld < u.out))
        return NOISE_EINVAL;
      OuterMat& m = g.m[k];
      m.a = u.a, m.b = u.b, m.grad = u.grad, m.a_ld = u.a_ld, m.b_ld = u.b_ld, m.out = u.out, m.in = u.in;
      m.tiles_i = (u.in + OUTER_TILE - 1) / OUTER_TILE;
      tiles += (long)((u.out + OUTER_TILE - 1) / OUTER_TILE) * m.tiles_i;
      if (tiles > 0x7fffffffL) return NOISE_ENOTSUP;
      m.tile_end = (int)tiles;
    }
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
  auto launch = [&](auto g, int base, int count) {
    g.n = count;
    g.beta1 = beta1, g.beta2 = beta2, g.eps = eps;
    long blocks = 0;
    for (int k = 0; k < count; ++k) {
      g.t[k] = tensors[base + k];
      blocks += (g.t[k].n + ADAM_BLOCK - 1) / ADAM_BLOCK;
      g.t[k].block_end = (int)blocks;
    }
    hipLaunchKernelGGL(adam_batch_kernel<decltype(g)::MAX_TENSORS>, dim3((unsigned)blocks), dim3(256), 0, s, g);
  };
  for (int base = 0; base < n; base += ADAM_MAX) {
    if (n == 1) launch(AdamBatchArgs<1>{}, base, 1);
    else launch(AdamBatchArgs<ADAM_MAX>{}, base, std::min(ADAM_MAX, n - base));
    NOISE_CHECK_LAUNCH();
  }
  return NOISE_OK;
}
