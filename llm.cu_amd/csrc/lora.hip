// lora.hip — rank-16 adapter kernels: the dA/dB reductions over tokens, one
// multi-tensor AdamW over the whole fp32 adapter arena (which also refreshes
// the fp16 operand copies the GEMMs read), and the seeded initialiser.
//
// Reference: LoRA grads src/kernels/lora_backward.cu:50-90 (two TN GEMMs per
// adapter through matmul_tn_forward, src/kernels/matmul.cu:102-138, plus
// scale_add_inplace, src/kernels/lora.cu:10-18); AdamW
// src/kernels/lora.cu:206-246 (224 launches per step); init
// src/kernels/lora.cu:32-62 (cuRAND, not reproduced: this library draws its
// own seeded normals).
#include <algorithm>
#include <type_traits>

#include "ops.h"

namespace llmt {

namespace {

constexpr int R = 16;
constexpr int NTH = 256;

// One adapter-gradient job: out = (acc ? out : 0) + lscale * X^T G over the T
// token rows, for the ncols columns of X and the 16 columns of G.
//   dA [16, d_in]:  X = adapter input (xn or o, fp16), G = dh  -> out[r][c]
//   dB [d_out, 16]: X = upstream grad dy,              G = h   -> out[c][r]
// (dy as the fp16 GEMM operand, row t scaled by the power of two 1 / xs[t],
// which the G row takes back exactly).
struct LoraGradGrid {
  int block_start[kLoraJobs + 1];  // column blocks of each job within a layer
};

// The reduction on the matrix cores in fp32 (v_mfma_f32_16x16x4_f32:
// out[r][c] = sum over 4 tokens k of G[k][r] X[k][c], so no operand needs a
// transposition).  Lane l reads G[t + l / 16][l % 16] (times the row factor)
// as its A value and CPL consecutive columns c .., c = CPL (l % 16), of X[t +
// l / 16] as its B values of the CPL MFMA column tiles (tile nb, MFMA column
// n stands for column CPL n + nb), so both loads are contiguous rows.
//
// Bound by its loads (fp32 MFMA floor 0.34 ms for 28 layers at T = 4096, the
// bytes 0.4 ms): the loads of the next MG_U quads are kept as they come
// (fp16 X, G and its factor apart) and converted where they are used --
// converting at the load made every MFMA batch wait for the batch after it
// (28 layers at T = 4096 1043 -> 827 us with 2 waves, T = 512 142 -> 104).
// Splitting the tokens over a workgroup's waves instead of 256 columns over
// 56 workgroups took one layer from 213 to 38 us at T = 4096, 28 layers from
// 857 to 676 (T = 512 162 -> 91, T = 128 46 -> 35).
constexpr int MG_U = 4;  // token quads a wave loads ahead

// Tokens [t0, t1) of one wave.
template <int CPL>
__device__ __forceinline__ void lora_grad_acc(const LoraGradJob& jb, int t0, int t1, int col,
                                              floatx4 (&acc)[CPL]) {
  typedef _Float16 xvec __attribute__((ext_vector_type(CPL)));
  const int lane = threadIdx.x & 63, kq = lane >> 4, r = lane & 15;
  if (t0 >= t1) return;
  const _Float16* X = jb.X + col;
  const float* Gc = jb.G + r;
  float gv[MG_U], fv[MG_U];
  xvec xv[MG_U];
  auto load = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < MG_U; ++u) {
      const int tc = min(tb + 4 * u + kq, t1 - 1);
      fv[u] = jb.xs ? jb.xs[tc] : 1.0f;
      gv[u] = Gc[(long long)tc * jb.ldg];
      xv[u] = *reinterpret_cast<const xvec*>(X + (long long)tc * jb.ldx);
    }
  };
  load(t0);
  for (int tb = t0; tb < t1; tb += 4 * MG_U) {
    float g_c[MG_U];
    xvec x_c[MG_U];
#pragma unroll
    for (int u = 0; u < MG_U; ++u) {
      // tokens past t1 get a zero G value, so they add nothing
      g_c[u] = tb + 4 * u + kq < t1 ? gv[u] * fv[u] : 0.f;
      x_c[u] = xv[u];
    }
    if (tb + 4 * MG_U < t1) load(tb + 4 * MG_U);
#pragma unroll
    for (int u = 0; u < MG_U; ++u)
#pragma unroll
      for (int nb = 0; nb < CPL; ++nb)
        acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(g_c[u], (float)x_c[u][nb], acc[nb], 0, 0, 0);
  }
}

// W waves a workgroup split the tokens into contiguous ranges, all over the
// same GC = 16 CPL columns; the W partial 16 x GC blocks are added in LDS in
// wave order.
template <int W, int CPL>
__global__ __launch_bounds__(W * 64) void lora_grad_kernel(const LoraGradJob* __restrict__ jobs,
                                                           const LoraGradGrid G, int T,
                                                           float lscale, int accumulate) {
  constexpr int GC = 16 * CPL;
  const int bpl = G.block_start[kLoraJobs];
  const int layer = (int)blockIdx.x / bpl, lb = (int)blockIdx.x - layer * bpl;
  int j = 0;
#pragma unroll
  for (int i = 1; i < kLoraJobs; ++i)
    if (lb >= G.block_start[i]) j = i;
  const LoraGradJob jb = jobs[layer * kLoraJobs + j];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cb = (lb - G.block_start[j]) * GC;
  const int tw = ((T + 4 * W - 1) / (4 * W)) * 4;  // tokens a wave, whole quads
  const int cc = min(cb + CPL * (lane & 15), jb.ncols - CPL);
  floatx4 acc[CPL];
#pragma unroll
  for (int nb = 0; nb < CPL; ++nb) acc[nb] = floatx4{0.f, 0.f, 0.f, 0.f};
  lora_grad_acc<CPL>(jb, w * tw, min(T, (w + 1) * tw), cc, acc);
  // lane: ranks 4 (l / 16) + i of its CPL columns; the block in the order it
  // is stored in: out[col][16] (dB) or out[16][col] (dA)
  __shared__ __attribute__((aligned(16))) float red[W][R * GC];
  const int r0 = 4 * (lane >> 4), n = lane & 15;
  if (jb.out_is_B) {
#pragma unroll
    for (int nb = 0; nb < CPL; ++nb)
      *reinterpret_cast<floatx4*>(&red[w][(CPL * n + nb) * R + r0]) = acc[nb];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int nb = 0; nb < CPL; nb += 4)
        *reinterpret_cast<float4*>(&red[w][(r0 + i) * GC + CPL * n + nb]) =
            make_float4(acc[nb][i], acc[nb + 1][i], acc[nb + 2][i], acc[nb + 3][i]);
  }
  __syncthreads();
  for (int e = 4 * threadIdx.x; e < R * GC; e += 4 * W * 64) {
    float4 v = *reinterpret_cast<const float4*>(&red[0][e]);
#pragma unroll
    for (int q = 1; q < W; ++q) {
      const float4 x = *reinterpret_cast<const float4*>(&red[q][e]);
      v = make_float4(v.x + x.x, v.y + x.y, v.z + x.z, v.w + x.w);
    }
    const int col = cb + (jb.out_is_B ? e / R : e % GC);
    if (col >= jb.ncols) continue;
    float4* o = reinterpret_cast<float4*>(
        jb.out + (jb.out_is_B ? (long long)cb * R + e : (long long)(e / GC) * jb.ncols + col));
    const float4 prev = accumulate ? *o : make_float4(0.f, 0.f, 0.f, 0.f);
    *o = make_float4(prev.x + lscale * v.x, prev.y + lscale * v.y, prev.z + lscale * v.z,
                     prev.w + lscale * v.w);
  }
}

// Arena element i -> (shadow block offset within the layer, row, column,
// row length) of its fp16 copies; the packed copy (a GEMM B operand) holds it
// at packed_index(row, col, len), the row-major twin at row * len + col.
struct ShadowPos {
  long long base;  // layer base + block offset
  long long row, col;
  int len;
};
__device__ __forceinline__ ShadowPos shadow_pos(const AdamShadow& sh, long long i) {
  const long long l = i / sh.per_layer;
  long long j = i - l * sh.per_layer;
  int s = 0;
#pragma unroll
  for (int k = 1; k < 8; ++k)
    if (j >= sh.seg_off[k]) s = k;
  j -= sh.seg_off[s];
  const int p = s >> 1;  // q, k, v, o
  const long long base = l * sh.shadow_per_layer;
  if ((s & 1) == 0) {  // A [16, d_in]: row r, column cc
    const int d_in = sh.d_in[p];
    const long long r = j / d_in, cc = j - r * d_in;
    if (p < 3) return {base + sh.a_qkv, p * R + r, cc, d_in};
    return {base + sh.a_o, r, cc, d_in};
  }
  // B [d_out, 16]: element (o, r) -> row r, column o of B^T
  const long long o = j / R, r = j - o * R;
  if (p < 3) return {base + sh.bt_qkv, p * R + r, sh.col_off[p] + o, sh.nt};
  return {base + sh.bt_o, r, o, sh.d_out[3]};
}
__device__ __forceinline__ void shadow_store(const AdamShadow& sh, long long i, float v) {
  const ShadowPos q = shadow_pos(sh, i);
  const _Float16 h = (_Float16)v;
  sh.shadow[q.base + packed_index(q.row, q.col, q.len)] = h;
  sh.rm[q.base + q.row * q.len + q.col] = h;
  if (sh.at) {  // A of q, k, v: also at (layer, column, row) of the transposed copy
    const long long l = i / sh.per_layer, j = i - l * sh.per_layer;
    if (j < sh.seg_off[5] && (j < sh.seg_off[1] || (j >= sh.seg_off[2] && j < sh.seg_off[3]) ||
                              j >= sh.seg_off[4]))
      sh.at[(l * sh.d_in[0] + q.col) * (3 * R) + q.row] = h;
  }
}

// The AdamW update of one element (src/kernels/lora.cu:206-220):
//   m = b1 m + (1 - b1) g;  v = b2 v + (1 - b2) g^2;
//   p = p (1 - lr wd) - lr (m / bc1) / (sqrt(v / bc2) + eps).
// The bias corrections enter as reciprocals taken once (ib1 = 1 / bc1,
// ib2 = 1 / bc2), and the square root and the last reciprocal are the
// hardware v_sqrt_f32 / v_rcp_f32 (1 ulp each): the IEEE division and
// square-root sequences had made the kernel VALU-bound (about 200 VALU
// instructions a thread for four elements).  The update differs from the
// correctly rounded formula by a few ulp of itself.
struct AdamCoef {
  float b1, b2, c1, c2, ib1, ib2, decay, lr, eps;
};
__device__ __forceinline__ AdamCoef adam_coef(const AdamHp& hp) {
  return {hp.beta1, hp.beta2, 1.0f - hp.beta1, 1.0f - hp.beta2, 1.0f / hp.bc1, 1.0f / hp.bc2,
          1.0f - hp.lr * hp.wd, hp.lr, hp.eps};
}
__device__ __forceinline__ float adam_update(const AdamCoef& k, float p, float g, float& m,
                                             float& v) {
  m = k.b1 * m + k.c1 * g;
  v = k.b2 * v + k.c2 * g * g;
  const float denom = __builtin_amdgcn_sqrtf(v * k.ib2) + k.eps;
  return p * k.decay - k.lr * (m * k.ib1) * __builtin_amdgcn_rcpf(denom);
}

// One AdamW element update in place; returns the new parameter.
__device__ __forceinline__ float adamw_elem(float* __restrict__ p, const float* __restrict__ g,
                                            float* __restrict__ m, float* __restrict__ v,
                                            long long i, const AdamCoef& k) {
  float mi = m[i], vi = v[i];
  const float pi = adam_update(k, p[i], g[i], mi, vi);
  m[i] = mi;
  v[i] = vi;
  p[i] = pi;
  return pi;
}

// Any contiguous set of parameters, no shadows.
__global__ __launch_bounds__(NTH) void adamw_kernel(float* __restrict__ p,
                                                    const float* __restrict__ g,
                                                    float* __restrict__ m, float* __restrict__ v,
                                                    long long n,
                                                    const AdamHp* __restrict__ hpp) {
  const AdamCoef k = adam_coef(*hpp);
  for (long long i = (long long)blockIdx.x * NTH + threadIdx.x; i < n;
       i += (long long)gridDim.x * NTH)
    adamw_elem(p, g, m, v, i, k);
}

// The whole arena with its fp16 shadows, one launch: blockIdx.y = layer x 8
// + segment (q, k, v, o x A, B), blockIdx.x = a tile of kTile elements of
// that segment, so every block knows where its elements' shadow rows and
// columns are (32-bit index math only).  A thread moves four elements as
// 16-byte loads and stores of p, g, m, v (one 16-byte piece a thread over
// many blocks keeps the DRAM streams dense: a copy in this form measured
// 6.3 TB/s on MI355X against 4.6-5.6 TB/s grid-stride; here nontemporal
// loads and stores measured slower, 43 against 37 us).  Each tile covers
// the 16 shadow rows x 64 columns of two whole fragment-packed 16 x 32
// blocks, so a block writes complete 1 KB packed blocks and 128-byte pieces
// of the row-major twin (the same kernel over linear half-row tiles, whose
// packed stores leave partial lines, took 41 us):
// an A tile is rows r = 0..15 x columns c0 .. c0 + 63 of A (16 pieces of
// 256 bytes of the arena; thread = row t / 16, four columns); a B tile is
// the 64 rows o0 .. o0 + 63 of B [d_out, 16] (contiguous in the arena),
// transposed through LDS so that each thread stores four consecutive
// columns o of one row r of B^T.  update = 0 only refreshes the shadows
// from the parameters.
constexpr int kTile = 4 * NTH;
// Tiles a block (TPB): two where every segment is an even number of tiles
// (eight elements a thread, all 32 loads issued before the arithmetic:
// 37.3 against 37.9 us at one and 39 us at four), else one.

__device__ __forceinline__ floatx4 ld4v(const float* p) {
  return *reinterpret_cast<const floatx4*>(p);
}
__device__ __forceinline__ void st4v(float* p, floatx4 v) {
  *reinterpret_cast<floatx4*>(p) = v;
}

template <int TPB>
__global__ __launch_bounds__(NTH) void adamw_shadow_kernel(float* __restrict__ p,
                                                           const float* __restrict__ g,
                                                           float* __restrict__ m,
                                                           float* __restrict__ v,
                                                           const AdamHp* __restrict__ hpp,
                                                           int update, const AdamShadow sh) {
  __shared__ _Float16 bt[TPB][R][64 + 4];
  const int l = blockIdx.y >> 3, s = blockIdx.y & 7, q = s >> 1;
  const int n = (int)((s < 7 ? sh.seg_off[s + 1] : sh.per_layer) - sh.seg_off[s]);
  if (blockIdx.x * TPB * kTile >= n) return;
  const bool is_b = s & 1;
  // A: element (r, c0 + 4 (t % 16)) with r = t / 16; B: elements 4 t .. of the tile
  const int a_len = sh.d_in[q];
  const int ar = threadIdx.x >> 4;
  long long i[TPB];
  floatx4 pv[TPB];
#pragma unroll
  for (int u = 0; u < TPB; ++u) {
    const int tx = blockIdx.x * TPB + u;
    const int ac = tx * 64 + 4 * (threadIdx.x & 15);
    const int jt = is_b ? tx * kTile + 4 * threadIdx.x : ar * a_len + ac;
    i[u] = (long long)l * sh.per_layer + sh.seg_off[s] + jt;
    pv[u] = ld4v(p + i[u]);
  }
  if (update) {
    floatx4 gv[TPB], mv[TPB], vv[TPB];
#pragma unroll
    for (int u = 0; u < TPB; ++u) {
      gv[u] = ld4v(g + i[u]);
      mv[u] = ld4v(m + i[u]);
      vv[u] = ld4v(v + i[u]);
    }
    const AdamCoef k = adam_coef(*hpp);
#pragma unroll
    for (int u = 0; u < TPB; ++u) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float me = mv[u][e], ve = vv[u][e];
        pv[u][e] = adam_update(k, pv[u][e], gv[u][e], me, ve);
        mv[u][e] = me;
        vv[u][e] = ve;
      }
      st4v(p + i[u], pv[u]);
      st4v(m + i[u], mv[u]);
      st4v(v + i[u], vv[u]);
    }
  }
  const long long lb = (long long)l * sh.shadow_per_layer;
  if (!is_b) {
    // A [16, d_in]: element (r, c) -> row row0 + r, column c (row length d_in)
    const int row = (q < 3 ? q * R : 0) + ar;
    const long long base = lb + (q < 3 ? sh.a_qkv : sh.a_o);
#pragma unroll
    for (int u = 0; u < TPB; ++u) {
      const int ac = (blockIdx.x * TPB + u) * 64 + 4 * (threadIdx.x & 15);
      const half4 h = {(_Float16)pv[u][0], (_Float16)pv[u][1], (_Float16)pv[u][2],
                       (_Float16)pv[u][3]};
      *reinterpret_cast<half4*>(sh.shadow + base + packed_index(row, ac, a_len)) = h;
      *reinterpret_cast<half4*>(sh.rm + base + (long long)row * a_len + ac) = h;
    }
    if (q == 3 || !sh.at) return;  // block-uniform
    // q, k, v: the transposed copy [column][3 R], through LDS: thread t then
    // stores ranks 4 (t % 4) .. of column t / 4 of the tile (8 bytes)
    __shared__ _Float16 at_t[TPB][64][R + 4];
#pragma unroll
    for (int u = 0; u < TPB; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) at_t[u][4 * (threadIdx.x & 15) + e][ar] = (_Float16)pv[u][e];
    __syncthreads();
    const int oc = threadIdx.x >> 2, orq = 4 * (threadIdx.x & 3);
#pragma unroll
    for (int u = 0; u < TPB; ++u) {
      const int col = (blockIdx.x * TPB + u) * 64 + oc;
      const half4 t = {at_t[u][oc][orq], at_t[u][oc][orq + 1], at_t[u][oc][orq + 2],
                       at_t[u][oc][orq + 3]};
      *reinterpret_cast<half4*>(sh.at + ((long long)l * a_len + col) * (3 * R) + q * R + orq) = t;
    }
    return;
  }
  // B [d_out, 16]: element j = (o, r) -> row row0 + r, column col0 + o of
  // B^T (row length len); tile u holds o in [64 tx, 64 tx + 64)
  {
    const int o = threadIdx.x >> 2, r = 4 * (threadIdx.x & 3);
#pragma unroll
    for (int u = 0; u < TPB; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) bt[u][r + e][o] = (_Float16)pv[u][e];
  }
  __syncthreads();
  const int len = q < 3 ? sh.nt : sh.d_out[3];
  const int r = threadIdx.x >> 4, c4 = 4 * (threadIdx.x & 15);
  const int row = (q < 3 ? q * R : 0) + r;
  const long long base = lb + (q < 3 ? sh.bt_qkv : sh.bt_o);
#pragma unroll
  for (int u = 0; u < TPB; ++u) {
    const int col = (q < 3 ? sh.col_off[q] : 0) + 64 * (blockIdx.x * TPB + u) + c4;
    const half4 t = *reinterpret_cast<const half4*>(&bt[u][r][c4]);
    *reinterpret_cast<half4*>(sh.shadow + base + packed_index(row, col, len)) = t;
    *reinterpret_cast<half4*>(sh.rm + base + (long long)row * len + col) = t;
  }
}

// Counter-based normal draws: SplitMix64 of (seed, index) -> two 24-bit
// uniforms -> Box-Muller.  Deterministic for a given seed regardless of the
// launch shape.
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

__global__ __launch_bounds__(NTH) void lora_init_kernel(float* __restrict__ p,
                                                        float* __restrict__ m,
                                                        float* __restrict__ v, long long n,
                                                        unsigned long long seed, float a_std,
                                                        float b_std, const AdamShadow sh) {
  for (long long i = (long long)blockIdx.x * NTH + threadIdx.x; i < n;
       i += (long long)gridDim.x * NTH) {
    const unsigned long long z = splitmix64(seed * 0x100000001B3ull + (unsigned long long)i);
    const float u1 = ((float)(z >> 40) + 1.0f) * (1.0f / 16777216.0f);  // (0, 1]
    const float u2 = (float)((z >> 16) & 0xFFFFFF) * (1.0f / 16777216.0f);
    const float nrm = sqrtf(-2.0f * logf(u1)) * cospif(2.0f * u2);
    const long long j = i % sh.per_layer;
    int s = 0;
#pragma unroll
    for (int k = 1; k < 8; ++k)
      if (j >= sh.seg_off[k]) s = k;
    const float val = nrm * ((s & 1) ? b_std : a_std);
    p[i] = val;
    m[i] = 0.f;
    v[i] = 0.f;
    if (sh.shadow) shadow_store(sh, i, val);
  }
}

inline unsigned grid_for(long long n) {
  long long g = (n + NTH - 1) / NTH;
  return (unsigned)(g > 8192 ? 8192 : (g < 1 ? 1 : g));
}

}  // namespace

hipError_t lora_grad(const LoraGradJob* jobs, const LoraGradPlan& plan, int layers, int T,
                     float lscale, int accumulate, hipStream_t st) {
  if (layers < 1 || T < 1) {
    set_error("lora_grad: %d layers, T=%d", layers, T);
    return hipErrorInvalidValue;
  }
  int cols = 0;
  for (int i = 0; i < kLoraJobs; ++i) {
    if (plan.ncols[i] % 8) {
      set_error("lora_grad: job %d has %d columns (a multiple of 8 is required)", i, plan.ncols[i]);
      return hipErrorInvalidValue;
    }
    cols += plan.ncols[i];
  }
  auto go = [&](auto wc, auto cc) {
    constexpr int W = decltype(wc)::value, CPL = decltype(cc)::value;
    LoraGradGrid G{};
    for (int i = 0; i < kLoraJobs; ++i)
      G.block_start[i + 1] = G.block_start[i] + (plan.ncols[i] + 16 * CPL - 1) / (16 * CPL);
    hipLaunchKernelGGL((lora_grad_kernel<W, CPL>), dim3(layers * G.block_start[kLoraJobs]),
                       dim3(W * 64), 0, st, jobs, G, T, lscale, accumulate);
  };
  // 128 columns a workgroup (16-byte X loads, half the loads per MFMA) where
  // that still fills the CUs, 64 where it does not (one layer: 112 blocks);
  // as many waves over the tokens as it takes to fill the chip.  28 layers at
  // T = 4096, us: 64 columns 786 / 773 / 834 with 4 / 8 / 16 waves, 128
  // columns 676 / 683 / 699; one layer: 49 / 40 / 38 and 70 / 59 / 57.  At T =
  // 128 28 layers 35 with 2 or 4 waves, 41 with 8.
  using std::integral_constant;
  const int blocks = layers * (cols / 128);
  auto width = [&](auto wc) {
    if (blocks >= 192) go(wc, integral_constant<int, 8>());
    else go(wc, integral_constant<int, 4>());
  };
  if (blocks < 512 && T >= 1024) width(integral_constant<int, 16>());
  else if (blocks < 512 && T >= 64) width(integral_constant<int, 8>());
  else if (T >= 64) go(integral_constant<int, 4>(), integral_constant<int, 8>());
  else width(integral_constant<int, 2>());
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t adamw(float* p, const float* g, float* m, float* v, long long n, const AdamHp* hp,
                 int update, const AdamShadow& sh, hipStream_t st) {
  if (!sh.shadow) {
    if (!update) return hipSuccess;
    hipLaunchKernelGGL(adamw_kernel, dim3(grid_for(n)), dim3(NTH), 0, st, p, g, m, v, n, hp);
    LLMT_LAUNCH_CHECK();
    return hipSuccess;
  }
  if (sh.per_layer <= 0 || n % sh.per_layer || !sh.rm) {
    set_error("adamw: %lld parameters are not whole layers of %lld", n, sh.per_layer);
    return hipErrorInvalidValue;
  }
  // every segment is whole tiles (its A rows and B^T rows a multiple of 64
  // columns, 16-byte aligned), so the tiles never straddle segments
  long long seg = 0;
  bool pairs = true;  // every segment an even number of tiles
  for (int s = 0; s < 8; ++s) {
    const long long ns = (s < 7 ? sh.seg_off[s + 1] : sh.per_layer) - sh.seg_off[s];
    if (ns % kTile || sh.seg_off[s] % 4) {
      set_error("adamw: segment %d of %lld elements is not whole %d-element tiles", s, ns, kTile);
      return hipErrorInvalidValue;
    }
    pairs = pairs && ns % (2 * kTile) == 0;
    seg = std::max(seg, ns);
  }
  for (int q = 0; q < 4; ++q)
    if (sh.d_in[q] % 64 || sh.d_out[q] % 64) {
      set_error("adamw: adapter %d dims %d x %d not multiples of 64", q, sh.d_out[q], sh.d_in[q]);
      return hipErrorInvalidValue;
    }
  const dim3 grid((unsigned)(seg / (pairs ? 2 * kTile : kTile)), (unsigned)(n / sh.per_layer * 8));
  if (pairs)
    hipLaunchKernelGGL(adamw_shadow_kernel<2>, grid, dim3(NTH), 0, st, p, g, m, v, hp, update, sh);
  else
    hipLaunchKernelGGL(adamw_shadow_kernel<1>, grid, dim3(NTH), 0, st, p, g, m, v, hp, update, sh);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t lora_init(float* p, float* m, float* v, long long n, unsigned long long seed,
                     float a_std, float b_std, const AdamShadow& sh, hipStream_t st) {
  hipLaunchKernelGGL(lora_init_kernel, dim3(grid_for(n)), dim3(NTH), 0, st, p, m, v, n, seed,
                     a_std, b_std, sh);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

}  // namespace llmt
