// gemm.hip — "NT" GEMMs on fp16 MFMA (v_mfma_f32_16x16x32_f16) for
// gfx950, plus the layout kernels (fragment packing, transposes,
// conversions, the bit-exact int8 quantizer) and the split-K reduction used
// by the standalone GEMM entry points.
//
// Every frozen-weight product of the training step is expressed as
// C = A * B^T with both operands contiguous along the reduction dimension:
// the forward uses W [out, in] as B, the backward (dX = dY * W) uses the
// pre-transposed copy W^T [in, out] the library keeps next to W.  This is the
// MI355X-native replacement for the reference's three fp32 32x32-tiled
// kernels (src/kernels/matmul.cu:8-138): matmul_forward (NT), matmul_nn
// (dX) and, for LoRA, matmul_tn.
//
// Kernels.  B operands are stored fragment-packed (packed_index in common.h),
// so an MFMA fragment of B is one contiguous 1 KB (int8: 512 B) wherever it
// is read from.
//   gemm_ring_kernel  any M % 16 == 0, all row counts where the plan finds it
//                     cheaper (below 512 always): 16 MR x 16 NB tiles fed by
//                     LDS DMA, K split over workgroups so
//                     that a launch fills the CUs; the fp32 split partials
//                     are summed in split order by the consuming row
//                     epilogue (deterministic), and the standalone GEMM entry
//                     points reduce them with reduce_lora
//   gemm_dma_kernel   many rows: 256 x 256 tiles
//   gemm_nt_kernel    what the two do not take (K % 64 != 0, several int8
//                     segments, rows of A off a 16-byte boundary): B streamed
//                     into registers, A through LDS
// gemm_plan picks the kernel, the tile and the split from a cost model.
#include <math.h>
#include <stdlib.h>
#include <type_traits>

#include "ops.h"

namespace llmt {

static int env_int(const char* name, int dflt) {
  const char* v = getenv(name);
  return v && *v ? atoi(v) : dflt;
}

namespace {

#define LLMT_INLINE __attribute__((always_inline))

constexpr int KSTEP = 32;  // k per MFMA

template <int V>
using IC = std::integral_constant<int, V>;

constexpr int gcd_c(int a, int b) { return b == 0 ? a : gcd_c(b, a % b); }
constexpr int lcm_c(int a, int b) { return a / gcd_c(a, b) * b; }

// Packed int8 weights are stored biased, byte = x + 128 (x ^ 0x80; written by
// pack_i8), so that fp16 bits 0x64 | byte read as 1024 + x + 128, exact.
// v_perm_b32 picks bytes 0-3 from its second source and 4-7 from its
// first: each output dword [b_i, 0x64, b_i+1, 0x64] is one instruction.
__device__ __forceinline__ half8 i8x8_to_h8(u32x2 raw) {
  constexpr unsigned k64 = 0x64646464u, s01 = 0x04010400u, s23 = 0x04030402u;
  u32x4 bits;
  bits[0] = __builtin_amdgcn_perm(k64, raw[0], s01);
  bits[1] = __builtin_amdgcn_perm(k64, raw[0], s23);
  bits[2] = __builtin_amdgcn_perm(k64, raw[1], s01);
  bits[3] = __builtin_amdgcn_perm(k64, raw[1], s23);
  const half8 h = __builtin_bit_cast(half8, bits);
  return h - (_Float16)1152.0f;
}

// Four dwords at any fp16 element (one load all the same).
typedef u32x4 u32x4_h __attribute__((aligned(2)));

// Register-staged kernel.  One workgroup: output tile (MF*16) x (NW*NF*16)
// over k-steps [s0, s1) of its split.  The A tile goes through LDS in chunks
// of CHS k-steps (two LDS buffers); chunk c + ADIST is loaded into registers
// while chunk c is multiplied, so an A load has ADIST chunks of MFMA work to
// land.  B fragments stream through a RING-slot register ring, RING - 1
// k-steps ahead.  The main loop body covers UC chunks so that every LDS
// buffer, A register set and ring slot index is a compile-time constant.
// Chunks and k-steps past the end are clamped loads multiplied by zeroed B
// fragments (branch-free: the compiler then keeps the newer loads in flight
// across every wait).  With I8 a segment may be int8 (dequantised in
// registers at MFMA time, optionally times a per-k scale loaded alongside).
template <int MF, int NF, int NW, int CHS, int RING, int ADIST, bool I8>
__global__ __launch_bounds__(NW * 64) void gemm_nt_kernel(const GemmArgs g) {
  constexpr int MT = MF * 16;
  constexpr int NT = NW * 64;
  constexpr int CH = CHS * KSTEP;
  constexpr int PIECES = MT * (CH / 8);  // 16-byte A pieces per chunk
  constexpr int APT = (PIECES + NT - 1) / NT;
  constexpr int UC = lcm_c(lcm_c(2, ADIST), lcm_c(RING, CHS) / CHS);
  static_assert(ADIST == 1 || ADIST == 2, "A prefetch distance is one or two chunks");
  // A chunk in LDS in MFMA fragment order: fragment (k-step q, m-tile mi) is
  // 1 KB at (q * MF + mi) * 512 halves with lane l's 8 halves at l * 8, so
  // every ds_read_b128 of a wave is one contiguous, conflict-free 1 KB, and
  // the staging writes (thread i -> piece i) are contiguous too.
  __shared__ __attribute__((aligned(16))) _Float16 As[2][MT * CH];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int m0 = blockIdx.z * MT;
  const int ksteps = g.K / KSTEP;
  const int s0 = (int)((long long)blockIdx.y * ksteps / g.split);
  const int s1 = (int)((long long)(blockIdx.y + 1) * ksteps / g.split);
  const int nst = s1 - s0;
  const int nch = (nst + CHS - 1) / CHS;

  const char* bptr[NF];
  int bi8[NF];
  int ncol[NF];
  const _Float16* cscale[NF];
  const _Float16* kscale[NF];
  bool valid[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int nn = (blockIdx.x * NW + wave) * NF * 16 + f * 16;
    ncol[f] = nn;
    valid[f] = nn < g.N;
    int s = 0;
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i < g.nseg && nn >= g.seg_start[i]) s = i;
    const BSeg& sg = g.seg[s];
    // Invalid fragments read row block 0 of their segment (in bounds) and
    // are never stored.
    const long long rb16 = valid[f] ? (nn - g.seg_start[s]) >> 4 : 0;
    const int i8 = I8 ? sg.is_i8 : 0;
    bptr[f] = (const char*)sg.ptr + ((rb16 * ksteps) * 512 + lane * 8) * (i8 ? 1 : 2);
    bi8[f] = i8;
    cscale[f] = sg.colscale ? sg.colscale + (nn - g.seg_start[s]) : nullptr;
    kscale[f] = (I8 && sg.kscale) ? sg.kscale + (lane >> 4) * 8 : nullptr;
  }

  floatx4 acc[MF][NF];
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[i][f] = floatx4{0.f, 0.f, 0.f, 0.f};

  u32x4 ra[ADIST][APT];
  u32x4 rb[RING][NF];
  u32x4 rk[RING][NF];

  auto load_a = [&](int c, auto R) LLMT_INLINE {
    constexpr int set = decltype(R)::value;
    const int kb = (s0 + min(c, nch - 1) * CHS) * KSTEP;
#pragma unroll
    for (int i = 0; i < APT; ++i) {
      const int idx = tid + i * NT;  // LDS piece: fragment idx / 64, lane idx % 64
      if (PIECES % NT == 0 || idx < PIECES) {
        const int fr = idx >> 6, l = idx & 63;
        const int q = fr / MF, mi = fr % MF;
        const int r = mi * 16 + (l & 15);
        const int k = min(kb + q * KSTEP + (l >> 4) * 8, g.K - 8);
        ra[set][i] = *reinterpret_cast<const u32x4_h*>(g.A + (long long)(m0 + r) * g.lda + k);
      }
    }
  };
  auto store_a = [&](auto R, auto BUF) LLMT_INLINE {
    constexpr int set = decltype(R)::value;
    constexpr int buf = decltype(BUF)::value;
#pragma unroll
    for (int i = 0; i < APT; ++i) {
      const int idx = tid + i * NT;
      if (PIECES % NT == 0 || idx < PIECES)
        *reinterpret_cast<u32x4*>(&As[buf][idx * 8]) = ra[set][i];
    }
  };
  auto load_b = [&](int j, auto S) LLMT_INLINE {
    constexpr int st = decltype(S)::value;
    const long long ss = s0 + min(j, nst - 1);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      if (I8 && bi8[f]) {
        const u32x2 q = *reinterpret_cast<const u32x2*>(bptr[f] + ss * 512);
        rb[st][f] = u32x4{q[0], q[1], 0u, 0u};
        if (kscale[f]) rk[st][f] = *reinterpret_cast<const u32x4*>(kscale[f] + ss * KSTEP);
      } else {
        rb[st][f] = *reinterpret_cast<const u32x4*>(bptr[f] + ss * 1024);
      }
    }
  };
  auto bfrag = [&](int f, auto S) LLMT_INLINE -> half8 {
    constexpr int st = decltype(S)::value;
    half8 h;
    if (I8 && bi8[f]) {
      h = i8x8_to_h8(u32x2{rb[st][f][0], rb[st][f][1]});
      if (kscale[f]) {
        h = h * __builtin_bit_cast(half8, rk[st][f]);
      }
    } else {
      h = __builtin_bit_cast(half8, rb[st][f]);
    }
    return h;
  };
  // k-step j = (chunk base cb + u) * CHS + q: ring slot (u * CHS + q) % RING
  // and LDS buffer u % 2 are static within the unrolled body.
  auto kstep = [&](int cb, auto U, auto Q) LLMT_INLINE {
    constexpr int u = decltype(U)::value;
    constexpr int q = decltype(Q)::value;
    constexpr int pos = u * CHS + q;
    const int j = (cb + u) * CHS + q;
    load_b(j + RING - 1, IC<(pos + RING - 1) % RING>{});
    const bool live = j < nst;
    half8 b[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      b[f] = bfrag(f, IC<pos % RING>{});
      if (!live) b[f] = half8{};
    }
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
      const half8 a =
          *reinterpret_cast<const half8*>(&As[u % 2][((q * MF + mi) * 64 + lane) * 8]);
#pragma unroll
      for (int f = 0; f < NF; ++f) acc[mi][f] = mfma16(a, b[f], acc[mi][f]);
    }
  };
  auto chunk = [&](int cb, auto U) LLMT_INLINE {
    constexpr int u = decltype(U)::value;
    // chunk cb + u + ADIST goes to register set (u + ADIST) % ADIST = u % ADIST
    load_a(cb + u + ADIST, IC<u % ADIST>{});
    __builtin_amdgcn_sched_barrier(0);
    [&]<int... Q>(std::integer_sequence<int, Q...>) LLMT_INLINE {
      (kstep(cb, IC<u>{}, IC<Q>{}), ...);
    }(std::make_integer_sequence<int, CHS>{});
    // chunk cb + u + 1 was loaded ADIST - 1 chunks ago into set (u + 1) % ADIST
    store_a(IC<(u + 1) % ADIST>{}, IC<(u + 1) % 2>{});
    __syncthreads();
  };

  if (nst > 0) {
    load_a(0, IC<0>{});
    if constexpr (ADIST == 2) load_a(1, IC<1>{});
    [&]<int... P>(std::integer_sequence<int, P...>) LLMT_INLINE {
      (load_b(P, IC<P>{}), ...);
    }(std::make_integer_sequence<int, RING - 1>{});
    store_a(IC<0>{}, IC<0>{});
    __syncthreads();
    // The unrolled body stops at the last chunk (uniform exit), so a deep
    // ring costs no padded MFMA work on short K ranges.
    for (int c = 0; c < nch; c += UC) {
      [&]<int... U>(std::integer_sequence<int, U...>) LLMT_INLINE {
        ((c + U < nch ? (chunk(c, IC<U>{}), true) : false) && ...);
      }(std::make_integer_sequence<int, UC>{});
    }
  }

  float* C = g.C + (long long)blockIdx.y * g.split_stride;
  float cs[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) cs[f] = cscale[f] ? (float)cscale[f][lane & 15] : 1.0f;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    if (!valid[f]) continue;
    const int col = ncol[f] + (lane & 15);
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = m0 + mi * 16 + (lane >> 4) * 4 + v;
        C[(long long)row * g.ldc + col] = acc[mi][f][v] * cs[f];
      }
    }
  }
  if (g.rowstats) {
    // each row's (max, sum exp) over the workgroup's NW NF 16 columns: a
    // wave's pair from its 16-lane groups, the NW waves merged in wave order
    float2* sh = reinterpret_cast<float2*>(&As[0][0]);  // [MT][NW]
    static_assert(MT * NW * 8 <= 2 * MT * CH * 2, "pairs fit in the A buffers");
    __syncthreads();  // every wave is past its last A fragment read
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float x[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) x[f] = valid[f] ? acc[mi][f][v] * cs[f] : -INFINITY;
        const float2 p = softmax_pair16<NF>(x);
        if ((lane & 15) == 0) sh[(mi * 16 + (lane >> 4) * 4 + v) * NW + wave] = p;
      }
    __syncthreads();
    for (int r = tid; r < MT; r += NT) {
      float m = -INFINITY, s = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) softmax_merge(m, s, sh[r * NW + w].x, sh[r * NW + w].y);
      g.rowstats[(long long)(m0 + r) * gridDim.x + blockIdx.x] = make_float2(m, s);
    }
  }
}

constexpr int BM = 256;  // large-tile rows

// LDS-DMA kernel for the large-M GEMMs: the operands go from global memory
// straight into LDS (global_load_lds: lane l's 16 bytes land at offset 16 l
// of the wave's block; a fragment-packed fp16 fragment is 1 KB in lane order
// and an int8 one 512 B, moved by the first 32 lanes, so both arrive in MFMA
// fragment order with no register staging and no LDS store phase), through
// an S-stage ring of 32-wide K chunks: chunks up to c + S - 1 are in flight
// while chunk c is multiplied.  Each workgroup of eight waves owns a 256 x 256
// tile (2 x 4 waves of 128 x 64, 32 accumulator fragments a wave; the
// four-wave form with 128 x 128 a wave measured 12-20% slower at the C4
// shapes).  The fragments run one chunk ahead in registers: while the MFMAs
// of chunk c issue, chunk c + 1's fragments are read from LDS (each A
// fragment register refilled right after its last MFMA), so LDS latency and
// the int8 dequantisation (exact int8 -> fp16 from the biased bytes, one
// v_perm_b32 and one v_pk_add_f16 a dword, times the per-k scale if any)
// leave the critical path (C4 dX
// GEMMs 187.5 -> 183.5 us, the tail-folded ones 2-3% faster).  The waits are
// explicit: vmcnt counts this thread's DMA issues, which complete in order,
// and a plain s_barrier (no fence, which would drain every load) publishes
// the chunk to the other waves.
__device__ __forceinline__ void dma16(const void* src, _Float16* lds_blk) {
  __builtin_amdgcn_global_load_lds(src, (void __attribute__((address_space(3)))*)lds_blk, 16, 0, 0);
}
// s_waitcnt with vmcnt = N (lgkmcnt and expcnt left free), gfx9 encoding.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}


// TL: a trailing fp16 segment `tail` of at most 64 rows (the LoRA A or B^T
// rows of a projection, output columns tail_c0 ..) rides along: its 16-row
// fragment f is computed by the workgroups of column tile f, over their row
// block and K range (two extra MFMAs a wave per chunk, the fragment's 1 KB
// a chunk moved by eight lanes of every wave), instead of a separate launch
// that streamed the whole activation matrix again.
template <bool I8, bool KS, int S, int WNN, bool GLU = false, bool TL = false>
__global__ __launch_bounds__(WNN * 128) void gemm_dma_kernel(const GemmArgs g, int g_order,
                                                             const BSeg tail, int tail_c0) {
  // WNN waves across N (2: four waves of 128 x 128; 4: eight waves of 128 x 64)
  constexpr int NW = 2 * WNN, WC = 256 / WNN, NFR = WC / 16;  // wave columns, fragments
  constexpr int FPW = 16 / NW;                                 // A (and B) fragments each wave moves
  constexpr int ABYTES = 256 * KSTEP * 2;
  constexpr int BBYTES = 256 * KSTEP * (I8 ? 1 : 2);
  constexpr int KSBYTES = KS ? 256 : 0;
  constexpr int TOFF = ABYTES + BBYTES + KSBYTES;              // tail fragment slot
  constexpr int SBYTES = TOFF + (TL ? 1024 : 0);
  constexpr int OPS = 2 * FPW + (KS ? 1 : 0) + (TL ? 1 : 0);   // DMA issues per chunk per thread
  static_assert(!(TL && GLU), "no tail with the SwiGLU epilogue");
  static_assert(!TL || WNN == 4, "the tail fragment is split over four column waves");
  __shared__ __attribute__((aligned(1024))) char smem[S * SBYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WNN, wn = wave % WNN;
  const int ntn = (g.N + 255) / 256, ntm = (g.M + 255) / 256;
  int t = blockIdx.x, sidx = blockIdx.y, nsp = g.split, tn0 = 0, ntn_r = ntn;
  if (g.split_col > 0) {
    // column tiles [0, ntc) unsplit (workgroups 0 .. ntc ntm - 1), then the
    // rest split in two over K (split 0 of every such tile, then split 1)
    const int ntc = g.split_col / 256, nfull = ntc * ntm;
    if (t < nfull) {
      nsp = 1;
      sidx = 0;
      ntn_r = ntc;
    } else {
      t -= nfull;
      nsp = 2;
      tn0 = ntc;
      ntn_r = ntn - ntc;
      sidx = t / (ntn_r * ntm);
      t -= sidx * (ntn_r * ntm);
    }
  }
  const int nwg = ntn_r * ntm;
  if (g_order >= 1 && nwg % 8 == 0) t = (t % 8) * (nwg / 8) + t / 8;
  // Consecutive t of one XCD walk GM row blocks per column step, so the 32
  // tiles an XCD runs at once share 4 A row blocks and 8 B column blocks in
  // its L2 (not 1 and 32): the logits GEMM 3.05 -> 2.88 ms at C4.
  const int GM = ntm % 4 == 0 ? 4 : ntm % 2 == 0 ? 2 : 1;
  const int grp = t / (GM * ntn_r), tr = t % (GM * ntn_r);
  const int tm = grp * GM + tr % GM, tn = tn0 + tr / GM;
  const int n0 = tn * 256, m0 = tm * 256;
  const int ksteps = g.K / KSTEP;
  const int c0 = (int)((long long)sidx * ksteps / nsp);
  const int c1 = (int)((long long)(sidx + 1) * ksteps / nsp);

  // issue pointers: wave w moves A fragments FPW w .. and B fragments FPW w ..
  // of every chunk (plus, with KS, k-scales through lane 0 of waves 0-3)
  // (A fragments past M re-read the last one; their rows are not stored)
  const int mfr = (g.M - m0) >> 4;  // 16-row fragments with rows of A
  const _Float16* asrc[FPW];
#pragma unroll
  for (int j = 0; j < FPW; ++j)
    asrc[j] = g.A + (long long)(m0 + min(wave * FPW + j, mfr - 1) * 16 + (lane & 15)) * g.lda +
              (lane >> 4) * 8;
  const BSeg& sg = g.seg[0];
  constexpr int ES = I8 ? 1 : 2;
  const char* bsrc = (const char*)sg.ptr + (long long)lane * 16;  // lanes < 32 for int8
  // SwiGLU pairs: tile fragment f is gate (f even) or up (f odd) row block
  // 8 tn + f / 2, so a wave's fragments 2 p and 2 p + 1 cover the same columns
  long long boff[FPW];
#pragma unroll
  for (int j = 0; j < FPW; ++j) {
    const int f = wave * FPW + j;
    const int rb = GLU ? (f & 1) * (g.glu >> 4) + tn * 8 + (f >> 1)
                       : min((n0 >> 4) + f, (g.N >> 4) - 1);
    boff[j] = (long long)rb * ksteps * 512 * ES;
  }
  const _Float16* ksrc = KS ? sg.kscale + (wave & 3) * 8 : nullptr;
  // tail fragment of this column tile (tiles past the last fragment load the
  // last one, unused, so every wave issues the same number of DMAs)
  const int ntf = TL ? tail.rows / 16 : 0;
  const bool has_tail = TL && tn < ntf;
  const _Float16* tsrc =
      TL ? (const _Float16*)tail.ptr + (long long)min(tn, ntf - 1) * ksteps * 512 + (wave * 8 + lane) * 8
         : nullptr;
  auto issue = [&](int c) LLMT_INLINE {
    const int cc = min(c, c1 - 1);
    char* st = smem + (c % S) * SBYTES;
#pragma unroll
    for (int j = 0; j < FPW; ++j)
      dma16(asrc[j] + cc * KSTEP, reinterpret_cast<_Float16*>(st + (wave * FPW + j) * 1024));
#pragma unroll
    for (int j = 0; j < FPW; ++j) {
      const char* src = bsrc + boff[j] + (long long)cc * 512 * ES;
      _Float16* dst = reinterpret_cast<_Float16*>(st + ABYTES + (wave * FPW + j) * 512 * ES);
      if constexpr (I8) {
        if (lane < 32) dma16(src, dst);
      } else {
        dma16(src, dst);
      }
    }
    if constexpr (KS) {
      if (lane == 0 && wave < 4)
        dma16(ksrc + (long long)cc * KSTEP, reinterpret_cast<_Float16*>(st + ABYTES + BBYTES + wave * 16));
      else if (lane == 0)  // keep the per-thread DMA count uniform (a harmless re-read)
        dma16(ksrc + (long long)cc * KSTEP, reinterpret_cast<_Float16*>(st + ABYTES + BBYTES + 64 + (wave & 3) * 16));
    }
    if constexpr (TL) {  // wave w moves bytes 128 w .. 128 w + 127 of the fragment
      if (lane < 8) dma16(tsrc + (long long)cc * 512, reinterpret_cast<_Float16*>(st + TOFF + wave * 128));
    }
  };

  floatx4 acc[8][NFR];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < NFR; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  // tail: this wave's rows 16 (2 wn + j) .. of its 128-row half
  floatx4 acc_t[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};

  // Fragments one chunk ahead: after the barrier that publishes chunk
  // c + 1, each A fragment register of chunk c is refilled from chunk c + 1
  // right after its last MFMA, and chunk c + 1's B bytes (and k-scales,
  // tail fragment) are read at the top, dequantised after the last MFMA;
  // so LDS latency sits under the MFMAs and the registers stay one set.
  half8 a[8], b[NFR], bt, btn, ksn, at[2], atn[2];
  u32x2 bn8[NFR];
  half8 bn16[NFR];
  auto read_b = [&](const char* st) LLMT_INLINE {
    if constexpr (KS) ksn = *reinterpret_cast<const half8*>(st + ABYTES + BBYTES + (lane >> 4) * 16);
#pragma unroll
    for (int j = 0; j < NFR; ++j) {
      const int fr = wn * NFR + j;
      if constexpr (I8)
        bn8[j] = *reinterpret_cast<const u32x2*>(st + ABYTES + fr * 512 + lane * 8);
      else
        bn16[j] = *reinterpret_cast<const half8*>(st + ABYTES + fr * 1024 + lane * 16);
    }
    if constexpr (TL) {
      // the tail's fragment and the two A fragments it meets (rows
      // 16 (2 wn + j) of the wave's half), read on their own so the tail
      // MFMAs need no register selection
      btn = *reinterpret_cast<const half8*>(st + TOFF + lane * 16);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        atn[j] = *reinterpret_cast<const half8*>(st + (wm * 8 + 2 * wn + j) * 1024 + lane * 16);
    }
  };
  auto take_b = [&]() LLMT_INLINE {
#pragma unroll
    for (int j = 0; j < NFR; ++j) {
      if constexpr (I8) {
        b[j] = i8x8_to_h8(bn8[j]);
        if constexpr (KS) b[j] = b[j] * ksn;
      } else {
        b[j] = bn16[j];
      }
    }
    if constexpr (TL) {
      bt = btn;
      at[0] = atn[0];
      at[1] = atn[1];
    }
  };
  auto read_a = [&](const char* st, int i) LLMT_INLINE {
    a[i] = *reinterpret_cast<const half8*>(st + (wm * 8 + i) * 1024 + lane * 16);
  };
#pragma unroll
  for (int c = 0; c < S; ++c) issue(c0 + c);
  static_assert((S - 1) * OPS < 64, "vmcnt range");
  wait_vm<(S - 1) * OPS>();
  __builtin_amdgcn_s_barrier();
  {
    const char* st = smem + (c0 % S) * SBYTES;
    read_b(st);
#pragma unroll
    for (int i = 0; i < 8; ++i) read_a(st, i);
    take_b();
  }
  for (int c = c0; c < c1; ++c) {
    // vmcnt: chunk c + 1 landed; lgkmcnt 0: this wave's reads of chunk c
    // returned, so after the barrier chunk c's slot takes chunk c + S
    constexpr int N = (S - 2) * OPS;
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
    __builtin_amdgcn_s_barrier();
    issue(c + S);
    const char* st = smem + ((c + 1) % S) * SBYTES;
    read_b(st);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int j = 0; j < NFR; ++j) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
      read_a(st, i);
    }
    // the order the loop states: chunk c + 1's B (and scale, tail) reads
    // first, then per row its MFMAs followed by the read that refills its A
    // register (left alone, the compiler sank all eight A reads below the
    // last MFMA, exposing their latency at the barrier)
    __builtin_amdgcn_sched_group_barrier(0x100, (I8 ? NFR / 2 : NFR) + (KS ? 1 : 0) + (TL ? 3 : 0), 0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, NFR, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    if constexpr (TL) {
      if (has_tail) {
        acc_t[0] = mfma16(at[0], bt, acc_t[0]);
        acc_t[1] = mfma16(at[1], bt, acc_t[1]);
      }
    }
    // the dequantisation stays below the rows: hoisted up to the B reads
    // (as the compiler otherwise does with part of it) it waits on them
    // right at the top of the chunk.  VALU may not cross; MFMA, LDS, SALU
    // and memory instructions may.
    __builtin_amdgcn_sched_barrier(0);
    take_b();
  }
  wait_vm<0>();

  float* C = g.C + (long long)sidx * g.split_stride;
  const _Float16* cs = sg.colscale;
  if constexpr (GLU) {
    float sgu[NFR];
#pragma unroll
    for (int jj = 0; jj < NFR / 2; ++jj) {
      const int col = (tn * 8 + ((wn * NFR) >> 1) + jj) * 16 + (lane & 15);
      sgu[2 * jj] = cs ? (float)cs[col] : 1.0f;
      sgu[2 * jj + 1] = cs ? (float)cs[g.glu + col] : 1.0f;
    }
    const int col0 = (tn * 8 + ((wn * NFR) >> 1)) * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (wm * 8 + i >= mfr) break;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long long row = m0 + wm * 128 + i * 16 + (lane >> 4) * 4 + v;
        _Float16* grow = g.gu16 + row * (2LL * g.glu) + col0;
        _Float16* arow = g.glu16 + row * g.ldglu + col0;
#pragma unroll
        for (int jj = 0; jj < NFR / 2; ++jj) {
          const float gt = acc[i][2 * jj][v] * sgu[2 * jj], up = acc[i][2 * jj + 1][v] * sgu[2 * jj + 1];
          grow[16 * jj] = (_Float16)gt;
          grow[g.glu + 16 * jj] = (_Float16)up;
          arow[16 * jj] = (_Float16)(gt * sigmoid_rcp(gt) * up);
        }
      }
    }
    return;
  }
  if constexpr (TL) {
    if (has_tail) {
      const int col = tail_c0 + tn * 16 + (lane & 15);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (wm * 8 + 2 * wn + j >= mfr) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = m0 + wm * 128 + (2 * wn + j) * 16 + (lane >> 4) * 4 + v;
          C[(long long)row * g.ldc + col] = acc_t[j][v];
        }
      }
    }
  }
  float scj[NFR];
#pragma unroll
  for (int j = 0; j < NFR; ++j) {
    const int col = n0 + wn * WC + j * 16 + (lane & 15);
    scj[j] = cs && col < g.N ? (float)cs[col] : 1.0f;
  }
  // store addresses: a wave-uniform row base plus one 32-bit lane offset
  // for all stores (the compiler then steps one 64-bit address by ldc, one
  // add a store instead of a 64-bit multiply-add and an add: the fp16
  // logits GEMM at C4 2429 -> 2370 us; the same for the SwiGLU epilogue's
  // fp16 stores measured 1% slower)
  const int lo = (lane >> 4) * 4 * g.ldc + (lane & 15);
  float* const Cw = C + (long long)(m0 + wm * 128) * g.ldc + n0 + wn * WC;
#pragma unroll
  for (int j = 0; j < NFR; ++j) {
    if (n0 + wn * WC + j * 16 >= g.N) continue;  // N % 16 == 0: whole fragments
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (wm * 8 + i >= mfr) break;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float* const Cr = Cw + (long long)(i * 16 + v) * g.ldc + j * 16;
        Cr[lo] = acc[i][j][v] * scj[j];
      }
    }
  }
  if (g.rowstats) {
    // each row's (max, sum exp) over the tile's 256 columns: a wave's pair
    // over its WC columns from its 16-lane groups, the WNN waves of a row
    // block merged in order (the ring is free: every DMA has landed)
    float2* sh = reinterpret_cast<float2*>(smem);  // [256 rows][WNN]
    __syncthreads();  // every wave is past its last fragment read
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float x[NFR];
#pragma unroll
        for (int j = 0; j < NFR; ++j) {
          const int col = n0 + wn * WC + j * 16 + (lane & 15);
          x[j] = col < g.N ? acc[i][j][v] * scj[j] : -INFINITY;
        }
        const float2 p = softmax_pair16<NFR>(x);
        if ((lane & 15) == 0) sh[(wm * 128 + i * 16 + (lane >> 4) * 4 + v) * WNN + wn] = p;
      }
    __syncthreads();
    for (int r = tid; r < 256 && r < 16 * mfr; r += WNN * 128) {
      float m = -INFINITY, s = 0.f;
#pragma unroll
      for (int w = 0; w < WNN; ++w) softmax_merge(m, s, sh[r * WNN + w].x, sh[r * WNN + w].y);
      g.rowstats[(long long)(m0 + r) * ntn + tn] = make_float2(m, s);
    }
  }
}

// Stage-ring kernel: fp16 or int8 weights, any M % 16 == 0 (every GEMM of a
// step of one to a few sequences; of 4096 rows those whose last round of 256 x
// 256 tiles is badly filled).  A workgroup of eight waves owns 16 MR rows x
// 16 NB columns, K split over workgroups.
//
// What bounds it: up to M = 128 the weight stream and the fixed costs of a
// launch (about 5 us: the first round trip, the partial stores), above that
// the LDS: a 64-wide stage of a 128 x 128 tile is 512 cycles of MFMA a SIMD
// but 96 KB of LDS traffic (64 KB of fragment reads, 32 KB of DMA), 768
// cycles at 128 B/clk; with the operands re-read from L2 (no fresh memory
// traffic) a stage takes 0.41 us, with them 0.58.  Hence the wave layout: two
// groups of four waves take one k half of every stage each (their sums meet
// in LDS at the end), so a wave covers 64 x (8 NB) with half the fragment
// reads per MFMA that eight waves over the whole tile would need, and the
// fragments are read one stage ahead into registers (an A register is
// refilled right after its last MFMA), so the reads run beside the MFMAs.
//
// Both operands move global -> LDS with buffer loads that have an LDS
// destination, 16 bytes a lane: A as 128-byte row pieces (the 16-byte pieces
// XOR-swizzled by row so the fragment reads are bank-conflict free; rows past
// M lie outside the descriptor and arrive as zeros), B as whole fragments
// (one wave-uniform descriptor per row block, the stage offset a scalar).
// int8 rows stay bytes in LDS and are dequantised after the fragment read.
// An S-stage ring keeps S - 1 stages in flight; a stage is waited for with an
// explicit vmcnt (younger stages stay in flight) and a plain barrier.
//
// Measured on MI355X (cold operands, replayed in a graph) against the
// register-staged kernel, which streams all weights once per 16 rows where M
// is not a multiple of 32: M = 624 fp16 gate/up 180 -> 44 us, gate/up dX 196
// -> 43 us; M = 128 int8 (which that kernel also took) gate/up 111 -> 20 us,
// Q/K/V 60 -> 11 us; M = 512 fp16 against the 128 x 64 tiles this kernel
// replaced: gate/up 45 -> 36 us, its dX 43 -> 38 us, O 15 -> 14 us; the
// logits of M = 128 (128 x 256 tiles, 622 MB of weights) 172 -> 162 us, their
// dX 135 -> 130 us.
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer, 32-bit data format
typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ void buffer_lds16(__amdgpu_buffer_rsrc_t rs, void* lds, unsigned voff,
                                             unsigned soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, kRsrcWord3);
}
// slot of 16-byte piece p (0..7) of A row r in a stage
__device__ __forceinline__ int a_slot(int r, int p) { return p ^ ((r >> 1) & 7); }

// vmcnt(rem * OPS): the rem youngest stages (OPS DMA issues of this wave
// each) may still be in flight, everything older has landed.
template <int OPS, int MAXREM>
__device__ __forceinline__ void wait_stages(int rem) {
  [&]<int... R>(std::integer_sequence<int, R...>) LLMT_INLINE {
    (void)((rem == R ? (wait_vm<R * OPS>(), true) : false) || ...);
  }(std::make_integer_sequence<int, MAXREM + 1>{});
}

// Shape of a stage-ring tile: S stages, MR x NB fragments (16 rows / columns
// each) a workgroup, WR x (4 / WR) waves over them and two groups of four
// waves over the k halves of a stage.
template <int S_, int MR_, int NB_, int WR_, bool I8_>
struct RingCfg {
  static constexpr int S = S_, MR = MR_, NB = NB_, WR = WR_, WC = 4 / WR_;
  static constexpr bool I8 = I8_;
  static constexpr int FR = MR / WR, FC = NB / WC;  // fragments a wave
  // Fragments one stage ahead in registers, where a wave has enough MFMAs a
  // stage to cover the reads; the 32-row waves of the narrow 128-row tiles
  // (8 MFMAs a stage, HBM-bound) read a stage when it lands instead: at
  // M = 128 the O GEMM 7.5 -> 7.2 us, gate/up dX 17.6 -> 17.2.
  static constexpr bool AHEAD = WR < 4;
  static constexpr int AB = MR * 2048;              // A bytes a stage
  static constexpr int BB = NB * (I8 ? 1024 : 2048);
  static constexpr int KSB = I8 ? 256 : 0;          // per-k scales of a stage (int8)
  static constexpr int SB = AB + BB + KSB;
  static constexpr int XCH = 8 * (FR / 2) * FC * 1024;  // k-half exchange
  static constexpr int LDS = S * SB > XCH ? S * SB : XCH;
  static_assert(MR % WR == 0 && NB % WC == 0 && FR % 2 == 0, "whole fragments a wave");
  static_assert(LDS <= 160 * 1024, "ring fits the LDS");
};

// One output tile over stages [c0, c1) of 64 k.  B8: this tile's B rows are
// int8 (a GEMM with int8 weights has its fp16 LoRA rows in tiles of their
// own, half as many fragments wide so that they take the same LDS).
template <class C, bool B8, bool KS, bool GLU>
__device__ __forceinline__ void ring_tile(const GemmArgs& g, char* smem, int seg, int f0, int ct,
                                          int rb, int sp, int ntn) {
  constexpr int S = C::S, MR = C::MR, FR = C::FR;
  constexpr bool HALF = C::I8 && !B8;              // an fp16 tile of an int8 GEMM
  constexpr int NB = HALF ? C::NB / 2 : C::NB;
  constexpr int FC = HALF ? (C::FC + 1) / 2 : C::FC;
  constexpr int BK = B8 ? 512 : 1024;              // bytes of a B fragment (32 k)
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave >> 2, wq = wave & 3, wr = wq % C::WR, wc = wq / C::WR;
  const int m0 = rb * MR * 16;
  const int ksteps = g.K / KSTEP, nst = g.K / 64;
  const int c0 = (int)((long long)sp * nst / g.split);
  const int c1 = (int)((long long)(sp + 1) * nst / g.split);
  const BSeg& sg = g.seg[seg];

  // A: 2 MR pieces of 8 rows x 128 bytes a stage, wave w moves pieces
  // APW w ..; rows past M lie outside the descriptor and arrive as zeros
  constexpr int APW = (2 * MR + 7) / 8;
  const int naw = 2 * MR >= 8 ? APW : (wave < 2 * MR ? 1 : 0);
  const __amdgpu_buffer_rsrc_t ars =
      make_rsrc(g.A + (long long)m0 * g.lda, (unsigned)min(MR * 16, g.M - m0) * (unsigned)g.lda * 2u);
  unsigned aoff[APW];
#pragma unroll
  for (int i = 0; i < APW; ++i) {
    const int r = 8 * (APW * wave + i) + (lane >> 3);
    aoff[i] = (unsigned)((r * g.lda + a_slot(r, lane & 7) * 8) * 2);
  }
  // B: fp16 row blocks as two 1 KB fragments (k halves), wave w moves half
  // w / 4 of row blocks w % 4, w % 4 + 4, ..; int8 row blocks as one 1 KB
  // piece, wave w moves row blocks w, w + 8, ..
  constexpr int BST = B8 ? 8 : 4;
  constexpr int BPW = (NB + BST - 1) / BST;
  const int bw = B8 ? wave : wq;
  const int nbw = (NB - bw + BST - 1) / BST;
  __amdgpu_buffer_rsrc_t brs[BPW];
#pragma unroll
  for (int i = 0; i < BPW; ++i) {
    const int f = min(bw + BST * i, NB - 1);
    long long rbk;
    if constexpr (GLU) {
      const int pr = ct * (NB / 2) + (f >> 1);
      rbk = (f & 1) * (g.glu >> 4) + (pr < (g.glu >> 4) ? pr : 0);
      brs[i] = make_rsrc((const char*)sg.ptr + rbk * ksteps * BK, (unsigned)(ksteps * BK));
    } else if constexpr (C::I8) {
      rbk = f0 + f < (sg.rows >> 4) ? f0 + f : 0;
      brs[i] = make_rsrc((const char*)sg.ptr + rbk * ksteps * BK, (unsigned)(ksteps * BK));
    } else {  // fp16 tiles may straddle segments
      const int nn = 16 * (f0 + f);
      int s = 0;
#pragma unroll
      for (int q = 1; q < 4; ++q)
        if (q < g.nseg && nn >= g.seg_start[q]) s = q;
      rbk = nn < g.N ? (nn - g.seg_start[s]) >> 4 : 0;
      brs[i] = make_rsrc((const char*)g.seg[s].ptr + rbk * ksteps * BK, (unsigned)(ksteps * BK));
    }
  }
  const bool ksw = KS && B8 && wave == 7;  // wave 7 also moves the stage's 64 k scales
  const __amdgpu_buffer_rsrc_t krs = make_rsrc(KS && B8 ? sg.kscale : nullptr,
                                               KS && B8 ? (unsigned)(g.K * 2) : 0u);
  auto issue = [&](int c) LLMT_INLINE {
    char* st = smem + (c % S) * C::SB;
#pragma unroll
    for (int i = 0; i < APW; ++i)
      if (i < naw) buffer_lds16(ars, st + (APW * wave + i) * 1024, aoff[i], c * 128u);
#pragma unroll
    for (int i = 0; i < BPW; ++i)
      if (i < nbw) {
        if constexpr (B8)
          buffer_lds16(brs[i], st + C::AB + (bw + 8 * i) * 1024, lane * 16u, c * 1024u);
        else
          buffer_lds16(brs[i], st + C::AB + ((bw + 4 * i) * 2 + kg) * 1024, lane * 16u + kg * 1024u,
                       c * 2048u);
      }
    if constexpr (KS && B8) {
      if (ksw && lane < 8) buffer_lds16(krs, st + C::AB + C::BB, lane * 16u, c * 128u);
    }
  };
  // DMA issues a stage of this wave: OMIN .. OMAX
  constexpr int OMIN = (2 * MR >= 8 ? APW : 0) + NB / BST;
  constexpr int OMAX = APW + BPW + (KS && B8 ? 1 : 0);
  const int nops = naw + nbw + (ksw ? 1 : 0);
  auto wait_rem = [&](int rem) LLMT_INLINE {
    [&]<int... O>(std::integer_sequence<int, O...>) LLMT_INLINE {
      (void)((OMIN == OMAX || nops == OMIN + O ? (wait_stages<OMIN + O, S - 1>(rem), true) : false) || ...);
    }(std::make_integer_sequence<int, OMAX - OMIN + 1>{});
  };

  int aread[FR];
#pragma unroll
  for (int i = 0; i < FR; ++i) {
    const int r = 16 * (wr * FR + i) + (lane & 15);
    aread[i] = r * 128 + a_slot(r, 4 * kg + (lane >> 4)) * 16;
  }
  floatx4 acc[FR][FC];
#pragma unroll
  for (int i = 0; i < FR; ++i)
#pragma unroll
    for (int j = 0; j < FC; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  half8 a[FR], b[FC], bn[FC], ksn;
  u32x2 b8[FC];
  auto read_a = [&](const char* st, int i) LLMT_INLINE {
    a[i] = *reinterpret_cast<const half8*>(st + aread[i]);
  };
  auto read_b = [&](const char* st) LLMT_INLINE {
    if constexpr (KS && B8)
      ksn = *reinterpret_cast<const half8*>(st + C::AB + C::BB + kg * 64 + (lane >> 4) * 16);
#pragma unroll
    for (int j = 0; j < FC; ++j) {
      const int f = min(wc * FC + j, NB - 1);
      if constexpr (B8)
        b8[j] = *reinterpret_cast<const u32x2*>(st + C::AB + f * 1024 + kg * 512 + lane * 8);
      else
        bn[j] = *reinterpret_cast<const half8*>(st + C::AB + (f * 2 + kg) * 1024 + lane * 16);
    }
  };
  auto take_b = [&]() LLMT_INLINE {
#pragma unroll
    for (int j = 0; j < FC; ++j) {
      if constexpr (B8) {
        b[j] = i8x8_to_h8(b8[j]);
        if constexpr (KS) b[j] = b[j] * ksn;
      } else {
        b[j] = bn[j];
      }
    }
  };

  if constexpr (C::AHEAD) {
    for (int c = c0; c < c1 && c < c0 + S; ++c) issue(c);
    wait_rem(min(S, c1 - c0) - 1);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    {
      const char* st = smem + (c0 % S) * C::SB;
      read_b(st);
#pragma unroll
      for (int i = 0; i < FR; ++i) read_a(st, i);
      take_b();
    }
    for (int c = c0; c < c1 - 1; ++c) {
      // stage c + 1 landed, and this wave's reads of stage c returned: after
      // the barrier slot c % S takes stage c + S
      wait_rem(min(S - 2, c1 - 2 - c));
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (c + S < c1) issue(c + S);
      const char* st = smem + ((c + 1) % S) * C::SB;
      read_b(st);
#pragma unroll
      for (int i = 0; i < FR; ++i) {
#pragma unroll
        for (int j = 0; j < FC; ++j) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
        read_a(st, i);
      }
      // B reads first, then each row's MFMAs and the read that refills its A
      // register
      __builtin_amdgcn_sched_group_barrier(0x100, FC + (KS && B8 ? 1 : 0), 0);
#pragma unroll
      for (int i = 0; i < FR; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, FC, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      take_b();
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
      for (int j = 0; j < FC; ++j) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
  } else {
    for (int c = c0; c < c1 && c < c0 + S - 1; ++c) issue(c);
    for (int c = c0; c < c1; ++c) {
      // stage c landed for every wave, and every wave is past its reads of
      // stage c - 1, whose slot takes stage c + S - 1
      wait_rem(min(S - 2, c1 - 1 - c));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (c + S - 1 < c1) issue(c + S - 1);
      const char* st = smem + (c % S) * C::SB;
      read_b(st);
#pragma unroll
      for (int i = 0; i < FR; ++i) read_a(st, i);
      take_b();
#pragma unroll
      for (int j = 0; j < FC; ++j)
#pragma unroll
        for (int i = 0; i < FR; ++i) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
      asm volatile("" ::: "memory");
    }
  }

  // the two k halves meet: each wave hands the other group's half of its row
  // fragments over through the (now free) ring, adds what it gets to its own
  // half and stores it
  constexpr int FH = FR / 2;
  wait_vm<0>();
  __syncthreads();
  floatx4* xch = reinterpret_cast<floatx4*>(smem) + (size_t)wq * (2 * FH * FC * 64);
#pragma unroll
  for (int h = 0; h < FH; ++h)
#pragma unroll
    for (int j = 0; j < FC; ++j)
      xch[(((1 - kg) * FH + h) * FC + j) * 64 + lane] = kg ? acc[h][j] : acc[FH + h][j];
  __syncthreads();
  floatx4 o[FH][FC];
#pragma unroll
  for (int h = 0; h < FH; ++h)
#pragma unroll
    for (int j = 0; j < FC; ++j)
      o[h][j] = (kg ? acc[FH + h][j] : acc[h][j]) + xch[((kg * FH + h) * FC + j) * 64 + lane];
  const int row0 = m0 + (wr * FR + kg * FH) * 16;  // first row of this wave's half

  if constexpr (GLU) {
    const _Float16* cs = sg.colscale;
#pragma unroll
    for (int jj = 0; jj < FC / 2; ++jj) {
      const int pr = ct * (NB / 2) + wc * (FC / 2) + jj;
      if (pr >= (g.glu >> 4)) continue;
      const int col = pr * 16 + (lane & 15);
      const float sgt = cs ? (float)cs[col] : 1.0f, su = cs ? (float)cs[g.glu + col] : 1.0f;
#pragma unroll
      for (int h = 0; h < FH; ++h) {
        if (row0 + 16 * h >= g.M) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const long long row = row0 + 16 * h + (lane >> 4) * 4 + v;
          const float gt = o[h][2 * jj][v] * sgt, up = o[h][2 * jj + 1][v] * su;
          g.gu16[row * (2LL * g.glu) + col] = (_Float16)gt;
          g.gu16[row * (2LL * g.glu) + g.glu + col] = (_Float16)up;
          g.glu16[row * g.ldglu + col] = (_Float16)(gt * sigmoid_rcp(gt) * up);
        }
      }
    }
    return;
  }
  float* Cp = g.C + (long long)sp * g.split_stride;
  const int n0 = (C::I8 ? g.seg_start[seg] : 0) + 16 * f0;  // first column of the tile
  const int nend = C::I8 ? g.seg_start[seg] + sg.rows : g.N;
  // a wave-uniform row base plus one 32-bit lane offset for every store
  const int lo = (lane >> 4) * 4 * g.ldc + (lane & 15);
  float* const Cw = Cp + (long long)row0 * g.ldc;
#pragma unroll
  for (int j = 0; j < FC; ++j) {
    const int nn = n0 + 16 * (wc * FC + j);
    if (nn >= nend || wc * FC + j >= NB) continue;
    if constexpr (B8) {
      const _Float16* cs = sg.colscale;
      const float sc = cs ? (float)cs[nn - g.seg_start[seg] + (lane & 15)] : 1.0f;
#pragma unroll
      for (int h = 0; h < FH; ++h) o[h][j] *= sc;
    }
#pragma unroll
    for (int h = 0; h < FH; ++h) {
      if (row0 + 16 * h >= g.M) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float* const Cr = Cw + (long long)(16 * h + v) * g.ldc + nn;
        Cr[lo] = o[h][j][v];
      }
    }
  }
  if constexpr (!C::I8) {
    if (g.rowstats) {
      // each row's (max, sum exp) over the tile: a wave's pair over its
      // columns from its 16-lane groups, the column waves merged in order
      constexpr int WC = C::WC;
      float2* sh = reinterpret_cast<float2*>(smem);  // [16 MR][WC]
      __syncthreads();  // the exchange has been read
#pragma unroll
      for (int h = 0; h < FH; ++h)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float x[FC];
#pragma unroll
          for (int j = 0; j < FC; ++j)
            x[j] = n0 + 16 * (wc * FC + j) < nend ? o[h][j][v] : -INFINITY;
          const float2 p = softmax_pair16<FC>(x);
          if ((lane & 15) == 0)
            sh[((wr * FR + kg * FH + h) * 16 + (lane >> 4) * 4 + v) * WC + wc] = p;
        }
      __syncthreads();
      for (int r = threadIdx.x; r < MR * 16 && m0 + r < g.M; r += 512) {
        float m = -INFINITY, s = 0.f;
#pragma unroll
        for (int w = 0; w < WC; ++w) softmax_merge(m, s, sh[r * WC + w].x, sh[r * WC + w].y);
        g.rowstats[(long long)(m0 + r) * ntn + ct] = make_float2(m, s);
      }
    }
  }
}

// Tile (row block, column tile, split) of linear workgroup id t.  One row
// block: the split is fastest, so the K slices of a column tile spread over
// the XCDs (workgroup t runs on XCD t % 8) while each XCD reads only the A
// columns of its splits.  More: each XCD gets a contiguous run of tiles with
// the row block fastest, so a B tile is fetched into one XCD's L2 and read
// there by every row block.
template <class C, bool KS, bool GLU>
__global__ __launch_bounds__(512) void gemm_ring_kernel(const GemmArgs g, int nrb, int nct) {
  __shared__ __attribute__((aligned(1024))) char smem[C::LDS];
  int rb = 0, ct = blockIdx.y, sp = blockIdx.x;  // one row block: grid (split, column tile)
  if (nrb > 1) {
    int t = blockIdx.x;
    const int n = gridDim.x, x = t & 7, q = n >> 3, r = n & 7;
    t = x * q + min(x, r) + (t >> 3);
    rb = t % nrb;
    t /= nrb;
    ct = t % nct;
    sp = t / nct;
  }
  if constexpr (C::I8) {
    const int nm = GLU ? nct : (g.seg[0].rows + C::NB * 16 - 1) / (C::NB * 16);
    if (ct < nm) {
      ring_tile<C, true, KS, GLU>(g, smem, 0, ct * C::NB, ct, rb, sp, nct);
    } else if constexpr (!GLU) {
      ring_tile<C, false, false, false>(g, smem, 1, (ct - nm) * (C::NB / 2), ct, rb, sp, nct);
    }
  } else {
    ring_tile<C, false, false, GLU>(g, smem, 0, ct * C::NB, ct, rb, sp, nct);
  }
}

template <int MF, int NF, int NW, int CHS, int RING, int ADIST>
hipError_t launch_cfg(const GemmArgs& g, hipStream_t st) {
  const int ncols = NW * NF * 16;
  dim3 grid((g.N + ncols - 1) / ncols, g.split, g.M / (MF * 16));
  bool i8 = false;
  for (int i = 0; i < g.nseg; ++i) i8 = i8 || g.seg[i].is_i8;
  if (i8)
    hipLaunchKernelGGL((gemm_nt_kernel<MF, NF, NW, CHS, RING, ADIST, true>), grid, dim3(NW * 64), 0,
                       st, g);
  else
    hipLaunchKernelGGL((gemm_nt_kernel<MF, NF, NW, CHS, RING, ADIST, false>), grid, dim3(NW * 64),
                       0, st, g);
  return hipGetLastError();
}

// The register-staged kernel's pipeline: 4 waves a workgroup, 2 k-steps an
// LDS chunk, a 4-slot B ring, A prefetched one chunk ahead (measured the
// fastest of the variants tried on the logits GEMM and the int8 GEMMs).
constexpr int kNF = 2, kNW = 4;

template <int MF>
hipError_t launch_mf(const GemmArgs& g, hipStream_t st) {
  return launch_cfg<MF, kNF, kNW, 2, 4, 1>(g, st);
}

// Fixed-order split-K reduction fused with the LoRA up-projections:
//   out[m][n] = sum_s part[s][m][n] + lscale * sum_r h[m][r] * M_p(r, n - c0_p)
// for n inside adapter p's column range (adapters may share columns: each
// one covering n adds its term), where h (the rank-16 LoRA activations,
// x A^T forward or dy B backward) is itself a set of extra columns of the same
// GEMM, reduced here first, per 16-row block, into LDS.  M_p is B [n, 16]
// (forward: y += s h B^T) or A [16, n] (backward: dx += s dh A).
// Workgroup: 16 rows x 64 columns; thread = one row x four columns.  The
// kernel is latency-bound (the partials were just written), so every load
// it needs (adapter block, h partials, column partials; RB splits at a time)
// is issued before the first sum; sums run in split order (deterministic).
constexpr int RB = 16;  // partial loads in flight per thread

__device__ __forceinline__ float4 add4(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// sum_s p[s * ss] for s < split, in order, RB loads in flight
__device__ __forceinline__ float4 sum_splits(const float* p, int split, long long ss) {
  float4 v = *reinterpret_cast<const float4*>(p);
  for (int k = 1; k < split; k += RB) {
    float4 x[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
      x[i] = *reinterpret_cast<const float4*>(p + (long long)min(k + i, split - 1) * ss);
#pragma unroll
    for (int i = 0; i < RB; ++i)
      if (k + i < split) v = add4(v, x[i]);
  }
  return v;
}

__global__ __launch_bounds__(256) void reduce_lora_kernel(const ReduceArgs a) {
  __shared__ float hs[16][3 * 16 + 4];
  __shared__ float ms[3][16][64 + 1];  // this block's 64 columns of each adapter matrix
  const int m0 = blockIdx.y * 16;
  const int cb = blockIdx.x * 64;
  const int tid = threadIdx.x;
  // Adapter column ranges are multiples of 64 wide and aligned: a block is
  // entirely inside or outside each of them.
  int inside = 0;
  for (int q = 0; q < a.nlora; ++q)
    if (cb >= a.up[q].c0 && cb < a.up[q].c0 + a.up[q].n) inside |= 1 << q;
  // adapter blocks -> registers (12 values per thread per adapter)
  float mreg[3][4];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (!(inside >> q & 1)) continue;
    const LoraUp& u = a.up[q];
    const int jb = cb - u.c0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = tid + 256 * e;  // 0..1023
      mreg[q][e] = u.is_B ? u.M[(long long)(jb + (i >> 4)) * 16 + (i & 15)]
                          : u.M[(long long)(i >> 6) * u.n + jb + (i & 63)];
    }
  }
  // h partials: thread -> (row tid / 12, 4 h columns), 192 threads
  const int nh4 = 4 * a.nlora;  // float4 groups of h per row
  float4 hv = make_float4(0.f, 0.f, 0.f, 0.f);
  const bool hthread = inside && tid < 16 * nh4;
  const int hr = hthread ? tid / nh4 : 0, hg = hthread ? tid % nh4 : 0;
  if (hthread)
    hv = sum_splits(a.part + (long long)(m0 + hr) * a.ldp + a.up[hg >> 2].hcol + (hg & 3) * 4,
                    a.split, a.ss);
  const int t = tid >> 4;
  const int cc = (tid & 15) * 4;
  const int c = cb + cc;
  const bool live = c < a.N;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live) v = sum_splits(a.part + (long long)(m0 + t) * a.ldp + c, a.split, a.ss);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (!(inside >> q & 1)) continue;
    const bool isB = a.up[q].is_B;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = tid + 256 * e;
      if (isB) ms[q][i & 15][i >> 4] = mreg[q][e];
      else ms[q][i >> 6][i & 63] = mreg[q][e];
    }
  }
  if (hthread) {
    float* h = &hs[hr][(hg >> 2) * 16 + (hg & 3) * 4];
    h[0] = hv.x; h[1] = hv.y; h[2] = hv.z; h[3] = hv.w;
  }
  __syncthreads();
  if (!live) return;
  for (int q = 0; q < a.nlora; ++q) {
    if (!(inside >> q & 1)) continue;
    float l0 = 0.f, l1 = 0.f, l2 = 0.f, l3 = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float h = hs[t][q * 16 + r];
      l0 += h * ms[q][r][cc];
      l1 += h * ms[q][r][cc + 1];
      l2 += h * ms[q][r][cc + 2];
      l3 += h * ms[q][r][cc + 3];
    }
    v.x += a.lscale * l0;
    v.y += a.lscale * l1;
    v.z += a.lscale * l2;
    v.w += a.lscale * l3;
  }
  if (a.out_scale != 0.f && a.out_scale != 1.f) {
    v.x *= a.out_scale;
    v.y *= a.out_scale;
    v.z *= a.out_scale;
    v.w *= a.out_scale;
  }
  *reinterpret_cast<float4*>(a.out + (long long)(m0 + t) * a.ldo + c) = v;
}

// Pack rows [row0, row0 + R) x k [k0, k0 + C) of a fragment-packed B operand
// (row length K) from a row-major source (leading dimension lds): if
// transpose, element (i, j) of the destination block is src[j][i], else
// src[i][j].  One thread per 8-element piece; C % 8 == 0, k0 % 8 == 0.
// int8: zs (may be NULL) is the fp16 scale of each source row; a row whose
// scale is 0 is stored as zeros, so the packed values agree with the
// dequantised weights whichever side applies the scale.
template <typename T>
__global__ void pack_kernel(const T* __restrict__ src, long long lds, int transpose, int R, int C,
                            T* __restrict__ dst, long long K, int row0, int k0,
                            const _Float16* __restrict__ zs) {
  const long long np = (long long)R * (C / 8);
  for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < np;
       p += (long long)gridDim.x * blockDim.x) {
    int i, jp;
    if (transpose) {  // consecutive threads: consecutive destination rows
      i = (int)(p % R);
      jp = (int)(p / R);
    } else {
      i = (int)(p / (C / 8));
      jp = (int)(p % (C / 8));
    }
    T v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int sr = transpose ? jp * 8 + e : i;  // source row
      v[e] = transpose ? src[(long long)sr * lds + i] : src[(long long)i * lds + jp * 8 + e];
      if (zs && zs[sr] == (_Float16)0.0f) v[e] = T(0);
    }
    T* d = dst + packed_index(row0 + i, k0 + jp * 8, K);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (std::is_same_v<T, int8_t>)
        d[e] = (int8_t)((uint8_t)v[e] ^ 0x80u);  // biased: byte = x + 128
      else
        d[e] = v[e];
    }
  }
}

// 64x64 tiles through LDS; 256 threads.
__global__ void transpose_f16_kernel(const _Float16* __restrict__ src, int rows, int cols, int lds,
                                     _Float16* __restrict__ dst, int ldd) {
  __shared__ _Float16 tile[64][65];
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < 64; r += 4) {
    const int gr = r0 + r, gc = c0 + tx;
    if (gr < rows && gc < cols) tile[r][tx] = src[(long long)gr * lds + gc];
  }
  __syncthreads();
  for (int c = ty; c < 64; c += 4) {
    const int gc = c0 + c, gr = r0 + tx;
    if (gc < cols && gr < rows) dst[(long long)gc * ldd + gr] = tile[tx][c];
  }
}

__global__ void transpose_i8_kernel(const int8_t* __restrict__ src, int rows, int cols, int lds,
                                    int8_t* __restrict__ dst, int ldd) {
  __shared__ int8_t tile[64][68];
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < 64; r += 4) {
    const int gr = r0 + r, gc = c0 + tx;
    if (gr < rows && gc < cols) tile[r][tx] = src[(long long)gr * lds + gc];
  }
  __syncthreads();
  for (int c = ty; c < 64; c += 4) {
    const int gc = c0 + c, gr = r0 + tx;
    if (gc < cols && gr < rows) dst[(long long)gc * ldd + gr] = tile[tx][c];
  }
}

__global__ void f32_to_f16_kernel(const float* __restrict__ s, _Float16* __restrict__ d, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    d[i] = (_Float16)s[i];
}

__global__ void copy_rows_f16_kernel(const _Float16* __restrict__ s, int rows, int cols, int lds,
                                     _Float16* __restrict__ d, int ldd) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)rows * cols) return;
  const int r = (int)(i / cols), c = (int)(i % cols);
  d[(long long)r * ldd + c] = s[(long long)r * lds + c];
}

__global__ void fill_f32_kernel(float* d, float v, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    d[i] = v;
}

// src/kernels/quantize.cu:8-44, bit-exact: scale = max|w|/127 (IEEE fp32
// division), inv = 1/scale, q = rint(clamp(w*inv, -127, 127)) with
// round-half-to-even (v_rndne_f32).  One workgroup of 256 per row.
__global__ void quantize_rows_kernel(const float* __restrict__ w, int cols, int8_t* __restrict__ q,
                                     float* __restrict__ scale) {
  __shared__ float red[4];
  const long long base = (long long)blockIdx.x * cols;
  float m = 0.f;
  for (int c = threadIdx.x; c < cols; c += blockDim.x) m = fmaxf(m, fabsf(w[base + c]));
  m = block_max<4>(m, red);
  const float sc = m / 127.0f;
  if (threadIdx.x == 0) scale[blockIdx.x] = sc;
  const float inv = sc > 0.f ? 1.0f / sc : 0.f;
  for (int c = threadIdx.x; c < cols; c += blockDim.x) {
    float v = w[base + c] * inv;
    v = fminf(fmaxf(v, -127.f), 127.f);
    q[base + c] = (int8_t)rintf(v);
  }
}

__global__ void f32_scale_to_f16_kernel(const float* s, _Float16* d, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = (_Float16)s[i];
}

inline int grid1d(size_t n, int bs, int cap = 65536) {
  size_t g = (n + bs - 1) / bs;
  return (int)(g > (size_t)cap ? cap : (g == 0 ? 1 : g));
}

}  // namespace

void gemm_finalize_segments(GemmArgs& g) {
  int s = 0;
  for (int i = 0; i < g.nseg; ++i) {
    g.seg_start[i] = s;
    s += g.seg[i].rows;
  }
  for (int i = g.nseg; i <= 4; ++i) g.seg_start[i] = s;
  g.N = s;
}

// Depth of the register-staged fallback: LLMT_GEMM_SKINNY_STAGES = 0 selects
// it for fp16 M % 128 == 0; 3, 5 or 6 with LLMT_GEMM_SKINNY_NB (2, 3, 4, 6 or
// 8 column fragments) force that ring for tests and tuning.
static int skinny_stages() { return env_int("LLMT_GEMM_SKINNY_STAGES", 4); }

// ------------------------------------------------------------------ plan
// Every tile the library launches, with the modelled time of a launch in us:
//   launch + waves (wave + stages (stage + fill f)) + part split M N / 1e6
// waves: rounds of the 256 CUs that the workgroups take, f: how full they
// are (a fuller chip shares L2 and HBM), stages: 64-wide K stages of a
// workgroup.  Fitted on MI355X to 4,800 timings of the layer GEMMs of
// Qwen3-1.7B (M = 16 .. 4096, cold random operands): mean error 4%, and the
// tile and split picked from the model cost 0.6% over the best measured ones
// on average, 7% at worst.  The logits GEMM is outside of that: several rounds
// of column tiles that do not run in step, and the statistics (128 rows: 112 us
// modelled, 162-170 measured; the pick is within 1% of the best in the head).
enum { GK_NT = 0, GK_RING = 1, GK_BIG = 2 };
struct TileCost {
  int kind, i8, mr, nb;
  float launch, wave, stage, fill, part;
};
static const TileCost kTiles[] = {
    {GK_RING, 0, 2, 4, 3.607f, 0.219f, 0.200f, 0.069f, 0.815f},
    {GK_RING, 0, 2, 8, 2.544f, 1.642f, 0.275f, 0.162f, 0.633f},
    {GK_RING, 0, 4, 4, 4.288f, 0.002f, 0.178f, 0.089f, 0.814f},
    {GK_RING, 0, 4, 8, 2.784f, 1.773f, 0.292f, 0.166f, 0.579f},
    {GK_RING, 0, 8, 3, 2.839f, 1.055f, 0.323f, 0.034f, 1.122f},
    {GK_RING, 0, 8, 4, 3.067f, 0.888f, 0.342f, 0.062f, 1.058f},
    {GK_RING, 0, 8, 8, 3.380f, 1.277f, 0.403f, 0.206f, 0.814f},
    {GK_RING, 0, 8, 12, 4.222f, 1.775f, 0.520f, 0.270f, 0.679f},
    {GK_RING, 0, 8, 16, 4.392f, 2.099f, 0.720f, 0.278f, 0.600f},
    {GK_BIG, 0, 16, 16, 4.626f, 0.000f, 1.213f, 0.541f, 0.854f},
    {GK_RING, 1, 2, 4, 3.686f, 0.000f, 0.249f, 0.000f, 0.748f},
    {GK_RING, 1, 2, 8, 2.031f, 1.299f, 0.312f, 0.111f, 0.912f},
    {GK_RING, 1, 4, 4, 2.147f, 1.397f, 0.349f, 0.021f, 0.924f},
    {GK_RING, 1, 4, 8, 2.668f, 1.546f, 0.392f, 0.081f, 0.778f},
    {GK_RING, 1, 8, 8, 3.108f, 1.488f, 0.470f, 0.113f, 0.695f},
    {GK_RING, 1, 8, 12, 3.362f, 2.829f, 0.570f, 0.215f, 0.492f},
    {GK_RING, 1, 8, 16, 3.915f, 2.049f, 0.759f, 0.179f, 0.599f},
    {GK_BIG, 1, 16, 16, 4.076f, 1.263f, 1.343f, 0.403f, 0.791f},
};
struct GemmPlan {
  int kind, mr, nb, split;
};
// What the GEMM asks of its tile besides the product.
enum { GN_PLAIN = 0, GN_GLU = 1, GN_STATS = 2 };

// The cheapest tile and split (fixed > 0: with that split) of a GEMM.  A
// consumer reads every partial back (at 5.5 TB/s), and the row epilogues
// issue 2, 4 or 8 partials as one round trip, other counts as several.  In the
// step that consumer runs anyway; `reduce` says that the sum is a pass of its
// own that an unsplit GEMM does without (the standalone products): a launch,
// about 4 us with its gap, and the output written again.  (Planned as in the
// step, the standalone fp16 product M256 N4096 K2048 took 12.8 + 5.0 us in two
// parts against 13.2 unsplit, M384 15.1 + 6.6 against 15.4, M128 N14336 K4096
// 29.1 + 6.7 against 30.7.)
// N counts a trailing LoRA segment (N % 64 rows); on 256 x 256 tiles it
// rides along, with int8 weights it has column tiles of its own.
static GemmPlan gemm_plan(int M, int N, int K, bool i8, int need, int fixed, int max_split,
                          bool reduce = false) {
  GemmPlan best{GK_NT, 0, 0, 0};
  if (K % 64) return best;
  double best_t = 1e300;
  const int nst = K / 64, tail = N % 64, nmain = N - tail;
  for (const TileCost& c : kTiles) {
    if (c.i8 != (i8 ? 1 : 0)) continue;
    // SwiGLU: whole (gate, up) fragment pairs a wave (RingCfg::FC even)
    if (need == GN_GLU && c.kind == GK_RING && (c.nb % 2 || (c.mr == 2 && c.nb == 4))) continue;
    // the softmax pairs' array has room for tiles of 128 columns or more
    if (need == GN_STATS && c.nb < 8) continue;
    // 256-row tiles below 512 rows leave most of a tile empty
    if (c.kind == GK_BIG && (M < 512 || (need == GN_GLU && N % 256))) continue;
    const int rows = 16 * c.mr, cols = 16 * c.nb;
    int nct;
    if (c.kind == GK_BIG) nct = ((nmain ? nmain : N) + cols - 1) / cols;
    else if (i8) nct = (nmain + cols - 1) / cols + (tail + cols / 2 - 1) / (cols / 2);
    else nct = (N + cols - 1) / cols;
    const int tiles = nct * ((M + rows - 1) / rows);
    auto consider = [&](int split) {
      if (split < 1 || split > max_split || split > nst) return;
      const int wg = tiles * split, waves = (wg + 255) / 256, st = (nst + split - 1) / split;
      const double pm = (double)split * M * N * 1e-6, fill = wg / (256.0 * waves);
      double t = c.launch + waves * (c.wave + st * (c.stage + c.fill * fill)) + c.part * pm;
      t += pm * (4 / 5.5) + (split == 1 || split == 2 || split == 4 || split == 8 ? 0.0 : 0.8);
      if (reduce && split > 1) t += 4.0 + (double)M * N * 1e-6 * (4 / 5.5);
      if (t < best_t) {
        best_t = t;
        best = {c.kind, c.mr, c.nb, split};
      }
    };
    if (fixed > 0) {
      consider(fixed);
    } else {
      // at most two rounds of the CUs, at least two stages a workgroup
      const int most = nst / 2 > 1 ? nst / 2 : 1;
      const int s1 = 256 / tiles, s2 = 512 / tiles;
      consider(1);
      consider(s1 < most ? s1 : most);
      consider(s2 < most ? s2 : most);
      for (int s = 2; s <= 8; s *= 2)
        if (s <= s2 && s <= most) consider(s);
    }
  }
  return best;
}

// 256 x 256 tiles take one B segment plus at most one fp16 LoRA segment whose
// fragments fit on the column tiles (fragment f rides with tile f).
static bool big_segments(const GemmArgs& g) {
  if (g.nseg == 1) return true;
  return g.nseg == 2 && !g.seg[1].is_i8 && g.seg[1].rows <= 64 && g.seg_start[1] % 64 == 0 &&
         g.seg[1].rows / 16 <= (g.seg[0].rows + 255) / 256;
}
static bool ring_segments(const GemmArgs& g) {
  if (g.seg[0].is_i8) return g.nseg == 1 || (g.nseg == 2 && !g.seg[1].is_i8);
  for (int i = 1; i < g.nseg; ++i)
    if (g.seg[i].is_i8) return false;
  return true;
}

// The plan gemm_nt launches for g (g.split fixed by the caller).
static GemmPlan plan_of(const GemmArgs& g) {
  const GemmPlan nt{GK_NT, 0, 0, g.split};
  if (g.K % 64 || g.split > g.K / 64) return nt;
  if (g.split_col) return {GK_BIG, 16, 16, g.split};  // planned as 256 x 256 tiles, unsplit
  // the LDS-DMA kernels move 16-byte pieces of A's rows; a caller's rows that
  // start elsewhere (the standalone GEMMs, the head's hidden states) are read
  // by register loads, which have no such requirement
  if (((uintptr_t)g.A | (uintptr_t)g.lda * sizeof(_Float16)) % 16 && !g.glu) return nt;
  const bool i8 = g.seg[0].is_i8;
  if (!i8 && g.M % 128 == 0 && skinny_stages() == 0 && !g.glu) return nt;
  const int need = g.glu ? GN_GLU : g.rowstats ? GN_STATS : GN_PLAIN;
  GemmPlan p = gemm_plan(g.M, g.N, g.K, i8, need, g.split, g.split);
  if (p.kind == GK_BIG && !big_segments(g)) p = {GK_RING, 8, 8, g.split};
  if (p.kind == GK_RING && !ring_segments(g)) return nt;
  return p;
}

int gemm_rowstats_tiles(const GemmArgs& g) {
  if (g.split != 1 || g.nseg != 1 || g.glu || g.N < 16 || g.seg[0].is_i8) return 0;
  GemmArgs q = g;
  static float2 any;
  q.rowstats = &any;  // planned with the statistics, as it will be launched
  const GemmPlan p = plan_of(q);
  const int cols = p.kind == GK_NT ? kNW * kNF * 16 : 16 * p.nb;
  return (g.N + cols - 1) / cols;
}

// The last wave of an unsplit 256 x 256-tile GEMM: with tiles = full waves of
// the 256 CUs plus r more (r <= 128, whole column tiles), the last r tiles
// run as 2 r half-K workgroups, so the launch takes 1 + 1/2 wave-times of a
// tile instead of 2.  Their partial is an extra fp32 [M, r/ntm x 256] the
// consumer reads back.  (The plan takes 128 x 256 ring tiles for the
// down-projection dX of hidden 2048, intermediate 6144; the split is reached
// at other widths, for instance hidden 512, intermediate 4352, 8192 rows: 544
// tiles.)
int gemm_split_col(int M, int N, int K, bool i8) {
  if (N % 256 || K % 64 || K / 64 < 8) return 0;
  const GemmPlan p = gemm_plan(M, N, K, i8, GN_PLAIN, 0, 64);
  if (p.kind != GK_BIG || p.split != 1) return 0;
  const int ntm = (M + BM - 1) / BM, ntn = N / 256, tiles = ntm * ntn;
  const int rest = tiles % 256;
  if (tiles < 256 || rest == 0 || rest > 128 || rest % ntm) return 0;
  return (ntn - rest / ntm) * 256;
}

// Forced ring widths (tests, tuning): the splits that keep the grid near one
// workgroup per CU.
static int forced_split(int M, int N, int K, int nb) {
  const int tiles = ((N + 15) / 16 + nb - 1) / nb * (M / 128);
  int split = (K <= 4096 ? 192 : 256) / tiles;
  if (split > K / 128) split = K / 128;
  return split < 1 ? 1 : split;
}
static int forced_nb(int M, int K, bool i8) {
  if (i8 || M % 128 || K % 64) return 0;
  return env_int("LLMT_GEMM_SKINNY_NB", 0);
}

int gemm_pick_split(int M, int N, int K, int max_split, bool i8, bool reduce) {
  if (const int nb = forced_nb(M, K, i8)) {
    const int s = forced_split(M, N, K, nb);
    return s > max_split ? max_split : s;
  }
  const GemmPlan p = gemm_plan(M, N, K, i8, GN_PLAIN, 0, max_split, reduce);
  if (p.kind != GK_NT) return p.split;
  // the register-staged kernel: about 3/4 of the CUs, four k-steps or more a
  // split
  const int mt = (M % 128 == 0) ? M / 128 : 1;
  constexpr int tn = kNW * kNF * 16;
  const int ntiles = (N + tn - 1) / tn * mt;
  int split = ((K > 16384 ? 512 : 192) + ntiles / 2) / ntiles;
  const int kmax = (K / KSTEP) / 4;
  if (split > kmax) split = kmax;
  if (split > max_split) split = max_split;
  if (split < 1) split = 1;
  return split;
}

// GLU false: a tile that only plain GEMMs are launched on (the forced ones).
template <class C, bool GLU = true>
static hipError_t launch_ring(const GemmArgs& g, hipStream_t st) {
  const int nrb = (g.M + C::MR * 16 - 1) / (C::MR * 16);
  int nct;
  if (g.glu) {
    nct = (g.glu / 16 + C::NB / 2 - 1) / (C::NB / 2);
  } else if (C::I8) {
    nct = (g.seg[0].rows / 16 + C::NB - 1) / C::NB;
    if (g.nseg > 1) nct += (g.seg[1].rows / 16 + C::NB / 2 - 1) / (C::NB / 2);
  } else {
    nct = (g.N / 16 + C::NB - 1) / C::NB;
  }
  const dim3 grid = nrb == 1 ? dim3(g.split, nct) : dim3(nrb * nct * g.split);
  if (g.glu) {
    if constexpr (GLU && C::FC % 2 == 0) {
      hipLaunchKernelGGL((gemm_ring_kernel<C, false, true>), grid, dim3(512), 0, st, g, nrb, nct);
      return hipGetLastError();
    }
    set_error("gemm_nt: no SwiGLU epilogue on tiles of %d fragments", C::NB);
    return hipErrorInvalidValue;
  }
  if constexpr (C::I8) {
    if (g.seg[0].kscale) {
      hipLaunchKernelGGL((gemm_ring_kernel<C, true, false>), grid, dim3(512), 0, st, g, nrb, nct);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((gemm_ring_kernel<C, false, false>), grid, dim3(512), 0, st, g, nrb, nct);
  return hipGetLastError();
}

// Ring depths: what keeps enough weight bytes in flight (about 24 KB a CU)
// and fits the LDS.
static hipError_t launch_plan(const GemmArgs& g, const GemmPlan& p, hipStream_t st) {
  const bool i8 = g.seg[0].is_i8;
  const int key = p.mr * 100 + p.nb;
  if (i8) {
    switch (key) {
      case 204: return launch_ring<RingCfg<8, 2, 4, 1, true>>(g, st);
      case 208: return launch_ring<RingCfg<8, 2, 8, 1, true>>(g, st);
      case 404: return launch_ring<RingCfg<8, 4, 4, 2, true>>(g, st);
      case 408: return launch_ring<RingCfg<7, 4, 8, 2, true>>(g, st);
      case 812: return launch_ring<RingCfg<5, 8, 12, 2, true>>(g, st);
      case 816: return launch_ring<RingCfg<4, 8, 16, 2, true>>(g, st);
      default: return launch_ring<RingCfg<5, 8, 8, 2, true>>(g, st);
    }
  } else {
    switch (key) {
      case 204: return launch_ring<RingCfg<6, 2, 4, 1, false>>(g, st);
      case 208: return launch_ring<RingCfg<5, 2, 8, 1, false>>(g, st);
      case 404: return launch_ring<RingCfg<4, 4, 4, 2, false>>(g, st);
      case 408: return launch_ring<RingCfg<4, 4, 8, 2, false>>(g, st);
      case 803: return launch_ring<RingCfg<4, 8, 3, 4, false>>(g, st);
      case 804: return launch_ring<RingCfg<4, 8, 4, 4, false>>(g, st);
      case 812: return launch_ring<RingCfg<4, 8, 12, 2, false>>(g, st);
      case 816: return launch_ring<RingCfg<3, 8, 16, 2, false>>(g, st);
      default: return launch_ring<RingCfg<4, 8, 8, 2, false>>(g, st);
    }
  }
}
template <int S>
static hipError_t launch_forced(const GemmArgs& g, int nb, hipStream_t st) {
  switch (nb) {
    case 2: return launch_ring<RingCfg<S, 8, 2, 4, false>, false>(g, st);
    case 3: return launch_ring<RingCfg<S, 8, 3, 4, false>, false>(g, st);
    case 4: return launch_ring<RingCfg<S, 8, 4, 4, false>, false>(g, st);
  }
  if constexpr (S <= 5) {
    if (nb == 6) return launch_ring<RingCfg<S, 8, 6, 4, false>, false>(g, st);
    if (nb == 8) return launch_ring<RingCfg<S, 8, 8, 4, false>, false>(g, st);
  }
  set_error("gemm_nt: no %d-stage ring of %d fragments", S, nb);
  return hipErrorInvalidValue;
}

static hipError_t launch_big(const GemmArgs& g, hipStream_t st) {
  GemmArgs gm = g;
  const bool fold = g.nseg > 1;  // the LoRA rows ride along (fragment f with column tile f)
  const BSeg tl = fold ? g.seg[1] : BSeg{};
  const int tc0 = fold ? g.seg_start[1] : 0;
  gm.nseg = 1;
  gemm_finalize_segments(gm);
  const int ntm = (gm.M + BM - 1) / BM;
  // XCD-contiguous tile runs: workgroup b goes to XCD b % 8, and the tiles
  // sharing an A row block then share that XCD's L2 (+0.7% step rate at 4096
  // rows)
  const int order = 1;
  const bool i8 = gm.seg[0].is_i8, ks = gm.seg[0].kscale != nullptr;
  if (gm.split_col > 0 &&
      (gm.split != 2 || gm.split_col % 256 || gm.split_col >= gm.N || gm.N % 256 || gm.glu ||
       gm.rowstats || fold)) {
    set_error("gemm_nt: split_col %d needs split 2 and whole 256-column tiles (N = %d)",
              gm.split_col, gm.N);
    return hipErrorInvalidValue;
  }
  const dim3 gr = gm.split_col > 0
                      ? dim3(gm.split_col / 256 * ntm + 2 * (gm.N - gm.split_col) / 256 * ntm, 1)
                      : dim3((gm.N + 255) / 256 * ntm, gm.split);
  // ring depth 5 (int8) / 4 (fp16): 4 measured the same, 6 slower
  auto go = [&](auto i8c, auto ksc, auto gluc, auto tlc) {
    constexpr bool I8 = decltype(i8c)::value, KS = decltype(ksc)::value;
    constexpr bool GL = decltype(gluc)::value, TLc = decltype(tlc)::value;
    constexpr int SD = I8 ? 5 : 4;
    hipLaunchKernelGGL((gemm_dma_kernel<I8, KS, SD, 4, GL, TLc>), gr, dim3(512), 0, st, gm, order,
                       tl, tc0);
  };
  using BT = std::integral_constant<bool, true>;
  using BF = std::integral_constant<bool, false>;
  if (gm.glu) {
    if (!i8) go(BF(), BF(), BT(), BF());
    else go(BT(), BF(), BT(), BF());
  } else if (fold) {
    if (!i8) go(BF(), BF(), BF(), BT());
    else if (ks) go(BT(), BT(), BF(), BT());
    else go(BT(), BF(), BF(), BT());
  } else {
    if (!i8) go(BF(), BF(), BF(), BF());
    else if (ks) go(BT(), BT(), BF(), BF());
    else go(BT(), BF(), BF(), BF());
  }
  return hipGetLastError();
}

const char* gemm_kernel_name(const GemmArgs& g) {
  const GemmPlan p = plan_of(g);
  if (p.kind == GK_BIG) return g.glu ? "gemm_dma_glu" : g.nseg > 1 ? "gemm_dma+lora" : "gemm_dma";
  if (p.kind == GK_RING) return g.glu ? "gemm_ring_glu" : "gemm_ring";
  return "gemm_nt";
}

hipError_t gemm_nt(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.N <= 0 || g.M % 16 || g.K % KSTEP || g.K < KSTEP || g.split < 1 ||
      g.split > g.K / KSTEP || g.nseg < 1 || g.nseg > 4) {
    set_error("gemm_nt: unsupported shape M=%d N=%d K=%d split=%d", g.M, g.N, g.K, g.split);
    return hipErrorInvalidValue;
  }
  for (int i = 0; i < g.nseg; ++i) {
    if (g.seg[i].rows % 16) {
      set_error("gemm_nt: segment rows must be a multiple of 16 (%d)", g.seg[i].rows);
      return hipErrorInvalidValue;
    }
    // scales that the kernels do not apply
    if (g.seg[i].kscale && (g.glu || !g.seg[i].is_i8)) {
      set_error("gemm_nt: a per-k scale needs an int8 segment and no SwiGLU epilogue");
      return hipErrorInvalidValue;
    }
    if (g.seg[i].colscale && !g.seg[i].is_i8) {
      set_error("gemm_nt: a column scale needs an int8 segment");
      return hipErrorInvalidValue;
    }
  }
  const GemmPlan p = plan_of(g);
  if (g.glu && !(g.N == 2 * g.glu && g.glu % 16 == 0 && g.nseg == 1 && g.split == 1 && g.glu16 &&
                 g.gu16 && p.kind != GK_NT)) {
    set_error("gemm_nt: SwiGLU epilogue needs K %% 64 == 0, split 1, one segment, N = 2 x %d", g.glu);
    return hipErrorInvalidValue;
  }
  if (!g.glu && !g.C) {
    set_error("gemm_nt: no output");
    return hipErrorInvalidValue;
  }
  if (g.split_col && p.kind != GK_BIG) {
    set_error("gemm_nt: split_col needs the large-tile kernel");
    return hipErrorInvalidValue;
  }
  if (g.rowstats && gemm_rowstats_tiles(g) == 0) {
    set_error("gemm_nt: row statistics need split 1, one fp16 segment and no SwiGLU epilogue");
    return hipErrorInvalidValue;
  }
  hipError_t e;
  const int m16 = g.M / 16;
  const int nb = g.glu || g.rowstats ? 0 : forced_nb(g.M, g.K, g.seg[0].is_i8);
  if (p.kind == GK_RING && nb) {
    switch (skinny_stages()) {
      case 3: e = launch_forced<3>(g, nb, st); break;
      case 5: e = launch_forced<5>(g, nb, st); break;
      case 6: e = launch_forced<6>(g, nb, st); break;
      default: e = launch_forced<4>(g, nb, st); break;
    }
  }
  else if (p.kind == GK_RING) e = launch_plan(g, p, st);
  else if (p.kind == GK_BIG) e = launch_big(g, st);
  else if (m16 % 8 == 0) e = launch_mf<8>(g, st);
  else if (m16 % 4 == 0) e = launch_mf<4>(g, st);
  else if (m16 % 2 == 0) e = launch_mf<2>(g, st);
  else e = launch_mf<1>(g, st);
  if (e != hipSuccess && e != hipErrorInvalidValue) set_error("gemm_nt launch: %s", hipGetErrorString(e));
  return e;
}

hipError_t reduce_lora(const ReduceArgs& a, hipStream_t st) {
  if (a.M % 16 || a.N % 4 || a.ldp % 4 || a.ldo % 4 || a.nlora < 0 || a.nlora > 3 ||
      a.out == a.part) {
    set_error("reduce_lora: M %% 16, N/ldp/ldo %% 4, nlora <= 3 and out != part required");
    return hipErrorInvalidValue;
  }
  for (int q = 0; q < a.nlora; ++q)
    if (a.up[q].c0 % 64 || a.up[q].n % 64 || a.up[q].hcol % 4) {
      set_error("reduce_lora: adapter column ranges must be 64-aligned, h columns 4-aligned");
      return hipErrorInvalidValue;
    }
  dim3 grid((a.N + 63) / 64, a.M / 16);
  hipLaunchKernelGGL(reduce_lora_kernel, grid, dim3(256), 0, st, a);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t pack_f16(const _Float16* src, long long lds, int transpose, int R, int C, _Float16* dst,
                    long long K, int row0, int k0, hipStream_t st) {
  if (C % 8 || k0 % 8 || K % 32) {
    set_error("pack_f16: C, k0 must be multiples of 8 and K of 32");
    return hipErrorInvalidValue;
  }
  const long long np = (long long)R * (C / 8);
  hipLaunchKernelGGL(pack_kernel<_Float16>, dim3(grid1d(np, 256)), dim3(256), 0, st, src, lds,
                     transpose, R, C, dst, K, row0, k0, nullptr);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t pack_i8(const int8_t* src, long long lds, int transpose, int R, int C, int8_t* dst,
                   long long K, int row0, int k0, hipStream_t st, const _Float16* zs) {
  if (C % 8 || k0 % 8 || K % 32) {
    set_error("pack_i8: C, k0 must be multiples of 8 and K of 32");
    return hipErrorInvalidValue;
  }
  const long long np = (long long)R * (C / 8);
  hipLaunchKernelGGL(pack_kernel<int8_t>, dim3(grid1d(np, 256)), dim3(256), 0, st, src, lds,
                     transpose, R, C, dst, K, row0, k0, zs);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t transpose_f16(const _Float16* src, int rows, int cols, int lds, _Float16* dst, int ldd,
                         hipStream_t st) {
  dim3 grid((cols + 63) / 64, (rows + 63) / 64);
  hipLaunchKernelGGL(transpose_f16_kernel, grid, dim3(256), 0, st, src, rows, cols, lds, dst, ldd);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t transpose_i8(const int8_t* src, int rows, int cols, int lds, int8_t* dst, int ldd,
                        hipStream_t st) {
  dim3 grid((cols + 63) / 64, (rows + 63) / 64);
  hipLaunchKernelGGL(transpose_i8_kernel, grid, dim3(256), 0, st, src, rows, cols, lds, dst, ldd);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t f32_to_f16(const float* src, _Float16* dst, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(f32_to_f16_kernel, dim3(grid1d(n, 256)), dim3(256), 0, st, src, dst, n);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t copy_rows_f16(const _Float16* src, int rows, int cols, int lds, _Float16* dst, int ldd,
                         hipStream_t st) {
  const long long n = (long long)rows * cols;
  hipLaunchKernelGGL(copy_rows_f16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, src,
                     rows, cols, lds, dst, ldd);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t fill_f32(float* dst, float v, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(fill_f32_kernel, dim3(grid1d(n, 256)), dim3(256), 0, st, dst, v, n);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t quantize_rows_i8(const float* w, int rows, int cols, int8_t* q, float* scale,
                            hipStream_t st) {
  hipLaunchKernelGGL(quantize_rows_kernel, dim3(rows), dim3(256), 0, st, w, cols, q, scale);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

hipError_t f32_scale_to_f16(const float* s, _Float16* d, int n, hipStream_t st) {
  hipLaunchKernelGGL(f32_scale_to_f16_kernel, dim3((n + 255) / 256), dim3(256), 0, st, s, d, n);
  LLMT_LAUNCH_CHECK();
  return hipSuccess;
}

}  // namespace llmt
