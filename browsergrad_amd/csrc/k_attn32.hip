// Float32 attention forward on the matrix cores (gfx950), head dim <= 64.
//
// Replaces the reference's row-wise online-softmax WGSL kernel
// (packages/browsergrad-kernels/src/kernels/flash_attention.ts:45-211: one
// invocation per query row, every K/V row read from storage, f32 throughout,
// optional additive mask [1|B, 1|H, Sq, Sk], MAX_D = 64) behind
// bridge.flash_attention (realizer.ts:1122-1151), the typed
// ATTENTION_FORWARD and the semantic attention, and keeps its numerics:
// scores s = (q . k) * scale (+ mask), online softmax with the running
// maximum starting at the -1e20 sentinel, output O / l with the l > 0 guard.
//
// Design (one 256-thread workgroup = 4 wavefronts x 32 queries of one
// (batch, head); K and V stream through LDS in 64-key tiles):
//   * S^T = K Q^T with v_mfma_f32_32x32x2_f32.  MFMA j of the d loop takes
//     d = 8 (j / 4) + 4 (lane / 32) + j % 4 on both operands, so a lane's
//     K operand for four MFMAs is one 16-byte LDS read and its Q operand sits
//     in registers for the whole loop (Q pre-multiplied by scale * log2 e,
//     which puts the softmax in the exp2 domain).
//   * The accumulator layout gives a lane 16 keys of one query (rows
//     8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32).  Those registers
//     are, unchanged, the B operands of O^T += V^T P^T: MFMA j of the key loop
//     takes key 8 (j / 4) + 4 (lane / 32) + j % 4 on both operands, so P never
//     leaves the registers; the V^T operand is one 4-byte LDS read per lane.
//   * The row maximum is exact for every 32-key half (f32 has no overflow
//     concern that would allow a lazy one): 16 maxima and one exchange with
//     lane ^ 32; the rescale of O and l costs 33 multiplies against 64 MFMAs
//     of 64 cycles per half.
//   * K rows (256 bytes) store 16-byte chunk c at c ^ (row % 16): the 16
//     lanes a ds_read_b128 serves together read 16 different rows at one
//     chunk, which then covers all 64 banks.  V rows store chunk c at
//     c ^ 8 (row / 4 % 2): the two half-wavefronts of a V read take rows four
//     apart at the same 32 columns, which then land on disjoint banks.
//   * Tiles are staged through registers with one tile of prefetch: the
//     global loads of tile t + 1 are issued before tile t's MFMAs and
//     written to the other LDS buffer after them (one barrier per tile).
//     A tile is 128 MFMAs of 64 cycles per wavefront, which covers HBM
//     latency many times over.
//   * Causal (top-left aligned, key j visible to query i iff j <= i): tiles
//     after the workgroup's last query are not loaded, a wavefront skips
//     halves wholly after its 32 queries, and only halves that cross the
//     diagonal or the key length are masked.  Heavy query blocks go first.
// Bound: fp32 MFMA (157.3 TFLOP/s dense); 4 * B * H * D * (visible pairs)
// FLOP per launch.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <initializer_list>

#include "common.cuh"
#include "core.h"
#include "split.cuh"

namespace {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kQW = 32;        // queries per wavefront
constexpr int kNW = 4;         // wavefronts per workgroup
constexpr int kBQ = kQW * kNW;  // queries per workgroup
constexpr int kBK = 64;        // keys per tile
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kMSentinel = -1.0e20f;  // flash_attention.ts:101 (m_i = -1.0e20)

struct Fa32Args {
  const float* q;
  const float* k;
  const float* v;
  const float* mask;  // NULL: no additive mask
  void* o;
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_sh, k_ss;
  int64_t v_sb, v_sh, v_ss;
  int64_t o_sb, o_sh, o_ss;
  int64_t m_sb, m_sh, m_ss;  // mask strides (batch, head, query row); keys contiguous
  int H, Sq, Sk, D;
  int n_qblocks;
  float sl2;      // scale * log2(e)
  int causal;
  int out_dtype;  // 0 f32, 1 f16, 2 bf16
};

__device__ __forceinline__ float16v mfma32(float a, float b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Value of lane ^ 32 (the other half-wavefront holds the same query).
__device__ __forceinline__ float xor32(float x) {
  const int v = __builtin_bit_cast(int, x);
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return __builtin_bit_cast(float, (threadIdx.x & 32) ? r[0] : r[1]);
}

__device__ __forceinline__ int k_slot(int row, int c) { return row * 64 + ((c ^ (row & 15)) << 2); }
__device__ __forceinline__ int v_slot(int row, int c) { return row * 64 + ((c ^ ((row & 4) << 1)) << 2); }

// Four floats of row `row` starting at column 4c of a [rows][D] operand
// (zeros past D or past the row count).  VEC: one 16-byte load (rows
// 16-byte aligned, D % 4 == 0).
template <bool VEC>
__device__ __forceinline__ float4v load4(const float* base, int64_t ss, int row, int nrows, int c, int D) {
  float4v r = {0.f, 0.f, 0.f, 0.f};
  if (row >= nrows || 4 * c >= D) return r;
  const float* p = base + int64_t(row) * ss + 4 * c;
  if constexpr (VEC) {
    return *reinterpret_cast<const float4v*>(p);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = 4 * c + i < D ? p[i] : 0.f;
    return r;
  }
}

// DP: head dim rounded up to 16, 32 or 64 (the MFMA d loop covers DP / 2
// values per half-wavefront; columns past D are zero in LDS and registers).  NT
// threads stage; the first kNW wavefronts compute.
// lds: two buffers of a K tile and a V tile, 64 rows x 256 bytes each.
constexpr int kFa32Lds = 2 * 2 * kBK * 256;

template <int DP, bool VEC, int NT>
__device__ __forceinline__ void fa32_tiles(const Fa32Args& P, float* lds) {
  constexpr int NG = DP / 8;             // 16-byte K reads per lane per half (4 MFMAs each)
  constexpr int NDB = DP > 32 ? 2 : 1;   // 32-row blocks of O^T
  constexpr int CH = DP / 4;             // 16-byte chunks per row that hold data
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int hi = lane >> 5;
  const int l32 = lane & 31;
  const int bh = blockIdx.x;
  const int qblk = P.n_qblocks - 1 - int(blockIdx.y);  // heavy (late) blocks first
  const int b = bh / P.H, h = bh % P.H;
  const int q0 = qblk * kBQ;
  const int q0w = q0 + w * kQW;
  const int qi = q0w + l32;

  const float* Qp = P.q + b * P.q_sb + h * P.q_sh;
  const float* Kp = P.k + b * P.k_sb + h * P.k_sh;
  const float* Vp = P.v + b * P.v_sb + h * P.v_sh;
  const float* Mp = P.mask ? P.mask + b * P.m_sb + h * P.m_sh : nullptr;

  const int nt_all = (P.Sk + kBK - 1) / kBK;
  const int nt = P.causal ? min(nt_all, (q0 + kBQ + kBK - 1) / kBK) : nt_all;

  // Q operand: qf[g][i] = Q[qi][8 g + 4 hi + i] * scale * log2(e).
  float qf[NG][4];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const float4v x = load4<VEC>(Qp, P.q_ss, qi, P.Sq, 2 * g + hi, P.D);
#pragma unroll
    for (int i = 0; i < 4; ++i) qf[g][i] = x[i] * P.sl2;
  }

  // Tile staging: thread t moves 16-byte units t, t + NT, ... of the K and
  // V tiles (unit u = row u / 16, chunk u % 16; chunks past DP / 4 stay 0).
  constexpr int UNITS = kBK * 16 / NT;
  float4v kst[UNITS], vst[UNITS];
  auto fetch = [&](int t) {
#pragma unroll
    for (int s = 0; s < UNITS; ++s) {
      const int u = threadIdx.x + s * NT;
      const int row = u >> 4, c = u & 15;
      const int key = t * kBK + row;
      kst[s] = c < CH ? load4<VEC>(Kp, P.k_ss, key, P.Sk, c, P.D) : float4v{0.f, 0.f, 0.f, 0.f};
      vst[s] = c < CH ? load4<VEC>(Vp, P.v_ss, key, P.Sk, c, P.D) : float4v{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto stash = [&](int buf) {
    float* kt = lds + buf * (2 * kBK * 64);
    float* vt = kt + kBK * 64;
#pragma unroll
    for (int s = 0; s < UNITS; ++s) {
      const int u = threadIdx.x + s * NT;
      const int row = u >> 4, c = u & 15;
      *reinterpret_cast<float4v*>(kt + k_slot(row, c)) = kst[s];
      *reinterpret_cast<float4v*>(vt + v_slot(row, c)) = vst[s];
    }
  };

  float16v acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[db][e] = 0.f;
  float m_run = kMSentinel, l_run = 0.f;
  const float mask_l2 = kLog2e;

  if (nt > 0) {
    fetch(0);
    stash(0);
  }
  __syncthreads();
  for (int t = 0; t < nt; ++t) {
    if (t + 1 < nt) fetch(t + 1);
    const float* kt = lds + (t & 1) * (2 * kBK * 64);
    const float* vt = kt + kBK * 64;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int j0 = t * kBK + hh * 32;
      if (NT > kNW * 64 && w >= kNW) continue;
      // A half wholly after the wavefront's last query adds nothing (causal).
      if (P.causal && j0 > q0w + kQW - 1) continue;
      if (j0 >= P.Sk) continue;
      float16v s;
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = 0.f;
      const int krow = hh * 32 + l32;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const float4v kf = *reinterpret_cast<const float4v*>(kt + k_slot(krow, 2 * g + hi));
#pragma unroll
        for (int i = 0; i < 4; ++i) s = mfma32(kf[i], qf[g][i], s);
      }
      // s[e]: key j0 + 8 (e / 4) + 4 hi + e % 4, query qi (log2 domain).
      const bool edge = (P.causal && j0 + 31 > q0w) || j0 + 32 > P.Sk;
      if (Mp) {
        const float* mrow = Mp + int64_t(min(qi, P.Sq - 1)) * P.m_ss;
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int kj = j0 + 8 * a + 4 * hi + c;
            s[4 * a + c] = kj < P.Sk ? __builtin_fmaf(mrow[kj], mask_l2, s[4 * a + c]) : s[4 * a + c];
          }
      }
      if (edge) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int kj = j0 + 8 * (e >> 2) + 4 * hi + (e & 3);
          if (kj >= P.Sk || (P.causal && kj > qi)) s[e] = -INFINITY;
        }
      }
      float mt = s[0];
#pragma unroll
      for (int e = 1; e < 16; ++e) mt = fmaxf(mt, s[e]);
      mt = fmaxf(mt, xor32(mt));
      const float m_new = fmaxf(m_run, mt);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[db][e] *= alpha;
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        s[e] = __builtin_amdgcn_exp2f(s[e] - m_new);
        s[e + 1] = __builtin_amdgcn_exp2f(s[e + 1] - m_new);
        l0 += s[e];
        l1 += s[e + 1];
      }
      l_run += l0 + l1;
      // O^T[32 db + lane % 32][q] += sum_j V[key(j)][32 db + lane % 32] P[q][key(j)].
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int vrow = hh * 32 + 8 * (j >> 2) + 4 * hi + (j & 3);
          const int col = 32 * db + l32;
          const float vf = vt[v_slot(vrow, col >> 2) + (col & 3)];
          acc[db] = mfma32(vf, s[j], acc[db]);
        }
    }
    if (t + 1 < nt) stash((t + 1) & 1);
    __syncthreads();
  }

  // O = acc / l (l > 0 guard, flash_attention.ts:125).  acc[db][e] holds
  // O^T[d = 32 db + 8 (e / 4) + 4 hi + e % 4][qi].
  const float lt = l_run + xor32(l_run);
  const float inv = lt > 0.f ? 1.0f / lt : 0.f;
  if (qi >= P.Sq || (NT > kNW * 64 && w >= kNW)) return;
  const int64_t obase = int64_t(b) * P.o_sb + int64_t(h) * P.o_sh + int64_t(qi) * P.o_ss;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int d = 32 * db + 8 * (e >> 2) + 4 * hi + (e & 3);
      if (d < P.D) bgk::store_from_f32(P.o, P.out_dtype, obase + d, acc[db][e] * inv);
    }
}

template <int DP, bool VEC>
__global__ void __launch_bounds__(kNW * 64, 2) fa32_fwd_kernel(Fa32Args P) {
  __shared__ float4v smem[kFa32Lds / 16];
  fa32_tiles<DP, VEC, kNW * 64>(P, reinterpret_cast<float*>(smem));
}

// ---- the same attention on the bf16 matrix core ------------------------------------
//
// split_fa32_fwd_kernel keeps the tiles and the numerics above and forms its
// products from three bf16 parts of Q, K, V and P (split.cuh): 24
// v_mfma_f32_32x32x16_bf16 of 32 cycles where float32 takes 32 MFMAs of 64.
//   * 512 threads: wavefront w takes queries 32 (w % 4) .. +31 and the 32-key
//     half w / 4 of every tile, with its own maximum, sum and output; the
//     halves merge through LDS at the end.  Four more wavefronts share the
//     cost of splitting a tile and halve the chain of a tile's products.
//   * K and V are split once per workgroup on the way to LDS, V transposed:
//     eight keys of one column per 16-byte unit, in the key order of a lane's
//     accumulator registers, so P again never leaves the registers.  Two
//     buffers; the split of tile t + 1 runs beside the score MFMAs of tile t
//     (seven vector instructions an MFMA), tile t + 2 loads meanwhile.
// Bound: neither pipe alone: per tile a SIMD's two wavefronts need about 3100
// cycles of the matrix core and 3000 of the vector unit (exponentials, the
// splits of P), which overlap only in the scores.  B4 H12 S1000 D64 causal 107
// -> 60 us, B8 H16 S2048 causal 614 -> 462, one head of 2048 163 -> 92 (a
// one-buffer form of four wavefronts, two workgroups a CU: 99 / 458 / 152).
// Error against float64, 2-norm, B4 H12 S1000: 2.2e-7 (fa32_fwd_kernel 3.3e-7).
// Q, K, V and P are split times kSplitScale (Q's factor and the scores' 2^-48
// cost nothing: they ride on the scale and on the subtraction of the maximum), so
// no value and no weight that float32 holds loses bits.  (A maximum kept 24 lower,
// which scales P for free, doubles the error: the exponents round at 24 instead
// of at 1.)  A workgroup whose sums are not finite redoes its queries in
// float32 as fa32_fwd_kernel does (fa32_tiles), with its bits.

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kSplitNT = 512;  // wavefront w: queries 32 (w % 4) .., keys 32 (w / 4) .. of every tile

template <int DP, bool VEC>
__global__ void __launch_bounds__(kSplitNT, 2) split_fa32_fwd_kernel(Fa32Args P, uint32_t k_bytes,
                                                                     uint32_t v_bytes) {
  constexpr int NC = DP / 16;            // 16-deep d steps of the scores
  constexpr int NDB = DP > 32 ? 2 : 1;   // 32-row blocks of O^T
  constexpr int KU = 2 * NC * 64;        // 16-byte units per plane: 64 keys x DP / 8 chunks
  constexpr int VU = 4 * NDB * 64;       // 32 NDB columns x 8 sets of eight keys
  constexpr int NK = (KU + kSplitNT - 1) / kSplitNT, NV = (VU + kSplitNT - 1) / kSplitNT;
  constexpr int BUF = 3 * (KU + VU);
  // (4 * 64 * 9 units hold the halves' merge, kFa32Lds bytes the float32 redo.)
  static_assert(kFa32Lds / 16 >= 4 * 64 * 9, "the redo's buffers cover the merge");
  __shared__ u32x4 smem[2 * BUF > kFa32Lds / 16 ? 2 * BUF : kFa32Lds / 16];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi = lane >> 5, l32 = lane & 31;
  const int bh = blockIdx.x;
  const int qblk = P.n_qblocks - 1 - int(blockIdx.y);  // heavy (late) blocks first
  const int b = bh / P.H, h = bh % P.H;
  const int q0 = qblk * kBQ, q0w = q0 + (w & 3) * kQW, qi = q0w + l32;
  const int hh = w >> 2;
  const float* Qp = P.q + b * P.q_sb + h * P.q_sh;
  const float* Kp = P.k + b * P.k_sb + h * P.k_sh;
  const float* Vp = P.v + b * P.v_sb + h * P.v_sh;
  const float* Mp = P.mask ? P.mask + b * P.m_sb + h * P.m_sh : nullptr;
  const int nt_all = (P.Sk + kBK - 1) / kBK;
  const int nt = P.causal ? min(nt_all, (q0 + kBQ + kBK - 1) / kBK) : nt_all;
  const float q_scale = P.sl2 * bgk::kSplitScale;

  // B operand of the scores: Q[qi][16 c + 8 hi + j] * scale * log2(e).
  bgk::bf16x8 qf[NC][3];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float x[8];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float4v v = load4<VEC>(Qp, P.q_ss, qi, P.Sq, 4 * c + 2 * hi + i, P.D);
#pragma unroll
      for (int j = 0; j < 4; ++j) x[4 * i + j] = v[j] * q_scale;
    }
    u32x4 p1, p2, p3;
    bgk::split8(x, 1.f, p1, p2, p3);
    // Pinned here, beside the loads of Q and the first tile: sunk to the scores the
    // split of Q adds 0.35 us to a call (one head of 65 queries and keys 13.0 us, 12.6
    // so, 12.75 pinned after the last load of Q).
    asm volatile("" : "+v"(p1), "+v"(p2), "+v"(p3));
    qf[c][0] = __builtin_bit_cast(bgk::bf16x8, p1);
    qf[c][1] = __builtin_bit_cast(bgk::bf16x8, p2);
    qf[c][2] = __builtin_bit_cast(bgk::bf16x8, p3);
  }

  // Staging: K unit (key, 8-deep chunk), V unit (column, set of eight keys:
  // set 2 g + x holds keys 16 g + 4 x + {0..3, 8..11}).  Buffer loads: rows
  // past Sk and columns past D take an offset beyond the head's span and read 0.
  const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)Kp, (short)0, int(k_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)Vp, (short)0, int(v_bytes), 0x00020000);
  // (An offset of the high bit is beyond any span; it is or-ed in, which keeps
  // the loads free of branches.  Tiles past the last one read nothing but 0.)
  const uint32_t k_row = uint32_t(P.k_ss) * 4, v_row = uint32_t(P.v_ss) * 4;
  auto oob = [](bool ok) { return ok ? 0u : 0x80000000u; };
  uint32_t k_at[NK], k_out[NK][VEC ? 2 : 8], v_at[NV], v_out[NV];
#pragma unroll
  for (int s = 0; s < NK; ++s) {
    const int u = tid + s * kSplitNT, c = 8 * (u % (2 * NC));
    k_at[s] = uint32_t(u / (2 * NC)) * k_row + c * 4;
#pragma unroll
    for (int i = 0; i < (VEC ? 2 : 8); ++i) k_out[s][i] = oob((KU % kSplitNT == 0 || u < KU) && c + (VEC ? 4 : 1) * i < P.D);
  }
#pragma unroll
  for (int s = 0; s < NV; ++s) {
    const int u = tid + s * kSplitNT, d = u % (32 * NDB), set = u / (32 * NDB);
    v_at[s] = uint32_t(16 * (set >> 1) + 4 * (set & 1)) * v_row + d * 4;
    v_out[s] = oob((VU % kSplitNT == 0 || u < VU) && d < P.D);
  }
  float kx[NK][8], vx[NV][8];
  auto fetch = [&](int t) {
    const int left = P.Sk - t * kBK;  // rows of the tile that exist
    const uint32_t k_tile = left > 0 ? uint32_t(t * kBK) * k_row : 0u, v_tile = left > 0 ? uint32_t(t * kBK) * v_row : 0u;
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const uint32_t off = k_at[s] + k_tile, row = oob((tid + s * kSplitNT) / (2 * NC) < left);
      if constexpr (VEC) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rk, (off + 16 * i) | row | k_out[s][i], 0, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j) kx[s][4 * i + j] = __uint_as_float(v[j]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          kx[s][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rk, (off + 4 * j) | row | k_out[s][j], 0, 0));
      }
    }
#pragma unroll
    for (int s = 0; s < NV; ++s) {
      const int set = (tid + s * kSplitNT) / (32 * NDB), key0 = 16 * (set >> 1) + 4 * (set & 1);
      const uint32_t off = v_at[s] + v_tile;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int kj = (j & 3) + 8 * (j >> 2);
        vx[s][j] = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(rv, (off + kj * v_row) | v_out[s] | oob(key0 + kj < left), 0, 0));
      }
    }
  };
  auto put = [&](u32x4* st, int plane, const float (&x)[8]) {
    u32x4 p1, p2, p3;
    bgk::split8(x, bgk::kSplitScale, p1, p2, p3);
    st[0] = p1;
    st[plane] = p2;
    st[2 * plane] = p3;
  };
  auto stash = [&](int buf) {
    u32x4* st = smem + buf * BUF;
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const int u = tid + s * kSplitNT, key = u / (2 * NC), c = u % (2 * NC);
      if (KU % kSplitNT == 0 || u < KU)
        put(st + ((key >> 5) * NC + (c >> 1)) * 64 + (c & 1) * 32 + ((key & 31) ^ ((c & 1) * 8)), KU, kx[s]);
    }
#pragma unroll
    for (int s = 0; s < NV; ++s) {
      const int u = tid + s * kSplitNT, d = u % (32 * NDB), set = u / (32 * NDB);
      if (VU % kSplitNT == 0 || u < VU)
        put(st + 3 * KU + ((set >> 1) * NDB + (d >> 5)) * 64 + (set & 1) * 32 + ((d & 31) ^ ((set & 1) * 8)), VU,
            vx[s]);
    }
  };
  // Parts (i, j) of the six products, small ones first.
  constexpr int QA[6] = {2, 0, 1, 1, 0, 0}, QB[6] = {0, 2, 1, 0, 1, 0};
  const int lu = lane ^ (hi << 3);

  float16v acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[db][e] = 0.f;
  float m_run = kMSentinel, l_run = 0.f;
  float16v s;
  float mv[16];  // mask of the half, loaded ahead of the products (row and key clamped)
  // Scores of tile t, and beside their MFMAs the split of tile t + 1 from the
  // loaded registers into the other buffer.  (A half that the causal mask hides
  // computes scores that are not used.)
  auto scores = [&](int t) {
    if (Mp) {
      const float* mrow = Mp + int64_t(min(qi, P.Sq - 1)) * P.m_ss;
#pragma unroll
      for (int e = 0; e < 16; ++e) mv[e] = mrow[min(t * kBK + hh * 32 + 8 * (e >> 2) + 4 * hi + (e & 3), P.Sk - 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
    const u32x4* ks = smem + (t & 1) * BUF + hh * NC * 64 + lu;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      bgk::bf16x8 kf[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) kf[p] = __builtin_bit_cast(bgk::bf16x8, ks[p * KU + c * 64]);
#pragma unroll
      for (int p = 0; p < 6; ++p)
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[QA[p]], qf[c][QB[p]], s, 0, 0, 0);
    }
    stash((t + 1) & 1);
    __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
    for (int q = 0; q < 6 * NC; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
      if (q % 6 == 1) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Step t loads tile t + 2, takes tile t's softmax and P V, and after the
  // barrier (its buffer is free, tile t + 1's is whole) tile t + 1's scores.
  fetch(0);
  stash(0);
  fetch(1);
  __syncthreads();
  if (nt > 0) scores(0);
  for (int t = 0; t < nt; ++t) {
    fetch(t + 2);
    __builtin_amdgcn_sched_barrier(0);
    const u32x4* vs = smem + (t & 1) * BUF + 3 * KU + 2 * hh * NDB * 64 + lu;
    const int j0 = t * kBK + hh * 32;
    // A half wholly after the wavefront's queries, or past Sk, adds nothing.
    if (!(P.causal && j0 > q0w + kQW - 1) && j0 < P.Sk) {
      // s[e]: key j0 + 8 (e / 4) + 4 hi + e % 4, query qi (log2 domain, times 2^48).
      const bool edge = (P.causal && j0 + 31 > q0w) || j0 + 32 > P.Sk;
      if (Mp) {
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = __builtin_fmaf(mv[e], kLog2e / bgk::kSplitUnscale, s[e]);
      }
      if (edge) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int kj = j0 + 8 * (e >> 2) + 4 * hi + (e & 3);
          if (kj >= P.Sk || (P.causal && kj > qi)) s[e] = -INFINITY;
        }
      }
      float mt = s[0];
#pragma unroll
      for (int e = 1; e < 16; ++e) mt = fmaxf(mt, s[e]);
      mt = fmaxf(mt, xor32(mt));
      const float m_new = fmaxf(m_run, mt * bgk::kSplitUnscale);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {  // (NaN counts)
        l_run *= alpha;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[db][e] *= alpha;
      }
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        s[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], bgk::kSplitUnscale, -m_new));
        s[e + 1] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e + 1], bgk::kSplitUnscale, -m_new));
        l0 += s[e];
        l1 += s[e + 1];
      }
      l_run += l0 + l1;
      // O^T[32 db + lane % 32][q] += V^T P^T over 16 keys an MFMA: registers
      // 8 m .. 8 m + 7 are, split and packed, its B operand.
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        float px[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) px[j] = s[8 * m + j];
        u32x4 pp[3];
        bgk::split8(px, bgk::kSplitScale, pp[0], pp[1], pp[2]);
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          bgk::bf16x8 vf[3];
#pragma unroll
          for (int p = 0; p < 3; ++p)
            vf[p] = __builtin_bit_cast(bgk::bf16x8, vs[p * VU + (m * NDB + db) * 64]);
#pragma unroll
          for (int p = 0; p < 6; ++p)
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[QA[p]], __builtin_bit_cast(bgk::bf16x8, pp[QB[p]]),
                                                             acc[db], 0, 0, 0);
        }
      }
    }
    __syncthreads();
    if (t + 1 < nt) scores(t + 1);
  }

  // The two key halves of a query block merge through LDS.
  float* red = reinterpret_cast<float*>(smem) + (w & 3) * 64 * 36 + lane;
  __syncthreads();
  if (hh == 1) {
    red[0] = m_run;
    red[64] = l_run;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) red[(2 + 16 * db + e) * 64] = acc[db][e];
  }
  __syncthreads();
  bool redo = false;
  if (hh == 0) {
    const float m = fmaxf(m_run, red[0]);
    const float f0 = __builtin_amdgcn_exp2f(m_run - m), f1 = __builtin_amdgcn_exp2f(red[0] - m);
    l_run = l_run * f0 + red[64] * f1;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[db][e] = acc[db][e] * f0 + red[(2 + 16 * db + e) * 64] * f1;
        redo |= !(fabsf(acc[db][e]) <= 3.402823466e38f);
      }
  }
  const int64_t ohead = int64_t(b) * P.o_sb + int64_t(h) * P.o_sh;
  const float lt = l_run + xor32(l_run);
  const float inv = lt > 0.f ? bgk::kSplitUnscale / lt : 0.f;
  redo |= hh == 0 && !(lt <= 3.402823466e38f);
  redo = __syncthreads_or(redo);
  if (redo) {
    fa32_tiles<DP, VEC, kSplitNT>(P, reinterpret_cast<float*>(smem));
    return;
  }
  if (hh == 1 || qi >= P.Sq) return;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int d = 32 * db + 8 * (e >> 2) + 4 * hi + (e & 3);
      if (d < P.D) bgk::store_from_f32(P.o, P.out_dtype, ohead + int64_t(qi) * P.o_ss + d, acc[db][e] * inv);
    }
}

}  // namespace
namespace bg {

// 16-byte loads of Q, K and V rows: D % 4 == 0, strides in whole 16-byte
// units, and the operands' first elements 16-byte aligned (ptrs_aligned).
static bool fa32_vec(const bg_attention_desc& d, bool ptrs_aligned) {
  return ptrs_aligned && d.d % 4 == 0 && d.q_ss % 4 == 0 && d.k_ss % 4 == 0 && d.v_ss % 4 == 0 &&
         d.q_sb % 4 == 0 && d.q_sh % 4 == 0 && d.k_sb % 4 == 0 && d.k_sh % 4 == 0 && d.v_sb % 4 == 0 &&
         d.v_sh % 4 == 0;
}

// True when the f32 MFMA kernel takes this attention (head dim <= 64).
bool fa32_supported(const bg_attention_desc& d) {
  return d.in_dtype == BG_F32 && d.d >= 1 && d.d <= 64 && d.batch * d.heads <= 0x7fffffff &&
         d.sq <= int64_t(65535) * kBQ && d.sk <= (int64_t(1) << 30) && d.sq <= (int64_t(1) << 30);
}

// The split kernel from two key tiles on (one tile: 16 queries and keys 10.2
// against 8.7 us, 64: 11.5 against 11.3), and where it needs more than one round
// of 256 workgroups (one a CU; the float32 kernel has two) only with more than
// three key tiles for a query block on average: first loads, merge and
// the uneven round cost more than the products save on few.  D64, split
// against float32 kernel: 256 heads of 128 queries and keys 17 against 19 us, 384
// heads 33 / 29, 1024 heads 67 / 60; 1024 heads of 8 queries and 128 keys 52 / 47,
// 192 keys 62 / 65, 256 keys 73 / 82; causal, 1024 heads of 256 155 / 139, of 320
// 239 / 238, of 512 395 / 411.  K and V of a head within a 32-bit buffer offset.
static bool fa32_split(const bg_attention_desc& d) {
  const int64_t lim = int64_t(1) << 31;
  const int64_t blocks = (d.sq + kBQ - 1) / kBQ, tiles = (d.sk + kBK - 1) / kBK;
  if (d.batch * d.heads * blocks > 256) {
    const int64_t cut = d.causal ? std::min(blocks, tiles / 2) : 0;  // block i sees 2 i + 2 tiles
    if (cut * (cut + 1) + (blocks - cut) * tiles <= 3 * blocks) return false;
  }
  return d.reserved != BG_ATTENTION_TILED && d.sk > kBK && ((d.sk - 1) * d.k_ss + d.d) * 4 < lim &&
         ((d.sk - 1) * d.v_ss + d.d) * 4 < lim && (d.sk + 2 * kBK) * d.k_ss * 4 < 2 * lim &&
         (d.sk + 2 * kBK) * d.v_ss * 4 < 2 * lim;
}

// q, k, v, o point at the first element of each operand (offsets applied);
// mask (f32, keys contiguous) is NULL or addressed by m_sb / m_sh / m_ss.
void launch_fa32(bg_ctx* ctx, const bg_attention_desc& d, const float* q, const float* k, const float* v,
                 const float* mask, int64_t m_sb, int64_t m_sh, int64_t m_ss, void* o) {
  if (!fa32_supported(d)) fail(BG_E_UNSUPPORTED, "flash_attention: f32 MFMA kernel takes head dim 1..64");
  Fa32Args A{};
  A.q = q;
  A.k = k;
  A.v = v;
  A.mask = mask;
  A.o = o;
  A.q_sb = d.q_sb; A.q_sh = d.q_sh; A.q_ss = d.q_ss;
  A.k_sb = d.k_sb; A.k_sh = d.k_sh; A.k_ss = d.k_ss;
  A.v_sb = d.v_sb; A.v_sh = d.v_sh; A.v_ss = d.v_ss;
  A.o_sb = d.o_sb; A.o_sh = d.o_sh; A.o_ss = d.o_ss;
  A.m_sb = m_sb; A.m_sh = m_sh; A.m_ss = m_ss;
  A.H = int(d.heads);
  A.Sq = int(d.sq);
  A.Sk = int(d.sk);
  A.D = int(d.d);
  A.n_qblocks = int((d.sq + kBQ - 1) / kBQ);
  A.sl2 = d.scale * kLog2e;
  A.causal = d.causal ? 1 : 0;
  A.out_dtype = d.out_dtype;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool vec = fa32_vec(d, al16(q) && al16(k) && al16(v));
  const dim3 grid(unsigned(d.batch * d.heads), unsigned(A.n_qblocks), 1);
  auto go = [&](auto kern) { dispatch(ctx, kern, grid, dim3(kNW * 64), 0, A); };
  if (fa32_split(d)) {
    const uint32_t kb = uint32_t(((d.sk - 1) * d.k_ss + d.d) * 4), vb = uint32_t(((d.sk - 1) * d.v_ss + d.d) * 4);
    auto sgo = [&](auto kern) { dispatch(ctx, kern, grid, dim3(kSplitNT), 0, A, kb, vb); };
    if (d.d <= 16) vec ? sgo(split_fa32_fwd_kernel<16, true>) : sgo(split_fa32_fwd_kernel<16, false>);
    else if (d.d <= 32) vec ? sgo(split_fa32_fwd_kernel<32, true>) : sgo(split_fa32_fwd_kernel<32, false>);
    else vec ? sgo(split_fa32_fwd_kernel<64, true>) : sgo(split_fa32_fwd_kernel<64, false>);
  } else if (d.d <= 16) {
    vec ? go(fa32_fwd_kernel<16, true>) : go(fa32_fwd_kernel<16, false>);
  } else if (d.d <= 32) {
    vec ? go(fa32_fwd_kernel<32, true>) : go(fa32_fwd_kernel<32, false>);
  } else {
    vec ? go(fa32_fwd_kernel<64, true>) : go(fa32_fwd_kernel<64, false>);
  }
  hip_check(hipGetLastError(), "f32 attention launch");
}

// The launch bg_attention_ex makes for an f32 attention whose operands
// start at their offsets inside this library's (256-byte aligned)
// allocations; zero strides mean contiguous [B, H, S, D] as there.
void plan_attention(const bg_attention_desc& d0, bg_launch_plan& out) {
  bg_attention_desc d = d0;
  if (d.batch <= 0 || d.heads <= 0 || d.sq <= 0 || d.sk <= 0 || d.d <= 0)
    fail(BG_E_INVALID, "flash_attention: b, h, sq, sk, d must be positive integers");
  auto fix = [&](int64_t& sb, int64_t& sh, int64_t& ss, int64_t s) {
    if (sb == 0 && sh == 0 && ss == 0) {
      ss = d.d;
      sh = s * d.d;
      sb = d.heads * s * d.d;
    }
  };
  fix(d.q_sb, d.q_sh, d.q_ss, d.sq);
  fix(d.k_sb, d.k_sh, d.k_ss, d.sk);
  fix(d.v_sb, d.v_sh, d.v_ss, d.sk);
  if (!fa32_supported(d))
    fail(BG_E_UNSUPPORTED, "attention launch plan: float32 attention with head dim 1..64 only");
  const bool ptrs = (d.q_off % 4) == 0 && (d.k_off % 4) == 0 && (d.v_off % 4) == 0;
  const int dp = d.d <= 16 ? 16 : d.d <= 32 ? 32 : 64;
  out = bg_launch_plan{};
  if (const int slices = attention_decode_slices(d, ptrs)) {
    const int nq = d.sq == 1 ? 1 : d.sq == 2 ? 2 : 4;
    out.tile_m = nq;
    out.tile_n = 1;
    out.tile_k = int32_t(d.d);
    out.k_slices = slices;
    const int waves = attention_decode_waves(d);
    out.lds_bytes = waves * nq * 66 * 4;
    out.workspace_bytes = slices > 1 ? d.batch * d.heads * slices * d.sq * (d.d + 2) * 4 : 0;
    out.n_launches = slices > 1 ? 2 : 1;
    auto entry = [&](int i, const char* family, std::initializer_list<int> targs, int64_t gx, int64_t gy, int threads) {
      bg_launch_plan_entry& e = out.launch[i];
      std::snprintf(e.family, sizeof e.family, "%s", family);
      e.n_targs = int(targs.size());
      std::copy(targs.begin(), targs.end(), e.targs);
      e.grid[0] = gx; e.grid[1] = gy; e.grid[2] = 1;
      e.block[0] = threads; e.block[1] = 1; e.block[2] = 1;
    };
    entry(0, "attention_decode_kernel", {BG_F32, nq, waves}, d.batch * d.heads, slices, waves * 64);
    if (slices > 1) entry(1, "attention_decode_merge_kernel", {BG_F32}, d.batch * d.heads * d.sq, 1, 64);
    return;
  }
  out.tile_m = kBQ;
  out.tile_n = kBK;
  out.tile_k = dp;
  out.k_slices = 1;
  out.lds_bytes = kFa32Lds;
  out.n_launches = 1;
  const bool split = fa32_split(d);
  if (split) out.lds_bytes = std::max(2 * 3 * 16 * (dp * 8 + (dp > 32 ? 512 : 256)), kFa32Lds);
  bg_launch_plan_entry& e = out.launch[0];
  std::snprintf(e.family, sizeof e.family, "%s", split ? "split_fa32_fwd_kernel" : "fa32_fwd_kernel");
  e.n_targs = 2;
  e.targs[0] = dp;
  e.targs[1] = fa32_vec(d, ptrs) ? 1 : 0;
  e.grid[0] = d.batch * d.heads;
  e.grid[1] = (d.sq + kBQ - 1) / kBQ;
  e.grid[2] = 1;
  e.block[0] = split ? kSplitNT : kNW * 64; e.block[1] = 1; e.block[2] = 1;
}

}  // namespace bg
