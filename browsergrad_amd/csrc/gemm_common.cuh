// Argument block, tile order and epilogue shared by the GEMM translation units.
#pragma once

#include "common.cuh"
#include "core.h"

namespace {

using namespace bgk;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf168 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));
// Native 16-byte vector (HIP's uint4 is a union-based struct, which keeps
// arrays of it from being promoted to registers).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct GemmArgs {
  const void* A;
  const void* B;
  const float* bias;
  void* C;
  int64_t M, N, K;
  int64_t lda, ldb, ldc;
  int64_t sa, sb, sc;  // batch strides (elements)
  int tiles_m, tiles_n;
  int round_dtype;  // 0 none, 1 f16, 2 bf16
  int act;          // BG_ACT_*
  int out_dtype;    // BG_F32 / BG_F16 / BG_BF16
  int vec_store;    // C rows can take 4-element vector stores (ldc % 4, alignment)
  const float* R;   // residual f32 [batch][M][N] added last (NULL: none)
  int64_t ldr, sr;  // its row and batch strides (elements)
};

// XCD-aware tile index -> (tile_m, tile_n).  Workgroups are dispatched
// round-robin over the 8 XCDs; the tiles of one XCD are made consecutive and
// then walked in groups of G tile-rows so neighbours share A and B panels.
__device__ __forceinline__ void tile_coords(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  if (total % 8 == 0) {
    const int per = total / 8;
    pid = (pid % 8) * per + pid / 8;
  }
  constexpr int G = 4;
  const int group = pid / (G * tiles_n);
  const int first_m = group * G;
  const int gsz = min(G, tiles_m - first_m);
  const int in_group = pid % (G * tiles_n);
  tm = first_m + in_group % gsz;
  tn = in_group / gsz;
}

__device__ __forceinline__ float epilogue_value(const GemmArgs& P, float v, float bias) {
  if (P.round_dtype) v = round_through(v, P.round_dtype);
  if (P.bias) v = v + bias;
  if (P.act == BG_ACT_RELU) v = v > 0.f ? v : 0.f;
  else if (P.act == BG_ACT_GELU_TANH) v = gelu_tanh(v);
  return v;
}

template <int OUT>
__device__ __forceinline__ void store_elem(char* p, float v) {
  if constexpr (OUT == BG_F32) *reinterpret_cast<float*>(p) = v;
  else if constexpr (OUT == BG_F16) *reinterpret_cast<uint16_t*>(p) = f32_to_f16_bits(v);
  else *reinterpret_cast<uint16_t*>(p) = f32_to_bf16_bits(v);
}

// Epilogue in registers, stored straight to C, one 32x32 accumulator tile
// (16 values per lane) at a time: [round to the 16-bit type] -> [+ bias[n]]
// -> [relu] -> store, each stage behind one uniform branch per tile.
// Scheduling fences between tiles keep the live set to one tile, so the
// accumulators never spill.  tanh-GELU (one exponential and one reciprocal
// per element) runs here for wavefront tiles of up to kGeluEpilogueTiles
// accumulator tiles; wider ones leave it to a separate f32 pass over C
// (run_matmul).
// 32x32 MFMA accumulator layout: lane l, register e holds row
// 8*(e/4) + 4*(l/32) + e%4, column l%32, so each store instruction writes 32
// consecutive columns of two rows.  Addresses are a uniform per-row base plus
// one 32-bit per-lane offset; nothing in the loop waits on memory.
// Largest per-wavefront accumulator tile count (TM * TN) whose epilogue
// evaluates GELU in registers.
constexpr int kGeluEpilogueTiles = 8;

template <int TM, int TN, bool FULL, int OUT>
__device__ __forceinline__ void epilogue_tiles(const GemmArgs& P, char* C, float16v (&acc)[TM][TN],
                                               int64_t row0, int64_t col0, const float (&bz)[TN]) {
  constexpr int ES = OUT == BG_F32 ? 4 : 2;
  const int lane = threadIdx.x & 63;
  const int half = lane >> 5;
  const int64_t cl = col0 + (lane & 31);
  char* corner = C + (row0 * P.ldc + col0) * ES;
  const uint32_t lane_off = uint32_t((4 * half * P.ldc + (lane & 31)) * ES);
  const int64_t row_bytes = P.ldc * ES;
  // Residual (f32, added after the activation): 16 values per tile, same
  // element layout as the accumulator tile.
  float rnext[16];
  const float* rbase = P.R ? P.R + int64_t(blockIdx.z) * P.sr + (row0 + 4 * half) * P.ldr + cl : nullptr;
  auto load_residual = [&](int ti, int tj) {
    const bool ok_c = FULL || cl + tj * 32 < P.N;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int rr = ti * 32 + 8 * (e >> 2) + (e & 3);
      rnext[e] = (FULL || (ok_c && row0 + rr + 4 * half < P.M)) ? rbase[rr * P.ldr + tj * 32] : 0.f;
    }
  };
  if (P.R) load_residual(0, 0);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      float v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = acc[i][j][e];
      if (P.round_dtype == 1) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = round_through(v[e], 1);
      } else if (P.round_dtype == 2) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = round_through(v[e], 2);
      }
      if (P.bias) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = v[e] + bz[j];
      }
      if (P.act == BG_ACT_RELU) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = v[e] > 0.f ? v[e] : 0.f;
      } else if constexpr (TM * TN <= kGeluEpilogueTiles) {
        // tanh-GELU on 16 values at a time (the tile fence below keeps the
        // compiler from interleaving tiles); wider wavefront tiles leave no
        // registers for it and take the separate f32 pass instead.
        if (P.act == BG_ACT_GELU_TANH) {
#pragma unroll
          for (int e = 0; e < 16; ++e) v[e] = gelu_tanh(v[e]);
        }
      }
      const bool col_ok = FULL || cl + j * 32 < P.N;
      if (P.R) {
        // The residual of this tile was loaded one tile ahead (before the
        // previous tile's stores), so its wait does not queue behind them.
        float cur[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) cur[e] = rnext[e];
        if (i * TN + j + 1 < TM * TN) load_residual((i * TN + j + 1) / TN, (i * TN + j + 1) % TN);
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = v[e] + cur[e];
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int rr = i * 32 + 8 * (e >> 2) + (e & 3);
        if (FULL || (col_ok && row0 + rr + 4 * half < P.M))
          store_elem<OUT>(corner + rr * row_bytes + lane_off + j * 32 * ES, v[e]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
}

template <int TM, int TN, bool FULL>
__device__ __forceinline__ void direct_epilogue(const GemmArgs& P, char* C, float16v (&acc)[TM][TN],
                                                int64_t row0, int64_t col0) {
  const int lane = threadIdx.x & 63;
  const int64_t cl = col0 + (lane & 31);
  float bz[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
    bz[j] = (P.bias && (FULL || cl + j * 32 < P.N)) ? P.bias[cl + j * 32] : 0.f;
  if (P.out_dtype == BG_F32) epilogue_tiles<TM, TN, FULL, BG_F32>(P, C, acc, row0, col0, bz);
  else if (P.out_dtype == BG_F16) epilogue_tiles<TM, TN, FULL, BG_F16>(P, C, acc, row0, col0, bz);
  else epilogue_tiles<TM, TN, FULL, BG_BF16>(P, C, acc, row0, col0, bz);
}

}  // namespace
