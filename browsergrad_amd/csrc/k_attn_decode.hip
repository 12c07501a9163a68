// Attention of one or two (f32: four) query rows per head (decode): a stream over K and V.
//
// The MFMA kernels give a workgroup 128 query rows of a (batch, head) and walk
// its keys tile by tile, so with a row or two they run a serial chain of tiles
// on a few CUs.  Here one workgroup of W wavefronts reads a (batch, head)'s K and V
// once, every wavefront with four K rows and four V rows of each lane group in
// flight; a group of 8 (16-bit) or 16 (f32) lanes holds a row, keeps its own
// running maximum, sum and output, and the groups are merged at the end, inside
// the wavefront and then over the wavefronts through LDS in order.  Few heads
// with long key runs are cut into key slices, merged by a second launch.
// Bound: HBM (K and V once), below about 50 MB the latency of a few rounds of
// loads.  D64, one row, kernel time against the tiled kernels:
//   8 x 12 heads, 1024 keys, f16     7.0 us (3.6 TB/s)    13.7 us
//   64 x 16 heads, 4096 keys, f16  178.6 us (6.0 TB/s)   323.1 us
//   8 x 12 heads, 1024 keys, f32    10.6 us (4.8 TB/s)    84.4 us
//   1 x 12 heads, 4096 keys, f32    20.8 us (slices)     315.3 us
#include <algorithm>
#include <type_traits>

#include "common.cuh"
#include "core.h"

namespace {

using namespace bgk;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct DecArgs {
  const char* q;
  const char* k;
  const char* v;
  void* o;
  float* part;  // [heads][slice][query][D + 2]: maximum, sum, output (NULL: one slice)
  int64_t q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss;
  int H, Sq, Sk, D, slices, ks;
  float sl2;  // scale * log2(e)
  int causal, round_scores, out_dtype;
};

// A lane's 16 bytes of a row as floats.
template <int DT, int E>
__device__ __forceinline__ void widen(const u32x4& r, float (&x)[E]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == BG_F32) {
      x[i] = __uint_as_float(r[i]);
    } else if constexpr (DT == BG_F16) {
      x[2 * i] = f16_bits_to_f32(uint16_t(r[i]));
      x[2 * i + 1] = f16_bits_to_f32(uint16_t(r[i] >> 16));
    } else {
      x[2 * i] = __uint_as_float(r[i] << 16);
      x[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
  }
}

// exp2(a - b) for a running maximum b that may still be -inf.
__device__ __forceinline__ float rel_exp2(float a, float b) {
  return __builtin_amdgcn_exp2f(a - (b == -INFINITY ? 0.f : b));
}

template <int DT, int NQ, int W>
__global__ void __launch_bounds__(W * 64) attention_decode_kernel(DecArgs P) {
  constexpr int ES = DT == BG_F32 ? 4 : 2;
  constexpr int E = 16 / ES;   // values per lane
  constexpr int L = 64 / E;    // lanes per row
  constexpr int R = 64 / L;    // rows per wavefront load
  constexpr int U = 4;         // rows per lane group in flight
  static_assert(W >= NQ, "one wavefront finishes a row");
  __shared__ float red[W][NQ][64 + 2];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane / L, c = lane % L;
  const int bh = blockIdx.x, slice = blockIdx.y;
  const int b = bh / P.H, h = bh % P.H;
  const bool col = c * E < P.D;
  const char* Q = P.q + (b * P.q_sb + h * P.q_sh + c * E) * ES;
  const char* K = P.k + (b * P.k_sb + h * P.k_sh + c * E) * ES;
  const char* V = P.v + (b * P.v_sb + h * P.v_sh + c * E) * ES;
  const int kbeg = slice * P.ks, kend = min(P.Sk, kbeg + P.ks);
  const int kq0 = P.causal ? min(kend, 1) : kend;  // keys that query 0 sees end here, query i sees i more

  float q[NQ][E], o[NQ][E], m[NQ], l[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    u32x4 r = {0u, 0u, 0u, 0u};
    if (col && i < P.Sq) r = *reinterpret_cast<const u32x4*>(Q + i * P.q_ss * ES);
    widen<DT, E>(r, q[i]);
#pragma unroll
    for (int e = 0; e < E; ++e) o[i][e] = 0.f;
    // f32: the reference's -1e20 start (flash_attention.ts:101)
    m[i] = DT == BG_F32 ? -1.0e20f : -INFINITY;
    l[i] = 0.f;
  }
  const int kall = P.causal ? min(kend, P.Sq) : kend;
  for (int k0 = kbeg + w * R * U; k0 < kall; k0 += W * R * U) {
    u32x4 kr[U], vr[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int row = k0 + u * R + g;
      kr[u] = vr[u] = u32x4{0u, 0u, 0u, 0u};
      if (col && row < kall) {
        kr[u] = *reinterpret_cast<const u32x4*>(K + int64_t(row) * P.k_ss * ES);
        vr[u] = *reinterpret_cast<const u32x4*>(V + int64_t(row) * P.v_ss * ES);
      }
    }
    float s[NQ][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float x[E];
      widen<DT, E>(kr[u], x);
      const int row = k0 + u * R + g;
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) d = __builtin_fmaf(q[i][e], x[e], d);
        d = dpp_add<0xB1>(d);
        d = dpp_add<0x4E>(d);
        d = dpp_add<0x141>(d);                         // mirror inside 8 lanes
        if constexpr (L == 16) d = dpp_add<0x140>(d);  // mirror inside 16 lanes
        if (DT != BG_F32 && P.round_scores) d = round_through(d, DT);
        const int lim = P.causal ? min(kend, kq0 + i) : kend;
        s[i][u] = row < lim ? d * P.sl2 : -INFINITY;
      }
    }
    float p[NQ][U];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      float mn = m[i];
#pragma unroll
      for (int u = 0; u < U; ++u) mn = fmaxf(mn, s[i][u]);
      const float alpha = rel_exp2(m[i], mn);
      m[i] = mn;
      l[i] *= alpha;
#pragma unroll
      for (int e = 0; e < E; ++e) o[i][e] *= alpha;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        p[i][u] = rel_exp2(s[i][u], mn);
        l[i] += p[i][u];
        if (DT != BG_F32) p[i][u] = round_through(p[i][u], DT);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float x[E];
      widen<DT, E>(vr[u], x);
#pragma unroll
      for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) o[i][e] = __builtin_fmaf(p[i][u], x[e], o[i][e]);
    }
  }
  // The lane groups of the wavefront, then the wavefronts.
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    float mw = m[i];
#pragma unroll
    for (int x = L; x < 64; x <<= 1) mw = fmaxf(mw, __shfl_xor(mw, x));
    const float f = rel_exp2(m[i], mw);
    l[i] *= f;
#pragma unroll
    for (int x = L; x < 64; x <<= 1) l[i] += __shfl_xor(l[i], x);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      o[i][e] *= f;
#pragma unroll
      for (int x = L; x < 64; x <<= 1) o[i][e] += __shfl_xor(o[i][e], x);
      if (g == 0) red[w][i][c * E + e] = o[i][e];
    }
    if (lane == 0) {
      red[w][i][64] = mw;
      red[w][i][65] = l[i];
    }
  }
  __syncthreads();
  const int i = threadIdx.x >> 6, d = threadIdx.x & 63;
  if (i >= P.Sq) return;  // Sq <= NQ <= W
  float mm = red[0][i][64];
#pragma unroll
  for (int x = 1; x < W; ++x) mm = fmaxf(mm, red[x][i][64]);
  float ls = 0.f, os = 0.f;
#pragma unroll
  for (int x = 0; x < W; ++x) {
    const float f = rel_exp2(red[x][i][64], mm);
    ls += red[x][i][65] * f;
    os += red[x][i][d] * f;
  }
  if (P.part) {
    float* out = P.part + ((int64_t(bh) * P.slices + slice) * P.Sq + i) * (P.D + 2);
    if (d == 0) {
      out[0] = mm;
      out[1] = ls;
    }
    if (d < P.D) out[2 + d] = os;
    return;
  }
  if (d < P.D)
    store_from_f32(P.o, P.out_dtype, b * P.o_sb + h * P.o_sh + i * P.o_ss + d,
                   DT == BG_F32 && !(ls > 0.f) && ls == ls ? 0.f : os / ls);
}

// One wavefront per (batch, head, query): merges the key slices in order.
template <int DT>
__global__ void __launch_bounds__(64) attention_decode_merge_kernel(DecArgs P) {
  const int bh = blockIdx.x / P.Sq, i = blockIdx.x % P.Sq, d = threadIdx.x;
  const int64_t step = int64_t(P.Sq) * (P.D + 2);
  const float* in = P.part + int64_t(bh) * P.slices * step + i * (P.D + 2);
  float mm = in[0];
  for (int x = 1; x < P.slices; ++x) mm = fmaxf(mm, in[x * step]);
  float ls = 0.f, os = 0.f;
  for (int x = 0; x < P.slices; ++x) {
    const float f = rel_exp2(in[x * step], mm);
    ls += in[x * step + 1] * f;
    if (d < P.D) os += in[x * step + 2 + d] * f;
  }
  if (d < P.D)
    store_from_f32(P.o, P.out_dtype, (bh / P.H) * P.o_sb + (bh % P.H) * P.o_sh + i * P.o_ss + d,
                   DT == BG_F32 && !(ls > 0.f) && ls == ls ? 0.f : os / ls);
}

}  // namespace

namespace bg {

// Key slices of a decode call, 0 where another kernel runs.  Strides are
// resolved; ptrs_aligned: Q, K and V start on 16 bytes.  One or two rows (f32
// four: its tiled kernel is far slower); with four 16-bit rows the vector work
// costs more than the matrix cores' (8 x 12 heads, 1024 keys: 16.2 against
// 13.8 us; 32 x 12, 4096 keys: 104 against 79).  From 64 keys: below, the tiled
// kernels walk one tile.  A workgroup streams about 100 GB/s, so fewer than 64
// heads with 1 MB of K and V each are cut into slices of 64 KB or more; their
// second launch costs about 4 us.
int attention_decode_slices(const bg_attention_desc& d, bool ptrs_aligned) {
  if (d.in_dtype != BG_F32 && d.in_dtype != BG_F16 && d.in_dtype != BG_BF16) return 0;
  const int64_t es = dtype_size(d.in_dtype), e = 16 / es;
  if (!ptrs_aligned || d.sq > (d.in_dtype == BG_F32 ? 4 : 2) || d.sk < 64 ||
      d.sk > (int64_t(1) << 30) || d.d > 64 || d.d % e != 0 ||
      d.batch * d.heads > 0x7fffffff || d.reserved == BG_ATTENTION_TILED)
    return 0;
  for (int64_t s : {d.q_sb, d.q_sh, d.q_ss, d.k_sb, d.k_sh, d.k_ss, d.v_sb, d.v_sh, d.v_ss})
    if (s % e != 0) return 0;
  const int64_t bh = d.batch * d.heads, bytes = 2 * d.sk * d.d * es;
  if (d.causal || bh >= 64 || bytes < (int64_t(1) << 20)) return 1;
  const int64_t n = std::min<int64_t>(256 / bh, bytes / (int64_t(64) << 10)), ks = (d.sk + n - 1) / n;
  return int((d.sk + ks - 1) / ks);
}

// Wavefronts of a workgroup.  Sixteen where a CU has one head, so that all its
// wavefronts read it; more heads than CUs, or short runs of keys, are better off
// with workgroups that end sooner (W of them merge through LDS, whatever the run):
// f16, D64, two rows, 16 / 8 / 4 wavefronts (tiled kernels): 1024 heads, 64 keys
// 17.7 / 10.7 / 6.5 us (11.1), 256 keys 24.0 / 16.5 / 15.1 (22.2), 1024 keys 50.3 /
// 42.8 / 42.5 (63.2); 512 heads, 1024 keys 28.0 / 24.2 / 24.0 (23.9); 96 heads, 192
// keys 6.5 / 6.2 / 6.2 (6.2), 1024 keys 10.8 / 11.2 / 13.4 (14.1).  One row: 1024
// heads, 64 keys 11.3 / 7.2 / 6.1 (11.0).  A float32 wavefront takes half the keys
// a step, so its runs are short up to 128 keys, and fewer than eight serve none
// but three and four rows: one row, D24, 272 heads, 512 keys 7.9 / - / 9.2 us; D64,
// 4096 heads, 128 keys 42.3 / 38.9 / 39.1; four rows, 272 heads, 64 keys 9.5 / 6.2
// / 6.2 (14.7), 1024 heads, 1024 keys 102 / 94 / 95 (292).
int attention_decode_waves(const bg_attention_desc& d) {
  const bool many = d.batch * d.heads > 256;
  if (d.in_dtype == BG_F32) return (many && d.sq > 2) || d.sk <= 128 ? 8 : 16;
  return many ? 4 : d.sk <= 512 ? 8 : 16;
}

bool launch_attention_decode(bg_ctx* ctx, const bg_attention_desc& d, const char* q, const char* k, const char* v,
                             void* o) {
  auto al16 = [](const char* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  int slices = attention_decode_slices(d, al16(q) && al16(k) && al16(v));
  if (slices == 0) return false;
  if (slices > 1 && stream_capturing(ctx)) slices = 1;
  DecArgs A{};
  A.q = q;
  A.k = k;
  A.v = v;
  A.o = o;
  A.q_sb = d.q_sb; A.q_sh = d.q_sh; A.q_ss = d.q_ss;
  A.k_sb = d.k_sb; A.k_sh = d.k_sh; A.k_ss = d.k_ss;
  A.v_sb = d.v_sb; A.v_sh = d.v_sh; A.v_ss = d.v_ss;
  A.o_sb = d.o_sb; A.o_sh = d.o_sh; A.o_ss = d.o_ss;
  A.H = int(d.heads);
  A.Sq = int(d.sq);
  A.Sk = int(d.sk);
  A.D = int(d.d);
  A.sl2 = d.scale * 1.4426950408889634f;
  A.causal = d.causal ? 1 : 0;
  A.round_scores = d.round_scores ? 1 : 0;
  A.out_dtype = d.out_dtype;
  const int64_t bh = d.batch * d.heads;
  A.slices = slices;
  A.ks = int((d.sk + slices - 1) / slices);
  if (A.slices > 1) A.part = static_cast<float*>(scratch(ctx, size_t(bh * A.slices * d.sq * (d.d + 2)) * 4, 3));
  const dim3 grid(unsigned(bh), unsigned(A.slices));
  auto by_q = [&](auto dt, auto waves) {
    constexpr int DT = decltype(dt)::value, W = decltype(waves)::value;
    if constexpr (DT != BG_F32 || W > 4) {
      if (d.sq == 1) dispatch(ctx, attention_decode_kernel<DT, 1, W>, grid, dim3(W * 64), 0, A);
      else if (d.sq == 2) dispatch(ctx, attention_decode_kernel<DT, 2, W>, grid, dim3(W * 64), 0, A);
      else if constexpr (DT == BG_F32) dispatch(ctx, attention_decode_kernel<DT, 4, W>, grid, dim3(W * 64), 0, A);
    }
    if (A.part) dispatch(ctx, attention_decode_merge_kernel<DT>, dim3(unsigned(bh * d.sq)), dim3(64), 0, A);
  };
  auto by_waves = [&](auto dt) {
    switch (attention_decode_waves(d)) {
      case 4: by_q(dt, std::integral_constant<int, 4>{}); break;
      case 8: by_q(dt, std::integral_constant<int, 8>{}); break;
      default: by_q(dt, std::integral_constant<int, 16>{});
    }
  };
  if (d.in_dtype == BG_F32) by_waves(std::integral_constant<int, BG_F32>{});
  else if (d.in_dtype == BG_F16) by_waves(std::integral_constant<int, BG_F16>{});
  else by_waves(std::integral_constant<int, BG_BF16>{});
  return true;
}

}  // namespace bg
