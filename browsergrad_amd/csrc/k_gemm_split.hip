// float32 GEMM on the bf16 matrix core (split.cuh): six bf16 MFMAs stand for a
// float32 product, at a sixteenth of the float32 MFMA's time each.
#include <algorithm>
#include <cstdio>

#include "gemm_common.cuh"
#include "split.cuh"

namespace {

constexpr uint32_t kOob = 0x80000000u;  // >= num_records: load returns 0
constexpr int kStages = 3;

// One workgroup: WGM x WGN wavefronts, a BM x BN tile of C, a ring of three
// stages of 16 k in LDS.  A stage is three bf16 planes of A (BM rows) and of B
// (BN columns), each in 1 KB blocks of 32 rows whose 16-byte unit
// 32 c + (r ^ 8 c) keeps k = 8 c .. 8 c + 7 of row r: a fragment read is 64
// consecutive units and meets no bank conflict.  The values pass through
// registers, where they are split once per workgroup (7 vector instructions a
// value, beside the MFMAs).  DUAL: the five small products of a pair go to
// accumulators of their own, so that only the sum of the first ones rounds at
// the size of the result (one rounding per 16 k instead of six).
//
// Bound: the matrix core, and with 256 x 256 tiles its power: 4096 x 4096 x
// 4096 takes 621 us (1309 by gemm32_kernel) with the MFMAs busy 70% of the
// cycles at a clock that has fallen to 1.85 GHz.  16x16x32 MFMAs keep 2.2 GHz
// but ran 590-640 us: their stages of 32 k leave LDS for two only, and two
// barriers a stage.  Error against float64 at that size, 2-norm: 1.0e-6
// (gemm32_kernel 1.15e-6); DUAL 3.9e-7.
template <int BM, int BN, int WGM, int WGN, bool DUAL, bool TRANS_B, bool ALIGNED>
__global__ void __launch_bounds__(64 * WGM * WGN, 2) gemm32_split_kernel(GemmArgs P, uint32_t a_bytes,
                                                                         uint32_t b_bytes, int ks, float* part) {
  constexpr int NT = 64 * WGM * WGN;
  constexpr int WTM = BM / WGM, WTN = BN / WGN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int UA = 2 * BM, UB = 2 * BN;  // 16-byte units per plane
  constexpr int NA = (UA + NT - 1) / NT, NB = (UB + NT - 1) / NT;
  constexpr int STAGE = 3 * (UA + UB);
  static_assert(TM >= 2, "a step splits A beside its first row group and B beside its second");
  __shared__ u32x4 smem[kStages * STAGE];

  int tm_, tn_;
  tile_coords(blockIdx.x, P.tiles_m, P.tiles_n, tm_, tn_);
  const int64_t m0 = int64_t(tm_) * BM, n0 = int64_t(tn_) * BN;
  const int64_t batch = blockIdx.z;
  const float* A = static_cast<const float*>(P.A) + batch * P.sa;
  const float* B = static_cast<const float*>(P.B) + batch * P.sb;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)A, (short)0, int(a_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)B, (short)0, int(b_bytes), 0x00020000);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int kbeg = int(blockIdx.y) * ks;
  const int kend = min(int(P.K), kbeg + ks);
  const int nk = (kend - kbeg + 15) / 16;

  // Staging units: (row, 8-deep k chunk).  Row-major operands: neighbouring
  // lanes take the two chunks of a row (64 consecutive bytes); B as [K][N]:
  // lanes run along n, one chunk for the whole wavefront.
  uint32_t va[NA], vb[NB];
  int wa[NA], wb[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int u = i * NT + tid, r = u >> 1, c = u & 1;
    va[i] = u < UA && m0 + r < P.M ? uint32_t(((m0 + r) * P.lda + c * 8) * 4) : kOob;
    wa[i] = (r >> 5) * 64 + c * 32 + ((r & 31) ^ (c * 8));
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int u = i * NT + tid;
    const int r = TRANS_B ? u >> 1 : u % BN, c = TRANS_B ? u & 1 : u / BN;
    vb[i] = u < UB && n0 + r < P.N ? uint32_t((TRANS_B ? (n0 + r) * P.ldb + c * 8 : n0 + r) * 4) : kOob;
    wb[i] = (r >> 5) * 64 + c * 32 + ((r & 31) ^ (c * 8));
  }

  float xa[NA][8], xb[NB][8];
  // Eight k of one row; lim: how many k of the stage lie before kend.
  auto load_row = [&](__amdgpu_buffer_rsrc_t rs, uint32_t off, int k0, int lim, float (&x)[8]) {
    if constexpr (ALIGNED) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 * h, uint32_t(k0) * 4, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) x[4 * h + j] = __uint_as_float(v[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        x[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off + 4 * j, uint32_t(k0) * 4, 0));
    }
    if (lim < 16) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = j + 8 * (tid & 1) < lim ? x[j] : 0.f;
    }
  };
  auto load_stage = [&](int t) {
    const int k0 = kbeg + t * 16;
    const int lim = kend - k0;
#pragma unroll
    for (int i = 0; i < NA; ++i) load_row(ra, va[i], k0, lim, xa[i]);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if constexpr (TRANS_B) {
        load_row(rb, vb[i], k0, lim, xb[i]);
      } else {
        const int c = (i * NT + wave * 64) / BN;
        const uint32_t row = uint32_t(P.ldb) * 4, base = uint32_t(k0 + c * 8) * row;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          xb[i][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              rb, c * 8 + j < lim ? vb[i] : kOob, c * 8 + j < lim ? base + j * row : 0u, 0));
      }
    }
  };
  auto put = [&](u32x4* st, int plane, const float (&x)[8]) {
    u32x4 p1, p2, p3;
    split8(x, kSplitScale, p1, p2, p3);
    st[0] = p1;
    st[plane] = p2;
    st[2 * plane] = p3;
  };
  auto put_a = [&](int slot) {
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (UA % NT == 0 || i * NT + wave * 64 < UA) put(smem + slot * STAGE + wa[i], UA, xa[i]);
  };
  auto put_b = [&](int slot) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (UB % NT == 0 || i * NT + wave * 64 < UB) put(smem + slot * STAGE + 3 * UA + wb[i], UB, xb[i]);
  };

  const int lu = lane ^ ((lane >> 5) << 3);
  bf16x8 fa[2][3], fb[3][TN];
  auto read_a = [&](int slot, int i, bf16x8 (&f)[3]) {
    const u32x4* as = smem + slot * STAGE + wm * TM * 64 + lu;
#pragma unroll
    for (int q = 0; q < 3; ++q) f[q] = __builtin_bit_cast(bf16x8, as[q * UA + i * 64]);
  };
  auto read_b = [&](int slot, int q) {
    const u32x4* bs = smem + slot * STAGE + 3 * UA + wn * TN * 64 + lu;
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[q][j] = __builtin_bit_cast(bf16x8, bs[q * UB + j * 64]);
  };
  constexpr int TS = DUAL ? TN : 1;
  float16v acc[TM][TN], small[TM][TS];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[i][j][e] = 0.f;
        small[i][j % TS][e] = 0.f;
      }
  auto mul = [&](int i, int qa, int qb) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      float16v& c = DUAL && qa + qb > 0 ? small[i][j % TS] : acc[i][j];
      c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i & 1][qa], fb[qb][j], c, 0, 0, 0);
    }
  };

  load_stage(0);
  put_a(0);
  put_b(0);
  if (nk > 1) {
    load_stage(1);
    put_a(1);
    put_b(1);
    if (nk > 2) load_stage(2);
  }
  __syncthreads();
  read_a(0, 0, fa[0]);
#pragma unroll
  for (int q = 0; q < 3; ++q) read_b(0, q);
  // Step t multiplies stage t; the fragments of its first row group are in
  // registers.  Its one barrier comes after that group's MFMAs are issued: by
  // then every wavefront has done with the slot of stage t - 1, which takes
  // stage t + 2, and stage t + 1, written a step ago, may be read: the last
  // row group reads the next step's first fragments between its MFMAs.
  int slot = 0;
  for (int t = 0; t < nk; ++t) {
    const bool more = t + 2 < nk;
    const int nslot = slot == 2 ? 0 : slot + 1, wslot = slot == 0 ? 2 : slot - 1;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const bool last = i + 1 == TM;
      if (!last) read_a(slot, i + 1, fa[(i + 1) & 1]);
      else read_a(nslot, 0, fa[(i + 1) & 1]);
      mul(i, 2, 0);
      mul(i, 0, 2);
      if (last) read_b(nslot, 2);
      mul(i, 1, 1);
      mul(i, 0, 1);
      if (last) read_b(nslot, 1);
      mul(i, 1, 0);
      mul(i, 0, 0);
      if (last) read_b(nslot, 0);
      if (i == 0) {
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront's own LDS writes too
        __builtin_amdgcn_s_barrier();
        if (more) put_a(wslot);
      }
      if (i == 1) {
        if (more) put_b(wslot);
        if (t + 3 < nk) load_stage(t + 3);
      }
    }
    slot = nslot;
  }

  // Redo the tile in float32 where a sum is not finite.
  if constexpr (DUAL) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += small[i][j];
  }
  bool redo = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        redo |= !(fabsf(acc[i][j][e]) <= 3.402823466e38f);
        acc[i][j][e] *= kSplitUnscale;
      }
  if (__syncthreads_or(redo)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    // The same stages, as float32 in k-major rows of two LDS buffers.
    constexpr int LA = BM + 4, LB = BN + 4;
    load_stage(0);
    for (int t = 0; t < nk; ++t) {
      float* as = reinterpret_cast<float*>(smem) + (t & 1) * 16 * (LA + LB);
      float* bs = as + 16 * LA;
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const int u = i * NT + tid;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (UA % NT == 0 || i * NT + wave * 64 < UA) as[(8 * (u & 1) + j) * LA + (u >> 1)] = xa[i][j];
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int u = i * NT + tid;
        const int r = TRANS_B ? u >> 1 : u % BN, c = TRANS_B ? u & 1 : u / BN;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (UB % NT == 0 || i * NT + wave * 64 < UB) bs[(8 * c + j) * LB + r] = xb[i][j];
      }
      __syncthreads();
      if (t + 1 < nk) load_stage(t + 1);
      mul_stage_f32<LA, LB>(as + wm * WTM, bs + wn * WTN, acc);
    }
  }

  if (part) {  // one K slice: its float32 sums, finished by a second kernel
    GemmArgs Q{};
    Q.M = P.M;
    Q.N = P.N;
    Q.ldc = P.N;
    Q.out_dtype = BG_F32;
    const float bz[TN] = {};
    epilogue_tiles<TM, TN, false, BG_F32>(Q, reinterpret_cast<char*>(part + int64_t(blockIdx.y) * P.M * P.N), acc,
                                          m0 + wm * WTM, n0 + wn * WTN, bz);
    return;
  }
  char* C = static_cast<char*>(P.C) + batch * P.sc * (P.out_dtype == BG_F32 ? 4 : 2);
  direct_epilogue<TM, TN, false>(P, C, acc, m0 + wm * WTM, n0 + wn * WTN);
}

}  // namespace

namespace bg {

namespace {

// The tile shapes, and what one 16-deep step of a workgroup takes on MI355X
// (us; 4096 x 4096 x 4096 and 512 x 4096 x 4096 by 1 to 16 slices): with one
// workgroup on a CU, and with as many as fit beside each other (LDS).
struct Tile {
  int bm, bn, wgm, wgn, dual, per_cu;
  double one, full;
};
constexpr Tile kTiles[] = {
    {256, 256, 2, 4, 0, 1, 2.4, 2.4},
    {256, 128, 4, 2, 1, 1, 1.3, 1.3},
    {128, 128, 2, 2, 1, 2, 0.9, 1.5},
    {64, 128, 1, 4, 1, 2, 0.7, 1.0},
};
constexpr int64_t kMaxPartials = int64_t(64) << 20;

// Time of `tiles` tiles of m x n values in all and k with `slices` K slices: rounds of workgroups, each about
// three steps longer than its k for the first loads and the epilogue, 3 us of
// launch, and for slices a second launch and the partials' way to memory and
// back.
double model_us(const Tile& t, int64_t tiles, int64_t mn, uint32_t k, uint32_t slices) {
  const uint32_t steps = (k + 16 * slices - 1) / (16 * slices);
  const int64_t wgs = tiles * slices;
  const int64_t slots = 256 * t.per_cu, full = wgs / slots, rest = wgs % slots;
  const double step = full * t.full + (rest == 0 ? 0.0 : rest <= 256 ? t.one : t.full);
  return 3.0 + (steps + 3.0) * step + (slices > 1 ? 4.0 + 2e-6 * slices * mn : 0.0);
}

}  // namespace

// The split kernel against the float32 one: faster wherever it fits (4096 x
// 4096 x 4096 620 against 1300 us; 256 x 4096 x 4096 62 against 138;
// 1000 x 768 x 3072 46 against 382; 5 x 3000 x 700 12 against 16), except
// for small outputs with a short K, which the wide-K kernel does in one short
// launch (3 us and about 1 us per 128 k: 64 x 784 x 128 in 5.5 us), and up to
// 32 rows against a [K][N] B or one of at most 10M values, which the skinny
// kernel streams as fast or faster (1 x 4096 x 4096 22 against 27 us, 6 x
// 3072 x 3072 17.6 against 21; with B as [N][K] 1 x 4096 x 4096 takes 29
// against 23.5).  Operands must span less than 2 GiB (32-bit buffer offsets).
Gemm32Split gemm32_split(const bg_matmul_desc& d, bool wide, bool skinny, size_t room) {
  Gemm32Split g;
  if (d.reserved == BG_MATMUL_F32_UNSPLIT) return g;
  // Products of up to four terms stay float32: with one the dropped parts double
  // the largest error (512 x 512: 1.0 against 1.6 units of 2^-24, 256 x 256 tiles
  // 2.6), and with operands near 1 + 2^-8 the 2-norm is larger up to K = 4 (K = 2:
  // 5.3e-8 against 3.5e-8; K = 4: 5.1 against 4.8; K = 5: 4.2 against 5.2).
  if (d.k <= 4) return g;
  if (skinny && !wide && d.m <= 32 && (!d.trans_b || d.n * d.k <= int64_t(10) << 20)) return g;
  // The wide-K kernel's sizes, first without the model (a few hundred ns of the
  // call).  Up to k = 900: with up to 32 slices the model says at least 9.1 us + k /
  // 730, which is under 3 us + k / 128 only from k = 940 on.  Outputs of fewer than
  // 64 x 128 values stay there at any k, as before the split kernel; K slices
  // would serve long ones better (64 x 64: k = 1200 20.5 us either way, 2000 32.9
  // against 13.2, 65536 1126 against 103; B as [N][K] 14.4 / 12.4 and 537 / 93).
  if (wide && (d.m * d.n < 64 * 128 || d.k < 900)) return g;
  const int64_t as = ((d.m - 1) * d.lda + d.k) * 4;
  const int64_t bs = (d.trans_b ? (d.n - 1) * d.ldb + d.k : (d.k - 1) * d.ldb + d.n) * 4;
  if (as >= (int64_t(1) << 31) || bs >= (int64_t(1) << 31)) return g;
  double best = 0;
  for (int c = 0; c < int(sizeof kTiles / sizeof kTiles[0]); ++c) {
    const Tile& t = kTiles[c];
    const int64_t tiles = (d.m + t.bm - 1) / t.bm * ((d.n + t.bn - 1) / t.bn) * d.batch;
    for (int s : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32}) {
      if (s > 1 && (d.batch > 1 || d.k < 64 * s || s * d.m * d.n * 4 > kMaxPartials ||
                    size_t(s * d.m * d.n) * 4 + 256 > room))
        break;
      const double us = model_us(t, tiles, d.m * d.n, uint32_t(d.k), uint32_t(s));
      if (g.tile >= 0 && us >= best) continue;
      best = us;
      g.tile = c;
      g.slices = s;
    }
  }
  if (wide && best > 3.0 + d.k / 128.0) {
    g.tile = -1;
    return g;
  }
  g.ks = ((d.k + g.slices - 1) / g.slices + 15) / 16 * 16;
  g.slices = int((d.k + g.ks - 1) / g.ks);
  const Tile& t = kTiles[g.tile];
  g.tiles_m = int((d.m + t.bm - 1) / t.bm);
  g.tiles_n = int((d.n + t.bn - 1) / t.bn);
  return g;
}

void launch_gemm32_split(bg_ctx* ctx, const Gemm32Split& g, void* args, const bg_matmul_desc& d, bool aligned,
                         GemmWorkspace& ws) {
  GemmArgs& P = *static_cast<GemmArgs*>(args);
  P.tiles_m = g.tiles_m;
  P.tiles_n = g.tiles_n;
  float* part = g.slices > 1 ? static_cast<float*>(ws.get(size_t(g.slices) * P.M * P.N * 4, 3)) : nullptr;
  const bool tb = d.trans_b != 0;
  const uint32_t ab = uint32_t(((d.m - 1) * d.lda + d.k) * 4);
  const uint32_t bb = uint32_t((tb ? (d.n - 1) * d.ldb + d.k : (d.k - 1) * d.ldb + d.n) * 4);
  const dim3 grid(unsigned(g.tiles_m * g.tiles_n), unsigned(g.slices), unsigned(d.batch));
  auto go = [&](auto kern, int threads) { dispatch(ctx, kern, grid, dim3(threads), 0, P, ab, bb, int(g.ks), part); };
#define BG_SPLIT(BM_, BN_, GM_, GN_, DUAL_)                                                  \
  (tb ? (aligned ? go(gemm32_split_kernel<BM_, BN_, GM_, GN_, DUAL_, true, true>, 64 * GM_ * GN_)    \
                 : go(gemm32_split_kernel<BM_, BN_, GM_, GN_, DUAL_, true, false>, 64 * GM_ * GN_))  \
      : (aligned ? go(gemm32_split_kernel<BM_, BN_, GM_, GN_, DUAL_, false, true>, 64 * GM_ * GN_)   \
                 : go(gemm32_split_kernel<BM_, BN_, GM_, GN_, DUAL_, false, false>, 64 * GM_ * GN_)))
  switch (g.tile) {
    case 0: BG_SPLIT(256, 256, 2, 4, false); break;
    case 1: BG_SPLIT(256, 128, 4, 2, true); break;
    case 2: BG_SPLIT(128, 128, 2, 2, true); break;
    default: BG_SPLIT(64, 128, 1, 4, true); break;
  }
#undef BG_SPLIT
  if (part) finish_gemm_slices(ctx, &P, g.slices, part);
}

void plan_gemm32_split(const Gemm32Split& g, const bg_matmul_desc& d, bool aligned, bg_launch_plan& out) {
  const Tile& t = kTiles[g.tile];
  out.tile_m = t.bm;
  out.tile_n = t.bn;
  out.tile_k = 16;
  out.k_slices = g.slices;
  out.lds_bytes = kStages * 3 * 2 * (t.bm + t.bn) * 16;
  out.workspace_bytes = g.slices > 1 ? g.slices * d.m * d.n * 4 : 0;
  bg_launch_plan_entry& e = out.launch[0];
  std::snprintf(e.family, sizeof e.family, "%s", "gemm32_split_kernel");
  const int targs[] = {t.bm, t.bn, t.wgm, t.wgn, t.dual, d.trans_b ? 1 : 0, aligned ? 1 : 0};
  e.n_targs = 7;
  std::copy(targs, targs + 7, e.targs);
  e.grid[0] = int64_t(g.tiles_m) * g.tiles_n; e.grid[1] = g.slices; e.grid[2] = d.batch;
  e.block[0] = 64 * t.wgm * t.wgn; e.block[1] = 1; e.block[2] = 1;
}

}  // namespace bg
