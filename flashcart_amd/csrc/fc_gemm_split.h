// GEMM of float32 operands on the bf16 matrix cores (included by fc_linear.hip).
//
// Every operand is split into three bf16 numbers, x = h + m + l, each the nearest bf16 of what the
// ones before it leave: 3 x 8 significant bits hold the 24 of a float32, so the split is exact. Of
// the nine products of two split operands the six of relative size 1, 2^-8 and 2^-16 are formed
// (hh; hm, mh; hl, lh, mm) with float32 accumulation, hh in one accumulator and the small ones in
// another, added at the end. What is left out is below 2^-24 of a product. Measured against
// float64 with normal operands, relative 2-norm error at K = 128 / 896 / 8,192: 0.66 / 1.7 / 5.7e-7,
// against 2.0 / 5.4 / 17e-7 for v_mfma_f32_16x16x4f32, whose chain rounds after every product.
// Range: the parts of an operand are multiples of its last bit, at least 2^-149, but bf16's smallest
// subnormal is 2^-133; operands are therefore scaled by 2^20 as they are split (and results by 2^-40),
// which keeps all bits of every float32, subnormal ones included: the matrix instructions take subnormal
// parts as they are (relative error 5e-8 at K = 64 from operands of 2^-110 down to 2^-132, less below,
// where operands have fewer bits). Results that come out infinite or NaN (an infinite or NaN operand, an
// operand above 2^107, a sum above 2^88) are formed again on the float32 matrix cores, so those follow
// the IEEE rules as before.
//
// Rate: six bf16 MFMAs take 3/8 of the time of the float32 MFMAs they replace, plus 6.5 VALU
// instructions for each operand element that is split.
#pragma once

namespace fc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr float kSplitScale = 0x1p20f, kSplitUnscale = 0x1p-40f;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Split8 {
  bf16x8 h, m, l;
};

// Two float32 to bf16, round to nearest even, a in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  uint32_t u;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(u) : "v"(a), "v"(b));
  return u;
}

// Eight float32 values as three bf16 vectors (scaled by kSplitScale). Pairs share a conversion, and
// the rounded values come back as float32 by a shift and a mask: 13 instructions for two values.
__device__ __forceinline__ Split8 split8(const f32x4& p, const f32x4& q) {
  u32x4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = (i < 2 ? p[2 * i] : q[2 * i - 4]) * kSplitScale;
    const float b = (i < 2 ? p[2 * i + 1] : q[2 * i - 3]) * kSplitScale;
    h[i] = pack_bf16(a, b);
    const float ra = a - __uint_as_float(h[i] << 16), rb = b - __uint_as_float(h[i] & 0xffff0000u);
    m[i] = pack_bf16(ra, rb);
    l[i] = pack_bf16(ra - __uint_as_float(m[i] << 16), rb - __uint_as_float(m[i] & 0xffff0000u));
  }
  Split8 s;
  s.h = __builtin_bit_cast(bf16x8, h);
  s.m = __builtin_bit_cast(bf16x8, m);
  s.l = __builtin_bit_cast(bf16x8, l);
  return s;
}

__device__ __forceinline__ floatx16 mfma_bf16(const bf16x8& a, const bf16x8& b, const floatx16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Tiles of 128 x BN outputs, one per workgroup of four waves; each wave holds 32 rows x BN
// columns in 32x32x16 blocks. K advances by 32: lane (r, h) = (lane % 32, lane / 32) of a wave takes
// k = 16 h .. 16 h + 15 of A row r straight from global memory (64 contiguous bytes; no other wave
// needs that row) and splits them in registers; the weights' 32 x BN step is split once per
// workgroup into LDS, double buffered, in the order the MFMAs read it: block (column block j, half
// s) of 64 16-byte entries per part, entry (column % 32 ^ 4 (2 h + s)) + 32 h holding k = 16 h + 8 s
// .. + 7 (the XOR spreads the four 8-k groups of a column over the banks as they are written).
// Loads run one K step ahead. Two workgroups per CU: the splits of one run under the MFMAs of the
// other.
constexpr int kSplitWaves = 4, kSplitBM = 32 * kSplitWaves;

template <int BN, bool KB>
__global__ void __launch_bounds__(64 * kSplitWaves, 2) gemm_split_kernel(GemmBatch gb) {
  constexpr int NT = 64 * kSplitWaves, BM = kSplitBM, FN = BN / 32;
  constexpr int ITEMS = 4 * BN / NT;  // (column, 8 k) groups each thread splits per step
  constexpr int PART = FN * 2 * 64;   // entries per part
  static_assert(ITEMS >= 1 && 4 * BN % NT == 0 && FN % 2 == 0, "tile shape");
  __shared__ bf16x8 Bs[2][3 * PART];

  // Rank, row and column tile: the column tiles of a row tile go to one XCD (block b runs on XCD
  // b % 8; every rank's row tiles are padded to a multiple of 8), whose L2 then serves the A rows.
  const int b = blockIdx.x;
  int ri = 0;
#pragma unroll
  for (int q = 1; q < FC_MAX_RANKS; ++q)
    if (q < gb.n_ranks && b >= gb.r[q].tile_base) ri = q;
  ri = __builtin_amdgcn_readfirstlane(ri);
  const GemmRank& g = gb.r[ri];
  const int local = b - g.tile_base, i8 = local >> 3;
  const int mt = g.tiles_n == 1 ? local : (i8 / g.tiles_n) * 8 + (local & 7);
  const int nt = g.tiles_n == 1 ? 0 : i8 % g.tiles_n;
  if (mt >= g.tiles_m) return;
  const int r0 = mt * BM, c0 = nt * BN;
  const int K = g.K, N = g.N, M = g.M, comps = g.comps;

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, rl = lane & 31, h = lane >> 5;
  const float* a_ptr;
  {
    const int row = min(r0 + 32 * wave + rl, M - 1);
    const int n = row / comps, c = row - n * comps;
    a_ptr = g.A + (int64_t)n * g.a_row + (int64_t)c * g.a_comp + 16 * h;
  }
  const float* b_ptr[ITEMS];
  int b_dst[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int it = t + i * NT;
    const int o = KB ? it / BN : it & 3, col = KB ? it % BN : it >> 2;
    const int gcol = min(c0 + col, N - 1);
    b_ptr[i] = KB ? g.B + (int64_t)(8 * o) * N + gcol : g.B + (int64_t)gcol * K + 8 * o;
    b_dst[i] = ((col >> 5) * 2 + (o & 1)) * 64 + ((col & 31) ^ (4 * o)) + 32 * (o >> 1);
  }

  f32x4 ar[4], br[ITEMS][2];
  auto load_a = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ar[i] = *reinterpret_cast<const f32x4*>(a_ptr + k0 + 4 * i);
  };
  auto load_b = [&](int k0) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if constexpr (KB) {
        const float* p = b_ptr[i] + (int64_t)k0 * N;
#pragma unroll
        for (int q = 0; q < 8; ++q) br[i][q >> 2][q & 3] = p[q * (int64_t)N];
      } else {
        br[i][0] = *reinterpret_cast<const f32x4*>(b_ptr[i] + k0);
        br[i][1] = *reinterpret_cast<const f32x4*>(b_ptr[i] + k0 + 4);
      }
    }
  };
  auto store_b = [&](int buf) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const Split8 s = split8(br[i][0], br[i][1]);
      Bs[buf][b_dst[i]] = s.h;
      Bs[buf][PART + b_dst[i]] = s.m;
      Bs[buf][2 * PART + b_dst[i]] = s.l;
    }
  };

  floatx16 hi[FN], lo[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) hi[j][v] = lo[j][v] = 0.f;

  // Groups of six MFMAs on one 32 x 32 block; the next group's operands are read from LDS while a
  // group multiplies (the scheduling barrier keeps the reads there).
  auto compute = [&](int buf, const Split8 (&a)[2]) {
    auto fetch = [&](int q) {
      const int s = q / FN, j = q % FN;
      const bf16x8* p = Bs[buf] + j * 128 + s * 64 + (rl ^ (4 * (2 * h + s))) + 32 * h;
      Split8 f;
      f.h = p[0];
      f.m = p[PART];
      f.l = p[2 * PART];
      return f;
    };
    Split8 nxt = fetch(0);
#pragma unroll
    for (int q = 0; q < 2 * FN; ++q) {
      const int s = q / FN, j = q % FN;
      const Split8 c = nxt;
      if (q + 1 < 2 * FN) nxt = fetch(q + 1);
      __builtin_amdgcn_sched_barrier(0);
      lo[j] = mfma_bf16(a[s].l, c.h, lo[j]);
      hi[j] = mfma_bf16(a[s].h, c.h, hi[j]);
      lo[j] = mfma_bf16(a[s].h, c.l, lo[j]);
      lo[j] = mfma_bf16(a[s].m, c.m, lo[j]);
      lo[j] = mfma_bf16(a[s].m, c.h, lo[j]);
      lo[j] = mfma_bf16(a[s].h, c.m, lo[j]);
    }
  };
  // This step's A rows, split; the empty asm keeps the compiler from starting on them (and so
  // waiting for them) in the step before.
  auto take_a = [&](Split8 (&a)[2]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(ar[i]));
    a[0] = split8(ar[0], ar[1]);
    a[1] = split8(ar[2], ar[3]);
  };

  // One K step per turn: one barrier, after which the other buffer (written before it, last read
  // the turn before) is the current one. Loads are issued on every path of the loop (the last turn
  // loads weights that it has already), so that waits count them exactly.
  load_b(0);
  load_a(0);
  store_b(0);
  load_b(K > 32 ? 32 : 0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K - 32; k0 += 32) {
    Split8 a[2];
    take_a(a);
    __builtin_amdgcn_sched_barrier(0);  // the loads below go to the registers that the split has freed
    load_a(k0 + 32);
    __builtin_amdgcn_sched_barrier(0);
    compute(buf, a);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q) asm volatile("" : "+v"(br[i][q]));
    store_b(buf ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    load_b(min(k0 + 64, K - 32));
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    buf ^= 1;
  }
  {
    Split8 a[2];
    take_a(a);
    compute(buf, a);
  }

  // Epilogue: block rows 8 (v / 4) + 4 h + v % 4, column lane % 32.
  float probe = 0.f;  // NaN if any sum is infinite or NaN
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      hi[j][v] = (hi[j][v] + lo[j][v]) * kSplitUnscale;
      probe = fmaf(hi[j][v], 0.f, probe);
    }
  const int col0 = c0 + rl;
  const int row0 = r0 + 32 * wave + 4 * h;
  if (__any(probe != probe)) {
    // again in plain float32: lane half h takes k = 4 h .. 4 h + 3 of every 8
    const float* ap = a_ptr - 12 * h;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) hi[j][v] = 0.f;
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 8) {
      const f32x4 av = *reinterpret_cast<const f32x4*>(ap + k0);
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = min(col0 + 32 * j, N - 1), k = k0 + 4 * h;
        f32x4 bv;
#pragma unroll
        for (int q = 0; q < 4; ++q) bv[q] = KB ? g.B[(int64_t)(k + q) * N + col] : g.B[(int64_t)col * K + k + q];
#pragma unroll
        for (int q = 0; q < 4; ++q) hi[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[q], bv[q], hi[j], 0, 0, 0);
      }
    }
  }
  const float scale = g.scale;
  const bool all_cols = c0 + BN <= N;  // uniform
  float bias_v[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) bias_v[j] = (gb.bias && col0 + j * 32 < N) ? gb.bias[col0 + j * 32] : 0.f;
  // Rows are addressed from the tile's first node (a uniform base) with 32-bit byte offsets (split_ok
  // bounds them); every residual value is loaded before the first store.
  const int n0 = r0 / comps, cc0 = r0 - n0 * comps;
  const float inv_comps = 1.0f / (float)comps;
  gfloat* const Dt = uniform_gptr(g.D + (int64_t)n0 * g.d_row);
  const bool has_r = g.R != nullptr;
  const gfloat* const Rt = uniform_gptr(has_r ? g.R + (int64_t)n0 * g.d_row : g.D);
  uint32_t off[16];
#pragma unroll
  for (int vg = 0; vg < 4; ++vg) {
    // node and component of the row, counted from node n0: y / comps for y < BM + comps (exact in
    // float: (y + 1/2) / comps is at least 1 / (2 comps) from an integer)
    const int y = cc0 + 32 * wave + 4 * h + 8 * vg;
    int dn = (int)(((float)y + 0.5f) * inv_comps), c = y - dn * comps;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      off[4 * vg + q] = 4u * (uint32_t)(dn * (int)g.d_row + c * (int)g.d_comp + col0);
      if (++c == comps) {
        c = 0;
        ++dn;
      }
    }
  }
  auto row_ok = [&](int v) { return row0 + 8 * (v >> 2) + (v & 3) < M; };
  auto at = [&](gfloat* base, uint32_t o, int j) {
    return reinterpret_cast<gfloat*>(reinterpret_cast<gchar*>(base) + o) + j * 32;
  };
#pragma unroll
  for (int v = 0; v < 16; ++v)
#pragma unroll
    for (int j = 0; j < FN; ++j) hi[j][v] = fmaf(hi[j][v], scale, bias_v[j]);
  if (has_r) {
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        lo[j][v] = (row_ok(v) && (all_cols || col0 + j * 32 < N)) ? *at(const_cast<gfloat*>(Rt), off[v], j) : 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
      for (int j = 0; j < FN; ++j) hi[j][v] += lo[j][v];
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    if (!row_ok(v)) continue;
#pragma unroll
    for (int j = 0; j < FN; ++j)
      if (all_cols || col0 + j * 32 < N) __builtin_nontemporal_store(hi[j][v], at(Dt, off[v], j));
  }
}

template <int BN>
int launch_split_cfg(GemmBatch gb, int n_ranks, hipStream_t s) {
  int64_t total = 0;
  for (int l = 0; l < n_ranks; ++l) {
    GemmRank& g = gb.r[l];
    g.tiles_m = (g.M + kSplitBM - 1) / kSplitBM;
    g.tiles_n = (g.N + BN - 1) / BN;
    g.tile_base = (int32_t)total;
    total += (int64_t)((g.tiles_m + 7) / 8 * 8) * g.tiles_n;
  }
  if (total == 0) return FC_OK;
  if (total > 0x7fffffff) return FC_ERR_SHAPE;
  gb.n_ranks = n_ranks;
  gb.total_tiles = (int32_t)total;
  const dim3 grid((unsigned)total), block(64 * kSplitWaves);
  if (gb.trans_b) hipLaunchKernelGGL((gemm_split_kernel<BN, false>), grid, block, 0, s, gb);
  else hipLaunchKernelGGL((gemm_split_kernel<BN, true>), grid, block, 0, s, gb);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

}  // namespace fc
