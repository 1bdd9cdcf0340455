// Equivariant linear maps and dense layers of float32 operands on the matrix cores (MFMA): bf16 ones with split
// operands for most launches, fp32 ones for the others.
//
// Per rank l the equivariant map is a GEMM with M = n*(2l+1) rows (one per node and
// component), K = in_features*in_paths[l], N = out_features, and one weight matrix
// for every component (reference src/flashcart/o3/_linear.py:64-110). Rows are
// addressed as (node, component), so the packed (n, in_dim) feature rows are read in
// place; all ranks run in one launch.
//
// Four kernels. gemm_small_kernel serves launches of little work (small_ok). gemm_split_kernel
// (fc_gemm_split.h) serves every other launch whose ranks have K % 32 == 0 and 16-byte aligned rows and need
// no activation. gemm_pairsum_kernel serves the pair sums: direct global->LDS loads into a three-stage ring,
// persistent workgroups, v_mfma_f32_16x16x4f32 blocks.
// gemm_kernel serves the rest (activation prologue/epilogue of the dense layers, ragged K):
// Tiling (gfx950, wave64): 256-thread workgroups, BM x BN output tiles, waves arranged
// WM x WN, each wave accumulating (BM/WM) x (BN/WN) with v_mfma_f32_32x32x2f32 blocks.
// K advances in steps of 32 through LDS (a single buffer with two barriers per step in
// the tile shapes launched, which leaves room for four workgroups per CU): the next
// step's global loads are in flight while the current step's 16 MFMA k-pairs run.
// Full K steps load through one branch-free path (row pointers clamped
// to valid rows and masked afterwards): per-lane divergence between vector and scalar
// loads made the compiler wait on outstanding loads inside the load sequence.
// A rows (and B rows when the weight is k-contiguous, the forward) sit in LDS in the
// order the MFMA consumes them: k-step s takes k = 2s (lanes 0-31) and k = 2s+1
// (lanes 32-63), so position (k % 2) * 16 + k / 2 puts each half-wave's 16 values of
// the step sequence next to each other and a lane fetches four k-steps with one
// 128-bit LDS read; the row pitch of 36 floats makes those reads conflict-free (row
// stride 9 x 16 B). A column-contiguous weight (the input gradient) is stored k-major
// with 128-bit writes instead and read one k-step at a time.
// Blocks are ordered N-tile fastest and remapped so that consecutive tiles of one row
// block land on the same XCD (the hardware deals workgroups round-robin over the 8
// XCDs), so the A rows are fetched from HBM once and then hit that XCD's L2.
// float32 inputs and float32 accumulation throughout.
#include "fc_common.h"
#include <type_traits>  // std::true_type

namespace fc {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float kSiluScale = 1.6765324703310907f;  // RescaledSiLULayer, src/flashcart/nn/layers.py:23

struct GemmRank {
  const float* A;   // row r = (n, c): A + n*a_row + c*a_comp, K contiguous floats
  const float* B;   // weight
  float* D;         // row r: D + n*d_row + c*d_comp, N contiguous floats
  const float* P;   // dense dgrad: pre-activation (same layout as A), multiplies A by act'(P)
  float* pre;       // dense fwd: pre-activation output (same layout as D)
  const float* R;   // residual added to the result (same layout as D; may be D itself)
  int64_t a_row, a_comp, d_row, d_comp;
  const int32_t* a_lo;  // pair sum (gb.pair_sum) with gathered halves: A row r's halves are rows a_lo[r]
  const int32_t* a_hi;  // and a_hi[r] of A (a_row floats apart); NULL: A row r holds both halves
  int32_t M;        // rows = n * comps
  int32_t comps, K, N;
  float scale;
  int32_t tiles_m, tiles_n, tile_base;  // tile grid of this rank, first linear tile id
};

struct GemmBatch {
  GemmRank r[FC_MAX_RANKS];
  int32_t n_ranks, total_tiles;
  const float* bias;  // dense fwd only
  int32_t trans_b;    // 1: B(k, o) = W[o*K + k] (forward); 0: B(k, o) = W[k*N + o] (input gradient)
  int32_t act;        // 1: rescaled SiLU epilogue (fwd)
  int32_t act_bwd;    // 1: rescaled SiLU derivative prologue on A (dgrad)
  int32_t pair_sum;   // 1: A rows hold two K-long halves, multiplied as their sum (one rank, at most 64 columns)
};

__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + __expf(-x)); }

__device__ __forceinline__ float silu_grad_(float p) {
  const float s = sigmoidf_(p);
  return kSiluScale * s * (1.0f + p * (1.0f - s));
}

constexpr int GEMM_BK = 32;
constexpr int GEMM_PITCH = GEMM_BK + 4;

// LDS position of k (0..31) inside an operand row.
__device__ __forceinline__ constexpr int kpos(int k) { return (k & 1) * 16 + (k >> 1); }

template <int BM, int BN, int WM, int WN, int NBUF, bool KB>
__global__ void __launch_bounds__(256) gemm_kernel(GemmBatch gb) {
  static_assert(WM * WN == 4, "four waves");
  constexpr int BK = GEMM_BK, LP = GEMM_PITCH;
  constexpr int TM = BM / WM, TN = BN / WN;  // per-wave tile
  constexpr int FM = TM / 32, FN = TN / 32;  // 32x32 MFMA blocks per wave
  constexpr int A_LOADS = BM * BK / 1024;    // float4 per thread and K step
  constexpr int B_LOADS = BN * BK / 1024;
  static_assert(A_LOADS >= 1 && B_LOADS >= 1, "tile too small for 256 threads");
  __shared__ __attribute__((aligned(16))) float As[NBUF][BM * LP];
  constexpr int BSZ = KB ? BK * (BN + 4) : BN * LP;
  __shared__ __attribute__((aligned(16))) float Bs[NBUF][BSZ];
  __shared__ int64_t d_off[BM];  // output row offsets of this tile (-1 past the end)

  // XCD-aware remap: hardware block b runs on XCD b % 8; give each XCD a contiguous tile range.
  const int nb = gridDim.x;
  const int b = blockIdx.x;
  int tile = b;
  if (nb >= 8 && nb % 8 == 0) tile = (b % 8) * (nb / 8) + b / 8;
  if (tile >= gb.total_tiles) return;
  int ri = 0;
#pragma unroll
  for (int q = 1; q < FC_MAX_RANKS; ++q)
    if (q < gb.n_ranks && tile >= gb.r[q].tile_base) ri = q;
  const GemmRank& g = gb.r[ri];
  const int local = tile - g.tile_base;
  const int tm = local / g.tiles_n, tn = local % g.tiles_n;
  const int r0 = tm * BM, c0 = tn * BN;

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN;
  for (int m = t; m < BM; m += 256) {
    const int row = r0 + m;
    int64_t off = -1;
    if (row < g.M) {
      const int n = row / g.comps, c = row - n * g.comps;
      off = (int64_t)n * g.d_row + (int64_t)c * g.d_comp;
    }
    d_off[m] = off;
  }

  // ---- global loads: 8 threads per operand row, one float4 (4 consecutive k) each.
  // Row pointers are clamped to valid rows and masked afterwards, so that full K steps
  // take one branch-free path (no per-lane divergence between vector and scalar loads).
  const int lk4 = (t & 7) * 4;  // k offset of this thread inside a K step
  const float* a_ptr[A_LOADS];
  const float* p_ptr[A_LOADS];
  bool a_ok[A_LOADS];
  const bool use_p = gb.act_bwd && g.P;
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i) {
    const int row0 = r0 + (t >> 3) + 32 * i;
    a_ok[i] = row0 < g.M;
    const int row = a_ok[i] ? row0 : g.M - 1;
    const int n = row / g.comps, c = row - n * g.comps;
    a_ptr[i] = g.A + (int64_t)n * g.a_row + (int64_t)c * g.a_comp;
    p_ptr[i] = use_p ? g.P + (int64_t)n * g.a_row + (int64_t)c * g.a_comp : nullptr;
  }
  const bool a_vec = ((g.K & 3) == 0) && ((g.a_row & 3) == 0) && ((g.a_comp & 3) == 0) &&
                     (((uintptr_t)g.A & 15) == 0) && (!use_p || (((uintptr_t)g.P & 15) == 0));
  const bool b_vec = gb.trans_b ? (((g.K & 3) == 0) && (((uintptr_t)g.B & 15) == 0))
                                : (((g.N & 3) == 0) && (((uintptr_t)g.B & 15) == 0));
  // B operand rows: trans_b -> output column c0 + (t>>3) + 32 i (k contiguous);
  // otherwise k row k0 + t/(BN/4) + (1024/BN) i, 4 consecutive columns from bcol.
  const float* b_ptr[B_LOADS];
  bool b_ok[B_LOADS];
  const int bcol = c0 + (t % (BN / 4)) * 4;
#pragma unroll
  for (int i = 0; i < B_LOADS; ++i) {
    if (gb.trans_b) {
      const int col0 = c0 + (t >> 3) + 32 * i;
      b_ok[i] = col0 < g.N;
      b_ptr[i] = g.B + (int64_t)(b_ok[i] ? col0 : g.N - 1) * g.K;
    } else {
      b_ok[i] = bcol + 3 < g.N;
      b_ptr[i] = g.B + (b_ok[i] ? bcol : 0);
    }
  }

  auto slow4 = [&](const float* p, int k, int kmax) -> float4 {
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (k < kmax) v.x = p[k];
    if (k + 1 < kmax) v.y = p[k + 1];
    if (k + 2 < kmax) v.z = p[k + 2];
    if (k + 3 < kmax) v.w = p[k + 3];
    return v;
  };
  const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);

  float4 ra[A_LOADS], rb[B_LOADS];
  auto load_step = [&](int k0) {
    const bool full = k0 + BK <= g.K;  // uniform
    float4 pa[A_LOADS];
    if (full && a_vec) {
#pragma unroll
      for (int i = 0; i < A_LOADS; ++i) ra[i] = *reinterpret_cast<const float4*>(a_ptr[i] + k0 + lk4);
      if (use_p) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) pa[i] = *reinterpret_cast<const float4*>(p_ptr[i] + k0 + lk4);
      }
    } else {
#pragma unroll
      for (int i = 0; i < A_LOADS; ++i) {
        ra[i] = slow4(a_ptr[i], k0 + lk4, g.K);
        if (use_p) pa[i] = slow4(p_ptr[i], k0 + lk4, g.K);
      }
    }
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      if (use_p) {
        const float pp[4] = {pa[i].x, pa[i].y, pa[i].z, pa[i].w};
        float* vv = reinterpret_cast<float*>(&ra[i]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float s = sigmoidf_(pp[j]);
          vv[j] *= kSiluScale * s * (1.0f + pp[j] * (1.0f - s));
        }
      }
      if (!a_ok[i]) ra[i] = zero4;
    }
    if (gb.trans_b) {
      if (full && b_vec) {
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i) rb[i] = *reinterpret_cast<const float4*>(b_ptr[i] + k0 + lk4);
      } else {
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i) rb[i] = slow4(b_ptr[i], k0 + lk4, g.K);
      }
#pragma unroll
      for (int i = 0; i < B_LOADS; ++i)
        if (!b_ok[i]) rb[i] = zero4;
    } else {
#pragma unroll
      for (int i = 0; i < B_LOADS; ++i) {
        const int k = k0 + (t / (BN / 4)) + (1024 / BN) * i;
        if (full && b_vec && b_ok[i]) {
          rb[i] = *reinterpret_cast<const float4*>(b_ptr[i] + (int64_t)k * g.N);
        } else {
          rb[i] = k < g.K ? slow4(g.B + (int64_t)k * g.N, bcol, g.N) : zero4;
        }
      }
    }
  };
  auto store_step = [&](int buf) {
    float* as = As[buf];
    float* bs = Bs[buf];
    const int p0 = kpos(lk4);  // lk4 even: (v.x, v.z) at p0, (v.y, v.w) at p0 + 16
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      float* r = as + ((t >> 3) + 32 * i) * LP;
      *reinterpret_cast<float2*>(r + p0) = make_float2(ra[i].x, ra[i].z);
      *reinterpret_cast<float2*>(r + p0 + 16) = make_float2(ra[i].y, ra[i].w);
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
      if (gb.trans_b) {
        float* r = bs + ((t >> 3) + 32 * i) * LP;
        *reinterpret_cast<float2*>(r + p0) = make_float2(rb[i].x, rb[i].z);
        *reinterpret_cast<float2*>(r + p0 + 16) = make_float2(rb[i].y, rb[i].w);
      } else {
        const int kk = (t / (BN / 4)) + (1024 / BN) * i, col = (t % (BN / 4)) * 4;
        if constexpr (KB) {
          *reinterpret_cast<float4*>(bs + kk * (BN + 4) + col) = rb[i];
        } else {
          const int p = kpos(kk);
          bs[(col + 0) * LP + p] = rb[i].x;
          bs[(col + 1) * LP + p] = rb[i].y;
          bs[(col + 2) * LP + p] = rb[i].z;
          bs[(col + 3) * LP + p] = rb[i].w;
        }
      }
    }
  };

  floatx16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int half = (lane >> 5) * 16;
  const int nk = (g.K + BK - 1) / BK;
  load_step(0);
  store_step(0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = NBUF == 2 ? (kt & 1) : 0;
    if (kt + 1 < nk) load_step((kt + 1) * BK);
    const float* as = As[cur] + (wm * TM + (lane & 31)) * LP + half;
    const float* bs = KB ? Bs[cur] + (lane >> 5) * (BN + 4) + wn * TN + (lane & 31)
                         : Bs[cur] + (wn * TN + (lane & 31)) * LP + half;
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      float4 a4[FM], b4[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) a4[i] = *reinterpret_cast<const float4*>(as + i * 32 * LP + s4 * 4);
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        if constexpr (KB) {  // k-step s = 4 s4 + q reads row 2 s + lane/32
          const float* p = bs + j * 32 + (8 * s4) * (BN + 4);
          b4[j] = make_float4(p[0], p[2 * (BN + 4)], p[4 * (BN + 4)], p[6 * (BN + 4)]);
        } else {
          b4[j] = *reinterpret_cast<const float4*>(bs + j * 32 * LP + s4 * 4);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(reinterpret_cast<const float*>(&a4[i])[q],
                                                             reinterpret_cast<const float*>(&b4[j])[q], acc[i][j],
                                                             0, 0, 0);
    }
    if constexpr (NBUF == 1) __syncthreads();
    if (kt + 1 < nk) store_step(NBUF == 2 ? cur ^ 1 : 0);
    __syncthreads();
  }

  // ---- epilogue: D[row][col] with row = 8*(v/4) + 4*(lane/32) + v%4, col = lane%32 per 32x32 block
  float bias_v[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = c0 + wn * TN + j * 32 + (lane & 31);
    bias_v[j] = (gb.bias && col < g.N) ? gb.bias[col] : 0.f;
  }
  // The residual may alias D (in-place accumulation), so a lane reads its residual values
  // before storing to them; loading them inside the store loop would serialise every load
  // behind the preceding stores.
  if (r0 + BM <= g.M && c0 + BN <= g.N && !g.pre && gb.act == 0) {
    // interior tile with a plain epilogue (scale, bias, residual): no bound checks, and
    // residual reads in groups of 4 rows so the values in flight stay in few registers
    const int cl = c0 + wn * TN + (lane & 31);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
      for (int v4 = 0; v4 < 16; v4 += 4) {  // rows 8 (v4/4) + 4 (lane/32) + q of the 32-row block
        int64_t offs[4];
        float rvi[4][FN];
#pragma unroll
        for (int q = 0; q < 4; ++q) offs[q] = d_off[wm * TM + i * 32 + 8 * (v4 >> 2) + 4 * (lane >> 5) + q];
        if (g.R) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < FN; ++j) rvi[q][j] = g.R[offs[q] + cl + j * 32];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float* drow = g.D + offs[q] + cl;
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            float val = fmaf(acc[i][j][v4 + q], g.scale, bias_v[j]);
            if (g.R) val += rvi[q][j];
            drow[j * 32] = val;
          }
        }
      }
    }
    return;
  }
  float rv[FM][16][FN];
  if (g.R) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t off = d_off[wm * TM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)];
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int col = c0 + wn * TN + j * 32 + (lane & 31);
          rv[i][v][j] = (off >= 0 && col < g.N) ? g.R[off + col] : 0.f;
        }
      }
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t off = d_off[wm * TM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)];
      if (off < 0) continue;
      float* drow = g.D + off;
      float* prow = g.pre ? g.pre + off : nullptr;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = c0 + wn * TN + j * 32 + (lane & 31);
        if (col >= g.N) continue;
        float val = fmaf(acc[i][j][v], g.scale, bias_v[j]);
        if (prow) prow[col] = val;
        if (gb.act == 1) val = kSiluScale * val * sigmoidf_(val);
        if (g.R) val += rv[i][v][j];
        drow[col] = val;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------
// Pair-sum GEMM of at most 64 columns: D = scale (A_lo + A_hi) W^T, where every A row is the sum of two halves of K floats,
// A[r, 0:K] and A[r, K:2K], or rows a_lo[r] and a_hi[r] of A when the rank gives those index arrays;
// both halves go to LDS and are added as the MFMA operands are read, so the MFMA work is that of K
// (the radial output layer's input gradient over edge pairs, whose two edges share the layer's
// output row). Bound by reading A (9.4 GB at 540,083 pairs and K = 2,176: 1.9-2.1 ms; the split
// kernel's loads through registers take 2.24 ms there). Operands travel global -> LDS by direct loads
// (global_load_lds_dwordx4: no register staging, no LDS store phase) into a ring of three stages, so
// every wave has the next two K steps in flight while it multiplies the current one, with one barrier
// per K step. Persistent workgroups (two per CU) walk their tiles as one stream of K steps: the first
// steps of the next tile load during the current tile's epilogue. K % 32 == 0, 16-byte aligned rows.
//
// LDS layout per stage: rows of 8 chunks of 4 floats (one 32-float K step); chunk c of row r sits at
// position c ^ ((r / 2) % 8), so the rows read together at one chunk fall in distinct banks
// (SQ_LDS_BANK_CONFLICT reads 0).
// K-step mapping: 16x16x4 blocks take k = 16 s + 4 (lane / 16) + q in k-quad q of half s, in A and B
// alike, so each lane reads four k values as one 128-bit chunk.

__device__ __forceinline__ int pipe_swz(int r) { return (r >> 1) & 7; }
// One 16-byte direct load per lane into LDS at lds + 16 * lane (lds: byte offset, wave-uniform).
// Issued as inline assembly so that the compiler does not track it: it would otherwise wait for
// every outstanding direct load before any LDS read, which defeats the ring. The kernel orders
// these loads itself (explicit vmcnt waits and barriers below); the 'memory' clobber keeps the
// compiler from moving other memory accesses across them. M0 written by a scalar move needs
// one wait state before the load that reads it.
// M0 is a reserved register to the compiler; no other code of these kernels uses it (no
// indirect register indexing, no compiler-issued direct loads), so clobbering it is safe here.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_dma16(const float* src, uint32_t lds_off) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_off)
               : "memory", "m0");
}

// LDS byte address of a __shared__ array (a compile-time constant for a named array)
__device__ __forceinline__ uint32_t lds_addr(const float* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) float*)(p);
}
#pragma clang diagnostic pop

// barrier after which LDS reads see what other waves (and their completed direct loads) wrote;
// the empty asm stops the compiler from moving LDS accesses across it
__device__ __forceinline__ void pipe_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// s_waitcnt immediate (gfx9 encoding): vector-memory count <= vm, LDS count <= lgkm, no export wait
#define FC_WAITCNT_IMM(vm, lgkm) (((vm) & 0xF) | ((((vm) >> 4) & 3) << 14) | (0x7 << 4) | (((lgkm) & 0xF) << 8))

constexpr int PAIR_T = 64;  // output tile edge

__global__ void __launch_bounds__(256, 2) gemm_pairsum_kernel(GemmBatch gb) {
  constexpr int BM = PAIR_T, BN = PAIR_T, WM = 2, WN = 2, MI = 16;
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int FM = TM / MI, FN = TN / MI;  // MFMA blocks per wave
  constexpr int NV = 4;                      // accumulator values per lane and block
  typedef float accv __attribute__((ext_vector_type(NV)));
  constexpr int A_DMA = BM * 8 / 256;  // 16-byte chunks per thread and K step
  constexpr int B_DMA = BN * 8 / 256;
  constexpr int AH = 2;                // A halves
  constexpr int L = AH * A_DMA + B_DMA;  // direct loads per wave and K step
  __shared__ __attribute__((aligned(16))) float As0[AH * BM * 32];
  __shared__ __attribute__((aligned(16))) float As1[AH * BM * 32];
  __shared__ __attribute__((aligned(16))) float As2[AH * BM * 32];
  __shared__ __attribute__((aligned(16))) float Bs0[BN * 32];
  __shared__ __attribute__((aligned(16))) float Bs1[BN * 32];
  __shared__ __attribute__((aligned(16))) float Bs2[BN * 32];

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int G = gridDim.x, b = blockIdx.x;
  // This workgroup's row tiles: a contiguous range of 1/G of them. Workgroups of one XCD (hardware
  // block b runs on XCD b % 8) take neighbouring ranges, so an XCD's L2 serves one contiguous run of
  // A rows. (Uniform; kept in scalar registers so the tile loop's bookkeeping stays scalar.)
  const int v = (G >= 8 && G % 8 == 0) ? (b % 8) * (G / 8) + b / 8 : b;
  const GemmRank& g = gb.r[0];
  const int t_first = __builtin_amdgcn_readfirstlane((int)(((int64_t)v * gb.total_tiles + G - 1) / G));
  const int t_end = __builtin_amdgcn_readfirstlane((int)(((int64_t)(v + 1) * gb.total_tiles + G - 1) / G));

  // ---- producer: direct loads of K steps in tile order
  int p_tile = t_first, p_k = 0, n_issued = 0;
  const float* a_src[A_DMA];
  const float* a_src2[A_DMA];  // second halves
  const float* b_src[B_DMA];
  auto p_setup = [&]() {
    if (p_tile >= t_end) return;
#pragma unroll
    for (int j = 0; j < A_DMA; ++j) {
      const int s = (j * 4 + wave) * 64 + lane;
      const int row = s >> 3, c = (s & 7) ^ pipe_swz(row);
      const int grow = min(p_tile * BM + row, g.M - 1);
      if (g.a_lo) {
        // Gathered halves. Using these loads waits for every outstanding vector load, the
        // direct loads of the ring included (once per tile).
        a_src[j] = g.A + (int64_t)g.a_lo[grow] * g.a_row + 4 * c;
        a_src2[j] = g.A + (int64_t)g.a_hi[grow] * g.a_row + 4 * c;
        continue;
      }
      a_src[j] = g.A + (int64_t)grow * g.a_row + 4 * c;
      a_src2[j] = a_src[j] + g.K;
    }
#pragma unroll
    for (int j = 0; j < B_DMA; ++j) {
      const int s = (j * 4 + wave) * 64 + lane;
      const int col = s >> 3, c = (s & 7) ^ pipe_swz(col);
      const int gcol = min(col, g.N - 1);
      b_src[j] = g.B + (int64_t)gcol * g.K + 4 * c;
    }
  };
  // LDS byte addresses of the stage being filled (as, bs); this wave's 16-byte chunks of a
  // direct load land at + 1024 (j * 4 + wave), kept in scalar registers
  const uint32_t wave_lds = 1024u * (uint32_t)__builtin_amdgcn_readfirstlane(wave);
  auto p_issue = [&](uint32_t as, uint32_t bs) {
    if (p_tile >= t_end) return;
#pragma unroll
    for (int j = 0; j < A_DMA; ++j) lds_dma16(a_src[j] + p_k, as + 4096u * j + wave_lds);
#pragma unroll
    for (int j = 0; j < A_DMA; ++j) lds_dma16(a_src2[j] + p_k, as + 4u * BM * 32 + 4096u * j + wave_lds);
#pragma unroll
    for (int j = 0; j < B_DMA; ++j) lds_dma16(b_src[j] + p_k, bs + 4096u * j + wave_lds);
    ++n_issued;
    p_k += 32;
    if (p_k >= g.K) {
      p_k = 0;
      ++p_tile;
      p_setup();
    }
  };

  // ---- consumer
  int c_tile = t_first, c_k = 0, n_done = 0;
  accv acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < NV; ++v) acc[i][j][v] = 0.f;

  const int kg = lane >> 4;  // lane group along k
  // FIRST: the tile's first K step, whose first MFMA of each block starts from zero (the
  // accumulators need no clearing between tiles)
  auto compute = [&](const float* as, const float* bs, auto first_c) {
    constexpr bool FIRST = decltype(first_c)::value;
#pragma unroll
    for (int s4 = 0; s4 < 2; ++s4) {
      float4 a4[FM], b4[FN];
      const int ch = 4 * s4 + kg;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int row = wm * TM + i * MI + (lane & (MI - 1));
        a4[i] = *reinterpret_cast<const float4*>(as + row * 32 + 4 * (ch ^ pipe_swz(row)));
        const float4 hi = *reinterpret_cast<const float4*>(as + BM * 32 + row * 32 + 4 * (ch ^ pipe_swz(row)));
        a4[i].x += hi.x; a4[i].y += hi.y; a4[i].z += hi.z; a4[i].w += hi.w;
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = wn * TN + j * MI + (lane & (MI - 1));
        b4[j] = *reinterpret_cast<const float4*>(bs + col * 32 + 4 * (ch ^ pipe_swz(col)));
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const float a = reinterpret_cast<const float*>(&a4[i])[q];
            const float b = reinterpret_cast<const float*>(&b4[j])[q];
            const accv c = (FIRST && s4 == 0 && q == 0) ? accv{} : acc[i][j];
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
          }
    }
  };

  auto epilogue = [&]() {
    const int M = g.M, N = g.N, r0 = c_tile * BM;
    const float scale = g.scale;
    // Rows are addressed from the tile's first row (a uniform base) with 32-bit byte offsets (the
    // caller bounds them), columns j > 0 as immediate offsets.
    gfloat* const Dt = uniform_gptr(g.D + (int64_t)r0 * g.d_row);
    const int col0 = wn * TN + (lane & (MI - 1));  // this lane's column in block j = 0
    const bool all_cols = BN <= N;                          // uniform
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const int row = wm * TM + i * MI + 4 * (lane >> 4) + v;  // block row of value v
        if (r0 + row >= M) continue;
        const uint32_t off = 4u * (uint32_t)(row * (int)g.d_row + col0);
        gfloat* const d = reinterpret_cast<gfloat*>(reinterpret_cast<gchar*>(Dt) + off);
#pragma unroll
        for (int j = 0; j < FN; ++j)
          if (all_cols || col0 + j * MI < N) __builtin_nontemporal_store(acc[i][j][v] * scale, d + j * MI);
      }
  };

  // One K step: wait for this wave's loads of the step (the step issued after it may stay in
  // flight), barrier (every wave's loads have landed and every wave is done with the stage
  // the new loads overwrite), refill that stage, multiply, and finish the tile at its end.
  bool more = c_tile < t_end;
  auto step = [&](const float* as, const float* bs, uint32_t pas, uint32_t pbs) {
    if (n_issued - n_done >= 2) __builtin_amdgcn_s_waitcnt(FC_WAITCNT_IMM(L, 0));
    else __builtin_amdgcn_s_waitcnt(FC_WAITCNT_IMM(0, 0));
    pipe_barrier();
    p_issue(pas, pbs);
    if (c_k == 0) compute(as, bs, std::true_type{});
    else compute(as, bs, std::false_type{});
    ++n_done;
    c_k += 32;
    if (c_k >= g.K) {
      epilogue();
      c_k = 0;
      ++c_tile;
      more = c_tile < t_end;
    }
  };

  p_setup();
  p_issue(lds_addr(As0), lds_addr(Bs0));
  p_issue(lds_addr(As1), lds_addr(Bs1));
  while (more) {
    step(As0, Bs0, lds_addr(As2), lds_addr(Bs2));
    if (!more) break;
    step(As1, Bs1, lds_addr(As0), lds_addr(Bs0));
    if (!more) break;
    step(As2, Bs2, lds_addr(As1), lds_addr(Bs1));
  }
}

// Whether gemm_split_kernel takes the batch.
static bool split_ok(const GemmBatch& gb, int n_ranks) {
  if (gb.act || gb.act_bwd) return false;
  for (int l = 0; l < n_ranks; ++l) {
    const GemmRank& g = gb.r[l];
    if (g.pre || g.P || g.K < 32 || (g.K & 31) || (g.a_row & 3) || (g.a_comp & 3)) return false;
    // 32-bit byte offsets of the epilogue's stores from the tile's first output node (128-row tiles)
    if ((int64_t)129 * g.d_row + (int64_t)g.comps * g.d_comp + g.N >= (int64_t(1) << 30)) return false;
    if (g.d_row > 0x7fffffff || g.d_comp > 0x7fffffff) return false;
    if (((uintptr_t)g.A & 15) || (gb.trans_b && ((uintptr_t)g.B & 15))) return false;
  }
  return true;
}

static int launch_pairsum(GemmBatch gb, hipStream_t s) {
  const GemmRank& g = gb.r[0];
  if (g.K < 32 || (g.K & 31) || (g.a_row & 3) || ((uintptr_t)g.A & 15) || ((uintptr_t)g.B & 15)) return FC_ERR_SHAPE;
  if (g.N > PAIR_T || 64 * g.d_row + g.N >= (int64_t(1) << 29)) return FC_ERR_SHAPE;  // one column tile; byte offsets
  const int64_t total = (g.M + (int64_t)PAIR_T - 1) / PAIR_T;
  if (total == 0) return FC_OK;
  gb.total_tiles = (int32_t)total;
  int64_t grid = 2 * (int64_t)device_cu_count();
  if (grid > total) grid = total;
  if (grid >= 8) grid -= grid % 8;
  hipLaunchKernelGGL(gemm_pairsum_kernel, dim3((unsigned)grid), dim3(256), 0, s, gb);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

// GEMM of few rows (a unit cell, a molecule): the tiles above would leave most of the chip idle and
// walk K serially. Here a workgroup owns a 16 x 16 output block and its four waves each take a quarter of K,
// straight from global memory into v_mfma_f32_16x16x4f32 operands (lane (r, q) = (lane % 16, lane / 16)
// loads k = 16 c + 4 q .. + 3 of A row r and of output column r), U chunks of 16 k in flight at once,
// no LDS until the four partial blocks are added in wave order. Takes every batch whose rows of 4 k are
// aligned, with the dense layers' activation prologue and epilogue; PS as in gemm_pairsum_kernel.
template <bool KB, bool PS, int U>
__global__ void __launch_bounds__(256) gemm_small_kernel(GemmBatch gb) {
  __shared__ float red[4][16][17];
  const int b = blockIdx.x;
  int ri = 0;
#pragma unroll
  for (int q = 1; q < FC_MAX_RANKS; ++q)
    if (q < gb.n_ranks && b >= gb.r[q].tile_base) ri = q;
  ri = __builtin_amdgcn_readfirstlane(ri);
  const GemmRank& g = gb.r[ri];
  const int local = b - g.tile_base;
  const int r0 = (local / g.tiles_n) * 16, c0 = (local % g.tiles_n) * 16;
  const int K = g.K, N = g.N, M = g.M;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, r = lane & 15, kq = 4 * (lane >> 4);
  const int row = min(r0 + r, M - 1), col = min(c0 + r, N - 1);
  const int n = row / g.comps;
  const int64_t a_off = (int64_t)n * g.a_row + (int64_t)(row - n * g.comps) * g.a_comp;
  const float *ap, *ap2 = nullptr;
  const float* const pp = gb.act_bwd && g.P ? g.P + a_off : nullptr;
  if (PS && g.a_lo) {
    ap = g.A + (int64_t)g.a_lo[row] * g.a_row;
    ap2 = g.A + (int64_t)g.a_hi[row] * g.a_row;
  } else {
    ap = g.A + a_off;
    if (PS) ap2 = ap + K;
  }
  const float* const bp = KB ? g.B + col : g.B + (int64_t)col * K;
  // chunks of 16 k: wave w takes the w-th quarter of them
  const int chunks = (K + 15) >> 4, per = (chunks + 3) >> 2;
  const int ch0 = wave * per, ch1 = min(ch0 + per, chunks);
  // one accumulator per chunk in flight, added pairwise at the end: shorter chains of roundings, and the
  // matrix instructions of the chunks do not wait for each other
  f32x4 acc[U];
#pragma unroll
  for (int i = 0; i < U; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int ch = ch0; ch < ch1; ch += U) {
    f32x4 av[U], bv[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      // a group of 4 k past the end reads the row's first (every K takes 4 or more) and counts as zero
      const int k = 16 * (ch + i) + kq;
      const bool ok = ch + i < ch1 && k < K;
      const int ks = ok ? k : 0;
      av[i] = *reinterpret_cast<const f32x4*>(ap + ks);
      if constexpr (PS) av[i] += *reinterpret_cast<const f32x4*>(ap2 + ks);
      if (pp) {
        const f32x4 p = *reinterpret_cast<const f32x4*>(pp + ks);
#pragma unroll
        for (int q = 0; q < 4; ++q) av[i][q] *= silu_grad_(p[q]);
      }
      if constexpr (KB) {
#pragma unroll
        for (int q = 0; q < 4; ++q) bv[i][q] = bp[(int64_t)(ks + q) * N];
      } else {
        bv[i] = *reinterpret_cast<const f32x4*>(bp + ks);
      }
      if (!ok) {
#pragma unroll
        for (int q = 0; q < 4; ++q) av[i][q] = bv[i][q] = 0.f;
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < U; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i][q], bv[i][q], acc[i], 0, 0, 0);
  }
#pragma unroll
  for (int w = 1; w < U; w *= 2)
#pragma unroll
    for (int i = 0; i + w < U; i += 2 * w) acc[i] += acc[i + w];
#pragma unroll
  for (int v = 0; v < 4; ++v) red[wave][4 * (lane >> 4) + v][r] = acc[0][v];
  __syncthreads();
  const int orow = r0 + (t >> 4), ocol = c0 + (t & 15);
  if (orow >= M || ocol >= N) return;
  float x = (red[0][t >> 4][t & 15] + red[1][t >> 4][t & 15]) + (red[2][t >> 4][t & 15] + red[3][t >> 4][t & 15]);
  x = fmaf(x, g.scale, gb.bias ? gb.bias[ocol] : 0.f);
  const int on = orow / g.comps;
  const int64_t off = (int64_t)on * g.d_row + (int64_t)(orow - on * g.comps) * g.d_comp + ocol;
  if (g.pre) g.pre[off] = x;
  if (gb.act) x = kSiluScale * x * sigmoidf_(x);
  if (g.R) x += g.R[off];
  g.D[off] = x;
}

// Chunks of 16 k in flight in a wave of gemm_small_kernel: those that fall to it of the batch's longest K, up to 8.
static int small_unroll(int max_k) {
  const int per = ((max_k + 15) / 16 + 3) / 4;
  return per <= 1 ? 1 : per <= 2 ? 2 : per <= 4 ? 4 : 8;
}

// Whether gemm_small_kernel takes the batch: aligned groups of 4 k, and little enough work that the
// latency of the tiled kernels, which walk all of K in one workgroup, costs more than reading every
// operand 16 rows at a time. Work in 16 x 16 x 16 blocks, each wave's chunks of every rank rounded up to the unroll
// of the longest: the small kernel takes 2.5 us and 1 us for every 3,200, the tiled ones at least 3.4 us and 0.85 us for
// every 32 k. (128-wide maps, l <= 3: 32 nodes 7.1 -> 3.1 us, 256 nodes 7.3 us either way, 512 nodes 7.6 against
// 12.7; K = 512 to 896: 32 nodes 27.3 -> 7.1 us, 256 nodes 32 against 36; K = 320, 192, 64, 128 into 64 columns, where
// rounding doubles to octuples the work: 100 nodes 12.5 -> 8.2 us, 300 nodes 15.4 against 13.2, 900 nodes 38 against 13.)
static bool small_ok(const GemmBatch& gb, int n_ranks) {
  int max_k = 0;
  for (int l = 0; l < n_ranks; ++l) {
    const GemmRank& g = gb.r[l];
    if ((g.K & 3) || (g.a_row & 3) || (g.a_comp & 3) || ((uintptr_t)g.A & 15) || ((uintptr_t)g.P & 15) ||
        (gb.trans_b && ((uintptr_t)g.B & 15)))
      return false;
    if (g.K > max_k) max_k = g.K;
  }
  const int u = small_unroll(max_k);
  int64_t blocks = 0;
  for (int l = 0; l < n_ranks; ++l) {
    const GemmRank& g = gb.r[l];
    const int64_t per = ((g.K + 15) / 16 + 3) / 4;  // chunks of a wave
    blocks += (int64_t)((g.M + 15) / 16) * ((g.N + 15) / 16) * 4 * ((per + u - 1) / u * u);
  }
  return blocks <= 3200 + 85 * (int64_t)max_k;
}

static int launch_small(GemmBatch gb, int n_ranks, hipStream_t s) {
  int64_t total = 0;
  int max_k = 0;
  for (int l = 0; l < n_ranks; ++l) {
    GemmRank& g = gb.r[l];
    g.tiles_m = (g.M + 15) / 16;
    g.tiles_n = (g.N + 15) / 16;
    g.tile_base = (int32_t)total;
    total += (int64_t)g.tiles_m * g.tiles_n;
    if (g.K > max_k) max_k = g.K;
  }
  if (total == 0) return FC_OK;
  gb.n_ranks = n_ranks;
  gb.total_tiles = (int32_t)total;
  const dim3 grid((unsigned)total), block(256);
  auto launch = [&](auto u) {
    constexpr int U = decltype(u)::value;
    if (gb.pair_sum) hipLaunchKernelGGL((gemm_small_kernel<false, true, U>), grid, block, 0, s, gb);
    else if (gb.trans_b) hipLaunchKernelGGL((gemm_small_kernel<false, false, U>), grid, block, 0, s, gb);
    else hipLaunchKernelGGL((gemm_small_kernel<true, false, U>), grid, block, 0, s, gb);
  };
  const int u = small_unroll(max_k);
  if (u == 1) launch(std::integral_constant<int, 1>{});
  else if (u == 2) launch(std::integral_constant<int, 2>{});
  else if (u == 4) launch(std::integral_constant<int, 4>{});
  else launch(std::integral_constant<int, 8>{});
  FC_LAUNCH_CHECK();
  return FC_OK;
}

template <int BM, int BN, int WM, int WN, int NBUF>
int launch_gemm_cfg(GemmBatch gb, int n_ranks, hipStream_t s) {
  int64_t total = 0;
  for (int l = 0; l < n_ranks; ++l) {
    GemmRank& g = gb.r[l];
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    g.tile_base = (int32_t)total;
    total += (int64_t)g.tiles_m * g.tiles_n;
  }
  if (total == 0) return FC_OK;
  if (total > 0x7fffffff) return FC_ERR_SHAPE;
  gb.n_ranks = n_ranks;
  gb.total_tiles = (int32_t)total;
  const int64_t grid = (total + 7) / 8 * 8;  // a multiple of 8 enables the XCD remap
  if (gb.trans_b) hipLaunchKernelGGL((gemm_kernel<BM, BN, WM, WN, NBUF, false>), dim3((unsigned)grid), dim3(256), 0, s, gb);
  else hipLaunchKernelGGL((gemm_kernel<BM, BN, WM, WN, NBUF, true>), dim3((unsigned)grid), dim3(256), 0, s, gb);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

}  // namespace fc
#include "fc_gemm_split.h"
namespace fc {

int launch_gemm(GemmBatch gb, int n_ranks, hipStream_t s) {
  int max_n = 0;
  int64_t max_m = 0;
  for (int l = 0; l < n_ranks; ++l) {
    if (gb.r[l].N > max_n) max_n = gb.r[l].N;
    if (gb.r[l].M > max_m) max_m = gb.r[l].M;
    if (gb.r[l].M < 0) return FC_ERR_SHAPE;
  }
  if (max_m == 0 || max_n == 0 || n_ranks == 0) return FC_OK;
  if (small_ok(gb, n_ranks)) return launch_small(gb, n_ranks, s);
  if (gb.pair_sum) return launch_pairsum(gb, s);
  if (split_ok(gb, n_ranks)) {
    // 128-column tiles where they fill the chip (two workgroups per CU) and the map is wider than 64;
    // 64-column tiles otherwise: twice the workgroups (256 nodes, K of 512 to 896 per rank: 43.6 ->
    // 30.0 us; at 25,000 nodes the wider tiles are the faster ones, 656 -> 606 us)
    int64_t tiles = 0;
    for (int l = 0; l < n_ranks; ++l) tiles += (int64_t)((gb.r[l].M + 127) / 128) * ((gb.r[l].N + 127) / 128);
    if (max_n > 64 && tiles >= 2 * (int64_t)device_cu_count()) return launch_split_cfg<128>(gb, n_ranks, s);
    return launch_split_cfg<64>(gb, n_ranks, s);
  }
  // Activation prologue or epilogue, ragged K or unaligned rows (M = n (2l+1) rows): 128 x 64 tiles
  // (waves stacked along M) for the wider input gradients, 64 x 128 (waves side by side along N) for
  // the forward, 64 x 64 for maps at most 64 wide (twice the workgroups, so short-K launches fill the
  // chip). All hold four workgroups per CU, whose prologues and epilogues overlap each other's MFMA
  // work better than two 128 x 128 tiles.
  if (max_n <= 64) return launch_gemm_cfg<64, 64, 2, 2, 1>(gb, n_ranks, s);
  if (!gb.trans_b) return launch_gemm_cfg<128, 64, 4, 1, 1>(gb, n_ranks, s);
  return launch_gemm_cfg<64, 128, 1, 4, 1>(gb, n_ranks, s);
}

// dst[r, off:off+width] = src ? src[r, off:off+width] : 0 (same row stride): one wave per
// row, lanes along the columns (no per-element division)
__global__ void fill_rows_kernel(int64_t rows, int64_t row_stride, int64_t off, int64_t width,
                                 const float* __restrict__ src, float* __restrict__ dst) {
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int64_t base = r * row_stride + off;
  for (int64_t c = threadIdx.x & 63; c < width; c += 64) dst[base + c] = src ? src[base + c] : 0.f;
}

// Output columns the map does not produce: zero, or the residual's values.
int fill_columns(int64_t rows, int64_t row_stride, int64_t off, int64_t width, const float* residual, float* dst,
                 hipStream_t s) {
  if (rows * width == 0 || residual == dst) return FC_OK;
  hipLaunchKernelGGL(fill_rows_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, rows, row_stride, off, width,
                     residual, dst);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

static int check_linear(const fc_linear_desc* d) {
  if (!d) return FC_ERR_NULL;
  if (d->in_l_max < 0 || d->out_l_max < 0) return FC_ERR_BAD_DESC;
  if (d->in_l_max >= FC_MAX_RANKS || d->out_l_max >= FC_MAX_RANKS) return FC_ERR_UNSUPPORTED_L;
  if (d->in_features < 1 || d->out_features < 1) return FC_ERR_BAD_DESC;
  const int common = d->in_l_max < d->out_l_max ? d->in_l_max : d->out_l_max;
  for (int l = 0; l <= d->in_l_max; ++l)
    if (d->in_paths[l] < 1) return FC_ERR_BAD_DESC;
  for (int l = 0; l <= common; ++l)
    if (!d->weight[l]) return FC_ERR_NULL;
  return FC_OK;
}

struct LinearLayout {
  int64_t in_dim, out_dim, in_off[FC_MAX_RANKS], out_off[FC_MAX_RANKS];
  int common;
};

static LinearLayout linear_layout(const fc_linear_desc* d) {
  LinearLayout L{};
  L.common = d->in_l_max < d->out_l_max ? d->in_l_max : d->out_l_max;
  int64_t o = 0;
  for (int l = 0; l <= d->in_l_max; ++l) {
    L.in_off[l] = o;
    o += (int64_t)(2 * l + 1) * d->in_features * d->in_paths[l];
  }
  L.in_dim = o;
  o = 0;
  for (int l = 0; l <= d->out_l_max; ++l) {
    L.out_off[l] = o;
    o += (int64_t)(2 * l + 1) * d->out_features;
  }
  L.out_dim = o;
  return L;
}

}  // namespace fc

using namespace fc;

extern "C" int fc_linear_fwd(const fc_linear_desc* d, int64_t n, const float* x, float alpha,
                             const float* residual, float* out, void* stream) {
  int st = check_linear(d);
  if (st != FC_OK) return st;
  if (n == 0) return FC_OK;
  if (!x || !out) return FC_ERR_NULL;
  if (n * (2 * FC_MAX_RANKS - 1) > 0x7fffffff) return FC_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  const LinearLayout L = linear_layout(d);
  GemmBatch gb{};
  gb.trans_b = 1;
  for (int l = 0; l <= L.common; ++l) {
    GemmRank& g = gb.r[l];
    const int K = d->in_features * d->in_paths[l];
    g.A = x + L.in_off[l];
    g.a_row = L.in_dim;
    g.a_comp = K;
    g.B = d->weight[l];
    g.D = out + L.out_off[l];
    g.R = residual ? residual + L.out_off[l] : nullptr;
    g.d_row = L.out_dim;
    g.d_comp = d->out_features;
    g.comps = 2 * l + 1;
    g.M = (int32_t)(n * g.comps);
    g.K = K;
    g.N = d->out_features;
    g.scale = alpha * d->scale[l];
  }
  st = launch_gemm(gb, L.common + 1, s);
  if (st != FC_OK) return st;
  if (L.common < d->out_l_max)
    return fill_columns(n, L.out_dim, L.out_off[L.common + 1], L.out_dim - L.out_off[L.common + 1], residual, out,
                        s);
  return FC_OK;
}

extern "C" int fc_linear_dgrad(const fc_linear_desc* d, int64_t n, const float* go, float alpha,
                               const float* residual, float* gx, void* stream) {
  int st = check_linear(d);
  if (st != FC_OK) return st;
  if (n == 0) return FC_OK;
  if (!go || !gx) return FC_ERR_NULL;
  if (n * (2 * FC_MAX_RANKS - 1) > 0x7fffffff) return FC_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  const LinearLayout L = linear_layout(d);
  GemmBatch gb{};
  gb.trans_b = 0;
  for (int l = 0; l <= L.common; ++l) {
    GemmRank& g = gb.r[l];
    const int Kin = d->in_features * d->in_paths[l];
    g.A = go + L.out_off[l];
    g.a_row = L.out_dim;
    g.a_comp = d->out_features;
    g.B = d->weight[l];
    g.D = gx + L.in_off[l];
    g.R = residual ? residual + L.in_off[l] : nullptr;
    g.d_row = L.in_dim;
    g.d_comp = Kin;
    g.comps = 2 * l + 1;
    g.M = (int32_t)(n * g.comps);
    g.K = d->out_features;
    g.N = Kin;
    g.scale = alpha * d->scale[l];
  }
  st = launch_gemm(gb, L.common + 1, s);
  if (st != FC_OK) return st;
  if (L.common < d->in_l_max)
    return fill_columns(n, L.in_dim, L.in_off[L.common + 1], L.in_dim - L.in_off[L.common + 1], residual, gx, s);
  return FC_OK;
}

namespace fc {

// ---- Wide output, K = 64: out (n x m) = scale * x (n x 64) @ W^T, W (m x 64), m >> 64 (the
// radial MLP's output layer, m = paths x channels). Writing the output is as costly as the
// MFMA work here, so each workgroup keeps its 128 x 64 block of x, split into bf16 parts
// (fc_gemm_split.h), in registers and walks the output columns in chunks of 64 whose weights are
// split once per workgroup into LDS, double buffered; the next chunk's weights load while the
// current one is multiplied. Four waves stacked along the rows, 32 x 64 outputs each per chunk.
// A launch of few row blocks splits the columns over blockIdx.y as well.
// Measured against float32 matrix instructions before it (m = 2,176): radial MLP of 540,083 rows
// 1,697 -> 1,299 us (1,377 with stores that are not nontemporal; 4.7 GB written), of 140,000 rows
// 553 -> 397 us, of 672 rows, where the columns are split, 94 -> 20 us; error against float64
// 2.5e-7 -> 2.0e-7.
constexpr int WIDE_BM = 128, WIDE_BN = 64, WIDE_K = 64, WIDE_P = 68;
constexpr int WIDE_PART = 2 * 4 * 64;  // LDS entries per part of a weight chunk

// This wave's 32 rows of x: lane (r, h) = (lane % 32, lane / 32) holds k = 16 c + 8 h .. + 7 of row r in
// chunk c, split and (for sums that come out infinite or NaN) as they are.
struct WideA {
  Split8 s[4];
  f32x4 x[8];
};
__device__ __forceinline__ void wide_load_a(const float* row, int h, WideA& a) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int q = 0; q < 2; ++q) a.x[2 * c + q] = *reinterpret_cast<const f32x4*>(row + 16 * c + 8 * h + 4 * q);
    a.s[c] = split8(a.x[2 * c], a.x[2 * c + 1]);
  }
}

// Output part shared by the wide kernels: rows r0 .. r0 + 127, the column chunks of this blockIdx.y.
// Bs holds two weight chunks: block (column block j, k chunk c) of 64 16-byte entries per part, entry
// (column % 32 ^ 2 (2 c + h)) + 32 h holding k = 16 c + 8 h .. + 7. Every thread of the workgroup calls it.
// FULL: every row and column of the block is in range, so the stores are unconditional and the
// compiler can count them as outstanding where it waits for the next weight chunk. LONG: rows of
// kWideLong elements or more, whose offsets are formed in 64 bits as they are needed.
constexpr int kWideLong = 1 << 22;  // (from here on a block's byte offsets, 128 m 4, leave 31 bits)
template <bool FULL, bool LONG = false>
__device__ __forceinline__ void wide_body(const WideA& a, bf16x8 (*Bs)[3 * WIDE_PART], int64_t n, int m,
                                          const float* __restrict__ w, float scale, float* __restrict__ out,
                                          int64_t r0) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, rl = lane & 31, h = lane >> 5;
  const int nch_all = (m + WIDE_BN - 1) / WIDE_BN;
  const int ch0 = (int)((int64_t)nch_all * blockIdx.y / gridDim.y);
  const int ch1 = (int)((int64_t)nch_all * (blockIdx.y + 1) / gridDim.y);
  if (ch0 >= ch1) return;  // uniform

  f32x4 br[2][2];
  auto load_b = [&](int ch) {  // 64 weight rows x 8 groups of 8 k, two per thread
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int it = t + 256 * i, o = it & 7;
      const int col = min(ch * WIDE_BN + (it >> 3), m - 1);
      const float* p = w + (int64_t)col * WIDE_K + 8 * o;
      br[i][0] = *reinterpret_cast<const f32x4*>(p);
      br[i][1] = *reinterpret_cast<const f32x4*>(p + 4);
    }
  };
  auto store_b = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int it = t + 256 * i, o = it & 7, col = it >> 3;
      const int e = ((col >> 5) * 4 + (o >> 1)) * 64 + ((col & 31) ^ (2 * o)) + 32 * (o & 1);
#pragma unroll
      for (int q = 0; q < 2; ++q) asm volatile("" : "+v"(br[i][q]));
      const Split8 s = split8(br[i][0], br[i][1]);
      Bs[buf][e] = s.h;
      Bs[buf][WIDE_PART + e] = s.m;
      Bs[buf][2 * WIDE_PART + e] = s.l;
    }
  };
  // offset of this lane's 16 output rows from the block's first element, so that a store is a wave-uniform
  // base plus a 32-bit offset
  uint32_t voff[16];  // bytes
  if constexpr (!LONG) {
#pragma unroll
    for (int v = 0; v < 16; ++v)
      voff[v] = (uint32_t)((wave * 32 + 4 * h + 8 * (v >> 2) + (v & 3)) * m + rl) * 4u;
  }
  gfloat* const blk = uniform_gptr(out + r0 * m);
  const int64_t row0 = r0 + wave * 32 + 4 * h;

  load_b(ch0);
  store_b(0);
  load_b(min(ch0 + 1, ch1 - 1));
  __syncthreads();
  int buf = 0;
  for (int ch = ch0; ch < ch1; ++ch) {
    floatx16 hi[2], lo[2];
    auto fetch = [&](int q) {  // group q: k chunk q / 2, column block q % 2
      const int c = q >> 1, j = q & 1;
      const bf16x8* p = Bs[buf] + (j * 4 + c) * 64 + (rl ^ (2 * (2 * c + h))) + 32 * h;
      Split8 f;
      f.h = p[0];
      f.m = p[WIDE_PART];
      f.l = p[2 * WIDE_PART];
      return f;
    };
    Split8 nxt = fetch(0);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int c = q >> 1, j = q & 1;
      const Split8 b = nxt;
      if (q + 1 < 8) nxt = fetch(q + 1);
      __builtin_amdgcn_sched_barrier(0);
      lo[j] = mfma_bf16(a.s[c].l, b.h, c == 0 ? floatx16{} : lo[j]);
      hi[j] = mfma_bf16(a.s[c].h, b.h, c == 0 ? floatx16{} : hi[j]);
      lo[j] = mfma_bf16(a.s[c].h, b.l, lo[j]);
      lo[j] = mfma_bf16(a.s[c].m, b.m, lo[j]);
      lo[j] = mfma_bf16(a.s[c].m, b.h, lo[j]);
      lo[j] = mfma_bf16(a.s[c].h, b.m, lo[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    // the next chunk's weights to the other buffer (last read before the barrier that ended the
    // turn before); loads are issued on every path, so that waits count them exactly
    store_b(buf ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    load_b(min(ch + 2, ch1 - 1));
    __builtin_amdgcn_sched_barrier(0);
    const int c0 = ch * WIDE_BN;
    float probe = 0.f;  // NaN if any sum is infinite or NaN
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        hi[j][v] = (hi[j][v] + lo[j][v]) * kSplitUnscale;
        probe = fmaf(hi[j][v], 0.f, probe);
      }
    float late = scale;
    if (__any(probe != probe)) {
      // Again in plain float32, with the weights scaled first: x W may overflow where scale x W does not.
      late = 1.f;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float* p = w + (int64_t)min(c0 + 32 * j + rl, m - 1) * WIDE_K + 8 * h;
        hi[j] = floatx16{};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const f32x4 bv = *reinterpret_cast<const f32x4*>(p + 16 * (q >> 1) + 4 * (q & 1));
#pragma unroll
          for (int i = 0; i < 4; ++i)
            hi[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x[q][i], bv[i] * scale, hi[j], 0, 0, 0);
        }
      }
    }
    gfloat* const base = blk + c0;
    if constexpr (FULL) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          __builtin_nontemporal_store(hi[j][v] * late,
                                      reinterpret_cast<gfloat*>(reinterpret_cast<gchar*>(base) + voff[v]) + j * 32);
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          if (row0 + 8 * (v >> 2) + (v & 3) < n && c0 + j * 32 + rl < m) {
            gfloat* const p = LONG ? base + (int64_t)(wave * 32 + 4 * h + 8 * (v >> 2) + (v & 3)) * m + rl
                                   : reinterpret_cast<gfloat*>(reinterpret_cast<gchar*>(base) + voff[v]);
            p[j * 32] = hi[j][v] * late;
          }
    }
    __syncthreads();
    buf ^= 1;
  }
}

template <bool LONG>  // (a kernel of its own: the body is long, and code that is not run costs small calls time too)
__device__ __forceinline__ void wide_out(const WideA& a, bf16x8 (*Bs)[3 * WIDE_PART], int64_t n, int m,
                                         const float* __restrict__ w, float scale, float* __restrict__ out, int64_t r0) {
  if constexpr (LONG) wide_body<false, true>(a, Bs, n, m, w, scale, out, r0);
  else if (r0 + WIDE_BM <= n && m % WIDE_BN == 0) wide_body<true>(a, Bs, n, m, w, scale, out, r0);
  else wide_body<false>(a, Bs, n, m, w, scale, out, r0);
}

// Row blocks x column parts of the wide kernels. Each part repeats the block's work before its columns, `fixed` column
// chunks' worth (4 for the radial MLP, whose parts all form the hidden layers, 1 for a dense layer). Two workgroups on
// a CU take `pair` fifths of one's time (8 and 7), k more 0.8 k times. The number of parts with the least time by that,
// for up to two row blocks a CU. Radial MLP, microseconds, one part / as many as 512 workgroups have room for / this rule:
// 235 blocks, 160 columns 23 / 34 / 23, 2,176 columns 89 / 87 / 73; 128 blocks 22 / 24 / 19 and 84 / 51 / 51; 6 blocks
// 19 / 15 / 15 and 82 / 16 / 16. Dense layer, 235 blocks, 2,176 columns 78 / 74 / 63.
static dim3 wide_grid(int64_t blocks, int m, int fixed, int pair) {
  const int64_t chunks = (m + (int64_t)WIDE_BN - 1) / WIDE_BN, cus = device_cu_count();
  int64_t parts = 1, least = -1;
  for (int64_t p = 1; p <= chunks && (p == 1 || (blocks <= 2 * cus && blocks * p <= 8 * cus)); ++p) {
    const int64_t per_cu = (blocks * p + cus - 1) / cus;
    const int64_t time = (fixed + (chunks + p - 1) / p) * (per_cu <= 1 ? 5 : per_cu == 2 ? pair : 4 * per_cu);
    if (least < 0 || time < least) {
      least = time;
      parts = p;
    }
  }
  return dim3((unsigned)blocks, (unsigned)parts);
}

template <bool LONG>
__global__ void __launch_bounds__(256, 2) gemm_wide_kernel(int64_t n, int m, const float* __restrict__ x,
                                                            const float* __restrict__ w, float scale,
                                                            float* __restrict__ out) {
  __shared__ bf16x8 Bs[2][3 * WIDE_PART];
  const int t = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.x * WIDE_BM, row = r0 + 32 * (t >> 6) + (t & 31);
  WideA a;
  wide_load_a(x + (row < n ? row : n - 1) * WIDE_K, (t >> 5) & 1, a);  // rows past n are not stored
  wide_out<LONG>(a, Bs, n, m, w, scale, out, r0);
}

// ---- Radial MLP with two hidden layers of 64 (reference InteractionLayer.radial_mlp,
// src/flashcart/nn/layers.py:258-267, applied at :357-363):
//   pre1 = s0 x W0^T, h1 = silu(pre1), pre2 = s1 h1 W1^T, h2 = silu(pre2), out = s2 h2 W2^T
// with silu the rescaled SiLU and x (n, n_in), n_in <= 64. The forward forms h1 and h2 of a
// 128-row block in LDS and hands h2 to the wide output part, so neither hidden layer goes
// through HBM. The backward (input gradient only) recomputes the hidden layers from x
// (n_in floats per row) instead of reading saved pre-activations.

// acc[j] (j < NJ) = A rows of this wave (as) x weight rows of column block j (bs + 32 j
// rows), k = 0..63: MFMA step s contracts k = s (lanes 0-31) and k = 32 + s (lanes 32-63).
// Only the first ns4 groups of four steps run: with K <= 32 the rest multiply zero padding
// (K = n_in, the first hidden layer), so ns4 = ceil(K / 4) there and 8 otherwise.
template <int NJ>
__device__ __forceinline__ void mfma_k64(const float* as, const float* bs, floatx16 (&acc)[2], int ns4 = 8) {
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
  // operands of group s4 + 1 are read from LDS while group s4 multiplies
  float4 a4n = *reinterpret_cast<const float4*>(as), b4n[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) b4n[j] = *reinterpret_cast<const float4*>(bs + j * 32 * WIDE_P);
#pragma unroll
  for (int s4 = 0; s4 < 8; ++s4) {
    if (s4 >= ns4) break;  // uniform
    const float4 a4 = a4n;
    float4 b4[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) b4[j] = b4n[j];
    if (s4 + 1 < ns4) {
      a4n = *reinterpret_cast<const float4*>(as + 4 * (s4 + 1));
#pragma unroll
      for (int j = 0; j < NJ; ++j) b4n[j] = *reinterpret_cast<const float4*>(bs + j * 32 * WIDE_P + 4 * (s4 + 1));
    }
    __builtin_amdgcn_sched_barrier(0);  // keep those reads ahead of this group's MFMAs
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(reinterpret_cast<const float*>(&a4)[q],
                                                      reinterpret_cast<const float*>(&b4[j])[q], acc[j], 0, 0, 0);
  }
}

// The same product with B stored the other way round: bt = W + (lane & 31) + half * WIDE_P for a
// weight square W[k][j] (k-major rows), so lane j of block jb reads W[k][jb * 32 + j] for its four
// k values (four scalar LDS reads, the same bytes as one float4): the input gradients multiply by
// the weight matrices the forward staged, without staging their transposes.
template <int NJ>
__device__ __forceinline__ void mfma_k64_t(const float* as, const float* bt, floatx16 (&acc)[2]) {
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
  auto read_b = [&](int s4, float4 (&b)[NJ]) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float* p = bt + 4 * s4 * WIDE_P + j * 32;
      b[j] = make_float4(p[0], p[WIDE_P], p[2 * WIDE_P], p[3 * WIDE_P]);
    }
  };
  float4 a4n = *reinterpret_cast<const float4*>(as), b4n[NJ];
  read_b(0, b4n);
#pragma unroll
  for (int s4 = 0; s4 < 8; ++s4) {
    const float4 a4 = a4n;
    float4 b4[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) b4[j] = b4n[j];
    if (s4 + 1 < 8) {
      a4n = *reinterpret_cast<const float4*>(as + 4 * (s4 + 1));
      read_b(s4 + 1, b4n);
    }
    __builtin_amdgcn_sched_barrier(0);  // keep those reads ahead of this group's MFMAs
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(reinterpret_cast<const float*>(&a4)[q],
                                                      reinterpret_cast<const float*>(&b4[j])[q], acc[j], 0, 0, 0);
  }
}

// Row (within the wave's 32 rows) of accumulator element v of this lane.
__device__ __forceinline__ int acc_row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }

__device__ __forceinline__ float silu_r(float z) { return kSiluScale * z * sigmoidf_(z); }
__device__ __forceinline__ float silu_r_grad(float z) {
  const float sg = sigmoidf_(z);
  return kSiluScale * sg * (1.0f + z * (1.0f - sg));
}

// x block (rows r0 .. r0 + 127 that exist; they are contiguous in x) -> As, zero-padded to 64
// columns; rows past n stay zero (never stored). W0 (64 x n_in) -> B0 and W1 (64 x 64) -> B1 as
// weight rows (zero-padded k). Every thread issues all of its global loads before its first LDS
// store, so the load latency is paid once.
__device__ __forceinline__ void mlp_stage_x(float* As, int64_t n, int n_in, const float* __restrict__ x, int64_t r0) {
  const int t = threadIdx.x;
  const int rows = n - r0 < WIDE_BM ? (int)(n - r0) : WIDE_BM;
  const int cnt = rows * n_in;
  const float* xb = x + r0 * n_in;
  // row of element e: e / n_in, exact in float for e < 2^13 ((e + 1/2) / n_in is at least
  // 1 / (2 n_in) from an integer), without an integer division per element
  const float inv_in = 1.0f / (float)n_in;
  // in chunks of eight values per thread (one chunk for up to 16 inputs), so few registers stay
  // reserved for the staging
  for (int base = 0; base < WIDE_BM * n_in; base += 8 * 256) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int e = base + t + 256 * i;
      v[i] = e < cnt ? xb[e] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int e = base + t + 256 * i;
      if (e < WIDE_BM * n_in) {
        const int q = (int)(((float)e + 0.5f) * inv_in);
        As[q * WIDE_P + (e - q * n_in)] = v[i];
      }
    }
  }
  for (int e = t; e < WIDE_BM * (WIDE_K - n_in); e += 256) {
    const int q = e / (WIDE_K - n_in);
    As[q * WIDE_P + n_in + (e - q * (WIDE_K - n_in))] = 0.f;
  }
}

__device__ __forceinline__ void mlp_stage_weights(float* B0, float* B1, int n_in, const float* __restrict__ w0,
                                                  const float* __restrict__ w1) {
  const int t = threadIdx.x;
  float a[16], b[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {  // element e = (r, c) of a 64 x 64 square, c = e & 63 along memory
    const int e = t + 256 * i, r = e >> 6, c = e & 63;
    a[i] = w1[r * 64 + c];
    b[i] = c < n_in ? w0[r * n_in + c] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int e = t + 256 * i, r = e >> 6, c = e & 63;
    B0[r * WIDE_P + c] = b[i];  // W0 row r (output), k = c
    B1[r * WIDE_P + c] = a[i];  // W1 row r, k = c
  }
}

// The wave's 32 x 64 accumulator block -> f(value) into its own rows of As.
template <class F>
__device__ __forceinline__ void acc_to_rows(const floatx16 (&acc)[2], float* As, int wave, int lane, F f) {
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v)
      As[(wave * 32 + acc_row(v, lane)) * WIDE_P + j * 32 + (lane & 31)] = f(acc[j][v]);
}

// HIDDEN: stop after the second hidden layer and write its activation h2 (n x 64) instead of
// the output layer (the first interaction layer's species density takes h2 itself).
template <bool HIDDEN, bool LONG = false>
__global__ void __launch_bounds__(256, 2) radial_mlp_fwd_kernel(int64_t n, int n_in, const float* __restrict__ x,
                                                                 const float* __restrict__ w0, float s0,
                                                                 const float* __restrict__ w1, float s1, int m,
                                                                 const float* __restrict__ w2, float s2,
                                                                 float* __restrict__ out) {
  // the hidden layers' operands, then the output layer's weight chunks
  union Lds {
    struct {
      float As[WIDE_BM * WIDE_P];
      float Bs[2][WIDE_BN * WIDE_P];
    } f;
    bf16x8 wide[2][3 * WIDE_PART];
    __device__ Lds() {}
  };
  __shared__ __attribute__((aligned(16))) char raw[sizeof(Lds)];
  Lds& lds = *reinterpret_cast<Lds*>(raw);
  float* const As = lds.f.As;
  auto Bs = lds.f.Bs;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t r0 = (int64_t)blockIdx.x * WIDE_BM;
  mlp_stage_x(As, n, n_in, x, r0);
  mlp_stage_weights(Bs[0], Bs[1], n_in, w0, w1);
  __syncthreads();
  const int half = (lane >> 5) * (WIDE_K / 2);
  const float* as = As + (wave * 32 + (lane & 31)) * WIDE_P + half;
  floatx16 acc[2];
  const int ns4_in = n_in <= 32 ? (n_in + 3) / 4 : 8;
  mfma_k64<2>(as, Bs[0] + (lane & 31) * WIDE_P + half, acc, ns4_in);
  __syncthreads();  // every wave's reads of the x rows are done (each wave rewrites only its own rows)
  acc_to_rows(acc, As, wave, lane, [&](float a) { return silu_r(a * s0); });
  __syncthreads();
  mfma_k64<2>(as, Bs[1] + (lane & 31) * WIDE_P + half, acc);
  if constexpr (HIDDEN) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t row = r0 + wave * 32 + acc_row(v, lane);
        if (row < n) out[row * 64 + j * 32 + (lane & 31)] = silu_r(acc[j][v] * s1);
      }
    return;
  }
  __syncthreads();  // reads of h1 done before it is overwritten
  acc_to_rows(acc, As, wave, lane, [&](float a) { return silu_r(a * s1); });
  __syncthreads();
  WideA a;
  wide_load_a(As + (wave * 32 + (lane & 31)) * WIDE_P, lane >> 5, a);
  __syncthreads();  // reads of h2 and of both weight matrices done before the weight chunks overwrite them
  wide_out<LONG>(a, lds.wide, n, m, w2, s2, out, r0);
}

// Input gradient of the two hidden layers: given gh2 = dL/dh2 (n, 64),
//   dpre2 = gh2 * silu'(pre2), dh1 = s1 dpre2 W1, dpre1 = dh1 * silu'(pre1), dx = s0 dpre1 W0.
// PAIRS: gh2 holds two rows per input row (rows 2r and 2r + 1, summed).
template <bool PAIRS = false>
__global__ void __launch_bounds__(256, 2) radial_mlp_bwd_kernel(int64_t n, int n_in, const float* __restrict__ x,
                                                                 const float* __restrict__ w0, float s0,
                                                                 const float* __restrict__ w1, float s1,
                                                                 const float* __restrict__ gh2,
                                                                 float* __restrict__ gx) {
  __shared__ __attribute__((aligned(16))) float As[WIDE_BM * WIDE_P];
  __shared__ __attribute__((aligned(16))) float B0[WIDE_BN * WIDE_P];
  __shared__ __attribute__((aligned(16))) float B1[WIDE_BN * WIDE_P];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // Persistent: workgroup b takes row blocks b, b + G, ...; the weights are staged once, and the
  // next block's dL/dh2 loads while the current block's last two products run.
  const int64_t nblk = (n + WIDE_BM - 1) / WIDE_BM;
  int64_t blk = blockIdx.x;
  if (blk >= nblk) return;  // uniform
  // this lane's dL/dh2 values of block b (accumulator layout); rows past n contribute nothing
  auto load_g2 = [&](int64_t b, float (&g)[2][16]) {
    const int64_t rb = b * WIDE_BM;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t row = rb + wave * 32 + acc_row(v, lane);
        if constexpr (PAIRS)
          g[j][v] = row < n ? gh2[2 * row * 64 + j * 32 + (lane & 31)] + gh2[(2 * row + 1) * 64 + j * 32 + (lane & 31)]
                            : 0.f;
        else
          g[j][v] = row < n ? gh2[row * 64 + j * 32 + (lane & 31)] : 0.f;
      }
  };
  float g2[2][16];
  load_g2(blk, g2);
  mlp_stage_weights(B0, B1, n_in, w0, w1);
  const int half = (lane >> 5) * (WIDE_K / 2);
  const float* as = As + (wave * 32 + (lane & 31)) * WIDE_P + half;
  // dh1 = dpre2 W1 and dx = dpre1 W0 read the weight rows staged for the forward layers
  const float* w1t = B1 + (lane & 31) + half * WIDE_P;
  const float* w0t = B0 + (lane & 31) + half * WIDE_P;
  const int ns4_in = n_in <= 32 ? (n_in + 3) / 4 : 8;
  const int nj = n_in <= 32 ? 1 : 2;  // dx has n_in columns: one 32-column block when n_in <= 32
  for (; blk < nblk; blk += gridDim.x) {
    const int64_t r0 = blk * WIDE_BM;
    mlp_stage_x(As, n, n_in, x, r0);
    __syncthreads();  // x rows (and, the first time, the weights) staged
    floatx16 acc[2], d1[2];
    mfma_k64<2>(as, B0 + (lane & 31) * WIDE_P + half, acc, ns4_in);
    // one sigmoid per pre-activation serves both silu'(pre1) (kept) and h1 = silu(pre1) (to LDS)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float z = acc[j][v] * s0, sg = sigmoidf_(z);
        d1[j][v] = kSiluScale * sg * (1.0f + z * (1.0f - sg));
        acc[j][v] = kSiluScale * z * sg;
      }
    __syncthreads();
    acc_to_rows(acc, As, wave, lane, [](float a) { return a; });
    __syncthreads();
    mfma_k64<2>(as, B1 + (lane & 31) * WIDE_P + half, acc);
    // dpre2 = gh2 * silu'(pre2)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[j][v] = g2[j][v] * silu_r_grad(acc[j][v] * s1);
    if (blk + gridDim.x < nblk) load_g2(blk + gridDim.x, g2);  // in flight during the rest of this block
    __syncthreads();  // reads of h1 done: stage dpre2
    acc_to_rows(acc, As, wave, lane, [](float a) { return a; });
    __syncthreads();
    mfma_k64_t<2>(as, w1t, acc);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[j][v] = acc[j][v] * s1 * d1[j][v];
    __syncthreads();
    acc_to_rows(acc, As, wave, lane, [](float a) { return a; });
    __syncthreads();
    if (nj == 1) mfma_k64_t<1>(as, w0t, acc);
    else mfma_k64_t<2>(as, w0t, acc);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t row = r0 + wave * 32 + acc_row(v, lane);
        const int col = j * 32 + (lane & 31);
        if (j < nj && row < n && col < n_in) gx[row * n_in + col] = acc[j][v] * s0;
      }
    __syncthreads();  // every wave's reads of this block's rows done before the next block's x
  }
}

}  // namespace fc

extern "C" int fc_dense_fwd(int64_t n, int32_t k, int32_t m, const float* x, const float* w, float scale,
                            const float* bias, int32_t act, float* pre_act, float* out, void* stream) {
  if (n < 0 || k < 1 || m < 1 || act < 0 || act > 1) return FC_ERR_BAD_DESC;
  if (n == 0) return FC_OK;
  if (!x || !w || !out) return FC_ERR_NULL;
  if (n > 0x7fffffff) return FC_ERR_SHAPE;
  if (k == WIDE_K && m >= 4 * WIDE_BN && !bias && act == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0) {
    const int64_t blocks = (n + WIDE_BM - 1) / WIDE_BM;
    const auto kernel = m < kWideLong ? gemm_wide_kernel<false> : gemm_wide_kernel<true>;
    hipLaunchKernelGGL(kernel, wide_grid(blocks, m, 1, 7), dim3(256), 0, (hipStream_t)stream, n, m, x, w, scale, out);
    FC_LAUNCH_CHECK();
    return FC_OK;
  }
  GemmBatch gb{};
  gb.trans_b = 1;
  gb.bias = bias;
  gb.act = act;
  GemmRank& g = gb.r[0];
  g.A = x; g.a_row = k; g.a_comp = 0;
  g.B = w;
  g.D = out; g.d_row = m; g.d_comp = 0;
  g.pre = pre_act;
  g.comps = 1; g.M = (int32_t)n; g.K = k; g.N = m; g.scale = scale;
  return launch_gemm(gb, 1, (hipStream_t)stream);
}

extern "C" int fc_dense_fwd_pairsum(int64_t n, int32_t k, int32_t m, const float* x, const int32_t* rows_lo,
                                    const int32_t* rows_hi, const float* w, float scale, float* out, void* stream) {
  if (n < 0 || k < 1 || m < 1 || m > 64) return FC_ERR_BAD_DESC;
  if (n == 0) return FC_OK;
  if (!x || !w || !out) return FC_ERR_NULL;
  if ((rows_lo == nullptr) != (rows_hi == nullptr)) return FC_ERR_NULL;
  if (n > 0x7fffffff || (k & 31) || (m & 3) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return FC_ERR_SHAPE;
  GemmBatch gb{};
  gb.trans_b = 1;
  gb.pair_sum = 1;
  GemmRank& g = gb.r[0];
  g.A = x; g.a_row = (rows_lo ? 1 : 2) * (int64_t)k; g.a_comp = 0;
  g.a_lo = rows_lo; g.a_hi = rows_hi;
  g.B = w;
  g.D = out; g.d_row = m; g.d_comp = 0;
  g.comps = 1; g.M = (int32_t)n; g.K = k; g.N = m; g.scale = scale;
  return launch_gemm(gb, 1, (hipStream_t)stream);
}

extern "C" int fc_radial_mlp_fwd(int64_t n, int32_t n_in, const float* x, const float* w0, float s0,
                                 const float* w1, float s1, int32_t m, const float* w2, float s2, float* out,
                                 void* stream) {
  if (n < 0 || n_in < 1 || n_in > WIDE_K || m < 1) return FC_ERR_BAD_DESC;
  if (n == 0) return FC_OK;
  if (!x || !w0 || !w1 || !w2 || !out) return FC_ERR_NULL;
  if (((uintptr_t)w2 & 15) != 0) return FC_ERR_SHAPE;  // weight chunks load as float4
  const int64_t blocks = (n + WIDE_BM - 1) / WIDE_BM;
  if (blocks > 0x7fffffff) return FC_ERR_SHAPE;
  const auto kernel = m < kWideLong ? radial_mlp_fwd_kernel<false, false> : radial_mlp_fwd_kernel<false, true>;
  hipLaunchKernelGGL(kernel, wide_grid(blocks, m, 4, 8), dim3(256), 0, (hipStream_t)stream, n, (int)n_in, x, w0, s0, w1, s1,
                     (int)m, w2, s2, out);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

extern "C" int fc_radial_mlp_hidden_fwd(int64_t n, int32_t n_in, const float* x, const float* w0, float s0,
                                        const float* w1, float s1, float* h2, void* stream) {
  if (n < 0 || n_in < 1 || n_in > WIDE_K) return FC_ERR_BAD_DESC;
  if (n == 0) return FC_OK;
  if (!x || !w0 || !w1 || !h2) return FC_ERR_NULL;
  const int64_t blocks = (n + WIDE_BM - 1) / WIDE_BM;
  if (blocks > 0x7fffffff) return FC_ERR_SHAPE;
  hipLaunchKernelGGL(radial_mlp_fwd_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, n,
                     (int)n_in, x, w0, s0, w1, s1, 64, (const float*)nullptr, 1.0f, h2);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

// persistent workgroups of the radial MLP backward: two per CU (their LDS), at most one per block
static int64_t mlp_bwd_grid(int64_t blocks) {
  const int64_t g = 2 * (int64_t)device_cu_count();
  return blocks < g ? blocks : g;
}

extern "C" int fc_radial_mlp_bwd(int64_t n, int32_t n_in, const float* x, const float* w0, float s0,
                                 const float* w1, float s1, const float* grad_h2, float* grad_x, void* stream) {
  if (n < 0 || n_in < 1 || n_in > WIDE_K) return FC_ERR_BAD_DESC;
  if (n == 0) return FC_OK;
  if (!x || !w0 || !w1 || !grad_h2 || !grad_x) return FC_ERR_NULL;
  const int64_t blocks = (n + WIDE_BM - 1) / WIDE_BM;
  if (blocks > 0x7fffffff) return FC_ERR_SHAPE;
  hipLaunchKernelGGL(radial_mlp_bwd_kernel<false>, dim3((unsigned)mlp_bwd_grid(blocks)), dim3(256), 0,
                     (hipStream_t)stream, n, (int)n_in, x, w0, s0, w1, s1, grad_h2, grad_x);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

extern "C" int fc_radial_mlp_bwd_pairsum(int64_t n, int32_t n_in, const float* x, const float* w0, float s0,
                                         const float* w1, float s1, const float* grad_h2, float* grad_x,
                                         void* stream) {
  if (n < 0 || n_in < 1 || n_in > WIDE_K) return FC_ERR_BAD_DESC;
  if (n == 0) return FC_OK;
  if (!x || !w0 || !w1 || !grad_h2 || !grad_x) return FC_ERR_NULL;
  const int64_t blocks = (n + WIDE_BM - 1) / WIDE_BM;
  if (blocks > 0x7fffffff) return FC_ERR_SHAPE;
  hipLaunchKernelGGL(radial_mlp_bwd_kernel<true>, dim3((unsigned)mlp_bwd_grid(blocks)), dim3(256), 0,
                     (hipStream_t)stream, n, (int)n_in, x, w0, s0, w1, s1, grad_h2, grad_x);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

extern "C" int fc_dense_dgrad(int64_t n, int32_t k, int32_t m, const float* go, const float* pre_act,
                              const float* w, float scale, int32_t act, float* gx, void* stream) {
  if (n < 0 || k < 1 || m < 1 || act < 0 || act > 1) return FC_ERR_BAD_DESC;
  if (n == 0) return FC_OK;
  if (!go || !w || !gx || (act == 1 && !pre_act)) return FC_ERR_NULL;
  if (n > 0x7fffffff) return FC_ERR_SHAPE;
  GemmBatch gb{};
  gb.trans_b = 0;
  gb.act_bwd = act;
  GemmRank& g = gb.r[0];
  g.A = go; g.a_row = m; g.a_comp = 0;
  g.P = act ? pre_act : nullptr;
  g.B = w;
  g.D = gx; g.d_row = k; g.d_comp = 0;
  g.comps = 1; g.M = (int32_t)n; g.K = m; g.N = k; g.scale = scale;
  return launch_gemm(gb, 1, (hipStream_t)stream);
}

namespace fc {

// ---- Elementwise products with the rescaled SiLU's derivatives (second-order backward of the
// dense layers): out1 = a f'(pre) + add, out2 = a b f''(pre), with f(x) = kSiluScale x sigmoid(x),
//   f'(x)  = kSiluScale s (1 + x (1 - s)),   f''(x) = kSiluScale s (1 - s) (2 + x (1 - 2 s)),
// s = sigmoid(x). One pass over the operands for both products (one sigmoid per element).
__device__ __forceinline__ void silu_mix_one(float a, float b, float p, float add, bool w1, bool w2, float* o1,
                                             float* o2) {
  const float s = sigmoidf_(p);
  if (w1) *o1 = fmaf(a, kSiluScale * s * (1.0f + p * (1.0f - s)), add);
  if (w2) *o2 = a * b * (kSiluScale * s * (1.0f - s) * (2.0f + p * (1.0f - 2.0f * s)));
}

__global__ void __launch_bounds__(256) silu_grad_mix_kernel(int64_t n, const float* __restrict__ a,
                                                            const float* __restrict__ b,
                                                            const float* __restrict__ pre,
                                                            const float* __restrict__ add, float* __restrict__ out1,
                                                            float* __restrict__ out2, bool vec) {
  const bool w1 = out1 != nullptr, w2 = out2 != nullptr;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (vec) {  // n % 4 == 0 and every pointer 16-byte aligned
    for (int64_t q = t0; q < n / 4; q += stride) {
      const float4 av = reinterpret_cast<const float4*>(a)[q];
      const float4 pv = reinterpret_cast<const float4*>(pre)[q];
      const float4 bv = w2 ? reinterpret_cast<const float4*>(b)[q] : make_float4(0.f, 0.f, 0.f, 0.f);
      const float4 dv = (w1 && add) ? reinterpret_cast<const float4*>(add)[q] : make_float4(0.f, 0.f, 0.f, 0.f);
      float4 r1, r2;
      silu_mix_one(av.x, bv.x, pv.x, dv.x, w1, w2, &r1.x, &r2.x);
      silu_mix_one(av.y, bv.y, pv.y, dv.y, w1, w2, &r1.y, &r2.y);
      silu_mix_one(av.z, bv.z, pv.z, dv.z, w1, w2, &r1.z, &r2.z);
      silu_mix_one(av.w, bv.w, pv.w, dv.w, w1, w2, &r1.w, &r2.w);
      if (w1) reinterpret_cast<float4*>(out1)[q] = r1;
      if (w2) reinterpret_cast<float4*>(out2)[q] = r2;
    }
    return;
  }
  for (int64_t i = t0; i < n; i += stride) {
    float r1, r2;
    silu_mix_one(a[i], w2 ? b[i] : 0.f, pre[i], (w1 && add) ? add[i] : 0.f, w1, w2, &r1, &r2);
    if (w1) out1[i] = r1;
    if (w2) out2[i] = r2;
  }
}

}  // namespace fc

extern "C" int fc_silu_grad_mix(int64_t n, const float* a, const float* b, const float* pre, const float* add,
                                float* out1, float* out2, void* stream) {
  using namespace fc;
  if (n < 0) return FC_ERR_BAD_DESC;
  if (n == 0 || (!out1 && !out2)) return FC_OK;
  if (!a || !pre || (out2 && !b)) return FC_ERR_NULL;
  auto al = [](const void* p) { return p == nullptr || ((uintptr_t)p & 15) == 0; };
  const bool vec = (n & 3) == 0 && al(a) && al(b) && al(pre) && al(add) && al(out1) && al(out2);
  const int64_t work = vec ? n / 4 : n;
  const int64_t cap = (int64_t)device_cu_count() * 8;
  const int64_t blocks = (work + 255) / 256 < cap ? (work + 255) / 256 : cap;
  hipLaunchKernelGGL(silu_grad_mix_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, n, a, b, pre,
                     add, out1, out2, vec);
  FC_LAUNCH_CHECK();
  return FC_OK;
}

namespace fc {

// ---- Weight gradients (training): dW[o, j] = scale * sum_r A'[r, o] * B[r, j] over every row
// r = (node, component) of a rank, with A = grad_out (A' = A * act'(pre) for a dense layer
// with the fused SiLU) and B = the layer input; optionally db[o] = sum_r A'[r, o].
// The rows of a rank block are read in place from the packed feature rows (no gather copy).
// The row range is split over workgroups for parallelism (rows_per_split each); with more
// than one split every workgroup writes its unscaled partial block to a workspace and a
// second kernel sums the partials in split order, so results do not depend on scheduling.
struct WgradProblem {
  const float* A;  // row r = (n, c): A + n*a_row + c*a_comp, O floats
  const float* P;  // pre-activation in A's layout (SiLU derivative prologue) or null
  const float* B;  // row r: B + n*b_row + c*b_comp, J floats
  float* D;        // (O, J) row-major
  float* Db;       // (O) bias gradient or null
  int64_t a_row, a_comp, b_row, b_comp;
  int64_t R, rows_per_split;
  int32_t comps, O, J;
  float scale;
  int32_t tiles_o, tiles_j, splits, wg_base;
  int64_t part_off, partb_off;  // workspace offsets (floats) of the partial blocks
};

// One block of partial sums to reduce: dst[k] = scale * sum_s src[s * stride + k], k < count.
struct WgradSection {
  const float* src;
  float* dst;
  int64_t count, stride, base;  // base: first element in the reduce grid (multiple of 256)
  int32_t splits;
  float scale;
};

struct WgradBatch {
  WgradProblem p[FC_MAX_RANKS];
  WgradSection sec[2 * FC_MAX_RANKS];
  int32_t n, total_wg, n_sec;
  int64_t total_elems;
  float* part;
};

// Split operands on the bf16 matrix cores (fc_gemm_split.h): the contraction runs over rows, so thread
// (column, o) of a step loads rows 8 o .. 8 o + 7 of its column (a wave reads whole row segments, and the
// rows' addresses are scalar), splits them and writes them to LDS as the MFMAs read them: block (column
// block, half s) of 64 16-byte entries per part, entry (column % 32 ^ 4 o) + 32 (o / 2), s = o % 2. Four waves
// 2 x 2, each (TO / 2) x (TJ / 2) outputs in 32x32x16 blocks; the next step's rows load during the current
// step's MFMAs.
// Weight gradients of the product linear (K = 512 to 896, N = 128; with the reduction), against the float32
// matrix instructions before it: 25,000 nodes 1,197 -> 858 us, 6,691 nodes 287 -> 227 us; 64-wide maps, l <= 2:
// 25,000 nodes 99 -> 71 us, 6,700 nodes 37 us either way. With 64 x 64 tiles a launch has 0.5 to 1 us more to do before
// its first rows are there (row cursors and addresses in scalar registers): 8 rows 5.1 -> 5.9 us, 300 rows 18.0 -> 19.0.
// Steps that do not exist are not loaded (8 rows 6.7 us with one); loads at one place of the loop, for half the
// code, gained nothing there and cost 3% at 25,000 rows.
// Few outputs leave little work to the splits of many inputs: 16,384 -> 16, 40,000 rows 950 -> 1,230 us, 2,560 -> 32,
// 25,000 nodes with l <= 2 873 -> 930; up to 900 inputs a rank it is even or faster.
template <int TO, int TJ, bool ACT>
__global__ void __launch_bounds__(256, 2) wgrad_kernel(WgradBatch wb) {
  constexpr int RK = 32;                    // rows per step
  constexpr int FO = TO / 64, FJ = TJ / 64;  // 32 x 32 blocks per wave
  constexpr int AI = TO / 64, BI = TJ / 64;  // (column, 8 rows) items per thread and step
  constexpr int AP = TO * 4, BP = TJ * 4;    // LDS entries per part
  __shared__ bf16x8 As[3 * AP];
  __shared__ bf16x8 Bs[3 * BP];
  const int b = blockIdx.x;
  if (b >= wb.total_wg) return;
  int pi = 0;
#pragma unroll
  for (int q = 1; q < FC_MAX_RANKS; ++q)
    if (q < wb.n && b >= wb.p[q].wg_base) pi = q;
  const WgradProblem& g = wb.p[pi];
  const int local = b - g.wg_base;
  const int tiles = g.tiles_o * g.tiles_j;
  const int split = local / tiles, tile = local - split * tiles;
  const int to = tile / g.tiles_j, tj = tile - to * g.tiles_j;
  const int o0 = to * TO, j0 = tj * TJ, comps = g.comps;
  const int r_begin = (int)(split * g.rows_per_split);
  const int r_end = (int)(r_begin + g.rows_per_split < g.R ? r_begin + g.rows_per_split : g.R);
  const int t = threadIdx.x, lane = t & 63, rl = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wo = wave >> 1, wj = wave & 1;
  const bool do_bias = g.Db && tj == 0;

  // this thread's column of each operand and the first of its row groups (the same for a whole wave)
  const int acol = t % TO, bcol = t % TJ;
  const int aw = wave / (TO / 64), bw = wave / (TJ / 64);
  const int acl = min(o0 + acol, g.O - 1), bcl = min(j0 + bcol, g.J - 1);
  float av[AI][8], pv[ACT ? AI : 1][8], bv[BI][8];
  // Row group cursors: (node, component) of the group's first row, advanced by 32 rows a step with
  // scalar additions (a division per row would cost more than the split).
  const int step_n = RK / comps, step_c = RK - step_n * comps;
  struct Cursor {
    int n, c;
  };
  auto cursor = [&](int r) {
    const int n = (int)((uint32_t)r / (uint32_t)comps);
    return Cursor{__builtin_amdgcn_readfirstlane(n), __builtin_amdgcn_readfirstlane(r - n * comps)};
  };
  auto advance = [&](Cursor& k) {
    k.n += step_n;
    k.c += step_c;
    if (k.c >= comps) {
      k.c -= comps;
      ++k.n;
    }
  };
  // eight rows of one operand column from a cursor; `left` of them exist (uniform), the others read the last
  auto load_rows = [&](const float* base, int64_t row_stride, int64_t comp_stride, Cursor k, int left, int col,
                       float (&v)[8]) {
    const gfloat* p = uniform_gptr(base + (int64_t)k.n * row_stride + (int64_t)k.c * comp_stride);
    const int64_t wrap = row_stride - (int64_t)(comps - 1) * comp_stride;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      v[q] = p[col];
      const bool last = ++k.c == comps;
      if (last) k.c = 0;
      if (q + 1 < left) p += last ? wrap : comp_stride;
    }
  };
  Cursor ka[AI], kb[BI];
  auto seek = [&](int r0) {
#pragma unroll
    for (int i = 0; i < AI; ++i) ka[i] = cursor(min(r0 + 8 * (aw + (256 / TO) * i), r_end - 1));
#pragma unroll
    for (int i = 0; i < BI; ++i) kb[i] = cursor(min(r0 + 8 * (bw + (256 / TJ) * i), r_end - 1));
  };
  auto load = [&](int r0) {  // the step's rows, and the cursors on to the next step
    if (r0 + RK > r_end) {
      asm volatile("");  // keeps this a branch: its divisions would otherwise run at every step
      seek(r0);          // (groups past the end start at the last row)
    }
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      const int left = r_end - (r0 + 8 * (aw + (256 / TO) * i));
      load_rows(g.A, g.a_row, g.a_comp, ka[i], left, acl, av[i]);
      if constexpr (ACT) load_rows(g.P, g.a_row, g.a_comp, ka[i], left, acl, pv[i]);
      advance(ka[i]);
    }
#pragma unroll
    for (int i = 0; i < BI; ++i) {
      load_rows(g.B, g.b_row, g.b_comp, kb[i], r_end - (r0 + 8 * (bw + (256 / TJ) * i)), bcl, bv[i]);
      advance(kb[i]);
    }
  };
  float bsum = 0.f;
  auto put = [&](bf16x8* lds, int part, int col, int o, const float (&v)[8]) {
    const int e = ((col >> 5) * 2 + (o & 1)) * 64 + ((col & 31) ^ (4 * o)) + 32 * (o >> 1);
    const Split8 s = split8(f32x4{v[0], v[1], v[2], v[3]}, f32x4{v[4], v[5], v[6], v[7]});
    lds[e] = s.h;
    lds[part + e] = s.m;
    lds[2 * part + e] = s.l;
  };
  auto store = [&](int r0) {
    const bool whole = r0 + RK <= r_end;  // uniform
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      const int o = aw + (256 / TO) * i;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        asm volatile("" : "+v"(av[i][q]));
        if constexpr (ACT) {
          asm volatile("" : "+v"(pv[i][q]));
          av[i][q] *= silu_grad_(pv[i][q]);
        }
        if (!whole && r0 + 8 * o + q >= r_end) av[i][q] = 0.f;
        if (do_bias) bsum += av[i][q];
      }
      put(As, AP, acol, o, av[i]);
    }
#pragma unroll
    for (int i = 0; i < BI; ++i) {
      const int o = bw + (256 / TJ) * i;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        asm volatile("" : "+v"(bv[i][q]));
        if (!whole && r0 + 8 * o + q >= r_end) bv[i][q] = 0.f;
      }
      put(Bs, BP, bcol, o, bv[i]);
    }
  };

  floatx16 hi[FO][FJ], lo[FO][FJ];
#pragma unroll
  for (int i = 0; i < FO; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j) hi[i][j] = lo[i][j] = floatx16{};

  if (r_begin < r_end) {
    if (r_begin + RK <= r_end) seek(r_begin);  // (else load does)
    load(r_begin);
  }
  for (int r0 = r_begin; r0 < r_end; r0 += RK) {
    store(r0);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    if (r0 + RK < r_end) load(r0 + RK);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int e = s * 64 + (rl ^ (4 * (2 * h + s))) + 32 * h;
      Split8 fa[FO], fb[FJ];
#pragma unroll
      for (int i = 0; i < FO; ++i) {
        const bf16x8* p = As + (wo * FO + i) * 128 + e;
        fa[i].h = p[0]; fa[i].m = p[AP]; fa[i].l = p[2 * AP];
      }
#pragma unroll
      for (int j = 0; j < FJ; ++j) {
        const bf16x8* p = Bs + (wj * FJ + j) * 128 + e;
        fb[j].h = p[0]; fb[j].m = p[BP]; fb[j].l = p[2 * BP];
      }
#pragma unroll
      for (int i = 0; i < FO; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j) {
          lo[i][j] = mfma_bf16(fa[i].l, fb[j].h, lo[i][j]);
          hi[i][j] = mfma_bf16(fa[i].h, fb[j].h, hi[i][j]);
          lo[i][j] = mfma_bf16(fa[i].h, fb[j].l, lo[i][j]);
          lo[i][j] = mfma_bf16(fa[i].m, fb[j].m, lo[i][j]);
          lo[i][j] = mfma_bf16(fa[i].m, fb[j].h, lo[i][j]);
          lo[i][j] = mfma_bf16(fa[i].h, fb[j].m, lo[i][j]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
  }

  float probe = 0.f;  // NaN if any sum is infinite or NaN
#pragma unroll
  for (int i = 0; i < FO; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        hi[i][j][v] = (hi[i][j][v] + lo[i][j][v]) * kSplitUnscale;
        probe = fmaf(hi[i][j][v], 0.f, probe);
      }
  if (__any(probe != probe)) {  // again in plain float32, two rows a step (lane half h takes row r + h)
#pragma unroll
    for (int i = 0; i < FO; ++i)
#pragma unroll
      for (int j = 0; j < FJ; ++j) hi[i][j] = floatx16{};
#pragma unroll 1
    for (int r = r_begin; r < r_end; r += 2) {
      const bool ok = r + h < r_end;
      const int row = ok ? r + h : r, n = row / comps, c = row - n * comps;
      float fa[FO], fb[FJ];
#pragma unroll
      for (int i = 0; i < FO; ++i) {
        const int64_t off = (int64_t)n * g.a_row + (int64_t)c * g.a_comp + min(o0 + (wo * FO + i) * 32 + rl, g.O - 1);
        fa[i] = g.A[off];
        if constexpr (ACT) fa[i] *= silu_grad_(g.P[off]);
        if (!ok) fa[i] = 0.f;
      }
#pragma unroll
      for (int j = 0; j < FJ; ++j) {
        fb[j] = g.B[(int64_t)n * g.b_row + (int64_t)c * g.b_comp + min(j0 + (wj * FJ + j) * 32 + rl, g.J - 1)];
        if (!ok) fb[j] = 0.f;
      }
#pragma unroll
      for (int i = 0; i < FO; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j) hi[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], hi[i][j], 0, 0, 0);
    }
  }

  // ---- epilogue: D[o][j] with o = 8*(v/4) + 4*(lane/32) + v%4, j = lane%32 per 32x32 block
  const bool direct = g.splits == 1;
  float* dst = direct ? g.D : wb.part + g.part_off + (int64_t)split * g.O * g.J;
  const float sc = direct ? g.scale : 1.0f;
#pragma unroll
  for (int i = 0; i < FO; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int o = o0 + (wo * FO + i) * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
      if (o >= g.O) continue;
#pragma unroll
      for (int j = 0; j < FJ; ++j) {
        const int jj = j0 + (wj * FJ + j) * 32 + rl;
        if (jj < g.J) dst[(int64_t)o * g.J + jj] = hi[i][j][v] * sc;
      }
    }
  if (do_bias) {  // the row groups of a column, added in order
    float* red = reinterpret_cast<float*>(As);
    red[t] = bsum;
    __syncthreads();
    if (t < TO && o0 + t < g.O) {
      float s = 0.f;
#pragma unroll
      for (int q = 0; q < 256 / TO; ++q) s += red[q * TO + t];
      (direct ? g.Db : wb.part + g.partb_off + (int64_t)split * g.O)[o0 + t] = s;
    }
  }
}

// D = scale * sum over splits of the partial blocks (and Db = sum of the partial bias sums).
// Every workgroup covers 256 consecutive elements of one section (a weight or bias block;
// section starts are padded to multiples of 256): 64 threads x 4 elements per split lane,
// four split lanes (splits q, q+4, q+8, ...) whose sums are combined in a fixed order, so
// each thread keeps four independent loads in flight and the result is deterministic.
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(WgradBatch wb) {
  __shared__ float red[4][256];
  const int64_t e0 = (int64_t)blockIdx.x * 256;
  int si = 0;
  for (int q = 1; q < wb.n_sec; ++q)
    if (e0 >= wb.sec[q].base) si = q;
  const WgradSection& sc = wb.sec[si];
  const int t = threadIdx.x, c = t & 63, lane_split = t >> 6;
  const int64_t k = e0 - sc.base + 4 * c;  // first of this thread's four elements
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int sp = lane_split; sp < sc.splits; sp += 4) {
    const float* src = sc.src + (int64_t)sp * sc.stride;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (k + q < sc.count) acc[q] += src[k + q];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) red[lane_split][4 * c + q] = acc[q];
  __syncthreads();
  if (lane_split == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = 4 * c + q;
      if (k + q < sc.count) sc.dst[k + q] = ((red[0][i] + red[1][i]) + (red[2][i] + red[3][i])) * sc.scale;
    }
  }
}

// Tile shape, splits and workspace layout; returns the workspace size in floats.
static int64_t plan_wgrad(WgradBatch& wb, int* TO, int* TJ) {
  int max_o = 0, max_j = 0;
  for (int q = 0; q < wb.n; ++q) {
    if (wb.p[q].O > max_o) max_o = wb.p[q].O;
    if (wb.p[q].J > max_j) max_j = wb.p[q].J;
  }
  *TO = max_o >= 128 ? 128 : 64;
  *TJ = max_j >= 128 ? 128 : 64;
  int64_t work = 0, all_tiles = 0;
  for (int q = 0; q < wb.n; ++q) {
    WgradProblem& g = wb.p[q];
    g.tiles_o = (g.O + *TO - 1) / *TO;
    g.tiles_j = (g.J + *TJ - 1) / *TJ;
    work += (int64_t)g.tiles_o * g.tiles_j * g.R;
    all_tiles += (int64_t)g.tiles_o * g.tiles_j;
  }
  // At most 512 workgroups (one round of two per CU: every tile's row range rounds up to one more part, so
  // that many are set aside), at least 256 rows each (a partial block costs as much as reading 128 rows of
  // both operands). Two rounds write and add twice the partial blocks: 6,691 nodes 238 against 227 us, 162
  // against 180 us for the K = 384 to 640 map; two workgroups more than a round holds cost a third round.
  const int64_t want = 2 * (int64_t)device_cu_count();
  const int64_t parts = all_tiles < want / 2 ? want - all_tiles : want / 2;
  int64_t rps = (work + parts - 1) / parts;
  if (rps < 256) rps = 256;
  rps = (rps + 31) / 32 * 32;
  int64_t wg = 0, ws = 0;
  for (int q = 0; q < wb.n; ++q) {
    WgradProblem& g = wb.p[q];
    g.rows_per_split = rps;
    g.splits = (int32_t)(g.R > 0 ? (g.R + rps - 1) / rps : 1);
    g.wg_base = (int32_t)wg;
    wg += (int64_t)g.splits * g.tiles_o * g.tiles_j;
    if (g.splits > 1) {
      g.part_off = ws;
      ws += (int64_t)g.splits * g.O * g.J;
      g.partb_off = ws;
      if (g.Db) ws += (int64_t)g.splits * g.O;
    }
  }
  wb.total_wg = (int32_t)wg;
  return ws;
}

// The reduce grid: one section per weight (and bias) block that was split.
static void wgrad_sections(WgradBatch& wb) {
  wb.n_sec = 0;
  int64_t base = 0;
  auto add = [&](const float* src, float* dst, int64_t count, int64_t stride, int32_t splits, float scale) {
    WgradSection& sc = wb.sec[wb.n_sec++];
    sc.src = src; sc.dst = dst; sc.count = count; sc.stride = stride; sc.splits = splits; sc.scale = scale;
    sc.base = base;
    base += (count + 255) / 256 * 256;
  };
  for (int q = 0; q < wb.n; ++q) {
    const WgradProblem& g = wb.p[q];
    if (g.splits == 1) continue;
    const int64_t nw = (int64_t)g.O * g.J;
    add(wb.part + g.part_off, g.D, nw, nw, g.splits, g.scale);
    if (g.Db) add(wb.part + g.partb_off, g.Db, g.O, g.O, g.splits, 1.0f);
  }
  wb.total_elems = base;
}

static int launch_wgrad(WgradBatch wb, float* workspace, int64_t workspace_floats, hipStream_t s) {
  int TO, TJ;
  const int64_t need = plan_wgrad(wb, &TO, &TJ);
  if (wb.total_wg == 0) return FC_OK;
  if (need > 0 && (!workspace || workspace_floats < need)) return FC_ERR_WORKSPACE;
  wb.part = workspace;
  wgrad_sections(wb);
  const dim3 grid((unsigned)wb.total_wg), block(256);
  auto launch = [&](auto act) {
    constexpr bool ACT = decltype(act)::value;
    if (TO == 128 && TJ == 128) hipLaunchKernelGGL((wgrad_kernel<128, 128, ACT>), grid, block, 0, s, wb);
    else if (TO == 128) hipLaunchKernelGGL((wgrad_kernel<128, 64, ACT>), grid, block, 0, s, wb);
    else if (TJ == 128) hipLaunchKernelGGL((wgrad_kernel<64, 128, ACT>), grid, block, 0, s, wb);
    else hipLaunchKernelGGL((wgrad_kernel<64, 64, ACT>), grid, block, 0, s, wb);
  };
  if (wb.p[0].P) launch(std::true_type{});  // a dense layer's batch of one
  else launch(std::false_type{});
  FC_LAUNCH_CHECK();
  if (need > 0) {
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((unsigned)((wb.total_elems + 255) / 256)), dim3(256), 0, s, wb);
    FC_LAUNCH_CHECK();
  }
  return FC_OK;
}

static void linear_wgrad_batch(const fc_linear_desc* d, int64_t n, const float* go, const float* x, float alpha,
                               float* const* gw, WgradBatch& wb) {
  const LinearLayout L = linear_layout(d);
  wb = WgradBatch{};
  for (int l = 0; l <= L.common; ++l) {
    if (!gw || !gw[l]) continue;
    WgradProblem& g = wb.p[wb.n++];
    g.A = go + L.out_off[l];
    g.a_row = L.out_dim;
    g.a_comp = d->out_features;
    g.B = x + L.in_off[l];
    g.b_row = L.in_dim;
    g.b_comp = (int64_t)d->in_features * d->in_paths[l];
    g.D = gw[l];
    g.comps = 2 * l + 1;
    g.R = n * g.comps;
    g.O = d->out_features;
    g.J = d->in_features * d->in_paths[l];
    g.scale = alpha * d->scale[l];
  }
}

static void dense_wgrad_batch(int64_t n, int32_t k, int32_t m, const float* go, const float* pre_act, int32_t act,
                              const float* x, float scale, float* gw, float* gb, WgradBatch& wb) {
  wb = WgradBatch{};
  wb.n = 1;
  WgradProblem& g = wb.p[0];
  g.A = go; g.a_row = m; g.a_comp = 0;
  g.P = act ? pre_act : nullptr;
  g.B = x; g.b_row = k; g.b_comp = 0;
  g.D = gw; g.Db = gb;
  g.comps = 1; g.R = n; g.O = m; g.J = k; g.scale = scale;
}

}  // namespace fc

extern "C" int64_t fc_linear_wgrad_workspace(const fc_linear_desc* d, int64_t n, float* const* grad_w) {
  const int st = check_linear(d);
  if (st != FC_OK) return -st;
  if (n < 0) return -FC_ERR_SHAPE;
  // only which entries are non-NULL matters here (NULL array: every rank)
  float* all[FC_MAX_RANKS];
  for (int l = 0; l < FC_MAX_RANKS; ++l) all[l] = reinterpret_cast<float*>(16);
  WgradBatch wb;
  linear_wgrad_batch(d, n, nullptr, nullptr, 1.f, grad_w ? grad_w : all, wb);
  int TO, TJ;
  return plan_wgrad(wb, &TO, &TJ);
}

extern "C" int fc_linear_wgrad(const fc_linear_desc* d, int64_t n, const float* go, const float* x, float alpha,
                               float* const* grad_w, float* workspace, int64_t workspace_floats, void* stream) {
  int st = check_linear(d);
  if (st != FC_OK) return st;
  if (n < 0) return FC_ERR_SHAPE;
  if (!grad_w) return FC_ERR_NULL;
  if (n * (2 * FC_MAX_RANKS - 1) > 0x7fffffff) return FC_ERR_SHAPE;
  const int common = d->in_l_max < d->out_l_max ? d->in_l_max : d->out_l_max;
  if (n == 0) {  // no rows: zero gradients (a fill kernel, so the call can be graph-captured)
    for (int l = 0; l <= common; ++l)
      if (grad_w[l]) {
        const int64_t sz = (int64_t)d->out_features * d->in_features * d->in_paths[l];
        st = fill_columns(1, sz, 0, sz, nullptr, grad_w[l], (hipStream_t)stream);
        if (st != FC_OK) return st;
      }
    return FC_OK;
  }
  if (!go || !x) return FC_ERR_NULL;
  WgradBatch wb;
  linear_wgrad_batch(d, n, go, x, alpha, grad_w, wb);
  if (wb.n == 0) return FC_OK;
  return launch_wgrad(wb, workspace, workspace_floats, (hipStream_t)stream);
}

extern "C" int64_t fc_dense_wgrad_workspace(int64_t n, int32_t k, int32_t m, int32_t with_bias) {
  if (n < 0 || k < 1 || m < 1) return -FC_ERR_BAD_DESC;
  WgradBatch wb;
  dense_wgrad_batch(n, k, m, nullptr, nullptr, 0, nullptr, 1.f, reinterpret_cast<float*>(16),
                    with_bias ? reinterpret_cast<float*>(16) : nullptr, wb);
  int TO, TJ;
  return plan_wgrad(wb, &TO, &TJ);
}

extern "C" int fc_dense_wgrad(int64_t n, int32_t k, int32_t m, const float* go, const float* pre_act, int32_t act,
                              const float* x, float scale, float* gw, float* gb, float* workspace,
                              int64_t workspace_floats, void* stream) {
  if (n < 0 || k < 1 || m < 1 || act < 0 || act > 1) return FC_ERR_BAD_DESC;
  if (!gw) return FC_ERR_NULL;
  if (n == 0) {  // no rows: zero gradients (a fill kernel, so the call can be graph-captured)
    const int st = fill_columns(1, (int64_t)k * m, 0, (int64_t)k * m, nullptr, gw, (hipStream_t)stream);
    if (st != FC_OK || !gb) return st;
    return fill_columns(1, m, 0, m, nullptr, gb, (hipStream_t)stream);
  }
  if (!go || !x || (act == 1 && !pre_act)) return FC_ERR_NULL;
  if (n > 0x7fffffff - 256) return FC_ERR_SHAPE;  // row indices are 32-bit in the kernel
  WgradBatch wb;
  dense_wgrad_batch(n, k, m, go, pre_act, act, x, scale, gw, gb, wb);
  return launch_wgrad(wb, workspace, workspace_floats, (hipStream_t)stream);
}
