// fp32 products on v_mfma_f32_32x32x2_f32 (fp32 operands, products and sums), and the chain
// proposals' cell built on them: the ChainDraftCell of flashgrpo/models/medusa_heads.py:12-42,
//   mixed = LayerNorm(state) . Ws^T + LayerNorm(token) . Wt^T
//   out   = state + sigmoid(gate) * (SiLU(mixed) . Wo^T + bo)
// run outside autocast in the heads' fp32 parameters (flash_medusa_decoder.py:435-539).
//
// One workgroup of 4 waves per 64 x 64 output tile and part of K, a wave's 32 x 32 block in 16
// registers. K advances 32 per step through a double buffer in LDS (rows padded to 44 floats: the
// 16-byte fragment reads of 16 rows lie on distinct banks, counted as 0 conflicts), the next step's
// four 16-byte loads per thread in flight during the current one's 16 MFMAs. A lane's 16-byte
// fragment holds 4 consecutive k of its row; MFMA e of the four takes element e of both operands,
// which is the same k for both. B's rows are the first operand, so a lane ends with 4 consecutive
// columns of one row.
// Bound by the fp32 matrix rate (256 flop per clock and CU, 154 TFLOP/s in a loop of nothing else):
// 45 KB of LDS leave three workgroups per CU, so a SIMD has three waves to fill its matrix core
// from. In a loop of one launch 768 x 512 x 8192 takes 67 us (96 TFLOP/s, the matrix cores busy 73% of a
// CU's time) and 768 x 4096 x 512 with the cell's epilogue 37 (steps of 64 at two workgroups per CU: 79 and
// 52); in the proposal step, behind an LM head that has streamed 1 GB, 82.0 and 46.2 (79 and 70 TFLOP/s).
// Neither an order of the items that keeps 87% of the lines in an XCD's L2, nor two steps
// in flight, nor a start of K that differs between tiles moved it further. The fp32 Medusa block of
// 96 x 4096 x 4096 with its norm and combine: 118 -> 54 us, of 4 heads 430 -> 186 (fmaf tiles before).
#include "fg_f32.h"

#include <algorithm>

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kT = 64;           // output tile
constexpr int kKT = 32;          // K per step
constexpr int kCUs = 256;
constexpr int kRow = kKT + 12;   // floats per LDS row
constexpr int kU = kT * kKT / 4 / 256;  // 16-byte chunks per thread, step and operand

struct TileArgs {
  fg::F32Gemm g;
  int tiles_m, tiles, items, per_xcd, steps, steps_per_part;
  float* out;           // parts, or the chain cell's new states [M, N]
  const float* state;   // [M, N] row stride ld_state
  int64_t ld_state;
  const float* bias;    // [N]
  const float* gate;    // scalar
};

template <bool CHAIN>
__global__ void __launch_bounds__(256, 4) f32_tile_kernel(TileArgs a) {
  __shared__ __attribute__((aligned(16))) float xs[2][kT * kRow];
  __shared__ __attribute__((aligned(16))) float ws[2][kT * kRow];
  const fg::F32Gemm& g = a.g;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, half = lane >> 5;
  // workgroup b runs on XCD b % 8, which takes a contiguous run of (part, batch, tile) items, tiles
  // along M first: its workgroups walk the same K window together and share it in their L2
  const int item = (int)(blockIdx.x % 8) * a.per_xcd + (int)(blockIdx.x / 8);
  if (item >= a.items) return;  // whole workgroup: before any barrier
  const int tile = item % a.tiles, pz = item / a.tiles;
  const int part = pz / g.batch, z = pz % g.batch;
  const int m0 = tile % a.tiles_m * kT, n0 = tile / a.tiles_m * kT;
  const int wm = wave & 1, wn = wave >> 1;
  const int s0 = part * a.steps_per_part, s1 = min(a.steps, s0 + a.steps_per_part);
  const float* A = g.A + z * g.a_batch;
  const float* B = g.B + z * g.b_batch;
  // loader: chunk u of this thread is row (tid + 256 u) / 8, columns 4 (tid % 8) .. + 3
  const int lr = tid >> 3, lc = (tid & 7) * 4;
  const float* xsrc[kU];
  const float* wsrc[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    xsrc[u] = A + (int64_t)min(m0 + lr + 32 * u, g.M - 1) * g.lda;
    wsrc[u] = B + (int64_t)min(n0 + lr + 32 * u, g.N - 1) * g.ldb;
  }
  const int k_b2 = g.B2 ? g.k_b2 : g.K;
  const int64_t b2 = g.B2 ? ((intptr_t)g.B2 - (intptr_t)g.B) / (int64_t)sizeof(float) - k_b2 : 0;
  floatx4 xr[kU], wr[kU];
  const auto load = [&](int step) __attribute__((always_inline)) {
    const int k = step * kKT + lc;
    const int64_t wk = k < k_b2 ? k : k + b2;
    const bool in = k < g.K;  // the last step's columns past K count as 0
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      xr[u] = in ? *(const floatx4*)(xsrc[u] + k) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      wr[u] = in ? *(const floatx4*)(wsrc[u] + wk) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  const auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      *(floatx4*)&xs[buf][(lr + 32 * u) * kRow + lc] = xr[u];
      *(floatx4*)&ws[buf][(lr + 32 * u) * kRow + lc] = wr[u];
    }
  };
  floatx16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  const auto multiply = [&](int buf) __attribute__((always_inline)) {
    const float* x = xs[buf] + (wm * 32 + l32) * kRow + half * 4;
    const float* w = ws[buf] + (wn * 32 + l32) * kRow + half * 4;
#pragma unroll
    for (int k = 0; k < kKT; k += 8) {
      const floatx4 xv = *(const floatx4*)(x + k), wv = *(const floatx4*)(w + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[e], xv[e], acc, 0, 0, 0);
    }
  };
  load(s0);
  store(0);
  for (int t = s0; t + 1 < s1; ++t) {
    const int buf = (t - s0) & 1;
    load(t + 1);
    __syncthreads();  // step t is in LDS and every wave is done with step t - 1
    multiply(buf);
    store(buf ^ 1);
  }
  __syncthreads();
  multiply((s1 - 1 - s0) & 1);
  const int m = m0 + wm * 32 + l32;
  if (m >= g.M) return;
  const float gate = CHAIN ? *a.gate : 0.0f;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int n = n0 + wn * 32 + v * 8 + half * 4;
    if (n >= g.N) continue;
    float4 o = make_float4(acc[4 * v], acc[4 * v + 1], acc[4 * v + 2], acc[4 * v + 3]);
    if constexpr (CHAIN) {
#pragma clang fp contract(off)
      // rounded where the module rounds: the projection with its bias, the product, the sum
      const float4 b = *(const float4*)(a.bias + n);
      const float4 st = *(const float4*)(a.state + (int64_t)m * a.ld_state + n);
      o = make_float4(st.x + gate * (o.x + b.x), st.y + gate * (o.y + b.y), st.z + gate * (o.z + b.z),
                      st.w + gate * (o.w + b.w));
      *(float4*)(a.out + (int64_t)m * g.N + n) = o;
    } else {
      *(float4*)(a.out + (((int64_t)part * g.batch + z) * g.M + m) * g.N + n) = o;
    }
  }
}

int launch_tiles(TileArgs a, int splits, bool chain, hipStream_t s) {
  const fg::F32Gemm& g = a.g;
  FG_REQUIRE(g.M > 0 && g.N > 0 && g.K > 0 && g.batch > 0 && g.K % 4 == 0 && g.N % 4 == 0, "f32 gemm: shape");
  FG_REQUIRE(g.lda % 4 == 0 && g.ldb % 4 == 0 && g.a_batch % 4 == 0 && g.b_batch % 4 == 0 &&
                 ((uintptr_t)g.A & 15) == 0 && ((uintptr_t)g.B & 15) == 0 && ((uintptr_t)a.out & 15) == 0 &&
                 (!g.B2 || (((uintptr_t)g.B2 & 15) == 0 && g.k_b2 % 4 == 0 && g.k_b2 > 0 && g.k_b2 < g.K)),
             "f32 gemm: 16-byte aligned rows");
  a.tiles_m = (g.M + kT - 1) / kT;
  a.steps = (g.K + kKT - 1) / kKT;
  a.steps_per_part = (a.steps + splits - 1) / splits;
  a.tiles = a.tiles_m * ((g.N + kT - 1) / kT);
  FG_REQUIRE((int64_t)a.tiles * splits * g.batch < (1 << 30), "f32 gemm: too many tiles");
  a.items = a.tiles * splits * g.batch;
  a.per_xcd = (a.items + 7) / 8;
  const dim3 grid((unsigned)a.per_xcd * 8);
  if (chain) hipLaunchKernelGGL(f32_tile_kernel<true>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(f32_tile_kernel<false>, grid, dim3(256), 0, s, a);
  return fg::check_launch("f32 gemm");
}

// mid = SiLU(sum of the parts, in order), 4 columns per thread; the module's fp32 expression.
__global__ void __launch_bounds__(256) chain_mid_kernel(const float* __restrict__ parts, int splits, int64_t quads,
                                                        float* __restrict__ mid) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= quads) return;
  float4 v = ((const float4*)parts)[i];
  for (int p = 1; p < splits; ++p) {
    const float4 q = ((const float4*)parts)[p * quads + i];
    v.x += q.x; v.y += q.y; v.z += q.z; v.w += q.w;
  }
  ((float4*)mid)[i] = make_float4(v.x / (1.0f + expf(-v.x)), v.y / (1.0f + expf(-v.y)), v.z / (1.0f + expf(-v.z)),
                                  v.w / (1.0f + expf(-v.w)));
}

struct ChainPlan {
  int splits;
  size_t x, parts, mid;  // floats: the normalised inputs, the first product's parts, its activation
};
ChainPlan chain_plan(int rows, int hidden, int bottleneck) {
  ChainPlan p;
  p.splits = fg::f32_splits(rows, bottleneck, 2 * hidden, 1);
  p.x = (size_t)rows * 2 * hidden;
  p.parts = (size_t)p.splits * rows * bottleneck;
  p.mid = (size_t)rows * bottleneck;
  return p;
}

}  // namespace

namespace fg {

int f32_splits(int M, int N, int K, int batch) {
  const int64_t tiles = (int64_t)batch * ((M + kT - 1) / kT) * ((N + kT - 1) / kT);
  const int steps = (K + kKT - 1) / kKT;
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int sp = 1; sp <= std::min(steps / 2 + 1, 16); ++sp) {
    const int per = (steps + sp - 1) / sp;
    const int64_t rounds = (tiles * ((steps + per - 1) / per) + kCUs - 1) / kCUs;
    const int64_t cost = rounds * (per + 2) * (rounds == 1 ? 3 : 2);
    if (cost < best_cost) best_cost = cost, best = sp;
  }
  const int per = (steps + best - 1) / best;
  return (steps + per - 1) / per;  // no empty part
}

int f32_gemm_parts(const F32Gemm& g, int splits, float* parts, hipStream_t s) {
  TileArgs a{};
  a.g = g;
  a.out = parts;
  return launch_tiles(a, splits, false, s);
}

}  // namespace fg

extern "C" {

size_t fg_chain_cell_step_workspace(int rows, int hidden, int bottleneck) {
  if (rows <= 0 || hidden <= 0 || bottleneck <= 0) return 0;
  const ChainPlan p = chain_plan(rows, hidden, bottleneck);
  return (p.x + p.parts + p.mid) * sizeof(float) + 64;
}

int fg_chain_cell_step(const float* state, int64_t ld_state, const void* token, int64_t ld_token, int token_dtype,
                       int rows, int hidden, int bottleneck, const float* state_w, const float* state_b, const float* token_w,
                       const float* token_b, float eps, const float* state_proj_w, const float* token_proj_w, const float* out_w, 
                       const float* out_b, const float* gate, float* out, void* workspace, size_t workspace_bytes, void* stream) {
  FG_REQUIRE(state && token && state_w && state_b && token_w && token_b && state_proj_w && token_proj_w && out_w && out_b &&
                 gate && out && workspace,
             "fg_chain_cell_step: null pointer");
  FG_REQUIRE(rows > 0 && hidden > 0 && hidden % 8 == 0 && hidden <= 8192 && bottleneck > 0 && bottleneck % 4 == 0,
             "fg_chain_cell_step: hidden must be a multiple of 8 up to 8192, bottleneck of 4");
  FG_REQUIRE(ld_state % 4 == 0 && ((uintptr_t)state & 15) == 0 && ((uintptr_t)state_proj_w & 15) == 0 &&
                 ((uintptr_t)token_proj_w & 15) == 0 && ((uintptr_t)out_w & 15) == 0 && ((uintptr_t)out_b & 15) == 0 && ((uintptr_t)out & 15) == 0,
             "fg_chain_cell_step: 16-byte aligned rows");
  FG_REQUIRE(workspace_bytes >= fg_chain_cell_step_workspace(rows, hidden, bottleneck),
             "fg_chain_cell_step: workspace too small");
  const ChainPlan p = chain_plan(rows, hidden, bottleneck);
  float* x = (float*)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);
  float* parts = x + p.x;
  float* mid = parts + p.parts;
  hipStream_t s = (hipStream_t)stream;
  int rc = fg::chain_cell_norm(state, ld_state, fg::kF32, token, ld_token, token_dtype, rows, hidden, state_w, state_b,
                               token_w, token_b, eps, x, s);
  if (rc) return rc;
  // both projections as one product over the two halves of K
  const fg::F32Gemm first{x,          2 * hidden, 0, state_proj_w, hidden, 0, rows, bottleneck, 2 * hidden, 1,
                          token_proj_w, hidden};
  rc = fg::f32_gemm_parts(first, p.splits, parts, s);
  if (rc) return rc;
  const int64_t quads = (int64_t)rows * bottleneck / 4;
  hipLaunchKernelGGL(chain_mid_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, parts, p.splits, quads,
                     mid);
  rc = fg::check_launch("fg_chain_cell_step");
  if (rc) return rc;
  TileArgs a{};
  a.g = fg::F32Gemm{mid, bottleneck, 0, out_w, bottleneck, 0, rows, hidden, bottleneck, 1};
  a.out = out;
  a.state = state;
  a.ld_state = ld_state;
  a.bias = out_b;
  a.gate = gate;
  return launch_tiles(a, 1, true, s);
}

}  // extern "C"
