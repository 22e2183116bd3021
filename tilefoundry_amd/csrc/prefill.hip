// Prompt passes: hundreds to thousands of prompt rows through a layer at once.
//
// A decode step's kernels are made for at most 32 rows: a prompt taken through
// them reads every weight once per 32 tokens and every cached key once per row.
// Here a pass takes all its rows (up to 4,096, of one or several sequences)
// through each layer together:
//   k_gemm_panels    projections: weights in the skinny GEMMs' packed blocks,
//                    activations in panel order (panel.h), f32 partial sums or a
//                    SwiGLU epilogue
//   k_panel_qkv      q/k norm, RoPE, cache append
//   k_panel_attn     causal attention over the paged cache on the matrix cores
//   k_panel_add_norm residual add and the next RMSNorm
//   k_panel_swiglu   SwiGLU over K-split gate/up sums
// Rounding points are the HIR's (ref_src/model.py:125-234); attention's two
// products are exact, as the reference's own fast path takes them (T.gemm,
// examples/qwen3_1_7b-tilelang/fast/kernels.py:418-501).

#include <type_traits>

#include "host_common.h"
#include "panel.h"
#include "tf_decode.h"
#include "tf_hybrid.h"

using namespace tfd;
using namespace tfd_host;

namespace {

// One 16-row x 32-k block of packed weights: as loaded, and as a matrix-core
// operand (e4m3fn codes decode exactly to bf16; their row scale multiplies the sum).
template <bool kFp8>
struct PanelW {
  using Raw = u32x4;
  static __device__ __forceinline__ Raw load(const void* W, int64_t block, int lane) {
    return load16((const bf16*)W + block * 512 + lane * 8);
  }
  static __device__ __forceinline__ u32x4 value(const Raw& r) { return r; }
};
template <>
struct PanelW<true> {
  using Raw = u32x2;
  static __device__ __forceinline__ Raw load(const void* W, int64_t block, int lane) {
    return *(const __attribute__((address_space(1))) u32x2*)((const uint8_t*)W + block * 512 +
                                                             lane * 8);
  }
  static __device__ __forceinline__ u32x4 value(const Raw& r) { return fp8x8_to_bf16(r); }
};

// ---------------------------------------------------------------------------
// Y[m][n] = sum_k X[m][k] W[n][k] for M rows in panel order.  A block of four
// waves takes TM x 16 rows and 4 x TN x 16 columns over its K slice; a wave owns
// TN column tiles for all the block's rows.  The weights go straight from memory
// to the wave's registers (packed blocks are matrix-core operands as they lie,
// and no other wave of the block reads them), DB K steps ahead; the rows, which
// every wave reads, pass through LDS, KC steps at a time in two buffers.
//
// The weight is the A operand and the row the B operand, so a lane ends up with
// four consecutive columns of one row: a partial is one 16-byte store, and a
// SwiGLU's (gate, up) pairs sit in one lane.
//
// Bound: at thousands of rows the matrix cores and LDS (a wave reads eight row
// blocks per 32 matrix products), below 128 rows the weights' stream and LDS (every
// row block is read for each column tile).  At four column tiles a wave's registers
// are held to 256 so that two blocks share a compute unit: with one, 4,000 x 2048 x
// 12288 took 266 us.  Measured, weights cold (M x K x N): 4,000 x 2048 x 12288 178 us
// (1,130 TFLOP/s), 4,000 x 6144 x 2048 95 us (1,060); 91 x 2048 x 12288 17.0 us (3.0 TB/s
// of weights); 17 x 2048 x 4096 5.1 us.  The skinny GEMM took 126 launches for the 4,000
// rows, 15 us each for 2048 x 12288.
//
// grid: 8 x ceil(tiles / 8) blocks.  Consecutive tiles (eight row blocks by a
// few column blocks) go to one XCD, so that the operands its blocks share stay in
// its L2.
// ---------------------------------------------------------------------------
enum PanelEpi { kPanPartial = 0, kPanSwiglu = 1 };

template <int TM, int TN, int KC, int DB, int kEpi, bool kFp8 = false>
__global__ __launch_bounds__(kBlock, 2) void k_gemm_panels(const bf16* __restrict__ X,
                                                        const void* __restrict__ W, int M, int K,
                                                        int N, int slices,
                                                        const float* __restrict__ wscale,
                                                        void* __restrict__ out) {
  using WL = PanelW<kFp8>;
  constexpr int kPasses = KC * TM / 4;       // 16-byte loads per thread of one LDS chunk
  static_assert(DB % KC == 0 && TM % 2 == 0 && KC * TM % 4 == 0, "tile shape");
  __shared__ __align__(16) uint8_t xs[2][KC * TM * 1024];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int nm = (M + TM * 16 - 1) / (TM * 16);
  const int ntiles = (N + 15) / 16;
  const int nn = (ntiles + 4 * TN - 1) / (4 * TN);
  const int total = nm * nn * slices, per = (total + 7) / 8;
  const int g = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || g >= total) return;
  const int slice = g / (nm * nn), rest = g % (nm * nn);
  const int grp = rest / (8 * nn), within = rest % (8 * nn);
  const int gm = min(8, nm - grp * 8);
  const int mb = grp * 8 + within % gm, nb = within / gm;

  const int ksteps = K / 32;
  const int steps = ksteps / slices, s0 = slice * steps;
  const int panels = (M + 31) / 32;

  // the block's rows: this thread's 16-byte pieces of a chunk (2 KiB per panel
  // and step; a panel past the last one repeats it, its rows are not stored)
  const bf16* xsrc[kPasses];
#pragma unroll
  for (int q = 0; q < kPasses; ++q) {
    const int blk = q * 2 + (tid >> 7);
    const int st = blk / (TM / 2), pn = min(mb * (TM / 2) + blk % (TM / 2), panels - 1);
    xsrc[q] = X + ((int64_t)pn * ksteps + s0 + st) * 1024 + (tid & 127) * 8;
  }
  int64_t wt[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t)
    wt[t] = (int64_t)min((nb * 4 + wave) * TN + t, ntiles - 1) * ksteps + s0;

  u32x4 xr[kPasses];
  typename WL::Raw b[DB][TN];
  auto load_x = [&](int step) {
#pragma unroll
    for (int q = 0; q < kPasses; ++q) xr[q] = load16(xsrc[q] + (int64_t)step * 1024);
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int q = 0; q < kPasses; ++q)
      *reinterpret_cast<u32x4*>(&xs[buf][q * 4096 + tid * 16]) = xr[q];
  };
  load_x(0);
#pragma unroll
  for (int u = 0; u < DB; ++u)
#pragma unroll
    for (int t = 0; t < TN; ++t) b[u][t] = WL::load(W, wt[t] + u, lane);
  f32x4 c[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int t = 0; t < TN; ++t) c[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  stage(0);
  __syncthreads();
  int cur = 0;
  // DB steps from step k0 on; with kMore every slot is refilled behind its use
  // and the next chunk of rows follows (the last body has nothing ahead)
  auto body = [&](int k0, auto more) {
#pragma unroll
    for (int u0 = 0; u0 < DB; u0 += KC) {
      constexpr bool kMore = decltype(more)::value;
      const bool next = kMore || u0 + KC < DB;
      if (next) load_x(k0 + u0 + KC);
#pragma unroll
      for (int v = 0; v < KC; ++v) {
        const int u = u0 + v;
        u32x4 a[TM];
#pragma unroll
        for (int m = 0; m < TM; ++m)
          a[m] = *reinterpret_cast<const u32x4*>(&xs[cur][(v * TM + m) * 1024 + lane * 16]);
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          const u32x4 w = WL::value(b[u][t]);
#pragma unroll
          for (int m = 0; m < TM; ++m) c[m][t] = mfma(w, a[m], c[m][t]);
        }
        if (kMore)
#pragma unroll
          for (int t = 0; t < TN; ++t)
            b[u][t] = WL::load(W, wt[t] + k0 + u + DB, lane);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (next) {
        cur ^= 1;
        stage(cur);
        __syncthreads();
      }
    }
  };
  for (int k0 = 0; k0 + DB < steps; k0 += DB) body(k0, std::true_type{});
  body(steps - DB, std::false_type{});

  const int r = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int row = (mb * TM + m) * 16 + r;
    if (row >= M) continue;
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      const int n = ((nb * 4 + wave) * TN + t) * 16 + 4 * kq;
      if (n >= N) continue;
      if (kEpi == kPanSwiglu) {
        const float g0 = rbf(c[m][t].x), u0 = rbf(c[m][t].y);
        const float g1 = rbf(c[m][t].z), u1 = rbf(c[m][t].w);
        *reinterpret_cast<uint32_t*>((bf16*)out + panel_off(row, n / 2, N / 2)) =
            pack2(rbf(silu_f(g0)) * u0, rbf(silu_f(g1)) * u1);
      } else {
        f32x4 y = c[m][t];
        if (kFp8) y *= *reinterpret_cast<const f32x4*>(wscale + n);
        *reinterpret_cast<f32x4*>((float*)out + ((int64_t)slice * M + row) * N + n) = y;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// After the q/k/v projection (model.py:172-190, 339-352): per head RMSNorm and
// RoPE of the queries (times the score scale) and keys, keys and values appended
// at the row's position of its sequence's pages.  A wave per (row, head vector).
// ---------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(kBlock) void k_panel_qkv(
    const float* __restrict__ part, int slices, int M, int heads, int kv_heads,
    const bf16* __restrict__ gq, const bf16* __restrict__ gk, const bf16* __restrict__ cos_t,
    const bf16* __restrict__ sin_t, int rope_rows, const int* __restrict__ pos,
    const int* __restrict__ seq, const int* __restrict__ page_table, int max_pages,
    bf16* __restrict__ kpool, bf16* __restrict__ vpool, int num_pages, float scale, float eps,
    bf16* __restrict__ q_out, int* err) {
  constexpr int kHalf = D / 2;
  const int m = blockIdx.x, lane = threadIdx.x & (kWave - 1);
  const int v = blockIdx.y * kWavesPerBlock + threadIdx.x / kWave;
  if (v >= heads + 2 * kv_heads) return;
  const int N = (heads + 2 * kv_heads) * D;
  const int P = pos[m];
  const bool isq = v < heads, isv = v >= heads + kv_heads;
  if (P < 0 || P >= rope_rows || P >= max_pages * kPage) {
    if (lane == 0) raise_error(err, kErrPosRange);
    return;
  }
  const bool act = lane < kHalf;
  const int li = act ? lane : 0;
  const float* x = part + (int64_t)m * N + v * D;
  const int64_t stride = (int64_t)M * N;
  const float x0 = act ? slice_sum(x + li, stride, slices) : 0.f;
  const float x1 = act ? slice_sum(x + li + kHalf, stride, slices) : 0.f;
  float o0 = x0, o1 = x1;
  if (!isv) {
    const bf16* gam = isq ? gq : gk;
    float ss = x0 * x0;
    ss += x1 * x1;
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / (float)D + eps);
    const int64_t row = (int64_t)P * D;
    const float n0 = rbf(rbf(x0 * r) * bf2f(gam[li]));
    const float n1 = rbf(rbf(x1 * r) * bf2f(gam[li + kHalf]));
    o0 = rbf(n0 * bf2f(cos_t[row + li]) + (-n1) * bf2f(sin_t[row + li]));
    o1 = rbf(n1 * bf2f(cos_t[row + li + kHalf]) + n0 * bf2f(sin_t[row + li + kHalf]));
  }
  if (!act) return;
  if (isq) {
    bf16* q = q_out + ((int64_t)m * heads + v) * D;
    q[li] = f2bf(o0 * scale);
    q[li + kHalf] = f2bf(o1 * scale);
    return;
  }
  const int page = page_table[(int64_t)seq[m] * max_pages + P / kPage];
  if (page < 0 || page >= num_pages) {
    if (lane == 0) raise_error(err, kErrPageRange);
    return;
  }
  const int h = isv ? v - heads - kv_heads : v - heads;
  bf16* pool = isv ? vpool : kpool;
  bf16* o = pool + (((int64_t)page * kv_heads + h) * kPage + P % kPage) * D;
  o[li] = f2bf(o0);
  o[li + kHalf] = f2bf(o1);
}

// ---------------------------------------------------------------------------
// The hybrids' attention layers before their scores.  Granite (granite model.py:
// 310-340): queries, keys and values as projected.  Qwen3.5 (torch_ref.py:335-395):
// per-head RMSNorm and rotate-half RoPE on the first `rot` dims in f32, the queries
// scaled; the row's own score q . k of its unrounded key; the output gates apart.
// A block per (row, kv head).
// ---------------------------------------------------------------------------
template <int D, int G, bool kF32>
__global__ __launch_bounds__(kBlock) void k_panel_gqa_append(
    const bf16* __restrict__ proj, int ldp, int heads, int kv_heads, const bf16* __restrict__ gq,
    const bf16* __restrict__ gk, const bf16* __restrict__ cos_t, const bf16* __restrict__ sin_t,
    int rope_rows, int rot, const int* __restrict__ pos, const int* __restrict__ seq,
    const int* __restrict__ page_table, int max_pages, bf16* __restrict__ kpool,
    bf16* __restrict__ vpool, int num_pages, float scale, float eps, void* __restrict__ q_out,
    bf16* __restrict__ gate_out, float* __restrict__ self_s, int* err) {
  constexpr int kPer = D / kWave;
  __shared__ float x_s[G + 1][D];
  const int m = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  const int P = pos[m];
  if (P < 0 || P >= max_pages * kPage || (kF32 && P >= rope_rows)) {
    if (tid == 0) raise_error(err, kErrPosRange);
    return;
  }
  const int page = page_table[(int64_t)seq[m] * max_pages + P / kPage];
  const bool page_ok = page >= 0 && page < num_pages;
  if (!page_ok && tid == 0) raise_error(err, kErrPageRange);
  const bf16* row = proj + (int64_t)m * ldp;
  const int qw = kF32 ? 2 * D : D;           // a query head, and its gate
  const bf16* krow = row + (int64_t)heads * qw + h * D;
  const bf16* vrow = krow + (int64_t)kv_heads * D;
  const int64_t at = (((int64_t)(page_ok ? page : 0) * kv_heads + h) * kPage + P % kPage) * D;
  if (!kF32) {
    for (int i = tid; i < G * D / 8; i += kBlock)
      *reinterpret_cast<u32x4*>((bf16*)q_out + ((int64_t)m * heads + h * G) * D + i * 8) =
          load16(row + (int64_t)h * G * D + i * 8);
    if (page_ok && tid < D / 8) {
      *reinterpret_cast<u32x4*>(kpool + at + tid * 8) = load16(krow + tid * 8);
      *reinterpret_cast<u32x4*>(vpool + at + tid * 8) = load16(vrow + tid * 8);
    }
    return;
  }
  for (int r = wave; r < G + 1; r += kWavesPerBlock) {
    const bf16* src = r < G ? row + (int64_t)(h * G + r) * qw : krow;
    const bf16* gam = r < G ? gq : gk;
    float x[kPer], ss = 0.f;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      x[i] = bf2f(src[lane + kWave * i]);
      ss += x[i] * x[i];
    }
    ss = wave_sum(ss);
    const float rs = rsqrtf(ss / (float)D + eps);
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      x_s[r][lane + kWave * i] = x[i] * rs * bf2f(gam[lane + kWave * i]);
  }
  __syncthreads();
  const bf16* cs = cos_t + (int64_t)P * rot;
  const bf16* sn = sin_t + (int64_t)P * rot;
  float kv[kPer], y[kPer];
  auto rope = [&](int r, float (&o)[kPer]) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int d = lane + kWave * i;
      const float v = x_s[r][d];
      if (d < rot) {
        const float partner = d < rot / 2 ? -x_s[r][d + rot / 2] : x_s[r][d - rot / 2];
        o[i] = v * bf2f(cs[d]) + partner * bf2f(sn[d]);
      } else {
        o[i] = v;
      }
    }
  };
  rope(G, kv);
  if (wave == 0 && page_ok) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      kpool[at + lane + kWave * i] = f2bf(kv[i]);
      vpool[at + lane + kWave * i] = vrow[lane + kWave * i];
    }
  }
  for (int r = wave; r < G; r += kWavesPerBlock) {
    rope(r, y);
    const int64_t qh = (int64_t)m * heads + h * G + r;
    float a = 0.f;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      y[i] *= scale;
      a += y[i] * kv[i];
      ((float*)q_out)[qh * D + lane + kWave * i] = y[i];
      gate_out[qh * D + lane + kWave * i] = row[(int64_t)(h * G + r) * qw + D + lane + kWave * i];
    }
    a = wave_sum(a);
    if (lane == 0) self_s[qh] = a;
  }
}

// ---------------------------------------------------------------------------
// Causal attention of a prompt pass (model.py:190-212) over the paged cache,
// which already holds the pass's own keys and values.
//
// A block takes one tile of consecutive rows of a sequence (64 CT / G of them) and
// one kv head: 64 CT (query head, row) columns, 16 CT per wave, past the context in
// tiles of 64 positions.  S^T = K Q^T puts four consecutive positions of one
// column in a lane; packed, that is the B operand of O^T = V^T P^T as it stands
// if V^T's positions are stored in the same order, so the probabilities never
// leave their lane.  K and V tiles are read once per block, prefetched into
// registers while the tile before is used, V transposed on its way into LDS.
//
// Bound: one wave's chain through a tile (LDS reads, products, softmax, products) with
// three waves per SIMD to cover it; of the busy cycles 45% are VALU, 18% matrix cores
// and a third LDS.  4,000 rows take 141 us a layer, eight prompts of 88-700 tokens 27,
// 91 rows 8.7.  What mattered: LDS in operand order (row-major tiles spent three
// quarters of their LDS cycles in bank conflicts: 213, 35 and 10.6 us); 16 columns a
// wave, whose registers let three blocks share a compute unit and whose tiles are half as
// long (32 columns and two blocks: 164, 33 and 11.9); page ids read a tile ahead, and a
// rescale only when a maximum moves (302 us before both, with 32 columns).
//
// The decode kernels it takes the place of re-read every cached key for each row: a
// 4,001-token prompt through eight layers took 123.0 ms, here 4.88 ms; 91 tokens
// 2.18 and 0.99 ms, eight prompts of 88-700 tokens 51.4-71 and 4.07 ms (each with
// one decode step).
//
// Rounding: s = bf16(q . k), p = bf16(exp(bf16(s - m))) against the running
// maximum m (the HIR's final maximum from the tile that holds it on; sums and
// outputs are rescaled in f32), the row's own key as its own term at the end
// (model.py:198-212).
// ---------------------------------------------------------------------------
struct PanelTile {
  int row0, rows, seq, pos0;
};

// bf16(exp(x)) for bf16 x <= 0, before its rounding: 2^(x log2 e) on the transcendental
// unit, off by at most |x| 2^-24 + 2^-22 of the value.  Rounded to bf16 it is the correctly
// rounded exp(x) for every bf16 x whose result is a normal number, as expf's is
// (test_panel_attn_probabilities_are_exactly_rounded takes all 17,070 of them); where the
// value itself is summed in f32 it would not be, and those policies call expf (190 rows
// of Granite 12.2 us, 10.0 with this).
__device__ __forceinline__ float exp_for_bf16(float x) {
  return __builtin_amdgcn_exp2f(x * 1.44269504088896340736f);
}

// Eight f32 values as three bf16 operands: each takes the next eight bits.
__device__ __forceinline__ void split3(const f32x4& a, const f32x4& b, u32x4 (&o)[3]) {
  float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    o[i] = u32x4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] -= rbf(v[e]);
  }
}

// kPol: the models' arithmetics.  kAttnDense as above.  kAttnGranite: s = bf16(q . k)
// times the scale in f32, p = bf16(exp(s - m)) with its sum in f32 (granite
// model.py:310-366; the cache holds the row's own key exactly).  kAttnF32 (Qwen3.5):
// f32 queries, scores and probabilities; a matrix-core operand is 8 bits wide, so a
// query and a probability are each three operands whose sum is the f32 value to its
// last bit, and the row's own score (of its unrounded key) comes from `self_s`; the
// output is gated by sigmoid(gate).  CT: 16-column tiles per wave.
enum PanelAttnPolicy { kAttnDense = 0, kAttnGranite = 1, kAttnF32 = 2 };

template <int D, int G, int CT, int kPol>
__global__ __launch_bounds__(kBlock, D <= 128 ? (CT == 1 ? 3 : 2) : 1) void k_panel_attn(
    const void* __restrict__ q_in, const PanelTile* __restrict__ tiles, int heads, int kv_heads,
    const int* __restrict__ page_table, int max_pages, const bf16* __restrict__ kpool,
    const bf16* __restrict__ vpool, int num_pages, float scale,
    const float* __restrict__ self_s, const bf16* __restrict__ gate, bf16* __restrict__ out,
    int* err) {
  constexpr int QT = 64 * CT / G;            // rows of a tile
  constexpr int kQ = kPol == kAttnF32 ? 3 : 1;   // operands per query / probability
  constexpr int DS = D / 32, DT = D / 16;    // k steps of q.k, 16-row tiles of V^T
  constexpr int kCh = D / 8;                 // 16-byte chunks of a head row
  constexpr int kKPass = 64 * kCh / kBlock;  // K loads per thread and tile
  constexpr int kVThr = 16 * kCh;            // pieces of V: 4 positions x 8 dims each
  constexpr int kVPass = kVThr > kBlock ? kVThr / kBlock : 1;
  // Both tiles lie in operand order, 1 KiB per 16 x 32 block.  Lane l's 16 bytes are at
  // l ^ l / 16 ^ 4 (step % 4) in K and at l ^ (block % 8) in V^T, so that the lanes of a
  // write (pieces of a few rows) fall on as many banks as those of a read.
  __shared__ __align__(16) uint8_t ks[64 * D * 2];
  __shared__ __align__(16) uint8_t vt[64 * D * 2];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int r = lane & 15, kq = lane >> 4;
  const int h = blockIdx.x;
  const PanelTile tl = tiles[blockIdx.y];
  const int last = tl.pos0 + tl.rows - 1;    // the last row's position
  if (tl.pos0 < 0 || last >= max_pages * kPage) {
    if (tid == 0) raise_error(err, kErrPosRange);
    return;
  }
  const int* pt = page_table + (int64_t)tl.seq * max_pages;
  bool page_bad = false;
  // entries past the last row's page need not be set (a table may be filled as the
  // sequence grows): the tiles' read-ahead re-reads that one in their place
  auto page_at = [&](int i) {
    const int pg = pt[min(i, last / kPage)];
    const bool ok = pg >= 0 && pg < num_pages;
    page_bad |= !ok;
    return ok ? pg : 0;
  };

  // this wave's columns: c = 16 (CT wave + ct) + r -> query head c / QT, row c % QT
  u32x4 qf[CT][DS][kQ];
  int qpos[CT];
  float own[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int c = 16 * (CT * wave + ct) + r;
    const int row = min(c % QT, tl.rows - 1);
    qpos[ct] = tl.pos0 + row;
    const int64_t qh = (int64_t)(tl.row0 + row) * heads + h * G + c / QT;
    own[ct] = kPol == kAttnF32 ? self_s[qh] : 0.f;
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const int64_t at = qh * D + 32 * s + 8 * kq;
      if constexpr (kPol == kAttnF32) {
        const f32x4* qp = reinterpret_cast<const f32x4*>((const float*)q_in + at);
        split3(qp[0], qp[1], qf[ct][s]);
      } else {
        qf[ct][s][0] = load16((const bf16*)q_in + at);
      }
    }
  }

  u32x4 kr[kKPass], vr[kVPass][4];
  const int vc = tid % kCh;                  // V: 8-dim chunk; position group tid / kCh + ..
  // lane l holds the id of a tile's page l % 4, read a tile ahead of the loads that
  // need it (a page-table read in front of every load made a tile five round trips)
  auto v_at = [](int i) { return 32 * (i >> 3) + 16 * (i & 1) + 4 * ((i >> 1) & 3); };
  auto load_tile = [&](int j0, int pid) {
#pragma unroll
    for (int i = 0; i < kKPass; ++i) {
      const int c = tid + i * kBlock, p = c / kCh;
      const int page = __builtin_amdgcn_readlane(pid, (i * kBlock + wave * kWave) / kCh / kPage);
      kr[i] = load16(kpool + (((int64_t)page * kv_heads + h) * kPage + p % kPage) * D +
                     (c % kCh) * 8);
    }
    if (kVThr >= kBlock || tid < kVThr) {
#pragma unroll
      for (int g = 0; g < kVPass; ++g) {
        const int at = v_at((tid + g * kBlock) / kCh), p = j0 + at;
        const int page = __shfl(pid, at / kPage, kWave);
        const bf16* v0 = vpool + (((int64_t)page * kv_heads + h) * kPage + p % kPage) * D + vc * 8;
        // positions past the last row hold anything (their p is 0): their V reads as 0
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const u32x4 v = load16(v0 + i * D);
          vr[g][i] = p + i <= last ? v : u32x4{0u, 0u, 0u, 0u};
        }
      }
    }
  };
  auto stage_tile = [&]() {
#pragma unroll
    for (int i = 0; i < kKPass; ++i) {
      const int c = tid + i * kBlock;
      const int p = c / kCh, s = c % kCh / 4, l = 16 * (c % 4) + p % 16;
      *reinterpret_cast<u32x4*>(&ks[(p / 16 * DS + s) * 1024 + (l ^ (c % kCh & 15)) * 16]) = kr[i];
    }
    if (kVThr >= kBlock || tid < kVThr) {
      // positions in the order the probabilities come in: within 32, position
      // 16 t + 4 g + e sits at 8 g + 4 t + e
#pragma unroll
      for (int g = 0; g < kVPass; ++g) {
        const int vg = (tid + g * kBlock) / kCh;
        const int at = (vc / 2 * 2 + (vg >> 3)) * 1024 + 8 * (vg & 1);
        auto word = [&](int i, int d) {
          const u32x4 v = vr[g][i];
          return (d >> 1) == 0 ? v.x : (d >> 1) == 1 ? v.y : (d >> 1) == 2 ? v.z : v.w;
        };
#pragma unroll
        for (int d = 0; d < 8; ++d) {
          const uint32_t sel = (d & 1) ? 0x07060302u : 0x05040100u;
          const int l = 16 * ((vg >> 1) & 3) + 8 * (vc % 2) + d;
          *reinterpret_cast<u32x2*>(&vt[at + (l ^ (vc / 2 & 7)) * 16]) =
              u32x2{__builtin_amdgcn_perm(word(1, d), word(0, d), sel),
                    __builtin_amdgcn_perm(word(3, d), word(2, d), sel)};
        }
      }
    }
  };

  f32x4 o[DT][CT];
  float mx[CT], sum[CT], self[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    mx[ct] = kPanelNegInf;
    self[ct] = sum[ct] = 0.f;                // self: the own key's lane of a column's four
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  int pid = page_at(lane & 3);
  int own_page[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) own_page[ct] = kPol == kAttnDense ? page_at(qpos[ct] / kPage) : 0;
  load_tile(0, pid);
  pid = page_at(4 + (lane & 3));
  for (int j0 = 0; j0 <= last; j0 += 64) {
    stage_tile();
    __syncthreads();
    if (j0 + 64 <= last) {
      load_tile(j0 + 64, pid);
      pid = page_at(j0 / kPage + 8 + (lane & 3));
    }
    f32x4 st[4][CT];
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) st[p][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const u32x4 kf =
            *reinterpret_cast<const u32x4*>(&ks[(p * DS + s) * 1024 + (lane ^ kq ^ 4 * (s & 3)) * 16]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int i = kQ - 1; i >= 0; --i) st[p][ct] = mfma(kf, qf[ct][s][i], st[p][ct]);
      }
    u32x4 pb[2][CT][kQ];                     // the packed probabilities of 32 positions each
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int before = qpos[ct] - j0 - 4 * kq;   // position 16 p + e is past: 16 p + e < before
      float tm = kPanelNegInf;
      auto score = [&](float v) {
        return kPol == kAttnDense ? rbf(v) : kPol == kAttnGranite ? rbf(v) * scale : v;
      };
      if (j0 + 64 > tl.pos0) {               // a tile that reaches the diagonal
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float s = score(st[p][ct][e]);
            if (kPol == kAttnF32 && 16 * p + e == before) s = own[ct];
            if (16 * p + e == before) self[ct] = s;
            if (16 * p + e <= before) tm = fmaxf(tm, s);
            // dense: the own key is a term of its own, added at the end
            st[p][ct][e] = 16 * p + e < before + (kPol == kAttnDense ? 0 : 1) ? s : kPanelNegInf;
          }
      } else {
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            st[p][ct][e] = score(st[p][ct][e]);
            tm = fmaxf(tm, st[p][ct][e]);
          }
      }
      float lo, hi;
      pair16(tm, lo, hi);
      tm = fmaxf(lo, hi);
      pair32(tm, lo, hi);
      tm = fmaxf(lo, hi);
      const float m1 = fmaxf(mx[ct], tm);
      // once the tiles that hold the maxima are past, no column's maximum moves
      if (__any(m1 != mx[ct])) {
        const float alpha = expf(mx[ct] - m1);
        mx[ct] = m1;
        sum[ct] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[dt][ct][e] *= alpha;
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        f32x4 pe[2];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = st[2 * kk + p][ct][e] - m1;
            pe[p][e] = kPol == kAttnDense ? exp_for_bf16(rbf(x)) : expf(x);
            if (kPol != kAttnDense) sum[ct] += pe[p][e];
          }
        if constexpr (kPol == kAttnF32) {
          split3(pe[0], pe[1], pb[kk][ct]);
        } else {
          pb[kk][ct][0] = u32x4{pack2(pe[0].x, pe[0].y), pack2(pe[0].z, pe[0].w),
                                pack2(pe[1].x, pe[1].y), pack2(pe[1].z, pe[1].w)};
          if (kPol == kAttnDense) {          // the sum of the rounded probabilities
            const u32x4 w = pb[kk][ct][0];
            sum[ct] = dot2(w.x, 0x3f803f80u, sum[ct]);
            sum[ct] = dot2(w.y, 0x3f803f80u, sum[ct]);
            sum[ct] = dot2(w.z, 0x3f803f80u, sum[ct]);
            sum[ct] = dot2(w.w, 0x3f803f80u, sum[ct]);
          }
        }
      }
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const u32x4 vf =
            *reinterpret_cast<const u32x4*>(&vt[(dt * 2 + kk) * 1024 + (lane ^ (dt & 7)) * 16]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int i = kQ - 1; i >= 0; --i) o[dt][ct] = mfma(vf, pb[kk][ct][i], o[dt][ct]);
      }
    __syncthreads();
  }

  // A product takes every position of a tile into every row: an infinite or NaN value
  // past a row reaches it as 0 * inf, and the parts of a split infinite value cancel.
  // Either leaves a NaN, so a wave that holds one takes its columns again position by
  // position, each from its own past alone, as a step's lanes do (4,000 rows that all see
  // an infinity: 12 ms a layer, bound by one position's loads after another's; 15 when the
  // decode kernels took them).
  float probe = 0.f;
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    probe = fmaf(sum[ct], 0.f, probe);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 4; ++e) probe = fmaf(o[dt][ct][e], 0.f, probe);
  }
  if (__any(probe != 0.f)) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int c = 16 * (CT * wave + ct) + r;
      const int64_t q0 =
          ((int64_t)(tl.row0 + min(c % QT, tl.rows - 1)) * heads + h * G + c / QT) * D + 8 * kq;
      // the score of position p, the same in a column's four lanes
      auto score_of = [&](int p) {
        const bf16* kp =
            kpool + (((int64_t)page_at(p / kPage) * kv_heads + h) * kPage + p % kPage) * D + 8 * kq;
        float a = 0.f, lo, hi;
#pragma unroll 1
        for (int s = 0; s < DS; ++s) {
          const u32x4 w = load16(kp + 32 * s);
          if constexpr (kPol == kAttnF32) {
            const f32x4* qp = reinterpret_cast<const f32x4*>((const float*)q_in + q0 + 32 * s);
            const f32x4 x = qp[0], y = qp[1];
            a = fmaf(x.x, bf_lo(w.x), fmaf(x.y, bf_hi(w.x), a));
            a = fmaf(x.z, bf_lo(w.y), fmaf(x.w, bf_hi(w.y), a));
            a = fmaf(y.x, bf_lo(w.z), fmaf(y.y, bf_hi(w.z), a));
            a = fmaf(y.z, bf_lo(w.w), fmaf(y.w, bf_hi(w.w), a));
          } else {
            a = dot8(w, load16((const bf16*)q_in + q0 + 32 * s), a);
          }
        }
        pair16(a, lo, hi);
        a = lo + hi;
        pair32(a, lo, hi);
        a = lo + hi;
        if (kPol == kAttnF32) return p == qpos[ct] ? own[ct] : a;
        return kPol == kAttnDense ? rbf(a) : rbf(a) * scale;
      };
      float m = kPanelNegInf, l = 0.f, sn = 0.f;
#pragma unroll 1
      for (int p = 0; p <= last; ++p) {
        const float s = score_of(p);
        if (p <= qpos[ct]) m = fmaxf(m, s);
        if (p == qpos[ct]) sn = s;
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int p = 0; p <= last; ++p) {
        const float x = score_of(p) - m;
        if (p >= qpos[ct] + (kPol == kAttnDense ? 0 : 1)) continue;
        float w = expf(kPol == kAttnDense ? rbf(x) : x);
        if (kPol == kAttnDense) w = rbf(w);
        l += w;
        if (kPol == kAttnGranite) w = rbf(w);
        const bf16* vp = vpool +
            (((int64_t)page_at(p / kPage) * kv_heads + h) * kPage + p % kPage) * D + 4 * kq;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const u32x2 vw = *reinterpret_cast<const u32x2*>(vp + 16 * dt);
          o[dt][ct].x = fmaf(w, bf_lo(vw.x), o[dt][ct].x);
          o[dt][ct].y = fmaf(w, bf_hi(vw.x), o[dt][ct].y);
          o[dt][ct].z = fmaf(w, bf_lo(vw.y), o[dt][ct].z);
          o[dt][ct].w = fmaf(w, bf_hi(vw.y), o[dt][ct].w);
        }
      }
      mx[ct] = m;
      sum[ct] = kq == 0 ? l : 0.f;
      self[ct] = kq == 0 ? sn : 0.f;
    }
  }

#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int c = 16 * (CT * wave + ct) + r;
    float lo, hi, l = sum[ct], sn = self[ct];
    pair16(l, lo, hi);
    l = lo + hi;
    pair32(l, lo, hi);
    l = lo + hi;
    pair16(sn, lo, hi);                      // (a NaN of the own key stays one)
    sn = lo + hi;
    pair32(sn, lo, hi);
    sn = lo + hi;
    const float pn = rbf(expf(rbf(sn - mx[ct])));
    const float inv = 1.f / (kPol == kAttnDense ? rbf(rbf(l) + pn) : l);
    const int P = qpos[ct];
    const bf16* vrow = vpool + (((int64_t)own_page[ct] * kv_heads + h) * kPage + P % kPage) * D;
    const int row = c % QT;
    const int64_t m = tl.row0 + row;
    const int k0 = (h * G + c / QT) * D;
    const bool on = row < tl.rows;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      float y[4];
      if constexpr (kPol == kAttnDense) {
        const u32x2 vw = *reinterpret_cast<const u32x2*>(vrow + 16 * dt + 4 * kq);
        const float vn[4] = {bf_lo(vw.x), bf_hi(vw.x), bf_lo(vw.y), bf_hi(vw.y)};
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = rbf(rbf(o[dt][ct][e]) + rbf(pn * vn[e])) * inv;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = o[dt][ct][e] * inv;
      }
      if constexpr (kPol == kAttnF32) {
        const u32x2 gw = *reinterpret_cast<const u32x2*>(
            gate + (int64_t)(on ? m : tl.row0) * heads * D + k0 + 16 * dt + 4 * kq);
        const float gn[4] = {bf_lo(gw.x), bf_hi(gw.x), bf_lo(gw.y), bf_hi(gw.y)};
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] *= 1.f / (1.f + expf(-gn[e]));
      }
      if (on)
        *reinterpret_cast<u32x2*>(out + panel_off(m, k0 + 16 * dt + 4 * kq, heads * D)) =
            u32x2{pack2(y[0], y[1]), pack2(y[2], y[3])};
    }
  }
  if (page_bad) raise_error(err, kErrPageRange);
}

// ---------------------------------------------------------------------------
// h = resid + bf16(sum of the slices), and the next RMSNorm of h in panel order
// (model.py:125-137, 213-225).  A block per row; slices 0: h = resid as it is.
// Bound by one load's latency at few rows: four slices are requested together
// (32 x 2048, 4 slices: 4.6 us, 5.0 with one slice at a time).
// ---------------------------------------------------------------------------
template <int kCh>
__global__ __launch_bounds__(kBlock) void k_panel_add_norm(
    const float* __restrict__ part, int slices, const bf16* resid, bf16* h_out,
    const bf16* __restrict__ gamma, bf16* __restrict__ norm_out, int M, int n, float eps) {
  __shared__ float red[kWavesPerBlock];
  const int64_t m = blockIdx.x;
  const int tid = threadIdx.x, nch = n / 8;
  u32x4 x[kCh], gm[kCh];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < kCh; ++i) {
    const int c = min(tid + i * kBlock, nch - 1);
    const u32x4 rv = load16(resid + m * n + c * 8);
    gm[i] = load16(gamma + c * 8);
    float y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < slices; s0 += 4) {       // four slices' loads in flight
      f32x4 lo[4], hi[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int s = min(s0 + j, slices - 1);
        const f32x4* p = reinterpret_cast<const f32x4*>(part + ((int64_t)s * M + m) * n + c * 8);
        lo[j] = p[0];
        hi[j] = p[1];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (s0 + j < slices) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            y[e] += lo[j][e];
            y[e + 4] += hi[j][e];
          }
        }
    }
    const uint32_t w[4] = {rv.x, rv.y, rv.z, rv.w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = slices ? pack2(bf_lo(w[e]) + rbf(y[2 * e]), bf_hi(w[e]) + rbf(y[2 * e + 1])) : w[e];
    x[i] = u32x4{o[0], o[1], o[2], o[3]};
    if (tid + i * kBlock < nch) {
      if (h_out) *reinterpret_cast<u32x4*>(h_out + m * n + c * 8) = x[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = bf_lo(o[e]), b = bf_hi(o[e]);
        ss += a * a;
        ss += b * b;
      }
    }
  }
  ss = wave_sum(ss);
  if ((tid & (kWave - 1)) == 0) red[tid / kWave] = ss;
  __syncthreads();
  ss = red[0];
  for (int w = 1; w < kWavesPerBlock; ++w) ss += red[w];
  const float rs = 1.0f / sqrtf(ss / (float)n + eps);
#pragma unroll
  for (int i = 0; i < kCh; ++i) {
    const int c = tid + i * kBlock;
    if (c < nch)
      *reinterpret_cast<u32x4*>(norm_out + panel_off(m, c * 8, n)) =
          rms_norm_chunk(x[i], gm[i], rs);
  }
}

// SwiGLU of K-split gate/up sums: (gate, up) pairs in adjacent columns.
__global__ __launch_bounds__(kBlock) void k_panel_swiglu(const float* __restrict__ part,
                                                         int slices, int M, int N,
                                                         bf16* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;   // four columns each
  const int per = N / 4;
  if (i >= (int64_t)M * per) return;
  const int64_t m = i / per;
  const int n = (int)(i % per) * 4;
  f32x4 a = *reinterpret_cast<const f32x4*>(part + m * N + n);
  for (int s = 1; s < slices; ++s)
    a += *reinterpret_cast<const f32x4*>(part + ((int64_t)s * M + m) * N + n);
  const float h0 = rbf(silu_f(rbf(a.x))) * rbf(a.y), h1 = rbf(silu_f(rbf(a.z))) * rbf(a.w);
  *reinterpret_cast<uint32_t*>(out + panel_off(m, n / 2, N / 2)) = pack2(h0, h1);
}

// ---------------------------------------------------------------------------
// Tile shape and K slices of a panel GEMM: 16-row tiles per block (every row up
// to 128, else 128), column tiles per wave (more of them read LDS less per product;
// fewer make more blocks), and as few K slices as give most compute units a block --
// nine tenths of them where K is deep and a block runs long.  Measured (us), the rule's
// choice against the nearest others: 250 x 2048 x 4096 11.3 (2 tiles, 4 slices), 12.3 (1,
// 2), 13.5 (2, 2); 250 x 6144 x 2048 13.4 (2, 8), 18.2 (1, 3); 1,000 x 2048 x 12288 58.8
// (2, 1), 63.0 (4, 1); 1,300 x 2048 x 12288 86.1 (4, 1), 87.3 (2, 1); 4,000 x 2048 x 12288
// 177.6 (4, 1), 225 (2, 1).
// ---------------------------------------------------------------------------
struct PanelPlan {
  int tm, tn, slices;
};

PanelPlan panel_plan(int M, int K, int N) {
  PanelPlan p;
  const int cus = compute_units(), ntiles = (N + 15) / 16, ksteps = K / 32;
  p.tm = M <= 128 ? (M + 31) / 32 * 2 : 8;
  const int nm = (M + p.tm * 16 - 1) / (p.tm * 16);
  auto blocks = [&](int tn) { return (int64_t)nm * ((ntiles + 4 * tn - 1) / (4 * tn)); };
  p.tn = M <= 128 ? 1 : M <= 1024 ? 2 : 4;
  p.slices = 1;
  static const int kTry[] = {1, 2, 3, 4, 6, 8, 12};
  for (int s : kTry) {
    if (ksteps % s || (ksteps / s) % 8) continue;
    p.slices = s;
    if (blocks(p.tn) * s * 10 >= cus * (K > 4096 ? 9 : 7)) break;
  }
  return p;
}

}  // namespace

extern "C" {

int tfd_panel_gemm_slices(int M, int K, int N) {
  if (M <= 0 || K <= 0 || K % 256 || N <= 0 || N % 4) return 0;
  return panel_plan(M, K, N).slices;
}

static int panel_gemm(const void* x, const void* w, const float* wscale, int M, int K, int N,
                      int epilogue, void* out, void* stream) {
  if (!x || !w || !out) return fail(kBadArg, "panel_gemm: null pointer");
  if (M <= 0 || K <= 0 || K % 256 || N <= 0 || N % 4)
    return fail(kBadShape, "panel_gemm: M=%d K=%d (multiple of 256) N=%d (multiple of 4)", M, K, N);
  const PanelPlan p = panel_plan(M, K, N);
  if (epilogue == TFD_PANEL_SWIGLU ? ((N / 2) % 32 || p.slices != 1)
                                   : epilogue != TFD_PANEL_PARTIAL)
    return fail(kBadShape, "panel_gemm: epilogue %d with N=%d, %d slices", epilogue, N, p.slices);
  const int nm = (M + p.tm * 16 - 1) / (p.tm * 16), ntiles = (N + 15) / 16;
  const int64_t total = (int64_t)nm * ((ntiles + 4 * p.tn - 1) / (4 * p.tn)) * p.slices;
  const dim3 grid((unsigned)((total + 7) / 8 * 8));
  const int steps = K / 32 / p.slices;
  auto s = (hipStream_t)stream;
#define TFD_PANEL_RUN(TM, TN, KC, DB)                                                           \
  if (wscale)                                                                                   \
    hipLaunchKernelGGL((k_gemm_panels<TM, TN, KC, DB, kPanPartial, true>), grid, dim3(kBlock),  \
                       0, s, (const bf16*)x, w, M, K, N, p.slices, wscale, out);                \
  else if (epilogue == TFD_PANEL_SWIGLU)                                                        \
    hipLaunchKernelGGL((k_gemm_panels<TM, TN, KC, DB, kPanSwiglu>), grid, dim3(kBlock), 0, s,   \
                       (const bf16*)x, w, M, K, N, p.slices, nullptr, out);                     \
  else                                                                                          \
    hipLaunchKernelGGL((k_gemm_panels<TM, TN, KC, DB, kPanPartial>), grid, dim3(kBlock), 0, s,  \
                       (const bf16*)x, w, M, K, N, p.slices, nullptr, out)
#define TFD_PANEL_DEEP(TM, KC)                                                                  \
  if (steps % 16 == 0) { TFD_PANEL_RUN(TM, 1, KC, 16); } else { TFD_PANEL_RUN(TM, 1, KC, 8); }
  if (p.tn == 4) { TFD_PANEL_RUN(8, 4, 2, 2); }
  else if (p.tn == 2) { TFD_PANEL_RUN(8, 2, 4, 8); }
  else if (p.tm == 2) { TFD_PANEL_DEEP(2, 8) }
  else if (p.tm == 4) { TFD_PANEL_DEEP(4, 8) }
  else if (p.tm == 6) { TFD_PANEL_DEEP(6, 8) }
  else { TFD_PANEL_DEEP(8, 4) }
#undef TFD_PANEL_DEEP
#undef TFD_PANEL_RUN
  return launched("panel_gemm");
}

int tfd_panel_gemm_bf16(const void* x, const void* w, int M, int K, int N, int epilogue,
                        void* out, void* stream) {
  return panel_gemm(x, w, nullptr, M, K, N, epilogue, out, stream);
}

int tfd_panel_gemm_fp8(const void* x, const void* w, const float* scale, int M, int K, int N,
                       void* out, void* stream) {
  if (!scale) return fail(kBadArg, "panel_gemm_fp8: null scale");
  return panel_gemm(x, w, scale, M, K, N, TFD_PANEL_PARTIAL, out, stream);
}

int tfd_panel_swiglu(const float* part, int slices, int M, int N, void* out, void* stream) {
  if (!part || !out) return fail(kBadArg, "panel_swiglu: null pointer");
  if (slices <= 0 || M <= 0 || N <= 0 || N % 64)
    return fail(kBadShape, "panel_swiglu: slices=%d M=%d N=%d", slices, M, N);
  const int64_t work = (int64_t)M * (N / 4);
  hipLaunchKernelGGL(k_panel_swiglu, dim3((unsigned)((work + kBlock - 1) / kBlock)), dim3(kBlock),
                     0, (hipStream_t)stream, part, slices, M, N, (bf16*)out);
  return launched("panel_swiglu");
}

int tfd_panel_add_norm(const float* part, int slices, const void* resid, void* h_out,
                       const void* gamma, void* norm_out, int M, int n, float eps, void* stream) {
  if ((slices > 0 && !part) || !resid || !gamma || !norm_out)
    return fail(kBadArg, "panel_add_norm: null pointer");
  if (slices < 0 || M <= 0 || n <= 0 || n % 32 || n > 8192)
    return fail(kBadShape, "panel_add_norm: slices=%d M=%d n=%d", slices, M, n);
  const int per = (n / 8 + kBlock - 1) / kBlock;
  auto s = (hipStream_t)stream;
#define TFD_PANEL_NORM(C)                                                                       \
  hipLaunchKernelGGL((k_panel_add_norm<C>), dim3(M), dim3(kBlock), 0, s, part, slices,          \
                     (const bf16*)resid, (bf16*)h_out, (const bf16*)gamma, (bf16*)norm_out, M, n, \
                     eps)
  if (per == 1) TFD_PANEL_NORM(1);
  else if (per == 2) TFD_PANEL_NORM(2);
  else TFD_PANEL_NORM(4);
#undef TFD_PANEL_NORM
  return launched("panel_add_norm");
}

int tfd_panel_qkv_append(const float* part, int slices, int M, int heads, int kv_heads,
                         int head_dim, const void* gamma_q, const void* gamma_k,
                         const void* cos_table, const void* sin_table, int rope_rows,
                         const int32_t* pos, const int32_t* seq, const int32_t* page_table,
                         int max_pages, void* k_pool, void* v_pool, int num_pages, float scale,
                         float eps, void* q_out, int32_t* err, void* stream) {
  if (!part || !gamma_q || !gamma_k || !cos_table || !sin_table || !pos || !seq || !page_table ||
      !k_pool || !v_pool || !q_out)
    return fail(kBadArg, "panel_qkv_append: null pointer");
  if (slices <= 0 || M <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || max_pages <= 0 ||
      num_pages <= 0 || (head_dim != 128 && head_dim != 64))
    return fail(kBadShape, "panel_qkv_append: M=%d heads=%d kv_heads=%d head_dim=%d", M, heads,
                kv_heads, head_dim);
  const dim3 grid(M, (heads + 2 * kv_heads + kWavesPerBlock - 1) / kWavesPerBlock);
  auto s = (hipStream_t)stream;
#define TFD_PANEL_QKV(D)                                                                        \
  hipLaunchKernelGGL((k_panel_qkv<D>), grid, dim3(kBlock), 0, s, part, slices, M, heads, kv_heads, \
                     (const bf16*)gamma_q, (const bf16*)gamma_k, (const bf16*)cos_table,        \
                     (const bf16*)sin_table, rope_rows, pos, seq, page_table, max_pages,        \
                     (bf16*)k_pool, (bf16*)v_pool, num_pages, scale, eps, (bf16*)q_out, err)
  if (head_dim == 128) TFD_PANEL_QKV(128);
  else TFD_PANEL_QKV(64);
#undef TFD_PANEL_QKV
  return launched("panel_qkv_append");
}

int tfd_panel_attn_rows(int group) { return group > 0 && group <= 8 ? 64 / group : 0; }

int tfd_panel_attn(const void* q, const int32_t* tiles, int ntiles, int heads, int kv_heads,
                   int head_dim, const int32_t* page_table, int max_pages, const void* k_pool,
                   const void* v_pool, int num_pages, void* out, int32_t* err, void* stream) {
  if (!q || !tiles || !page_table || !k_pool || !v_pool || !out)
    return fail(kBadArg, "panel_attn: null pointer");
  if (ntiles <= 0 || ntiles > 65535 || heads <= 0 || kv_heads <= 0 || heads % kv_heads ||
      max_pages <= 0 || num_pages <= 0)
    return fail(kBadShape, "panel_attn: ntiles=%d heads=%d kv_heads=%d", ntiles, heads, kv_heads);
  const int G = heads / kv_heads;
  const dim3 grid(kv_heads, ntiles);
  auto s = (hipStream_t)stream;
#define TFD_PANEL_ATTN(D, GG)                                                                   \
  hipLaunchKernelGGL((k_panel_attn<D, GG, 1, kAttnDense>), grid, dim3(kBlock), 0, s, q,         \
                     (const PanelTile*)tiles, heads, kv_heads, page_table, max_pages,           \
                     (const bf16*)k_pool, (const bf16*)v_pool, num_pages, 1.f, nullptr, nullptr, \
                     (bf16*)out, err)
  if (head_dim == 128 && G == 2) TFD_PANEL_ATTN(128, 2);
  else if (head_dim == 64 && G == 2) TFD_PANEL_ATTN(64, 2);
  else if (head_dim == 128 && G == 1) TFD_PANEL_ATTN(128, 1);
  else return fail(kUnsupported, "panel_attn: head_dim=%d group=%d not built", head_dim, G);
#undef TFD_PANEL_ATTN
  return launched("panel_attn");
}

int tfd_panel_gqa(const TfdPanelGqaArgs* args, void* stream) {
  if (!args) return fail(kBadArg, "panel_gqa: null args");
  const TfdPanelGqaArgs& t = *args;
  const bool f32 = t.policy == TFD_POLICY_F32;
  if (!f32 && t.policy != TFD_POLICY_BF16) return fail(kBadArg, "panel_gqa: policy %d", t.policy);
  if (!t.proj || !t.pos || !t.seq || !t.tiles || !t.page_table || !t.k_pool || !t.v_pool ||
      !t.q || !t.out || (f32 && (!t.gamma_q || !t.gamma_k || !t.cos_table || !t.sin_table ||
                                 !t.gate || !t.self_scores)))
    return fail(kBadArg, "panel_gqa: null pointer");
  const int D = t.head_dim, G = t.kv_heads > 0 ? t.heads / t.kv_heads : 0;
  const int qw = f32 ? 2 * D : D;
  if (t.M <= 0 || t.ntiles <= 0 || t.ntiles > 65535 || t.kv_heads <= 0 || t.heads % t.kv_heads ||
      !(f32 ? D == 256 && G == 8 : D == 128 && G == 4) ||
      t.ldp < t.heads * qw + 2 * t.kv_heads * D || t.ldp % 8 || t.max_pages <= 0 ||
      t.num_pages <= 0 ||
      (f32 && (t.rot_dim <= 0 || t.rot_dim % 2 || t.rot_dim > D || t.rope_rows <= 0)))
    return fail(kBadShape, "panel_gqa: M=%d tiles=%d heads=%d kv_heads=%d head_dim=%d ldp=%d",
                t.M, t.ntiles, t.heads, t.kv_heads, D, t.ldp);
  auto s = (hipStream_t)stream;
#define TFD_PANEL_GQA(DD, GG, CT, F32, POL)                                                     \
  hipLaunchKernelGGL((k_panel_gqa_append<DD, GG, F32>), dim3(t.M, t.kv_heads), dim3(kBlock), 0, \
                     s, (const bf16*)t.proj, t.ldp, t.heads, t.kv_heads,                        \
                     (const bf16*)t.gamma_q, (const bf16*)t.gamma_k, (const bf16*)t.cos_table,  \
                     (const bf16*)t.sin_table, t.rope_rows, t.rot_dim, t.pos, t.seq,            \
                     t.page_table, t.max_pages, (bf16*)t.k_pool, (bf16*)t.v_pool, t.num_pages,  \
                     t.scale, t.eps, t.q, (bf16*)t.gate, t.self_scores, t.err);                 \
  hipLaunchKernelGGL((k_panel_attn<DD, GG, CT, POL>), dim3(t.kv_heads, t.ntiles), dim3(kBlock), \
                     0, s, t.q, (const PanelTile*)t.tiles, t.heads, t.kv_heads, t.page_table,   \
                     t.max_pages, (const bf16*)t.k_pool, (const bf16*)t.v_pool, t.num_pages,    \
                     t.scale, t.self_scores, (const bf16*)t.gate, (bf16*)t.out, t.err)
  if (f32) {
    TFD_PANEL_GQA(256, 8, 1, true, kAttnF32);
  } else {
    TFD_PANEL_GQA(128, 4, 2, false, kAttnGranite);
  }
#undef TFD_PANEL_GQA
  return launched("panel_gqa");
}

}  // extern "C"
