// Prompt passes of the hybrid models: M = seqs * T rows (T consecutive tokens of
// each sequence) through a layer at once, around the panel GEMMs and the panel
// attention of prefill.hip.
//
// Walking a prompt reads every dense weight, the picked experts and the whole
// recurrent state once per token.  Here the projections and the experts take all
// rows together, and only the recurrence itself runs token by token, with its
// state in registers:
//   k_panel_sum / k_panel_halves   K-split sums -> bf16 rows, SwiGLU
//   k_panel_mix                    residual stream + next norm (+ expert mix)
//   k_pmoe_group, k_pmoe_tiles     routed experts in tiles of up to 64 rows
//   k_pgdn_*                       gated DeltaNet: conv and norms, scan, gated norm
//   k_pmamba_*                     Mamba2: conv and dt, scan, gated norm
// Rounding is the decode kernels' (hybrid.hip), per policy.
//
// Measured (four layers, prompt to first logits, one sequence): Qwen3.5 at 250 tokens
// 58.4 ms walked, 1.92 ms in a pass; Granite at 190 tokens 65.9 and 1.78 ms.

#include "host_common.h"
#include "hybrid_common.h"
#include "panel.h"
#include "tf_decode.h"
#include "tf_hybrid.h"

using namespace tfd;
using namespace tfd_host;
using namespace tfd_hybrid;

namespace {

__global__ __launch_bounds__(kBlock) void k_panel_sum(const float* __restrict__ part, int slices,
                                                      int M, int N, void* __restrict__ out,
                                                      int ldo, int f32) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;   // four columns each
  const int per = N / 4;
  if (i >= (int64_t)M * per) return;
  const int64_t m = i / per;
  const int n = (int)(i % per) * 4;
  const f32x4 a = slice_sum4(part + m * N + n, (int64_t)M * N, slices);
  if (f32)
    *reinterpret_cast<f32x4*>((float*)out + m * ldo + n) = f32x4{rbf(a.x), rbf(a.y), rbf(a.z),
                                                                 rbf(a.w)};
  else
    *reinterpret_cast<u32x2*>((bf16*)out + m * ldo + n) = u32x2{pack2(a.x, a.y), pack2(a.z, a.w)};
}

// SwiGLU of [gate | up] sums, four columns of I each.
template <bool kF32>
__global__ __launch_bounds__(kBlock) void k_panel_halves(const float* __restrict__ part,
                                                         int slices, int M, int I,
                                                         bf16* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int per = I / 4;
  if (i >= (int64_t)M * per) return;
  const int64_t m = i / per;
  const int n = (int)(i % per) * 4;
  const int64_t stride = (int64_t)M * 2 * I;
  const f32x4 g = slice_sum4(part + m * 2 * I + n, stride, slices);
  const f32x4 u = slice_sum4(part + m * 2 * I + I + n, stride, slices);
  float h[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float s = silu_f(rbf(g[e]));
    h[e] = (kF32 ? s : rbf(s)) * rbf(u[e]);
  }
  *reinterpret_cast<u32x2*>(out + panel_off(m, n, I)) = u32x2{pack2(h[0], h[1]),
                                                              pack2(h[2], h[3])};
}

// ---------------------------------------------------------------------------
// Residual stream and next norm, a block per row.  The experts' mix adds the slots
// in slot order, then the shared expert, as k_moe_mix does; five slots' loads are in
// flight together (190 rows of ten slots, 4,096 columns: 20.2 us one by one, 15.8).
// ---------------------------------------------------------------------------
template <bool kF32, bool kMoe>
__global__ __launch_bounds__(kBlock) void k_panel_mix(TfdPanelMixArgs a) {
  constexpr int kMax4 = 8, kSlots = 5;       // n <= 8192; slots of the mix per round trip
  __shared__ float red[kWavesPerBlock];
  const int64_t m = blockIdx.x;
  const int tid = threadIdx.x, n = a.n, n4 = n / 4;
  auto block_sum = [&](float v) {
    v = wave_sum(v);
    __syncthreads();
    if ((tid & (kWave - 1)) == 0) red[tid / kWave] = v;
    __syncthreads();
    float t = red[0];
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; ++w) t += red[w];
    return t;
  };
  float sg = 1.f;
  if (kMoe && a.w_shared_scale) {
    float s = 0.f;
    for (int c = tid; c < n / 8; c += kBlock)
      s = dot8(load16((const bf16*)a.x_moe + m * n + c * 8),
               load16((const bf16*)a.w_shared_scale + c * 8), s);
    sg = sigmoid_f(rbf(block_sum(s)));
  }
  f32x4 v[kMax4];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < kMax4; ++i) {
    const int q = tid + kBlock * i;
    v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (q < n4) {
      const int c = 4 * q;
      if (kF32) {
        v[i] = *reinterpret_cast<const f32x4*>((const float*)a.stream_rows + m * n + c);
      } else {
        const u32x2 w = *reinterpret_cast<const u32x2*>((const bf16*)a.stream_rows + m * n + c);
        v[i] = f32x4{bf_lo(w.x), bf_hi(w.x), bf_lo(w.y), bf_hi(w.y)};
      }
      if (a.slices > 0) {
        f32x4 y = slice_sum4(a.part + m * n + c, (int64_t)a.M * n, a.slices);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = rbf(y[e]);
        if (kMoe) {
          f32x4 acc = {0.f, 0.f, 0.f, 0.f};
          for (int s0 = 0; s0 < a.k; s0 += kSlots) {       // their loads in flight together
            u32x2 w[kSlots];
            float wt[kSlots];
#pragma unroll
            for (int s = 0; s < kSlots; ++s) {
              const int64_t at = m * a.k + min(s0 + s, a.k - 1);
              w[s] = *reinterpret_cast<const u32x2*>((const bf16*)a.d + at * n + c);
              wt[s] = a.weights[at];
            }
#pragma unroll
            for (int s = 0; s < kSlots; ++s)
              if (s0 + s < a.k) {
                const float d[4] = {bf_lo(w[s].x), bf_hi(w[s].x), bf_lo(w[s].y), bf_hi(w[s].y)};
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += kF32 ? d[e] * wt[s] : rbf(d[e] * wt[s]);
              }
          }
#pragma unroll
          for (int e = 0; e < 4; ++e)
            y[e] = kF32 ? acc[e] + y[e] * sg : rbf(rbf(acc[e]) + y[e]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[i][e] = kF32 ? v[i][e] + y[e] : rbf(v[i][e] + rbf(y[e] * a.mult));
        if (kF32)
          *reinterpret_cast<f32x4*>((float*)a.stream_rows + m * n + c) = v[i];
        else
          *reinterpret_cast<u32x2*>((bf16*)a.stream_rows + m * n + c) =
              u32x2{pack2(v[i].x, v[i].y), pack2(v[i].z, v[i].w)};
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += v[i][e] * v[i][e];
  }
  if (!a.gamma) return;
  const float ms = block_sum(ss) / (float)n + a.eps;
  const float r = kF32 ? rsqrtf(ms) : 1.0f / sqrtf(ms);
#pragma unroll
  for (int i = 0; i < kMax4; ++i) {
    const int q = tid + kBlock * i;
    if (q < n4) {
      const int c = 4 * q;
      const u32x2 g = *reinterpret_cast<const u32x2*>((const bf16*)a.gamma + c);
      const u32x2 o = {pack2(v[i].x * r * bf_lo(g.x), v[i].y * r * bf_hi(g.x)),
                       pack2(v[i].z * r * bf_lo(g.y), v[i].w * r * bf_hi(g.y))};
      if (a.norm_panels) *reinterpret_cast<u32x2*>((bf16*)a.norm_panels + panel_off(m, c, n)) = o;
      if (a.norm_rows) *reinterpret_cast<u32x2*>((bf16*)a.norm_rows + m * n + c) = o;
    }
  }
}

// ---------------------------------------------------------------------------
// Routed experts.  One block sorts the (row, slot) entries by expert and cuts each
// expert's into tiles of up to 64.  groups: tiles, then per tile (expert, first
// entry, entries), then the entries (m * k + slot) by expert; the order inside an
// expert is the order of arrival, which no value depends on.
// ---------------------------------------------------------------------------
constexpr int kTileRows = 64;
constexpr int kPmoeExperts = 256;

struct MoeTable {
  int* tiles;                                // [..][3]
  int* entries;
};
__device__ __host__ __forceinline__ MoeTable moe_table(int32_t* groups, int E, int n) {
  return MoeTable{groups + 4, groups + 4 + 3 * (E + n / kTileRows)};
}

__global__ __launch_bounds__(1024) void k_pmoe_group(const int* __restrict__ idx, int n, int E,
                                                     int32_t* __restrict__ groups, int* err) {
  __shared__ int cnt[kPmoeExperts], first[kPmoeExperts], tile0[kPmoeExperts];
  const int tid = threadIdx.x;
  if (tid < kPmoeExperts) cnt[tid] = 0;
  __syncthreads();
  auto expert = [&](int i) {
    const int e = idx[i];
    if (e >= 0 && e < E) return e;
    raise_error(err, kErrTokenRange);        // served as expert 0
    return 0;
  };
  for (int i = tid; i < n; i += 1024) atomicAdd(&cnt[expert(i)], 1);
  __syncthreads();
  if (tid == 0) {
    int at = 0, t = 0;
    for (int e = 0; e < E; ++e) {
      first[e] = at;
      tile0[e] = t;
      at += cnt[e];
      t += (cnt[e] + kTileRows - 1) / kTileRows;
    }
    groups[0] = t;
  }
  __syncthreads();
  const MoeTable tb = moe_table(groups, E, n);
  if (tid < E)
    for (int j = 0, t = tile0[tid]; j < cnt[tid]; j += kTileRows, ++t) {
      tb.tiles[3 * t] = tid;
      tb.tiles[3 * t + 1] = first[tid] + j;
      tb.tiles[3 * t + 2] = min(kTileRows, cnt[tid] - j);
    }
  __syncthreads();
  if (tid < E) cnt[tid] = first[tid];
  __syncthreads();
  for (int i = tid; i < n; i += 1024) tb.entries[atomicAdd(&cnt[expert(i)], 1)] = i;
}

// A 16-column tile of an expert's weights, 128 K values (four K steps) at a time.
// Packed e4m3fn blocks are operands as they lie.  bf16 rows are loaded 256 bytes of
// a row at a time (four rows per load; 64-byte pieces of sixteen rows stream at half
// the rate) and turned into operands through LDS of the wave's own.
template <bool kFp8>
struct TileW;
template <>
struct TileW<true> {
  u32x2 raw[4];
  __device__ __forceinline__ void load(const void* w, int64_t row0, int K, int c, int lane) {
    const uint8_t* p = (const uint8_t*)w + ((row0 / 16) * (K / 32) + 4 * c) * 512 + lane * 8;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      raw[v] = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p + v * 512));
  }
  __device__ __forceinline__ void stage(bf16*, int) const {}
  __device__ __forceinline__ u32x4 value(const bf16*, int v, int) const {
    return fp8x8_to_bf16(raw[v]);
  }
};
constexpr int kRowS = 128 + 8;               // LDS row stride of 128 K values
template <>
struct TileW<false> {
  u32x4 raw[4];
  __device__ __forceinline__ void load(const void* w, int64_t row0, int K, int c, int lane) {
    const bf16* p = (const bf16*)w + (row0 + lane / 16) * K + c * 128 + (lane % 16) * 8;
#pragma unroll
    for (int v = 0; v < 4; ++v) raw[v] = load16_stream(p + (int64_t)4 * v * K);
  }
  __device__ __forceinline__ void stage(bf16* s, int lane) const {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      *reinterpret_cast<u32x4*>(&s[(4 * v + lane / 16) * kRowS + (lane % 16) * 8]) = raw[v];
  }
  __device__ __forceinline__ u32x4 value(const bf16* s, int v, int lane) const {
    return *reinterpret_cast<const u32x4*>(&s[(lane % 16) * kRowS + 32 * v + 8 * (lane / 16)]);
  }
};

// ---------------------------------------------------------------------------
// One projection of the routed experts.  A block takes a tile of up to 64 entries of
// an expert and 64 SwiGLU columns (each wave 16 gate and 16 up rows) or 128 output
// columns of the down projection (each wave 32); the rows pass through LDS, 128 K
// values at a time.
// Bound: the experts' weights, read once per tile (250 tokens of Qwen3.5 give 8
// entries per expert, so one tile each): gate/up 165 us for 1.07 GB (6.5 TB/s), down
// 92 us for 0.54 GB; Granite's at 190 tokens 97 us for 0.45 GB and 53 us for 0.23 GB.
// ---------------------------------------------------------------------------
struct PmoeArgs {
  const bf16* x;                             // gate/up: [M][H]; down: [entries][I]
  const void *w0, *w1;                       // gate, up; down: the same matrix twice
  const float *s0, *s1;
  int32_t* groups;
  bf16* out;                                 // gate/up: [entries][I]; down: [M * k][H]
  int K, N, k, E, n;                         // K, columns, slots, experts, entries
};

template <bool kFp8, bool kDown, bool kF32>
__global__ __launch_bounds__(kBlock) void k_pmoe_tiles(PmoeArgs a) {
  __shared__ __align__(16) bf16 xs[kTileRows * kRowS];
  __shared__ __align__(16) bf16 ws[kFp8 ? 1 : kWavesPerBlock * 2 * 16 * kRowS];
  __shared__ int ent[kTileRows];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  if ((int)blockIdx.y >= a.groups[0]) return;
  const MoeTable tb = moe_table(a.groups, a.E, a.n);
  const int e = tb.tiles[3 * blockIdx.y], first = tb.tiles[3 * blockIdx.y + 1];
  const int rows = tb.tiles[3 * blockIdx.y + 2];
  const int sub = (rows + 15) / 16;
  if (tid < kTileRows) ent[tid] = tb.entries[first + min(tid, rows - 1)];
  __syncthreads();
  const int c0 = (blockIdx.x * kWavesPerBlock + wave) * (kDown ? 32 : 16);
  const bool on = c0 < a.N;
  const int cA = on ? c0 : 0, cB = kDown ? cA + 16 : cA;
  const int64_t rA = (int64_t)e * a.N + cA, rB = (int64_t)e * a.N + cB;
  // this thread's pieces of the rows: 16 bytes each, 16 to a row
  const bf16* xp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = min(i * 16 + tid / 16, rows - 1);
    const int64_t row = kDown ? first + r : ent[r] / a.k;
    xp[i] = a.x + row * a.K + (tid % 16) * 8;
  }
  u32x4 xr[4];
  TileW<kFp8> wA, wB;
  auto load = [&](int c) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < sub) xr[i] = load16(xp[i] + c * 128);
    wA.load(a.w0, rA, a.K, c, lane);
    wB.load(a.w1, rB, a.K, c, lane);
  };
  bf16* wsA = ws + (kFp8 ? 0 : wave * 2 * 16 * kRowS);
  bf16* wsB = wsA + (kFp8 ? 0 : 16 * kRowS);
  f32x4 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  load(0);
  const int chunks = a.K / 128;
  for (int c = 0; c < chunks; ++c) {
    u32x4 opA[4], opB[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < sub)
        *reinterpret_cast<u32x4*>(&xs[(i * 16 + tid / 16) * kRowS + (tid % 16) * 8]) = xr[i];
    wA.stage(wsA, lane);
    wB.stage(wsB, lane);
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      opA[v] = wA.value(wsA, v, lane);
      opB[v] = wB.value(wsB, v, lane);
    }
    if (c + 1 < chunks) load(c + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < sub) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const u32x4 x = *reinterpret_cast<const u32x4*>(
              &xs[(i * 16 + lane % 16) * kRowS + 32 * v + 8 * (lane / 16)]);
          acc[i][0] = mfma(opA[v], x, acc[i][0]);
          acc[i][1] = mfma(opB[v], x, acc[i][1]);
        }
      }
    __syncthreads();
  }
  if (!on) return;
  const int r = lane % 16, kq = lane / 16;
  f32x4 scA = {1.f, 1.f, 1.f, 1.f}, scB = scA;
  if (kFp8) {
    scA = *reinterpret_cast<const f32x4*>(a.s0 + rA + 4 * kq);
    scB = *reinterpret_cast<const f32x4*>(a.s1 + rB + 4 * kq);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = i * 16 + r;
    if (t >= rows) continue;
    const f32x4 yA = acc[i][0] * scA, yB = acc[i][1] * scB;
    if (kDown) {
      bf16* o = a.out + (int64_t)ent[t] * a.N + cA + 4 * kq;
      *reinterpret_cast<u32x2*>(o) = u32x2{pack2(yA.x, yA.y), pack2(yA.z, yA.w)};
      *reinterpret_cast<u32x2*>(o + 16) = u32x2{pack2(yB.x, yB.y), pack2(yB.z, yB.w)};
    } else {
      float h[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float s = silu_f(rbf(yA[q]));
        h[q] = (kF32 ? s : rbf(s)) * rbf(yB[q]);
      }
      *reinterpret_cast<u32x2*>(a.out + (int64_t)(first + t) * a.N + cA + 4 * kq) =
          u32x2{pack2(h[0], h[1]), pack2(h[2], h[3])};
    }
  }
}

// ---------------------------------------------------------------------------
// Gated DeltaNet.  conv: a block per (row, key head) convolves the head's q and k and
// its value heads' channels and normalises q and k, as k_gdn_step does; the last
// three rows of a sequence leave the window.
// ---------------------------------------------------------------------------
constexpr int kGD = 128;
__global__ __launch_bounds__(kBlock) void k_pgdn_conv(TfdPanelGdnArgs a) {
  const int m = blockIdx.x, hk = blockIdx.y, tid = threadIdx.x;
  const int b = m / a.T, t = m % a.T, vpk = a.value_heads / a.key_heads;
  const int key = a.key_heads * kGD, val = a.value_heads * kGD, conv = 2 * key + val;
  const bf16* proj = (const bf16*)a.proj;
  const bf16* cw = (const bf16*)a.conv_w;
  const float* cin = a.conv_in + (int64_t)b * conv * 3;
  float* cout = a.conv_out + (int64_t)b * conv * 3;
  __shared__ float red[kWavesPerBlock];
  auto value = [&](int c, int i) {           // channel c of the sequence's row i of this pass
    return i >= 0 ? bf2f(proj[(int64_t)(b * a.T + i) * a.ldp + c]) : cin[(int64_t)c * 3 + 3 + i];
  };
  auto conv_silu = [&](int c) {
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) acc += value(c, t - 3 + j) * bf2f(cw[(int64_t)c * 4 + j]);
    if (t == a.T - 1) {
#pragma unroll
      for (int j = 0; j < 3; ++j) cout[(int64_t)c * 3 + j] = value(c, t - 2 + j);
    }
    return silu_f(acc);
  };
  const int d = tid % kGD, isk = tid / kGD;
  const float x = conv_silu(isk * key + hk * kGD + d);
  const float ss = wave_sum(x * x);
  if ((tid & (kWave - 1)) == 0) red[tid / kWave] = ss;
  __syncthreads();
  const float rs = rsqrtf(red[2 * isk] + red[2 * isk + 1] + a.l2_eps);
  a.qk[((int64_t)isk * a.seqs * a.T + m) * key + hk * kGD + d] =
      isk ? x * rs : x * (rs * rsqrtf((float)kGD));
  for (int c = tid; c < vpk * kGD; c += kBlock) {
    const int ch = hk * vpk * kGD + c;
    a.v[(int64_t)m * val + ch] = conv_silu(2 * key + ch);
  }
  if (tid < vpk) {
    const int hv = hk * vpk + tid;
    const bf16* row = proj + (int64_t)m * a.ldp + conv + val;
    const float braw = bf2f(row[hv]), araw = bf2f(row[a.value_heads + hv]);
    float* g = a.gates + ((int64_t)m * a.value_heads + hv) * 2;
    g[0] = expf(-expf(bf2f(((const bf16*)a.a_log)[hv])) *
                softplus_f(araw + bf2f(((const bf16*)a.dt_bias)[hv])));
    g[1] = sigmoid_f(braw);
  }
}

// The delta rule over the sequence's T tokens.  A value column of a head's state
// depends on no other column, so a block takes 32 columns of one (head, sequence),
// eight lanes to a column, sixteen key rows each in registers; the tokens' q, k, v and
// gates come through LDS, sixteen tokens at a time.
// Bound: the chain of a token (64 multiply-adds a lane and two eight-lane sums): 250
// tokens take 71 us, 0.28 us each; with the step's kernel a token's launch took 5.5.  One
// sequence's 128 blocks (32 heads) leave half the compute units without one.
constexpr int kScanT = 16;
__global__ __launch_bounds__(kBlock) void k_pgdn_scan(TfdPanelGdnArgs a) {
  const int hv = blockIdx.y, b = blockIdx.z, tid = threadIdx.x;
  const int cl = tid / 8, rg = tid % 8, col = blockIdx.x * 32 + cl;
  const int key = a.key_heads * kGD, val = a.value_heads * kGD;
  const int hk = hv / (a.value_heads / a.key_heads);
  const int64_t M = (int64_t)a.seqs * a.T, m0 = (int64_t)b * a.T;
  __shared__ __align__(16) float q_s[kScanT][kGD], k_s[kScanT][kGD];
  __shared__ float v_s[kScanT][32], g_s[kScanT][2];
  float* st = a.state + ((int64_t)b * a.value_heads + hv) * kGD * kGD + col;
  float s[16];                               // key rows 32 j + 4 rg + e
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] = st[(int64_t)(32 * (i / 4) + 4 * rg + i % 4) * kGD];
  f32x4 qr[2], kr[2];
  float vr[2], gr = 0.f;
  auto load = [&](int t0) {                  // tokens past the end repeat the last
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = tid + i * kBlock;
      const int64_t m = m0 + min(t0 + c / 32, a.T - 1);
      const float* p = a.qk + m * key + hk * kGD + (c % 32) * 4;
      qr[i] = *reinterpret_cast<const f32x4*>(p);
      kr[i] = *reinterpret_cast<const f32x4*>(p + M * key);
      vr[i] = a.v[m * val + hv * kGD + blockIdx.x * 32 + c % 32];
    }
    if (tid < 2 * kScanT)
      gr = a.gates[((m0 + min(t0 + tid / 2, a.T - 1)) * a.value_heads + hv) * 2 + tid % 2];
  };
  load(0);
  for (int t0 = 0; t0 < a.T; t0 += kScanT) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = tid + i * kBlock;
      *reinterpret_cast<f32x4*>(&q_s[c / 32][(c % 32) * 4]) = qr[i];
      *reinterpret_cast<f32x4*>(&k_s[c / 32][(c % 32) * 4]) = kr[i];
      v_s[c / 32][c % 32] = vr[i];
    }
    if (tid < 2 * kScanT) g_s[tid / 2][tid % 2] = gr;
    __syncthreads();
    if (t0 + kScanT < a.T) load(t0 + kScanT);
    const int n = min(kScanT, a.T - t0);
    for (int t = 0; t < n; ++t) {
      const float decay = g_s[t][0], beta = g_s[t][1];
      float kv[16], qv[16], rec = 0.f, rd = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 k4 = *reinterpret_cast<const f32x4*>(&k_s[t][32 * j + 4 * rg]);
        const f32x4 q4 = *reinterpret_cast<const f32x4*>(&q_s[t][32 * j + 4 * rg]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          kv[4 * j + e] = k4[e];
          qv[4 * j + e] = q4[e];
        }
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[i] *= decay;
        rec = fmaf(s[i], kv[i], rec);
      }
      rec = group_sum<8>(rec);
      const float delta = (v_s[t][cl] - rec) * beta;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[i] = fmaf(kv[i], delta, s[i]);
        rd = fmaf(s[i], qv[i], rd);
      }
      rd = group_sum<8>(rd);
      if (rg == 0) a.read[(m0 + t0 + t) * val + hv * kGD + col] = rd;
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) st[(int64_t)(32 * (i / 4) + 4 * rg + i % 4) * kGD] = s[i];
}

// The gated norm of the read-out per (row, value head), a wave each.
__global__ __launch_bounds__(kBlock) void k_pgdn_gate(TfdPanelGdnArgs a) {
  const int64_t m = blockIdx.x;
  const int h = blockIdx.y * kWavesPerBlock + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if (h >= a.value_heads) return;
  const int val = a.value_heads * kGD, conv = 2 * a.key_heads * kGD + val;
  const float* r = a.read + m * val + h * kGD + 2 * lane;
  const float x0 = r[0], x1 = r[1];
  const float ms = wave_sum(x0 * x0 + x1 * x1) / (float)kGD;
  const float rs = rsqrtf(ms + a.rms_eps);
  const uint32_t g = *reinterpret_cast<const uint32_t*>((const bf16*)a.gamma + 2 * lane);
  const uint32_t z = *reinterpret_cast<const uint32_t*>((const bf16*)a.proj + m * a.ldp + conv +
                                                        h * kGD + 2 * lane);
  *reinterpret_cast<uint32_t*>((bf16*)a.out + panel_off(m, h * kGD + 2 * lane, val)) =
      pack2(x0 * rs * bf_lo(g) * silu_f(bf_lo(z)), x1 * rs * bf_hi(g) * silu_f(bf_hi(z)));
}

// ---------------------------------------------------------------------------
// Mamba2.  conv: a block per row and 1,024 channels.
// ---------------------------------------------------------------------------
constexpr int kMP = 64, kMN = 128;
__global__ __launch_bounds__(kBlock) void k_pmamba_conv(TfdPanelMambaArgs a) {
  const int m = blockIdx.x, tid = threadIdx.x, b = m / a.T, t = m % a.T;
  const int exp_ = a.heads * kMP, conv = exp_ + 2 * kMN;
  const bf16* proj = (const bf16*)a.proj;
  const bf16* cw = (const bf16*)a.conv_w;
  const bf16* cin = (const bf16*)a.conv_in + (int64_t)b * conv * 3;
  bf16* cout = (bf16*)a.conv_out + (int64_t)b * conv * 3;
  auto value = [&](int c, int i) {
    return i >= 0 ? proj[(int64_t)(b * a.T + i) * a.ldp + exp_ + c] : cin[(int64_t)c * 3 + 3 + i];
  };
  for (int c = blockIdx.y * 1024 + tid; c < conv && c < (int)(blockIdx.y + 1) * 1024; c += kBlock) {
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      sum += rbf(bf2f(value(c, t - 3 + j)) * bf2f(cw[(int64_t)c * 4 + j]));
    if (t == a.T - 1) {
#pragma unroll
      for (int j = 0; j < 3; ++j) cout[(int64_t)c * 3 + j] = value(c, t - 2 + j);
    }
    const bf16 y = f2bf(silu_f(rbf(rbf(sum) + bf2f(((const bf16*)a.conv_b)[c]))));
    if (c < exp_)
      ((bf16*)a.x)[(int64_t)m * exp_ + c] = y;
    else
      ((bf16*)a.bc)[(int64_t)m * 2 * kMN + c - exp_] = y;
  }
  if (blockIdx.y == 0)
    for (int h = tid; h < a.heads; h += kBlock) {
      const float dt = rbf(softplus_f(rbf(bf2f(proj[(int64_t)m * a.ldp + exp_ + conv + h]) +
                                          bf2f(((const bf16*)a.dt_bias)[h]))));
      float* g = a.gates + ((int64_t)m * a.heads + h) * 2;
      g[0] = expf(dt * -expf(bf2f(((const bf16*)a.a_log)[h])));
      g[1] = dt;
    }
}

// The state update over the sequence's T tokens: a block takes 32 of a head's 64 state
// rows, eight lanes to a row, sixteen columns each in registers (columns 32 j + 4 ng
// + e); bf16(dt B) and C come through LDS, sixteen tokens at a time and read a token
// ahead.
// Bound: the VALU, one wave to a SIMD where a block runs: one sequence's 128 blocks (64
// heads) leave half the compute units without one (eleven operations a state and token with dt B
// formed by every row and one value to a conversion: 92 us for 190 tokens; six with two
// values to a conversion and C's products summed in pairs: 71, 0.37 a token).
__global__ __launch_bounds__(kBlock) void k_pmamba_scan(TfdPanelMambaArgs a) {
  const int h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x;
  const int pl = tid / 8, ng = tid % 8, p = blockIdx.x * 32 + pl;
  const int exp_ = a.heads * kMP;
  const int64_t m0 = (int64_t)b * a.T;
  __shared__ __align__(16) float b_s[kScanT][kMN];       // bf16(dt B)
  __shared__ __align__(16) bf16 c_s[kScanT][kMN];
  __shared__ float x_s[kScanT][32], g_s[kScanT];
  float* st = a.state + (((int64_t)b * a.heads + h) * kMP + p) * kMN + 4 * ng;
  float s[16];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(st + 32 * j);
#pragma unroll
    for (int e = 0; e < 4; ++e) s[4 * j + e] = v[e];
  }
  const float dsk = bf2f(((const bf16*)a.d_skip)[h]);
  u32x4 bcr[2];
  bf16 xr[2];
  float dtr[2], gr = 0.f;
  auto load = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = tid + i * kBlock;        // B | C: 32 pieces of 8 a token
      const int64_t m = m0 + min(t0 + c / 32, a.T - 1);
      dtr[i] = a.gates[(m * a.heads + h) * 2 + 1];
      bcr[i] = load16((const bf16*)a.bc + m * 2 * kMN + (c % 32) * 8);
      xr[i] = ((const bf16*)a.x)[m * exp_ + h * kMP + blockIdx.x * 32 + c % 32];
    }
    if (tid < kScanT) gr = a.gates[((m0 + min(t0 + tid, a.T - 1)) * a.heads + h) * 2];
  };
  load(0);
  for (int t0 = 0; t0 < a.T; t0 += kScanT) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = tid + i * kBlock, part = c % 32;
      if (part < 16) {
        const float dt = dtr[i];
        float* dst = &b_s[c / 32][part * 8];
        *reinterpret_cast<f32x4*>(dst) =
            f32x4{rbf(dt * bf_lo(bcr[i].x)), rbf(dt * bf_hi(bcr[i].x)),
                  rbf(dt * bf_lo(bcr[i].y)), rbf(dt * bf_hi(bcr[i].y))};
        *reinterpret_cast<f32x4*>(dst + 4) =
            f32x4{rbf(dt * bf_lo(bcr[i].z)), rbf(dt * bf_hi(bcr[i].z)),
                  rbf(dt * bf_lo(bcr[i].w)), rbf(dt * bf_hi(bcr[i].w))};
      } else {
        *reinterpret_cast<u32x4*>(&c_s[c / 32][(part - 16) * 8]) = bcr[i];
      }
      x_s[c / 32][c % 32] = bf2f(xr[i]);
    }
    if (tid < kScanT) g_s[tid] = gr;
    __syncthreads();
    if (t0 + kScanT < a.T) load(t0 + kScanT);
    const int n = min(kScanT, a.T - t0);
    f32x4 bn[4];                             // a token ahead of its use
    u32x2 cn[4];
    float dn, xn;
    auto fetch = [&](int t) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bn[j] = *reinterpret_cast<const f32x4*>(&b_s[t][32 * j + 4 * ng]);
        cn[j] = *reinterpret_cast<const u32x2*>(&c_s[t][32 * j + 4 * ng]);
      }
      dn = g_s[t];
      xn = x_s[t][pl];
    };
    fetch(0);
    for (int t = 0; t < n; ++t) {
      const float decay = dn, xp = xn;
      f32x4 bt[4];
      u32x2 ct[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bt[j] = bn[j];
        ct[j] = cn[j];
      }
      fetch(min(t + 1, kScanT - 1));
      float r2[2] = {0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) {        // two states per conversion and per dot
          float &u = s[4 * j + 2 * i], &w = s[4 * j + 2 * i + 1];
          const uint32_t in = pack2(bt[j][2 * i] * xp, bt[j][2 * i + 1] * xp);
          u = u * decay + bf_lo(in);
          w = w * decay + bf_hi(in);
          r2[i] = dot2(pack2(u, w), i == 0 ? ct[j].x : ct[j].y, r2[i]);
        }
      const float rd = group_sum<8>(r2[0] + r2[1]);
      if (ng == 0)
        ((bf16*)a.y)[(m0 + t0 + t) * exp_ + h * kMP + p] = f2bf(rbf(rd) + rbf(xp * dsk));
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    *reinterpret_cast<f32x4*>(st + 32 * j) = f32x4{s[4 * j], s[4 * j + 1], s[4 * j + 2],
                                                   s[4 * j + 3]};
}

// RMSNormGated over the inner width, a block per row (n <= 8192, n % 4 == 0).
__global__ __launch_bounds__(kBlock) void k_pmamba_norm(TfdPanelMambaArgs a) {
  constexpr int kMax4 = 8;
  __shared__ float red[kWavesPerBlock];
  const int64_t m = blockIdx.x;
  const int tid = threadIdx.x, n = a.heads * kMP, n4 = n / 4;
  f32x4 v[kMax4];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < kMax4; ++i) {
    const int q = tid + kBlock * i;
    v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (q < n4) {
      const u32x2 y = *reinterpret_cast<const u32x2*>((const bf16*)a.y + m * n + 4 * q);
      const u32x2 g = *reinterpret_cast<const u32x2*>((const bf16*)a.proj + m * a.ldp + 4 * q);
      v[i] = f32x4{bf_lo(y.x) * silu_f(bf_lo(g.x)), bf_hi(y.x) * silu_f(bf_hi(g.x)),
                   bf_lo(y.y) * silu_f(bf_lo(g.y)), bf_hi(y.y) * silu_f(bf_hi(g.y))};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += v[i][e] * v[i][e];
  }
  ss = wave_sum(ss);
  if ((tid & (kWave - 1)) == 0) red[tid / kWave] = ss;
  __syncthreads();
  float tot = red[0];
#pragma unroll
  for (int w = 1; w < kWavesPerBlock; ++w) tot += red[w];
  const float r = rsqrtf(tot / (float)n + a.eps);
#pragma unroll
  for (int i = 0; i < kMax4; ++i) {
    const int q = tid + kBlock * i;
    if (q < n4) {
      const u32x2 g = *reinterpret_cast<const u32x2*>((const bf16*)a.gamma + 4 * q);
      *reinterpret_cast<u32x2*>((bf16*)a.out + panel_off(m, 4 * q, n)) =
          u32x2{pack2(v[i].x * r * bf_lo(g.x), v[i].y * r * bf_hi(g.x)),
                pack2(v[i].z * r * bf_lo(g.y), v[i].w * r * bf_hi(g.y))};
    }
  }
}

unsigned blocks_for(int64_t work) { return (unsigned)((work + kBlock - 1) / kBlock); }

}  // namespace

extern "C" {

int tfd_panel_sum(const float* part, int slices, int M, int N, void* out, int ldo, int f32,
                  void* stream) {
  if (!part || !out) return fail(kBadArg, "panel_sum: null pointer");
  if (slices <= 0 || M <= 0 || N <= 0 || N % 4 || ldo < N || ldo % 4)
    return fail(kBadShape, "panel_sum: slices=%d M=%d N=%d ldo=%d", slices, M, N, ldo);
  hipLaunchKernelGGL(k_panel_sum, dim3(blocks_for((int64_t)M * (N / 4))), dim3(kBlock), 0,
                     (hipStream_t)stream, part, slices, M, N, out, ldo, f32);
  return launched("panel_sum");
}

int tfd_panel_swiglu_halves(const float* part, int slices, int M, int N, int policy, void* out,
                            void* stream) {
  if (!part || !out) return fail(kBadArg, "panel_swiglu_halves: null pointer");
  if (slices <= 0 || M <= 0 || N <= 0 || N % 64)
    return fail(kBadShape, "panel_swiglu_halves: slices=%d M=%d N=%d", slices, M, N);
  const dim3 grid(blocks_for((int64_t)M * (N / 8)));
  auto s = (hipStream_t)stream;
  if (policy == TFD_POLICY_F32)
    hipLaunchKernelGGL((k_panel_halves<true>), grid, dim3(kBlock), 0, s, part, slices, M, N / 2,
                       (bf16*)out);
  else
    hipLaunchKernelGGL((k_panel_halves<false>), grid, dim3(kBlock), 0, s, part, slices, M, N / 2,
                       (bf16*)out);
  return launched("panel_swiglu_halves");
}

int tfd_panel_mix(const TfdPanelMixArgs* args, void* stream) {
  if (!args) return fail(kBadArg, "panel_mix: null args");
  const TfdPanelMixArgs& t = *args;
  if (!t.stream_rows || (t.slices > 0 && !t.part) ||
      (t.moe && (!t.d || !t.weights || (t.w_shared_scale && !t.x_moe))))
    return fail(kBadArg, "panel_mix: null pointer");
  if (t.M <= 0 || t.n <= 0 || t.n % 32 || t.n > 8192 || t.slices < 0 ||
      (t.moe && (t.k <= 0 || t.slices <= 0)))
    return fail(kBadShape, "panel_mix: M=%d n=%d slices=%d k=%d", t.M, t.n, t.slices, t.k);
  auto s = (hipStream_t)stream;
  const bool f32 = t.policy == TFD_POLICY_F32;
  const dim3 grid(t.M), block(kBlock);
  if (f32 && t.moe) hipLaunchKernelGGL((k_panel_mix<true, true>), grid, block, 0, s, t);
  else if (f32) hipLaunchKernelGGL((k_panel_mix<true, false>), grid, block, 0, s, t);
  else if (t.moe) hipLaunchKernelGGL((k_panel_mix<false, true>), grid, block, 0, s, t);
  else hipLaunchKernelGGL((k_panel_mix<false, false>), grid, block, 0, s, t);
  return launched("panel_mix");
}

int tfd_panel_moe(const TfdPanelMoeArgs* args, void* stream) {
  if (!args) return fail(kBadArg, "panel_moe: null args");
  const TfdPanelMoeArgs& t = *args;
  if (!t.x || !t.idx || !t.w_gate || !t.w_up || !t.w_down || !t.groups || !t.hidden || !t.d ||
      (t.fp8 && (!t.s_gate || !t.s_up || !t.s_down)))
    return fail(kBadArg, "panel_moe: null pointer");
  if (t.M <= 0 || t.k <= 0 || t.experts <= 0 || t.experts > kPmoeExperts || t.H <= 0 ||
      t.H % 128 || t.H > 8192 || t.I <= 0 || t.I % 128 || (int64_t)t.M * t.k > (1 << 20))
    return fail(kBadShape, "panel_moe: M=%d k=%d experts=%d H=%d I=%d", t.M, t.k, t.experts, t.H,
                t.I);
  auto s = (hipStream_t)stream;
  const int n = t.M * t.k;
  hipLaunchKernelGGL(k_pmoe_group, dim3(1), dim3(1024), 0, s, t.idx, n, t.experts, t.groups,
                     t.err);
  const int most = (n < t.experts ? n : t.experts) + n / kTileRows;   // tiles at most
  PmoeArgs g{(const bf16*)t.x, t.w_gate, t.w_up, t.s_gate, t.s_up, t.groups, (bf16*)t.hidden,
             t.H, t.I, t.k, t.experts, n};
  PmoeArgs d{(const bf16*)t.hidden, t.w_down, t.w_down, t.s_down, t.s_down, t.groups,
             (bf16*)t.d, t.I, t.H, t.k, t.experts, n};
  const dim3 g1((t.I + 63) / 64, most), g2((t.H + 127) / 128, most), block(kBlock);
  const bool f32 = t.policy == TFD_POLICY_F32;
#define TFD_PMOE(FP8, F32)                                                       \
  hipLaunchKernelGGL((k_pmoe_tiles<FP8, false, F32>), g1, block, 0, s, g);       \
  hipLaunchKernelGGL((k_pmoe_tiles<FP8, true, F32>), g2, block, 0, s, d)
  if (t.fp8 && f32) { TFD_PMOE(true, true); }
  else if (t.fp8) { TFD_PMOE(true, false); }
  else if (f32) { TFD_PMOE(false, true); }
  else { TFD_PMOE(false, false); }
#undef TFD_PMOE
  return launched("panel_moe");
}

int tfd_panel_gdn(const TfdPanelGdnArgs* args, void* stream) {
  if (!args) return fail(kBadArg, "panel_gdn: null args");
  const TfdPanelGdnArgs& t = *args;
  if (!t.proj || !t.conv_in || !t.conv_out || t.conv_in == t.conv_out || !t.state || !t.conv_w ||
      !t.a_log || !t.dt_bias || !t.gamma || !t.qk || !t.v || !t.read || !t.gates || !t.out)
    return fail(kBadArg, "panel_gdn: null pointer, or conv_in == conv_out");
  if (t.seqs <= 0 || t.seqs > 65535 || t.T <= 0 || t.head_dim != kGD || t.key_heads <= 0 ||
      t.value_heads <= 0 || t.value_heads % t.key_heads || t.value_heads / t.key_heads > kBlock ||
      t.ldp % 2 ||
      t.ldp < (2 * t.key_heads + 2 * t.value_heads) * kGD + 2 * t.value_heads)
    return fail(kBadShape, "panel_gdn: seqs=%d T=%d heads=%d/%d head_dim=%d ldp=%d", t.seqs, t.T,
                t.key_heads, t.value_heads, t.head_dim, t.ldp);
  auto s = (hipStream_t)stream;
  const int M = t.seqs * t.T;
  hipLaunchKernelGGL(k_pgdn_conv, dim3(M, t.key_heads), dim3(kBlock), 0, s, t);
  hipLaunchKernelGGL(k_pgdn_scan, dim3(kGD / 32, t.value_heads, t.seqs), dim3(kBlock), 0, s, t);
  hipLaunchKernelGGL(k_pgdn_gate, dim3(M, (t.value_heads + 3) / 4), dim3(kBlock), 0, s, t);
  return launched("panel_gdn");
}

int tfd_panel_mamba(const TfdPanelMambaArgs* args, void* stream) {
  if (!args) return fail(kBadArg, "panel_mamba: null args");
  const TfdPanelMambaArgs& t = *args;
  if (!t.proj || !t.conv_in || !t.conv_out || t.conv_in == t.conv_out || !t.state || !t.conv_w ||
      !t.conv_b || !t.a_log || !t.dt_bias || !t.d_skip || !t.gamma || !t.x || !t.bc || !t.y ||
      !t.gates || !t.out)
    return fail(kBadArg, "panel_mamba: null pointer, or conv_in == conv_out");
  const int exp_ = t.heads * kMP, conv = exp_ + 2 * kMN;
  if (t.seqs <= 0 || t.seqs > 65535 || t.T <= 0 || t.heads <= 0 || exp_ > 8192 ||
      t.head_dim != kMP || t.state_dim != kMN || t.ldp < exp_ + conv + t.heads || t.ldp % 4)
    return fail(kBadShape, "panel_mamba: seqs=%d T=%d heads=%d x %d state=%d ldp=%d", t.seqs, t.T,
                t.heads, t.head_dim, t.state_dim, t.ldp);
  auto s = (hipStream_t)stream;
  const int M = t.seqs * t.T;
  hipLaunchKernelGGL(k_pmamba_conv, dim3(M, (conv + 1023) / 1024), dim3(kBlock), 0, s, t);
  hipLaunchKernelGGL(k_pmamba_scan, dim3(kMP / 32, t.heads, t.seqs), dim3(kBlock), 0, s, t);
  hipLaunchKernelGGL(k_pmamba_norm, dim3(M), dim3(kBlock), 0, s, t);
  return launched("panel_mamba");
}

}  // extern "C"
