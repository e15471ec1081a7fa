// gather_qmm: routed (MoE expert) 4-bit affine quantized matmul, gfx950.
//
// Semantics restated: mlx_ext::gather_qmm(x, w, scales, biases,
// lhs_indices, rhs_indices, transpose = true, 64, 4, sorted_indices)
// (crates/base-mlx-core/src/mlx_ext.rs:66-117), as QSwitchLinear::forward
// calls it for the experts of SwitchGlu with lhs_indices = None (crates/
// base-mlx-core/src/model/granite.rs:74-88, 181-201): W, s, b stack E
// experts ([E, N, K/8] u32, [E, N, K/64] bf16), and route r -- one (token,
// top-k slot) pair of the index array -- computes
//   y[r] = x[lhs(r)] . W[rhs(r)]^T               ([M, K] x [K, N] -> [M, N])
// with quantized_matmul's group decomposition, fp32 accumulation and a bf16
// result.  lhs(r) = lhs_indices[r] when given, else r / x_bcast: MLX's
// broadcast of x over the top-k axis (top_k for the gate/up projection,
// whose x [T, 1, 1, K] every slot of a token shares; 1 for the down
// projection, which has one input row block per route).  rhs(r) =
// rhs_indices[r] when given, else r.  sorted_indices only tells MLX the
// routes come grouped by expert; results do not depend on it.
//
// Work decomposition: a workgroup of 4 waves owns RB consecutive output
// rows of one route (grid = row tiles x routes); the expert id is read on
// the device, so a captured graph replays with new routes.  The route's x
// rows are staged once in LDS, pair-permuted with per-chunk sums (as the
// GEMV of qmv.hip stages them); each output row is served by S lanes that
// stride over its 64-wide groups (32 bytes of W, one s and one b per group
// and lane), with every W load of a lane issued before the staging.  With
// many routes an expert, gather_rows_kernel (below) takes each expert's
// routes together instead.
#include <math.h>

#include <algorithm>

#include "bmx_device.h"

namespace bmx {
namespace {

constexpr int kGThreads = 256;
constexpr int kGChunk = 80;   // LDS bytes per 32 x values: 64 data + 16 pad
constexpr int kGMaxNG = 8;    // groups per lane
constexpr int kGMaxM = 8;     // rows of x per route

struct GatherParams {
  const uint16_t* x;    // route r: rows [M, K] at x + lhs(r) * x_rstride
  const uint32_t* w;    // [E, N, K/8]
  const uint16_t* s;    // [E, N, K/64]
  const uint16_t* b;    // [E, N, K/64]
  const uint32_t* lhs;  // [R] x block of each route, or null: r / x_bcast
  const uint32_t* rhs;  // [R] expert of each route, or null: r
  uint16_t* y;          // route r: rows [M, N] at y + r * y_rstride
  int64_t x_rstride, y_rstride;
  int x_bcast, nxb, E, M, N, K;  // nxb: x blocks
  int S;                // lanes per output row (power of two, 1..64)
  int R;                // routes
  int run;              // by expert: tiles per unit
};

template <int MT>
__global__ void __launch_bounds__(kGThreads) gather_qmv_kernel(const GatherParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int K = p.K, G = K / 64, C = K / 32, W8 = K / 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lshift = __builtin_ctz(p.S);
  const int slot = lane >> lshift, sl = lane & (p.S - 1);
  const int slots = 64 >> lshift;
  const int rb = 4 * slots;
  const int route = blockIdx.y;
  // out-of-range expert and x block ids are clamped (a valid address for
  // every route)
  const int64_t e = min(p.rhs ? p.rhs[route] : static_cast<uint32_t>(route), static_cast<uint32_t>(p.E - 1));
  const int64_t xb = p.lhs ? min(p.lhs[route], static_cast<uint32_t>(p.nxb - 1)) : route / p.x_bcast;
  const uint16_t* xr = p.x + xb * p.x_rstride;
  const int row = blockIdx.x * rb + wave * slots + slot;
  const int64_t rr = min(row, p.N - 1);
  const uint32_t* wrow = p.w + (e * p.N + rr) * (K / 8);
  const uint16_t* srow = p.s + (e * p.N + rr) * G;
  const uint16_t* brow = p.b + (e * p.N + rr) * G;
  unsigned char* xs = smem;                                           // [MT][C] x kGChunk
  float* sxs = reinterpret_cast<float*>(smem + MT * C * kGChunk);     // [MT][C]

  // ---- W, s, b of this lane's groups g = sl + u * S (clamped, unconditional) ----
  uint4 w0[kGMaxNG], w1[kGMaxNG];
  uint16_t sv[kGMaxNG], bv[kGMaxNG];
#pragma unroll
  for (int u = 0; u < kGMaxNG; u++) {
    const int g = min(sl + (u << lshift), G - 1);
    w0[u] = *reinterpret_cast<const uint4*>(wrow + g * 8);
    w1[u] = *reinterpret_cast<const uint4*>(wrow + g * 8 + 4);
    sv[u] = srow[g];
    bv[u] = brow[g];
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- x rows into LDS: pair-permuted 16-byte units, per-chunk sums ----
  // (a chunk of 32 values is 4 consecutive units = 4 consecutive lanes)
  const int units = p.M * W8;
  for (int base = 0; base < MT * W8; base += kGThreads) {
    const int idx = base + static_cast<int>(threadIdx.x);
    const bool act = idx < units;
    const int m = act ? idx / W8 : 0;
    const int j = act ? idx - m * W8 : 0;
    uint4 d = make_uint4(0, 0, 0, 0);
    if (act) d = *reinterpret_cast<const uint4*>(xr + static_cast<int64_t>(m) * K + j * 8);
    const uint32_t dv[4] = {d.x, d.y, d.z, d.w};
    float part = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; q++) part += bf2f(dv[q] & 0xffffu) + bf2f(dv[q] >> 16);
    part += dpp_f32<0xB1>(part);
    part += dpp_f32<0x4E>(part);
    if (act) {
      *reinterpret_cast<uint4*>(xs + (m * C + (j >> 2)) * kGChunk + (j & 3) * 16) = permute_pairs(d);
      if ((j & 3) == 0) sxs[m * C + (j >> 2)] = part;
    }
  }
  __syncthreads();
  // ---- dot products: y[m] += s * D + (b - 128 s) * Sx per group ----
  const NibbleK nk = nibble_consts();
  float acc[MT];
#pragma unroll
  for (int m = 0; m < MT; m++) acc[m] = 0.0f;
#pragma unroll
  for (int u = 0; u < kGMaxNG; u++) {
    const int g = sl + (u << lshift);
    if (g < G) {
      const float s = bf2f(sv[u]);
      const float bb = bf2f(bv[u]) - 128.0f * s;
#pragma unroll
      for (int m = 0; m < MT; m++) {
        if (m >= p.M) break;
        const uint4* xp0 = reinterpret_cast<const uint4*>(xs + (m * C + 2 * g) * kGChunk);
        const uint4* xp1 = reinterpret_cast<const uint4*>(xs + (m * C + 2 * g + 1) * kGChunk);
        float d0 = 0.0f, d1 = 0.0f;
        d0 = word_dot(w0[u].x, xp0[0], d0, nk);
        d1 = word_dot(w0[u].y, xp0[1], d1, nk);
        d0 = word_dot(w0[u].z, xp0[2], d0, nk);
        d1 = word_dot(w0[u].w, xp0[3], d1, nk);
        d0 = word_dot(w1[u].x, xp1[0], d0, nk);
        d1 = word_dot(w1[u].y, xp1[1], d1, nk);
        d0 = word_dot(w1[u].z, xp1[2], d0, nk);
        d1 = word_dot(w1[u].w, xp1[3], d1, nk);
        const float sx = sxs[m * C + 2 * g] + sxs[m * C + 2 * g + 1];
        acc[m] += s * (d0 + d1);
        acc[m] += bb * sx;
      }
    }
  }
  // ---- reduce the S lanes of each row, store ----
#pragma unroll
  for (int m = 0; m < MT; m++) acc[m] = wave_sum_xor(acc[m], p.S);
  if (sl == 0 && row < p.N) {
    uint16_t* yr = p.y + static_cast<int64_t>(route) * p.y_rstride + row;
#pragma unroll
    for (int m = 0; m < MT; m++) {
      if (m >= p.M) break;
      yr[static_cast<int64_t>(m) * p.N] = f2bf(acc[m]);
    }
  }
}

// ---------------------------------------------------------------------------
// Many routes: every expert's weights read once for all of its rows.
//
// gather_qmv_kernel reads a route's whole weight matrix for that route
// alone, so with R routes over E experts the same weights come from memory
// (or the caches) R / E times.  Here a workgroup owns one unit -- a few tiles
// of 16 MT rows of one expert -- and kGCols output columns.  The first E grid
// rows are the experts' first units; the rows past them, as many as R routes
// can need, take the further units of whichever experts have more: each
// counts the routes of every expert (LDS counters) and finds its unit in the
// prefix sum of those.  So an expert is spread over as many workgroups as it
// has units, whatever share of the routes it takes (90% of 400 routes over
// 128 experts to one of them, 1536 x 2048: 255 us where one workgroup walked
// an expert's tiles, now 46), and workgroups without a unit end here.  No
// scratch memory, no second launch: a captured graph replays with new routes.
// The rows are multiplied
// on v_mfma_f32_16x16x32_bf16: A = x rows (from LDS), B = the nibbles as bf16
// integers 128 + q, lane l holding W row l % 16.  The group
// decomposition stays as in the per-route kernel, fp32 throughout:
//   acc = fma(s, D, acc) per group and output,
//   acc += (b - 128 s) Sx over four groups on v_mfma_f32_16x16x4_f32,
// with the group sums Sx taken once per workgroup while x is staged (pair
// order, so a nibble pair is one v_and_or; against Sx by products with a tile
// of ones in every wave and one FMA per output more, a third of the vector
// instructions less).  Rows past the count repeat the last row and are not
// stored; a row's result does not depend on its slot.
//
// What each operand needs decides where it comes from.  W is read once, so it
// goes straight to registers: 16 bytes per lane and step of two groups (64
// contiguous bytes per W row), a chunk of kGChunkK columns ahead.  x is shared
// by the 8 waves and comes through LDS in chunks, double-buffered, one barrier
// per chunk; s and b of the workgroup's 256 columns are one contiguous block
// per array and are staged whole.  (Read per lane and step instead, the 4-byte
// s and b pieces and the x rows were 85% of the L1 misses, and the kernel ran
// at the L2's rate: 226 MB of weights in 118 us.)
constexpr int kGChunkK = 256;    // columns of x per LDS chunk
constexpr int kGXS = kGChunkK + 8;  // LDS row stride of x (odd number of 16-byte units: no bank conflicts)
constexpr int kGWaves = 8, kGCols = 32 * kGWaves;  // waves and output columns per workgroup
constexpr int kGList = 1024;  // rows of a unit at most (their routes are listed in LDS)
constexpr int kGMaxE = 4096;  // experts with a counter (in the LDS that holds x later)
constexpr int kGFurther = 128;  // workgroups for units past the experts' first ones, about
constexpr int gather_rows_sbstride(int K) { return (K / 128) | 1; }
constexpr size_t gather_rows_lds(int mt, int K) {
  return 2ull * 16 * mt * kGXS * 2 + 2ull * 16 * mt * 4 * 4 + 8ull * kGCols * gather_rows_sbstride(K);
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// the 8 nibbles of a word as bf16 128 + q, in the order of permute_pairs
__device__ __forceinline__ bf16x8_t nibbles_bf16(uint32_t w, const NibbleK& k) {
  uint4 r;
  r.x = (w & k.mask) | k.magic;
  r.y = ((w >> 4) & k.mask) | k.magic;
  r.z = ((w >> 8) & k.mask) | k.magic;
  r.w = ((w >> 12) & k.mask) | k.magic;
  return __builtin_bit_cast(bf16x8_t, r);
}

// MT: 16-row tiles of x
template <int MT>
__global__ void __launch_bounds__(64 * kGWaves, MT == 4 ? 2 : 4) gather_rows_kernel(const GatherParams p) {
  constexpr int T = 64 * kGWaves, NT = 2, D = kGChunkK / 128;
  constexpr int XU = 16 * MT * (kGChunkK / 8) / T;  // 16-byte units of an x chunk per thread
  extern __shared__ __align__(16) unsigned char smem[];
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem);                             // [2][16 MT][kGXS]
  float* sxs = reinterpret_cast<float*>(smem + 2 * 16 * MT * kGXS * 2);         // [2][16 MT][4]: sums of a group
  uint2* sbs = reinterpret_cast<uint2*>(sxs + 2 * 16 * MT * 4);                 // [kGCols][sbstride]: s pair, b pair
  __shared__ uint16_t list[kGList + 1];
  __shared__ int wsum[kGWaves];
  __shared__ int unit_of[2];  // expert, unit of it
  const int K = p.K, S = K / 128, C = K / kGChunkK;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * kGCols;
  // ---- the experts of the routes; a thread's first ID (every T-th) stay in
  // registers ----
  constexpr int ID = 8;
  auto expert_of = [&](int r) {
    return static_cast<int>(min(p.rhs ? p.rhs[r] : static_cast<uint32_t>(r), static_cast<uint32_t>(p.E - 1)));
  };
  int id[ID];
  {
    uint32_t v[ID];  // (every load issued before one is waited for)
#pragma unroll
    for (int u = 0; u < ID; u++) v[u] = static_cast<uint32_t>(u * T + tid);
    if (p.rhs) {
#pragma unroll
      for (int u = 0; u < ID; u++) v[u] = p.rhs[min(u * T + tid, p.R - 1)];
    }
#pragma unroll
    for (int u = 0; u < ID; u++)
      id[u] = u * T + tid < p.R ? static_cast<int>(min(v[u], static_cast<uint32_t>(p.E - 1))) : -1;
  }
  // exclusive prefix sum over the workgroup's threads, and the total (a second
  // use needs a barrier after the first)
  int total = 0;
  auto prefix = [&](int v) {
    int incl = v;
    for (int off = 1; off < 64; off <<= 1) {
      const int w = __shfl_up(incl, off, 64);
      if (lane >= off) incl += w;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int before = incl - v;
    total = 0;
#pragma unroll
    for (int w = 0; w < kGWaves; w++) {
      if (w < wave) before += wsum[w];
      total += wsum[w];
    }
    return before;
  };
  // ---- this workgroup's unit: expert e, its rows from t0 on ----
  const int UM = p.run * 16 * MT;  // rows of a unit
  int e = blockIdx.y, t0 = 0;
  if (e >= p.E) {  // a further unit: thread i owns experts i EP .. + EP - 1
    int* counts = reinterpret_cast<int*>(smem);
    for (int i = tid; i < p.E; i += T) counts[i] = 0;
    if (tid == 0) unit_of[0] = -1;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < ID; u++)
      if (id[u] >= 0) atomicAdd(&counts[id[u]], 1);
    for (int r = ID * T + tid; r < p.R; r += T) atomicAdd(&counts[expert_of(r)], 1);
    __syncthreads();
    const int EP = (p.E + T - 1) / T, e0 = tid * EP, e1 = min(e0 + EP, p.E);
    auto further = [&](int i) { return max(counts[i] * p.M - 1, 0) / UM; };
    int mine = 0;
    for (int i = e0; i < e1; i++) mine += further(i);
    int at = e - p.E - prefix(mine);
    if (at >= 0 && at < mine) {  // one thread, if any
      int i = e0;
      for (int n = further(i); at >= n; n = further(i)) {
        at -= n;
        i++;
      }
      unit_of[0] = i;
      unit_of[1] = at + 1;
    }
    __syncthreads();
    e = unit_of[0];
    t0 = unit_of[1] * UM;
    if (e < 0) return;  // uniform: no such unit
  }
  int cnt = 0;
#pragma unroll
  for (int u = 0; u < ID; u++) cnt += id[u] == e;
  for (int r = ID * T + tid; r < p.R; r += T) cnt += expert_of(r) == e;
  int idx = prefix(cnt);
  const int rows = total * p.M;
  if (rows == 0) return;  // uniform

  // ---- this wave's W rows (word offsets inside the expert) ----
  const uint32_t* we = p.w + static_cast<int64_t>(e) * p.N * (K / 8);
  uint32_t wo[NT];
  int n[NT];
#pragma unroll
  for (int j = 0; j < NT; j++) {
    n[j] = n0 + (wave * NT + j) * 16 + li;
    wo[j] = static_cast<uint32_t>(min(n[j], p.N - 1)) * static_cast<uint32_t>(K / 8) + q * 4;
  }
  uint4 wr[D][NT];
  auto load_w = [&](int u, int step) {
#pragma unroll
    for (int j = 0; j < NT; j++) wr[u][j] = *reinterpret_cast<const uint4*>(we + (wo[j] + step * 16));
  };
  // ---- the unit's rows, t0 .. end - 1 of the expert's, as its routes first ..
  // last in thread order ----
  const int end = min(t0 + UM, rows), first = t0 / p.M, last = (end - 1) / p.M;
  if (cnt > 0) {
    idx -= first;
    auto put = [&](int r) {
      if (idx >= 0 && idx <= last - first) list[idx] = static_cast<uint16_t>(r);
      idx++;
    };
#pragma unroll
    for (int u = 0; u < ID; u++)
      if (id[u] == e) put(u * T + tid);
    for (int r = ID * T + tid; r < p.R; r += T)
      if (expert_of(r) == e) put(r);
  }
  __syncthreads();

  // ---- s and b of the workgroup's columns (a contiguous block of each) ----
  const int SB = gather_rows_sbstride(K);
  {
    const int64_t base = (static_cast<int64_t>(e) * p.N + n0) * S;  // in words: S = G / 2 per row
    const uint32_t* se = reinterpret_cast<const uint32_t*>(p.s) + base;
    const uint32_t* be = reinterpret_cast<const uint32_t*>(p.b) + base;
    const int words = min(kGCols, p.N - n0) * S;
    const float rcp = 1.0f / static_cast<float>(S);
    for (int i0 = 0; i0 < words; i0 += 4 * T) {
      uint32_t sv[4], bv[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int i = min(i0 + u * T + tid, words - 1);
        sv[u] = se[i];
        bv[u] = be[i];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int i = min(i0 + u * T + tid, words - 1);
        const int row = udiv_small(i, rcp);
        sbs[row * SB + i - row * S] = make_uint2(sv[u], bv[u]);
      }
    }
  }
  const NibbleK nk = nibble_consts();
  const f32x4_t zero{0.0f, 0.0f, 0.0f, 0.0f};

  for (int t = t0; t < end; t += 16 * MT) {
    // this thread's part of an x chunk: 16-byte units tid + k T of
    // [16 MT rows][kGChunkK / 8 units]
    constexpr int UR = kGChunkK / 8;  // units per row
    const uint16_t* xp[XU];
#pragma unroll
    for (int k = 0; k < XU; k++) {
      const int unit = tid + k * T;
      const int j = min(t + unit / UR, end - 1);
      const int lr = p.M == 1 ? j : j / p.M, m = j - lr * p.M;
      const int route = list[lr - first];
      const int64_t xb = p.lhs ? min(p.lhs[route], static_cast<uint32_t>(p.nxb - 1)) : route / p.x_bcast;
      xp[k] = p.x + xb * p.x_rstride + static_cast<int64_t>(m) * K + (unit % UR) * 8;
    }
    uint4 xr[XU];
    auto load_x = [&](int c) {
#pragma unroll
      for (int k = 0; k < XU; k++) xr[k] = *reinterpret_cast<const uint4*>(xp[k] + c * kGChunkK);
    };
    auto store_x = [&](int c) {
#pragma unroll
      for (int k = 0; k < XU; k++) {
        const int unit = tid + k * T, row = (c & 1) * 16 * MT + unit / UR;
        *reinterpret_cast<uint4*>(xs + row * kGXS + (unit % UR) * 8) = permute_pairs(xr[k]);
        // a group is 8 units = 8 consecutive lanes
        const float sum = lanes_sum(gemv_unit_sum(xr[k]), 8);
        if ((unit & 7) == 0) sxs[row * 4 + (unit % UR) / 8] = sum;
      }
    };
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++) acc[i][j] = zero;
    auto compute = [&](int u, int c) {
      // lanes q 0, 1 hold a row's 8 words of the step's first group, q 2, 3
      // of the second; after the swaps every lane holds words
      // 4 (q & 1) + 2 (q >> 1) + {0, 1} of each
      uint4 v[NT];
      uint32_t sw[NT];
#pragma unroll
      for (int j = 0; j < NT; j++) {
        const auto a = __builtin_amdgcn_permlane32_swap(wr[u][j].x, wr[u][j].z, false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(wr[u][j].y, wr[u][j].w, false, false);
        v[j] = make_uint4(a[0], b[0], a[1], b[1]);
        sw[j] = sbs[((wave * NT + j) * 16 + li) * SB + c * D + u].x;
      }
      const uint16_t* xt = xs + ((c & 1) * 16 * MT + li) * kGXS + u * 128 + (q & 1) * 32 + (q >> 1) * 16;
#pragma unroll
      for (int g = 0; g < 2; g++) {
        bf16x8_t xa[MT][2];
#pragma unroll
        for (int i = 0; i < MT; i++) {
          xa[i][0] = *reinterpret_cast<const bf16x8_t*>(xt + i * 16 * kGXS + g * 64);
          xa[i][1] = *reinterpret_cast<const bf16x8_t*>(xt + i * 16 * kGXS + g * 64 + 8);
        }
#pragma unroll
        for (int j = 0; j < NT; j++) {
          const bf16x8_t b0 = nibbles_bf16(g == 0 ? v[j].x : v[j].z, nk);
          const bf16x8_t b1 = nibbles_bf16(g == 0 ? v[j].y : v[j].w, nk);
          const float sv = __uint_as_float(g == 0 ? sw[j] << 16 : sw[j] & 0xffff0000u);
          f32x4_t d[MT];
#pragma unroll
          for (int i = 0; i < MT; i++) d[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][0], b0, zero, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < MT; i++) d[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][1], b1, d[i], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < MT; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = __builtin_fmaf(sv, d[i][r], acc[i][j][r]);
        }
      }
    };
    // + (b - 128 s) Sx of the chunk's four groups, lane (li, q): row li's
    // sum and column li's factor of group q
    auto bias = [&](int c) {
      float sx[MT];
#pragma unroll
      for (int i = 0; i < MT; i++) sx[i] = sxs[((c & 1) * 16 * MT + i * 16 + li) * 4 + q];
#pragma unroll
      for (int j = 0; j < NT; j++) {
        const uint2 sb = sbs[((wave * NT + j) * 16 + li) * SB + c * D + (q >> 1)];
        const float sv = __uint_as_float((q & 1) ? sb.x & 0xffff0000u : sb.x << 16);
        const float bv = __uint_as_float((q & 1) ? sb.y & 0xffff0000u : sb.y << 16);
        const float bb = __builtin_fmaf(-128.0f, sv, bv);
#pragma unroll
        for (int i = 0; i < MT; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[i], bb, acc[i][j], 0, 0, 0);
      }
    };
    // chunk c + 1: x into registers at the top of chunk c, ahead of the W
    // loads of its steps (loads complete in order, so the x stores at the
    // bottom leave those in flight), each W step into the registers the
    // step before it freed.  Loads past the last chunk repeat it.
    load_x(0);
#pragma unroll
    for (int u = 0; u < D; u++) load_w(u, u);
    store_x(0);
    __syncthreads();
    for (int c = 0; c < C; c++) {
      const int cn = min(c + 1, C - 1);
      load_x(cn);
#pragma unroll
      for (int u = 0; u < D; u++) {
        __builtin_amdgcn_sched_barrier(0);
        compute(u, c);
        __builtin_amdgcn_sched_barrier(0);
        load_w(u, cn * D + u);
      }
      bias(c);
      // chunk c - 1's buffer: its reads ended before the last barrier
      store_x(c + 1);
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int j = t + i * 16 + 4 * q + r;
        if (j >= end) continue;
        const int lr = p.M == 1 ? j : j / p.M, m = j - lr * p.M;
        uint16_t* yr = p.y + static_cast<int64_t>(list[lr - first]) * p.y_rstride + static_cast<int64_t>(m) * p.N;
#pragma unroll
        for (int k = 0; k < NT; k++)
          if (n[k] < p.N) yr[n[k]] = f2bf(acc[i][k][r]);
      }
  }
}

// units past the experts' first ones that R routes of M rows can make
int64_t gather_rows_further(int unit_rows, int M, int R) { return static_cast<int64_t>(R) * M / unit_rows; }

// Whether the routes of an expert are better multiplied together, from what
// both kernels take (us; 1 to 128 experts, 1 to 50 routes each, 200 x 256 to
// 14336 x 4096, 1 to 8 rows a route): per route every route's weights at the
// caches' rate, and each expert's once from memory; by expert the chain of K
// chunks that a workgroup walks, or each expert's weights once from memory.
// 1536 x 2048, per route and by expert: 8 experts 16 routes 7.6 and 16.6, 80
// routes 18.9 and 17.4; 32 experts 40 routes 16.7 and 18.3; 128 experts 160
// routes 40.7 and 34.6, 1280 routes 259 and 58.  It picks the slower one by
// more than 5% only near the line, at most 12% over those shapes (4 experts of
// 14336 x 4096, 6 routes: per route 33.1, by expert 29.5).
// (Below 1.25 routes an expert the weights are hardly read twice.)
bool gather_by_expert(int E, int M, int N, int K, int R) {
  if (4ll * R < 5ll * E) return false;
  const double mb = static_cast<double>(N) * K * 0.5625e-6, used = mb * E * (1.0 - exp(-static_cast<double>(R) / E));
  const double per_route = 3.7 + M * (0.2 + 0.35 * K / 1024.0) + R * (0.005 + (1.0 + 0.4 * (M - 1)) * mb / 9.5) +
                           used / 16.0;
  const double chain = 5.5 + 5.1 * K / 1024.0, by_expert = std::max(chain, 0.4 * chain + used / 4.3);
  return 1.06 * by_expert < per_route;
}

template <int MT>
int launch_gather_rows(GatherParams p, hipStream_t stream) {
  const size_t lds = gather_rows_lds(MT, p.K);
  if (int rc = allow_lds(gather_rows_kernel<MT>, lds)) return rc;
  const int cols = (p.N + kGCols - 1) / kGCols;
  // Tiles per unit: one where the CUs hold every unit there can be; else so
  // many that the further units are few, since an even routing leaves them
  // nothing to do (2664 routes over 128 experts, 1536 x 2048 and 2048 x 768:
  // 122 us with one tile a unit, 112 so; with 90% of the routes to one expert
  // the first takes 90 us so and 136, of 1125 with an expert to a workgroup)
  const int64_t most = gather_rows_further(16 * MT, p.M, p.R), rows = std::max(1, kGFurther / cols);
  p.run = 1;
  if (cols * (std::min(p.E, p.R) + most) > 256)
    p.run = static_cast<int>(std::min<int64_t>((most + rows - 1) / rows, kGList / (16 * MT)));
  if (p.run < 1) p.run = 1;
  const dim3 grid(cols, p.E + static_cast<unsigned>(gather_rows_further(p.run * 16 * MT, p.M, p.R)));
  hipLaunchKernelGGL(gather_rows_kernel<MT>, grid, dim3(64 * kGWaves), lds, stream, p);
  return check_launch("gather_qmm rows");
}

}  // namespace

int launch_gather_qmm(const uint16_t* x, const uint32_t* w, const uint16_t* s, const uint16_t* b,
                      const uint32_t* lhs, const uint32_t* rhs, uint16_t* y, int R, int x_bcast, int nxb,
                      int64_t x_rstride, int64_t y_rstride, int E, int M, int N, int K, hipStream_t stream) {
  if (R == 0) return BMX_OK;
  if (R < 0 || R > 65535 || E <= 0 || M <= 0 || N <= 0 || K <= 0 || x_bcast <= 0 || nxb <= 0)
    return set_error(BMX_E_SHAPE, "gather_qmm: bad sizes R=%d E=%d M=%d N=%d K=%d x_bcast=%d x blocks=%d", R, E, M,
                     N, K, x_bcast, nxb);
  if (K % 64) return set_error(BMX_E_SHAPE, "gather_qmm: K=%d not a multiple of the group size 64", K);
  if (M > kGMaxM) return set_error(BMX_E_UNSUPPORTED, "gather_qmm: M=%d rows per route (at most %d)", M, kGMaxM);
  const int G = K / 64;
  // lanes per row: the fewest (a power of two) that keep a lane at or under
  // kGMaxNG groups, then more while the grid is under 512 workgroups and
  // every lane keeps a group
  int S = 1;
  while (S < 64 && (G + S - 1) / S > kGMaxNG) S *= 2;
  if ((G + S - 1) / S > kGMaxNG)
    return set_error(BMX_E_UNSUPPORTED, "gather_qmm: K=%d above %d", K, 64 * 64 * kGMaxNG);
  auto tiles = [&](int s) { return static_cast<int64_t>((N + 4 * (64 / s) - 1) / (4 * (64 / s))) * R; };
  while (S < 64 && 2 * S <= G && tiles(S) < 512) S *= 2;
  const int mt = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : 8;
  const size_t lds = static_cast<size_t>(mt) * (K / 32) * (kGChunk + 4);
  if (lds > 160 * 1024) return set_error(BMX_E_UNSUPPORTED, "gather_qmm: M*K=%d too large", M * K);
  const int rb = 4 * (64 / S);
  GatherParams p{x, w, s, b, lhs, rhs, y, x_rstride, y_rstride, x_bcast, nxb, E, M, N, K, S, R, 1};
  if (E <= kGMaxE && K % kGChunkK == 0 && aligned(s, 4) && aligned(b, 4) &&
      gather_rows_lds(4, K) <= 160 * 1024 - 4096 && static_cast<int64_t>(N) * (K / 8) <= UINT32_MAX &&
      gather_by_expert(E, M, N, K, R)) {
    // the rows an expert gets on average decide the tile; shorter ones where
    // those leave CUs idle too (1536 x 2048, 8 experts, 400 routes: 32 rows
    // 20.8 us, 16 rows 17.8; 32 experts, 640 routes, 420 workgroups of 16
    // rows: 23.3 and 30.6)
    const int64_t rows = static_cast<int64_t>(R) * M;
    const int64_t avg = (rows + E - 1) / E, cols = (N + kGCols - 1) / kGCols;
    int t = avg <= 8 ? 1 : avg <= 48 ? 2 : 4;
    while (t > 1 && cols * (std::min(E, R) + gather_rows_further(8 * t, M, R)) <= 256) t /= 2;
    return t == 1   ? launch_gather_rows<1>(p, stream)
           : t == 2 ? launch_gather_rows<2>(p, stream)
                    : launch_gather_rows<4>(p, stream);
  }
  const dim3 grid((N + rb - 1) / rb, R);
  const void* kern = mt == 1   ? reinterpret_cast<const void*>(gather_qmv_kernel<1>)
                     : mt == 2 ? reinterpret_cast<const void*>(gather_qmv_kernel<2>)
                     : mt == 4 ? reinterpret_cast<const void*>(gather_qmv_kernel<4>)
                               : reinterpret_cast<const void*>(gather_qmv_kernel<8>);
  if (lds > 64 * 1024)
    if (int rc = allow_lds_ptr(kern, lds)) return rc;
  switch (mt) {
    case 1: hipLaunchKernelGGL(gather_qmv_kernel<1>, grid, dim3(kGThreads), lds, stream, p); break;
    case 2: hipLaunchKernelGGL(gather_qmv_kernel<2>, grid, dim3(kGThreads), lds, stream, p); break;
    case 4: hipLaunchKernelGGL(gather_qmv_kernel<4>, grid, dim3(kGThreads), lds, stream, p); break;
    default: hipLaunchKernelGGL(gather_qmv_kernel<8>, grid, dim3(kGThreads), lds, stream, p);
  }
  return check_launch("gather_qmm");
}

}  // namespace bmx

using namespace bmx;

extern "C" int bmx_gather_qmm(const bmx_bf16* x, const uint32_t* w, const bmx_bf16* scales, const bmx_bf16* biases,
                              const uint32_t* rhs_indices, bmx_bf16* out, int n_routes, int x_bcast, int n_experts,
                              int M, int N, int K, int group_size, int bits, void* stream) {
  if (!x || !w || !scales || !biases || !out || (!rhs_indices && n_routes > 0))
    return set_error(BMX_E_ARG, "gather_qmm: null pointer");
  if (bits != 4 || group_size != 64)
    return set_error(BMX_E_UNSUPPORTED, "gather_qmm: only bits=4, group_size=64 (got %d, %d)", bits, group_size);
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15)
    return set_error(BMX_E_ALIGN, "gather_qmm: x and w must be 16-byte aligned");
  const int nxb = x_bcast > 0 ? (n_routes + x_bcast - 1) / x_bcast : 0;  // x blocks the routes read
  return launch_gather_qmm(x, w, scales, biases, nullptr, rhs_indices, out, n_routes, x_bcast, nxb,
                           static_cast<int64_t>(M) * K, static_cast<int64_t>(M) * N, n_experts, M, N, K,
                           as_stream(stream));
}

extern "C" int bmx_gather_qmm_indexed(const bmx_bf16* x, const uint32_t* w, const bmx_bf16* scales,
                                      const bmx_bf16* biases, const uint32_t* lhs_indices,
                                      const uint32_t* rhs_indices, bmx_bf16* out, int n_routes, int n_x_blocks,
                                      int n_experts, int M, int N, int K, int transpose, int group_size, int bits,
                                      int sorted_indices, void* stream) {
  (void)sorted_indices;  // a grouping hint in MLX; the results do not depend on it
  if (!x || !w || !scales || !biases || !out) return set_error(BMX_E_ARG, "gather_qmm: null pointer");
  if (!transpose) return set_error(BMX_E_UNSUPPORTED, "gather_qmm: transpose=false is not supported");
  if (bits != 4 || group_size != 64)
    return set_error(BMX_E_UNSUPPORTED, "gather_qmm: only bits=4, group_size=64 (got %d, %d)", bits, group_size);
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15)
    return set_error(BMX_E_ALIGN, "gather_qmm: x and w must be 16-byte aligned");
  if (n_x_blocks <= 0 || n_routes < 0) return set_error(BMX_E_SHAPE, "gather_qmm: %d x blocks", n_x_blocks);
  // without lhs_indices the x blocks broadcast evenly over the routes
  if (!lhs_indices && n_routes % n_x_blocks)
    return set_error(BMX_E_SHAPE, "gather_qmm: %d routes over %d x blocks without lhs_indices", n_routes, n_x_blocks);
  // without rhs_indices route r uses expert r
  if (!rhs_indices && n_routes != n_experts)
    return set_error(BMX_E_SHAPE, "gather_qmm: %d routes and %d experts without rhs_indices", n_routes, n_experts);
  const int x_bcast = lhs_indices || n_routes == 0 ? 1 : n_routes / n_x_blocks;
  return launch_gather_qmm(x, w, scales, biases, lhs_indices, rhs_indices, out, n_routes, x_bcast, n_x_blocks,
                           static_cast<int64_t>(M) * K, static_cast<int64_t>(M) * N, n_experts, M, N, K,
                           as_stream(stream));
}
