// Greedy argmax and the elementwise ops of a Qwen3 block (gfx950).
//
// Semantics restated:
//   argmax / argmax_axis over the last axis (engine.rs:195-202,
//     speculative.rs:168-173, 289-293): index of the largest value, the
//     first such index on ties, as uint32;
//   mlp_block activation silu(g) * up (model/kernels.rs:73-74): each MLX op
//     rounds to bf16 -- sigmoid, g * sigmoid, then * up;
//   residual add `&x + &y` in bf16 (qwen3.rs:521, 541).
#include <math.h>

#include "bmx_device.h"

namespace bmx {
namespace {

constexpr int kArgThreads = 1024;

__device__ __forceinline__ bool better(float v, uint32_t i, float bv, uint32_t bi) {
  return v > bv || (v == bv && i < bi);
}

// (value, index) reduction across a workgroup of kArgThreads; the result is
// valid in thread 0.
__device__ __forceinline__ void block_best(float& bv, uint32_t& bi) {
  __shared__ float sv[kArgThreads / 64];
  __shared__ uint32_t si[kArgThreads / 64];
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(bv, off, 64);
    const uint32_t oi = __shfl_xor(bi, off, 64);
    if (better(ov, oi, bv, bi)) {
      bv = ov;
      bi = oi;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    sv[wave] = bv;
    si[wave] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kArgThreads / 64; w++)
      if (better(sv[w], si[w], bv, bi)) {
        bv = sv[w];
        bi = si[w];
      }
  }
}

// Row 0's token handed to the next decode step (see DecodeChain): the step's
// token and position advance in device memory, and the token goes to the
// next slot of the host ring as one system-scope store (straight to host
// memory, visible to the polling host without a copy or a stream sync).
__device__ __forceinline__ void chain_publish(const DecodeChain& ch, uint32_t tok) {
  int* io = ch.io;
  io[0] = static_cast<int>(tok);
  io[1] += 1;
  const unsigned k = static_cast<unsigned>(io[3]);
  io[3] = static_cast<int>(k + 1);
  __hip_atomic_store(ch.ring + (k & ch.mask), tok, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// One workgroup per row; rows of a multiple of 8 values at 16-byte alignment
// are read 8 values per load, B loads in flight per thread.  A row is one
// CU's work, so instructions bound it once the loads overlap: a thread keeps
// the largest value and the 16-byte unit it first stood in (three operations
// per pair of values and three per unit, against five per value with an
// index each), and looks the position up in that unit at the end.
// 5 rows of 151936: 14.6 -> 8.2 us.  W: waves per SIMD that the registers
// leave room for: 4 (one workgroup per CU, 10 loads) up to a row per CU, 8 (two,
// 8 loads) for more rows, whose second workgroups else wait for the first (300
// rows of 151937, not a multiple of 8: 57 us, 103 at 4).
template <int B, int W>
__global__ void __launch_bounds__(kArgThreads, W)
    argmax_kernel(const uint16_t* __restrict__ x, int64_t n, uint32_t* __restrict__ out, const DecodeChain ch) {
  const uint16_t* xr = x + static_cast<int64_t>(blockIdx.x) * n;
  float bv = -INFINITY;
  uint32_t bi = 0xffffffffu;
  if (n % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0) {
    const uint4* xv = reinterpret_cast<const uint4*>(xr);
    const int64_t nv = n / 8;
    int64_t bj = -1;
    for (int64_t j0 = threadIdx.x; j0 < nv; j0 += static_cast<int64_t>(kArgThreads) * B) {
      uint4 d[B];
#pragma unroll
      for (int u = 0; u < B; u++) d[u] = xv[min(j0 + static_cast<int64_t>(u) * kArgThreads, nv - 1)];
      // (a unit past the end repeats the row's last one: a thread that had not
      // read that may take its value here, and means it -- see the min below;
      // a NaN loses every comparison)
#pragma unroll
      for (int u = 0; u < B; u++) {
        const uint32_t w[4] = {d[u].x, d[u].y, d[u].z, d[u].w};
        float m = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float lo = __uint_as_float(w[e] << 16), hi = __uint_as_float(w[e] & 0xffff0000u);
          m = lo > m ? lo : m;
          m = hi > m ? hi : m;
        }
        if (m > bv) {
          bv = m;
          bj = j0 + static_cast<int64_t>(u) * kArgThreads;
        }
      }
    }
    // nothing above -inf: the first -inf this thread holds, if any (its other
    // values are NaN)
    for (int64_t j = threadIdx.x; bj < 0 && j < nv; j += kArgThreads) {
      const uint4 d = xv[j];
      const uint32_t w[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
      for (int e = 0; e < 4; e++)
        if ((w[e] & 0xffffu) == 0xff80u || (w[e] >> 16) == 0xff80u) bj = j;
    }
    if (bj >= 0) {
      bj = min(bj, nv - 1);
      const uint4 d = xv[bj];
      const uint32_t w[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
      for (int e = 7; e >= 0; e--)
        if (bf2f((w[e >> 1] >> (16 * (e & 1))) & 0xffffu) == bv) bi = static_cast<uint32_t>(bj * 8 + e);
    }
  } else {
    for (int64_t i = threadIdx.x; i < n; i += kArgThreads) {
      const float v = bf2f(xr[i]);
      if (better(v, static_cast<uint32_t>(i), bv, bi)) {
        bv = v;
        bi = static_cast<uint32_t>(i);
      }
    }
  }
  block_best(bv, bi);
  // all -inf / NaN rows: index 0
  if (threadIdx.x == 0) {
    const uint32_t tok = bi == 0xffffffffu ? 0u : bi;
    out[blockIdx.x] = tok;
    if (ch.io != nullptr && blockIdx.x == 0) chain_publish(ch, tok);
  }
}

// one workgroup per row over the per-workgroup partials (value bits, index)
// of the GEMV epilogue
__global__ void __launch_bounds__(kArgThreads)
    argmax_partials_kernel(const uint2* __restrict__ part, int nblk, uint32_t* __restrict__ out,
                           const DecodeChain ch) {
  const uint2* pr = part + static_cast<int64_t>(blockIdx.x) * nblk;
  float bv = -INFINITY;
  uint32_t bi = 0xffffffffu;
  constexpr int B = 8;
  for (int j0 = threadIdx.x; j0 < nblk; j0 += kArgThreads * B) {
    uint2 d[B];
#pragma unroll
    for (int u = 0; u < B; u++) {
      const int j = j0 + u * kArgThreads;
      d[u] = j < nblk ? pr[j] : make_uint2(0xff800000u, 0xffffffffu);
    }
#pragma unroll
    for (int u = 0; u < B; u++) {
      const float v = __uint_as_float(d[u].x);
      if (better(v, d[u].y, bv, bi)) {
        bv = v;
        bi = d[u].y;
      }
    }
  }
  block_best(bv, bi);
  if (threadIdx.x == 0) {
    const uint32_t tok = bi == 0xffffffffu ? 0u : bi;
    out[blockIdx.x] = tok;
    if (ch.io != nullptr && blockIdx.x == 0) chain_publish(ch, tok);
  }
}

__device__ __forceinline__ uint16_t silu_mul_one(uint16_t g, uint16_t u) {
  const float gv = bf2f(g);
  const float sg = round_bf(1.0f / (1.0f + expf(-gv)));
  return f2bf(round_bf(gv * sg) * bf2f(u));
}
__device__ __forceinline__ uint16_t add_one(uint16_t a, uint16_t b) { return f2bf(bf2f(a) + bf2f(b)); }

// y = OP(a, b) elementwise: 8 values (16 bytes) per thread and array where
// all three are 16-byte aligned and n is a multiple of 8, else one.
// One value per thread is bound by issuing memory instructions: add of 10.5M
// values 19.9 -> 10.7 us, silu_mul of 19.9M 33.3 -> 22.0 (119 MB: the rate of
// memory).  y may be a or b (each thread reads its values before it writes
// them).
template <uint16_t (*OP)(uint16_t, uint16_t), bool VEC>
__global__ void __launch_bounds__(256) elementwise_kernel(const uint16_t* a, const uint16_t* b, uint16_t* y, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if constexpr (VEC) {
    if (i * 8 >= n) return;
    const uint4 av = reinterpret_cast<const uint4*>(a)[i], bv = reinterpret_cast<const uint4*>(b)[i];
    const uint32_t aw[4] = {av.x, av.y, av.z, av.w}, bw[4] = {bv.x, bv.y, bv.z, bv.w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
      o[e] = static_cast<uint32_t>(OP(aw[e] & 0xffffu, bw[e] & 0xffffu)) |
             (static_cast<uint32_t>(OP(aw[e] >> 16, bw[e] >> 16)) << 16);
    reinterpret_cast<uint4*>(y)[i] = make_uint4(o[0], o[1], o[2], o[3]);
  } else {
    if (i < n) y[i] = OP(a[i], b[i]);
  }
}

// (small arrays spread over more CUs one value per thread: 8 values a thread
// from `from` values on)
template <uint16_t (*OP)(uint16_t, uint16_t)>
int launch_elementwise(const char* what, const uint16_t* a, const uint16_t* b, uint16_t* y, int64_t n, int64_t from,
                       hipStream_t stream) {
  if (n <= 0) return BMX_OK;
  const bool vec = n % 8 == 0 && n >= from && aligned(a, 16) && aligned(b, 16) && aligned(y, 16);
  const int64_t threads = vec ? n / 8 : n;
  const dim3 grid(static_cast<unsigned>((threads + 255) / 256));
  if (vec) hipLaunchKernelGGL((elementwise_kernel<OP, true>), grid, dim3(256), 0, stream, a, b, y, n);
  else hipLaunchKernelGGL((elementwise_kernel<OP, false>), grid, dim3(256), 0, stream, a, b, y, n);
  return check_launch(what);
}

// dst[i] = src[i] (token ids u32 -> i32 for the embedding gather)
__global__ void tokens_to_ids_kernel(const uint32_t* __restrict__ src, int32_t* __restrict__ dst, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = static_cast<int32_t>(src[i]);
}

}  // namespace

int launch_argmax(const uint16_t* x, int64_t rows, int64_t n, uint32_t* out, hipStream_t stream,
                  const DecodeChain* chain) {
  if (rows <= 0) return BMX_OK;
  if (n <= 0 || n > UINT32_MAX) return set_error(BMX_E_SHAPE, "argmax: n=%lld", (long long)n);
  if (rows > INT32_MAX) return set_error(BMX_E_SHAPE, "argmax: rows=%lld", (long long)rows);
  if (chain && (rows != 1 || !chain->io || !chain->ring)) return set_error(BMX_E_ARG, "argmax: chained hand-off of %lld rows", (long long)rows);
  const DecodeChain ch = chain ? *chain : DecodeChain{};
  const dim3 grid(static_cast<unsigned>(rows));
  if (rows <= 256) hipLaunchKernelGGL((argmax_kernel<10, 4>), grid, dim3(kArgThreads), 0, stream, x, n, out, ch);
  else hipLaunchKernelGGL((argmax_kernel<8, 8>), grid, dim3(kArgThreads), 0, stream, x, n, out, ch);
  return check_launch("argmax");
}

int launch_argmax_partials(const uint2* part, int rows, int nblk, uint32_t* out, hipStream_t stream,
                           const DecodeChain* chain) {
  if (rows <= 0) return BMX_OK;
  if (nblk <= 0) return set_error(BMX_E_SHAPE, "argmax partials: %d per row", nblk);
  if (chain && (rows != 1 || !chain->io || !chain->ring)) return set_error(BMX_E_ARG, "argmax: chained hand-off of %d rows", rows);
  const DecodeChain ch = chain ? *chain : DecodeChain{};
  hipLaunchKernelGGL(argmax_partials_kernel, dim3(rows), dim3(kArgThreads), 0, stream, part, nblk, out, ch);
  return check_launch("argmax_partials");
}

int launch_silu_mul(const uint16_t* g, const uint16_t* u, uint16_t* y, int64_t n, hipStream_t stream) {
  // one value per thread and 8, us: 359936 values 2.36 and 2.65, 749056 3.06
  // and 3.36, 1048576 3.62 and 3.60, 2097152 5.23 and 4.82
  return launch_elementwise<silu_mul_one>("silu_mul", g, u, y, n, 1 << 20, stream);
}

int launch_add(const uint16_t* a, const uint16_t* b, uint16_t* y, int64_t n, hipStream_t stream) {
  // one value per thread and 8, us: 262144 values 2.16 and 2.25, 524288 2.43
  // and 2.59, 749056 3.00 and 2.71, 2097152 4.84 and 3.59
  return launch_elementwise<add_one>("add", a, b, y, n, 10 << 16, stream);
}

int launch_tokens_to_ids(const uint32_t* src, int32_t* dst, int n, hipStream_t stream) {
  if (n <= 0) return BMX_OK;
  hipLaunchKernelGGL(tokens_to_ids_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, src, dst, n);
  return check_launch("tokens_to_ids");
}

}  // namespace bmx

using namespace bmx;

extern "C" int bmx_argmax_rows(const bmx_bf16* x, int64_t rows, int64_t n, uint32_t* out, void* stream) {
  if (!x || !out) return set_error(BMX_E_ARG, "argmax: null pointer");
  return launch_argmax(x, rows, n, out, as_stream(stream));
}

extern "C" int bmx_silu_mul(const bmx_bf16* gate, const bmx_bf16* up, bmx_bf16* y, int64_t n, void* stream) {
  if (!gate || !up || !y) return set_error(BMX_E_ARG, "silu_mul: null pointer");
  return launch_silu_mul(gate, up, y, n, as_stream(stream));
}

extern "C" int bmx_add(const bmx_bf16* a, const bmx_bf16* b, bmx_bf16* y, int64_t n, void* stream) {
  if (!a || !b || !y) return set_error(BMX_E_ARG, "add: null pointer");
  return launch_add(a, b, y, n, as_stream(stream));
}
