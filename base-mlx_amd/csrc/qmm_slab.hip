// qmm_slab: the dequantizing GEMM (qmm.hip has its semantics) for tens to a
// few hundred rows of x, gfx950 bf16 MFMA.
//
// At these sizes a product is a few microseconds of work that the tile
// kernel of qmm.hip spends on waiting: per 64 columns of K it waits for
// memory one step ahead and meets at two barriers (about 2 us a step), it
// multiplies 128-row tiles whatever M is, and its small grids split K into
// partials that a second launch adds.  What bounds the work itself is the
// rate at which one CU pulls tiles out of L2 (45 KB/us measured), so this
// kernel moves as little as it can and never waits for one slab at a time:
//   * tiles of 16 MT rows of x (MT from M) by BN columns on 8 or 16 waves (16
//     up to 48 rows: 9728 x 2560 at 37 rows 13.6 -> 12.1 us), WN along the
//     columns (32 each) and the rest along K, whose partial tiles meet in
//     LDS at the end: a full CU per tile without partials in memory;
//   * K in slabs of KS groups, everything by global_load_lds: x rows and the
//     packed W rows (KS 32-byte pieces of a row are contiguous in MLX's
//     layout) into a ring of up to six slabs, all but one in flight while
//     that is multiplied, one barrier per slab; s and b of the tile once,
//     before the first slab;
//   * W dequantized from its packed words straight into the MFMA B operand,
//     once per tile (the waves along K and along N hold distinct words).
//
// (Registers instead of LDS for x and W, every wave on its own groups of K
// and no barrier, was slower than the tile kernel from 37 rows on: 32 us
// against 24 for 9728 x 2560.  Each wave then fetches its own x, and code
// unrolled to keep groups in flight runs once, at the rate instructions come
// from memory.)
//
// The loads are inline assembly with hand-placed waits: the compiler cannot
// tell the ring's slots apart and would wait for every load in flight
// before each LDS read.  They have no register results; every s_waitcnt
// the compiler adds for its own loads only waits longer than it must.
#include <algorithm>

#include "qmm_device.h"

namespace bmx {
namespace {

// waits until at most min(K, behind) slabs' loads (L each) are outstanding
template <int K, int L>
__device__ __forceinline__ void wait_behind(int behind) {
  if constexpr (K == 0) {
    vm_wait<0>();
  } else {
    if (behind >= K) vm_wait<K * L>();
    else wait_behind<K - 1, L>(behind);
  }
}

// bytes of one ring slot, and of a workgroup (sb: bytes of s and b)
constexpr size_t slab_slot(int mt, int bn, int ks) { return 16ull * mt * ks * 128 + 1ull * bn * ks * 32; }
constexpr size_t slab_lds(int mt, int bn, int ks, int ring, size_t sb) {
  const size_t a = ring * slab_slot(mt, bn, ks) + sb, b = 16ull * mt * bn * ks * 4;  // (waves along K: ks)
  return a > b ? a : b;
}

// position of a W row's logical piece c in its slab row: c ^ w_swz(row), so
// 16 rows' reads of one group spread over all banks (2 KS pieces per row)
template <int KS>
__device__ __forceinline__ int w_swz(int r) {
  return KS == 8 ? r & 15 : KS == 4 ? (r >> 1) & 7 : (r >> 2) & 3;
}

// waves and groups per slab of a tile
constexpr int slab_waves(int mt) { return mt <= 3 ? 16 : 8; }
constexpr int slab_groups(int mt, int bn) { return slab_waves(mt) / (bn / 32); }
// ring slots: as many as fit beside the s and b, at most 6 (more in flight
// than that gained nothing)
constexpr size_t kSlabLds = 160 * 1024;
constexpr int slab_ring(int mt, int bn, size_t sb) {
  const size_t slot = slab_slot(mt, bn, slab_groups(mt, bn));
  return sb >= kSlabLds ? 0 : (kSlabLds - sb) / slot > 6 ? 6 : static_cast<int>((kSlabLds - sb) / slot);
}
constexpr int slab_ring_max(int mt, int bn) { return slab_ring(mt, bn, 0); }
constexpr size_t slab_sb(const SlabPlan& s) { return 4ull * s.bn * s.gps; }

// EPI: as qmm_kernel (MLX-layout weights).  MT: 16-row tiles of x; BN: W
// rows per tile (SwiGLU: BN / 2 gate / up pairs).
template <int EPI, int MT, int BN>
__global__ void __launch_bounds__(64 * slab_waves(MT), slab_waves(MT) / 4) qmm_slab_kernel(const QmmParams p, const int R) {
  constexpr int NT = 2, NW = slab_waves(MT), KS = slab_groups(MT, BN), RMAX = slab_ring_max(MT, BN);
  constexpr int WN = BN / 32, WK = NW / WN;
  constexpr int BM = 16 * MT, CN = EPI == QMM_SWIGLU ? BN / 2 : BN;
  static_assert(KS % WK == 0 && KS >= 2, "every wave along K has whole groups of a slab");
  // 16-byte pieces per row of a slab; instructions of 64 pieces, per wave
  constexpr int XP = KS * 8, WP = KS * 2;
  constexpr int XI = BM * XP / 64, WI = BN * WP / 64;
  constexpr int XW = (XI + NW - 1) / NW, WW = (WI + NW - 1) / NW;
  constexpr size_t SLOT = slab_slot(MT, BN, KS);
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, q = lane >> 4;
  const int wn = wave % WN, wk = wave / WN;
  const int M = p.M, K = p.K, G = K / 64;
  const int m0 = blockIdx.y * BM;
  int n0 = blockIdx.x * CN, N = p.N;
  const uint32_t* pw = p.w;
  const uint16_t *ps = p.s, *pb = p.b;
  uint16_t* py = p.y;
  if constexpr (EPI == QMM_STORE) {
    if (p.nseg > 1) {
      const int si = (n0 >= p.seg_n0[1]) + (p.nseg > 2 && n0 >= p.seg_n0[2]);
      pw = p.seg_w[si];
      ps = p.seg_s[si];
      pb = p.seg_b[si];
      py = p.seg_y[si];
      n0 -= p.seg_n0[si];
      N = p.seg_n0[si + 1] - p.seg_n0[si];
    }
  }
  const int gb = blockIdx.z * p.gps, ge = min(G, gb + p.gps);
  const int ns = (ge - gb + KS - 1) / KS;
  // tile row r of W: its matrix and row (SwiGLU: a wave's 32 rows are 16 gate
  // rows and the up rows of the same columns; rows past N repeat the last)
  auto w_row = [&](int r) {
    return min(n0 + (EPI == QMM_SWIGLU ? (r >> 5) * 16 + (r & 15) : r), N - 1);
  };
  auto is_up = [&](int r) { return EPI == QMM_SWIGLU && (r & 16) != 0; };

  // ---- s, b of the tile: [array][BN][SB words of two groups], word c of
  // row r at (c + r) mod SB (rows of one word column in distinct banks) ----
  const int SB = p.gps / 2;
  unsigned char* sbl = smem + R * SLOT;
  const uint32_t* s_lds = reinterpret_cast<const uint32_t*>(sbl);
  const uint32_t* b_lds = s_lds + BN * SB;
  {
    const float rcp = 1.0f / static_cast<float>(SB);
    const int per = BN * SB;  // words of one array, a multiple of 64
    for (int i = wave; i < per / 64; i += NW) {
      const int idx = i * 64 + lane, r = udiv_small(idx, rcp);
      int c = idx - r * SB - r % SB;
      if (c < 0) c += SB;
      const int64_t at = static_cast<int64_t>(w_row(r)) * G + min(gb + 2 * c, G - 2);
      const bool up = is_up(r);
      lds_load4((up ? p.s2 : ps) + at, __builtin_amdgcn_readfirstlane(lds_offset(sbl) + i * 256));
      lds_load4((up ? p.b2 : pb) + at, __builtin_amdgcn_readfirstlane(lds_offset(sbl) + (per + i * 64) * 4));
    }
  }

  // ---- this lane's pieces of a slab: instruction i = wave + NW k fills
  // pieces 64 i .. + 63 of the slot's x (W) part; the piece at position c of
  // row r is logical piece c ^ swizzle(r), so the operand reads below fall
  // in distinct banks ----
  const unsigned char *xsrc[XW], *wsrc[WW];
  int xg[XW], wg[WW];
  uint32_t xdst[XW], wdst[WW];
#pragma unroll
  for (int k = 0; k < XW; k++) {
    const int i = min(wave + NW * k, XI - 1), pc = i * 64 + lane, r = pc / XP;
    const int c = (pc % XP) ^ (r & 15);
    xg[k] = c >> 3;
    xsrc[k] = reinterpret_cast<const unsigned char*>(p.x + static_cast<int64_t>(min(m0 + r, M - 1)) * K) + (c & 7) * 16;
    xdst[k] = __builtin_amdgcn_readfirstlane(i * 1024);
  }
#pragma unroll
  for (int k = 0; k < WW; k++) {
    const int i = min(wave + NW * k, WI - 1), pc = i * 64 + lane, r = pc / WP;
    const int c = (pc % WP) ^ (w_swz<KS>(r));
    wg[k] = c >> 1;
    wsrc[k] = reinterpret_cast<const unsigned char*>((is_up(r) ? p.w2 : pw) + static_cast<int64_t>(w_row(r)) * (K / 8)) +
              (c & 1) * 16;
    wdst[k] = __builtin_amdgcn_readfirstlane(BM * KS * 128 + i * 1024);
  }
  const uint32_t ring0 = __builtin_amdgcn_readfirstlane(lds_offset(smem));
  auto issue = [&](int s, int slot) {
    const int g0 = gb + s * KS;
    const uint32_t base = ring0 + static_cast<uint32_t>(slot) * static_cast<uint32_t>(SLOT);
    // (groups past the end repeat the last; they are not multiplied)
#pragma unroll
    for (int k = 0; k < WW; k++) lds_load16(wsrc[k] + static_cast<int64_t>(min(g0 + wg[k], G - 1)) * 32, base + wdst[k]);
#pragma unroll
    for (int k = 0; k < XW; k++) lds_load16(xsrc[k] + static_cast<int64_t>(min(g0 + xg[k], G - 1)) * 128, base + xdst[k]);
  };

  f32x4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  int rot[NT];  // row mod SB of the lane's W rows
#pragma unroll
  for (int j = 0; j < NT; j++) rot[j] = (wn * 32 + j * 16 + li) % SB;

#pragma unroll 1
  for (int s = 0; s < min(R - 1, ns); s++) issue(s, s);
  int slot = 0;
#pragma unroll 1
  for (int s = 0; s < ns; s++) {
    // slab s has arrived once only the loads of the slabs behind it (at most
    // R - 2) are outstanding; after the barrier every wave's part has, and
    // slab s - 1 is no longer read
    wait_behind<RMAX - 2, XW + WW>(min(ns - 1 - s, R - 2));
    __syncthreads();
    if (s + R - 1 < ns) issue(s + R - 1, slot == 0 ? R - 1 : slot - 1);
    const unsigned char* xt = smem + slot * SLOT;
    const unsigned char* wt = xt + BM * KS * 128;
#pragma unroll
    for (int h = 0; h < KS / WK; h++) {
      const int lg = h * WK + wk, g = s * KS + lg;  // group of the slab, of the split
      if (gb + g < ge) {                            // uniform
        bf16x8_t b[NT][2];
#pragma unroll
        for (int j = 0; j < NT; j++) {
          const int r = wn * 32 + j * 16 + li;
          const int c = (2 * lg + (q >> 1)) ^ (w_swz<KS>(r));
          const uint2 w = *reinterpret_cast<const uint2*>(wt + (r * WP + c) * 16 + (q & 1) * 8);
          int cw = (g >> 1) + rot[j];
          if (cw >= SB) cw -= SB;
          const uint32_t sw = s_lds[r * SB + cw], bw = b_lds[r * SB + cw];
          const float sv = __uint_as_float((g & 1) ? sw & 0xffff0000u : sw << 16);
          const float bv = __uint_as_float((g & 1) ? bw & 0xffff0000u : bw << 16);
          b[j][0] = __builtin_bit_cast(bf16x8_t, qmm_dequant_word(w.x, sv, bv));
          b[j][1] = __builtin_bit_cast(bf16x8_t, qmm_dequant_word(w.y, sv, bv));
        }
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
          for (int t = 0; t < 2; t++) {
            const int r = i * 16 + li, c = (lg * 8 + 2 * q + t) ^ li;
            const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(xt + (r * XP + c) * 16);
#pragma unroll
            for (int j = 0; j < NT; j++)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[j][t], acc[i][j], 0, 0, 0);
          }
      }
    }
    slot = slot == R - 1 ? 0 : slot + 1;
  }

  // ---- the WK partial tiles through LDS: [wk][MT][WN][NT][lane] x 4 floats ----
  float4* red = reinterpret_cast<float4*>(smem);
  constexpr int TILES = MT * WN * NT;
  __syncthreads();  // every wave has read its last slab
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++)
      red[(wk * TILES + (i * WN + wn) * NT + j) * 64 + lane] =
          make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  __syncthreads();
  auto sum = [&](int tile) {
    float4 t = red[tile * 64 + lane];
#pragma unroll
    for (int w = 1; w < WK; w++) {
      const float4 v = red[(w * TILES + tile) * 64 + lane];
      t.x += v.x;
      t.y += v.y;
      t.z += v.z;
      t.w += v.w;
    }
    return t;
  };
  // lane holds column li, rows 4 q + r of a tile
  if constexpr (EPI == QMM_SWIGLU) {
    for (int u = wave; u < MT * WN; u += NW) {
      const int i = u / WN, n = n0 + (u % WN) * 16 + li;
      const float4 ga = sum(u * NT), ua = sum(u * NT + 1);
      const float gv[4] = {ga.x, ga.y, ga.z, ga.w}, uv[4] = {ua.x, ua.y, ua.z, ua.w};
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = m0 + i * 16 + 4 * q + r;
        if (m >= M || n >= N) continue;
        // silu(gate) * up, each MLX op rounding to bf16 (kernels.rs:73-74)
        const float g = round_bf(gv[r]), uu = round_bf(uv[r]);
        const float sg = round_bf(1.0f / (1.0f + expf(-g)));
        py[static_cast<int64_t>(m) * N + n] = f2bf(round_bf(g * sg) * uu);
      }
    }
    return;
  }
  for (int u = wave; u < TILES; u += NW) {
    const int i = u / (WN * NT), n = n0 + (u % (WN * NT)) * 16 + li;
    const float4 a = sum(u);
    const float av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = m0 + i * 16 + 4 * q + r;
      if (m >= M || n >= N) continue;
      const int64_t o = static_cast<int64_t>(m) * N + n;
      if (p.part) p.part[static_cast<int64_t>(blockIdx.z) * M * N + o] = av[r];
      else if (EPI == QMM_RESIDUAL) py[o] = f2bf(bf2f(p.res[o]) + round_bf(av[r]));
      else py[o] = f2bf(av[r]);
    }
  }
}

// ... and with several rounds of workgroups no more than lets a CU hold two
// (151936 x 2560: 16 rows 78 -> 65 us, 64 rows 117 -> 92)
int slab_slots(const SlabPlan& s, int64_t wgs) {
  const int most = slab_ring(s.mt, s.bn, slab_sb(s));
  if (wgs <= 256) return most;
  const int half = static_cast<int>((kSlabLds / 2 - std::min(kSlabLds / 2, slab_sb(s))) /
                                    slab_slot(s.mt, s.bn, slab_groups(s.mt, s.bn)));
  return half >= 2 ? std::min(half, most) : most;
}

template <int EPI, int MT, int BN>
int launch_one(const QmmParams& p, const SlabPlan& s, hipStream_t stream) {
  constexpr int cn = EPI == QMM_SWIGLU ? BN / 2 : BN, threads = 64 * slab_waves(MT);
  const dim3 grid((p.N + cn - 1) / cn, (p.M + 16 * MT - 1) / (16 * MT), s.splits);
  const int ring = slab_slots(s, static_cast<int64_t>(grid.x) * grid.y * grid.z);
  const size_t lds = slab_lds(MT, BN, slab_groups(MT, BN), ring, slab_sb(s));
  const auto kern = qmm_slab_kernel<EPI, MT, BN>;
  if (int rc = allow_lds(kern, lds)) return rc;
  hipLaunchKernelGGL(kern, grid, dim3(threads), lds, stream, p, ring);
  return check_launch("qmm_slab");
}

template <int EPI>
int launch_epi(const QmmParams& p, const SlabPlan& s, hipStream_t stream) {
  switch (s.mt * 2 + (s.bn == 128)) {
    case 2: return launch_one<EPI, 1, 64>(p, s, stream);
    case 3: return launch_one<EPI, 1, 128>(p, s, stream);
    case 4: return launch_one<EPI, 2, 64>(p, s, stream);
    case 5: return launch_one<EPI, 2, 128>(p, s, stream);
    case 6: return launch_one<EPI, 3, 64>(p, s, stream);
    case 7: return launch_one<EPI, 3, 128>(p, s, stream);
    case 8: return launch_one<EPI, 4, 64>(p, s, stream);
    case 9: return launch_one<EPI, 4, 128>(p, s, stream);
    case 10: return launch_one<EPI, 5, 64>(p, s, stream);
    case 11: return launch_one<EPI, 5, 128>(p, s, stream);
    case 12: return launch_one<EPI, 6, 64>(p, s, stream);
    case 13: return launch_one<EPI, 6, 128>(p, s, stream);
    case 14: return launch_one<EPI, 7, 64>(p, s, stream);
    case 16: return launch_one<EPI, 8, 64>(p, s, stream);
    default: return launch_one<EPI, 8, 128>(p, s, stream);
  }
}

}  // namespace

// The rule, from times of both kernels (us, tile kernel -> this one; weights
// from memory), where the LDS holds the whole split's s and b and two ring
// slots (long K: else the tile kernel, as 5120 x 25600 at 33..48 and 97..384
// rows, 83 and 87 us between 31.0 at 32 rows and 45.6 at 49; 4096 x 12288 at
// 225..256 and from 289 on; 2560 x 9728 from 337):
//   * up to 64 rows, any N: 9728 x 2560 20.7 -> 10.5 at 9 rows, 26.1 -> 16.4
//     at 64; 151936 x 2560 141 -> 63 at 9, 133 -> 92 at 64;
//   * more rows while the tiles are one round of the 256 CUs: 1024 x 2560
//     18.2 -> 12.2 at 200 rows, 33.8 -> 22.1 at 2048; 12288 x 4096 55.7 ->
//     47 at 200 (192 tiles); 4096 x 2560 42.8 -> 32.6 at 1024 (256 tiles),
//     but 55.1 -> 73 at 2048 (512 tiles);
//   * 64 columns per tile (half the x reuse, but twice the CUs) where those
//     tiles fit the round, with K split to fill it: 2560 x 9728 at 37 rows
//     29 -> 14.5 with 6 splits (unsplit 37), though 4096 x 12288 gains only
//     47.7 -> 46.5 at 200 rows (28.8 at 128); else 128 columns;
//   * not 128 columns in three or more row tiles that leave a fifth of the
//     CUs idle: 8192 x 5120 at 300 rows (192 tiles) 60.5 -> 64.
SlabPlan slab_plan(QmmEpilogue epi, int M, int N, int K, int max_splits) {
  SlabPlan s{false, 0, 0, 1, 0};
  if (M <= 8 || K % 128) return s;
  const int G = K / 64;
  const int per = epi == QMM_SWIGLU ? 2 : 1;  // W rows per output column
  // row tiles of up to 128 rows, equal heights
  const int t16 = (M + 15) / 16, rt = (t16 + 7) / 8;
  s.mt = (t16 + rt - 1) / rt;
  auto tiles = [&](int bn) { return (per * static_cast<int64_t>(N) + bn - 1) / bn * rt; };
  s.bn = tiles(64) <= 256 ? 64 : 128;
  // 112-row tiles of 128 columns run slower than 128-row ones (12288 x 4096,
  // 192 tiles: 224 rows 53.4 us, 256 rows 46.9; 64 columns: equal)
  if (s.bn == 128 && s.mt == 7) s.mt = 8;
  const int step = s.mt <= 3 ? 8 : 4;  // whole slabs
  s.gps = (G + step - 1) / step * step;
  if (epi != QMM_SWIGLU && s.bn == 64) {
    const int want = static_cast<int>(std::min<int64_t>({256 / tiles(64), max_splits, G / 8}));
    if (want > 1) {
      s.gps = ((G + want - 1) / want + step - 1) / step * step;
      s.splits = (G + s.gps - 1) / s.gps;
    }
  }
  if (rt > 65535 || tiles(s.bn) > INT32_MAX) return s;
  s.fits = (M <= 64 || (tiles(s.bn) <= 256 && !(s.bn == 128 && rt >= 3 && tiles(128) < 208))) &&
           slab_ring(s.mt, s.bn, slab_sb(s)) >= 2;
  return s;
}

int launch_qmm_slab(QmmEpilogue epi, const QmmParams& p, const SlabPlan& s, hipStream_t stream) {
  QmmParams q = p;
  q.gps = s.gps;
  if (s.splits == 1) q.part = nullptr;
  return epi == QMM_STORE      ? launch_epi<QMM_STORE>(q, s, stream)
         : epi == QMM_RESIDUAL ? launch_epi<QMM_RESIDUAL>(q, s, stream)
                               : launch_epi<QMM_SWIGLU>(q, s, stream);
}

}  // namespace bmx
