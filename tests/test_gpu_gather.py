"""GPU parity of gather_qmm (routed MoE expert qmm) against the CPU oracle:
within 2 bf16 ulps of the oracle's fp32-accumulated result per route, for
the Qwen3-30B-A3B-shaped decode projections (128 experts of gate|up
(1536, 2048) with x shared over the 8 routes of a token, down (2048, 768)
with one x block per route), ragged shapes, several rows of x per route,
repeated and out-of-range expert ids."""
import numpy as np
import pytest

from _util import bf16_to_f32, to_torch_bf16, torch_bf16_bits, u32_of

pytestmark = pytest.mark.gpu


def _experts(gpu, orc, seed, E, N, K):
    import torch

    dev = [gpu.init_qlinear(seed + e, N, K) for e in range(E)]
    w, s, b = (torch.stack([t[i] for t in dev]).contiguous() for i in range(3))
    return (w, s, b), (u32_of(w), torch_bf16_bits(s), torch_bf16_bits(b))


def _close(y_bits, ref_bits):
    y = bf16_to_f32(y_bits).astype(np.float64)
    r = bf16_to_f32(ref_bits).astype(np.float64)
    ok = np.abs(y - r) <= np.maximum(2 * np.abs(r) * 2.0 ** -7, 1e-4 * np.max(np.abs(r)))
    return ok.mean()


# (E, N, K, M, R, x_bcast)
CASES = [(128, 1536, 2048, 1, 8, 8), (128, 2048, 768, 1, 8, 1), (5, 100, 320, 3, 7, 1), (8, 256, 4096, 8, 4, 2),
         (3, 64, 64, 2, 6, 3)]


@pytest.mark.parametrize("E,N,K,M,R,x_bcast", CASES)
def test_gather_qmm(gpu, orc, E, N, K, M, R, x_bcast):
    import torch

    print(f"gather_qmm E={E} N={N} K={K} M={M} R={R} x_bcast={x_bcast}", flush=True)
    (w, s, b), (wq, sq, bq) = _experts(gpu, orc, 1000 + K, E, N, K)
    rng = np.random.default_rng(R * 31 + E)
    rhs = rng.integers(0, E, R).astype(np.uint32)
    rhs[-1] = rhs[0]  # a repeated expert
    x = gpu.fill_normal_bf16(2000 + M, (R // x_bcast, M, K))
    rhs_d = torch.from_numpy(rhs.view(np.int32)).cuda()
    y = gpu.gather_qmm(x, w, s, b, rhs_d, x_bcast)
    torch.cuda.synchronize()
    ref = orc.gather_qmm(torch_bf16_bits(x), wq, sq, bq, rhs, x_bcast)
    assert _close(torch_bf16_bits(y), ref) > 0.999
    # out-of-range ids: clamped to the last expert
    rhs2 = rhs.copy()
    rhs2[0] = E + 5
    y2 = gpu.gather_qmm(x, w, s, b, torch.from_numpy(rhs2.view(np.int32)).cuda(), x_bcast)
    rhs2[0] = E - 1
    y3 = gpu.gather_qmm(x, w, s, b, torch.from_numpy(rhs2.view(np.int32)).cuda(), x_bcast)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(torch_bf16_bits(y2), torch_bf16_bits(y3))


def test_gather_qmm_matches_qmatmul_per_route(gpu, orc):
    """A single route with x_bcast 1 is the plain quantized_matmul of its expert."""
    import torch

    E, N, K = 4, 384, 1024
    (w, s, b), _ = _experts(gpu, orc, 3000, E, N, K)
    x = gpu.fill_normal_bf16(3100, (1, 1, K))
    for e in range(E):
        y = gpu.gather_qmm(x, w, s, b, torch.tensor([e], dtype=torch.int32, device="cuda"))
        z = gpu.quantized_matmul(x[0], w[e], s[e], b[e])
        torch.cuda.synchronize()
        assert _close(torch_bf16_bits(y[0]), torch_bf16_bits(z)) == 1.0


def test_gather_qmm_errors(gpu):
    import torch

    w = torch.zeros(2, 16, 8, dtype=torch.int32, device="cuda")
    s = torch.zeros(2, 16, 1, dtype=torch.bfloat16, device="cuda")
    x = torch.zeros(1, 9, 64, dtype=torch.bfloat16, device="cuda")
    idx = torch.zeros(1, dtype=torch.int32, device="cuda")
    with pytest.raises(gpu.BmxError) as ei:  # 9 rows of x per route
        gpu.gather_qmm(x, w, s, s, idx)
    assert ei.value.code == gpu.BMX_E_UNSUPPORTED


def test_gather_qmm_indexed_lhs_and_rhs(gpu, orc):
    """mlx_gather_qmm with both index arrays: route r multiplies x block
    lhs[r] (repeated, permuted and one out-of-range id, clamped to the last
    block) by expert rhs[r]; checked against the oracle run on the x blocks
    gathered on the host."""
    import torch

    E, N, K, M, B, R = 6, 320, 1536, 2, 5, 9
    print(f"gather_qmm_indexed E={E} N={N} K={K} M={M} x blocks={B} R={R}", flush=True)
    (w, s, b), (wq, sq, bq) = _experts(gpu, orc, 4000, E, N, K)
    rng = np.random.default_rng(17)
    lhs = rng.integers(0, B, R).astype(np.uint32)
    lhs[2] = B + 3  # clamped to B - 1
    rhs = rng.integers(0, E, R).astype(np.uint32)
    x = gpu.fill_normal_bf16(4100, (B, M, K))
    dev = lambda a: torch.from_numpy(a.view(np.int32)).cuda()  # noqa: E731
    y = gpu.gather_qmm_indexed(x, w, s, b, dev(lhs), dev(rhs), sorted_indices=True)
    torch.cuda.synchronize()
    xg = torch_bf16_bits(x)[np.minimum(lhs, B - 1)]
    ref = orc.gather_qmm(xg, wq, sq, bq, rhs, 1)
    assert _close(torch_bf16_bits(y), ref) > 0.999
    # without lhs_indices the x blocks broadcast over the routes: the same
    # bits as bmx_gather_qmm with x_bcast = R / B
    x3 = gpu.fill_normal_bf16(4200, (3, M, K))
    rhs6 = dev(rng.integers(0, E, 6).astype(np.uint32))
    a = gpu.gather_qmm_indexed(x3, w, s, b, None, rhs6)
    c = gpu.gather_qmm(x3, w, s, b, rhs6, x_bcast=2)
    # without rhs_indices route r uses expert r (R = E)
    x6 = gpu.fill_normal_bf16(4300, (E, M, K))
    d = gpu.gather_qmm_indexed(x6, w, s, b, None, None)
    e = gpu.gather_qmm(x6, w, s, b, dev(np.arange(E, dtype=np.uint32)))
    torch.cuda.synchronize()
    np.testing.assert_array_equal(torch_bf16_bits(a), torch_bf16_bits(c))
    np.testing.assert_array_equal(torch_bf16_bits(d), torch_bf16_bits(e))


def test_gather_qmm_indexed_errors(gpu):
    import torch

    w = torch.zeros(2, 16, 8, dtype=torch.int32, device="cuda")
    s = torch.zeros(2, 16, 1, dtype=torch.bfloat16, device="cuda")
    x = torch.zeros(3, 1, 64, dtype=torch.bfloat16, device="cuda")
    idx = torch.zeros(4, dtype=torch.int32, device="cuda")
    cases = [(dict(lhs_indices=idx, rhs_indices=idx, transpose=False), gpu.BMX_E_UNSUPPORTED),
             (dict(lhs_indices=None, rhs_indices=idx), gpu.BMX_E_SHAPE),  # 4 routes over 3 x blocks
             (dict(lhs_indices=idx, rhs_indices=None), gpu.BMX_E_SHAPE)]  # 4 routes, 2 experts
    for kw, code in cases:
        with pytest.raises(gpu.BmxError) as ei:
            gpu.gather_qmm_indexed(x, w, s, s, **kw)
        assert ei.value.code == code, kw


# Where that is faster, an expert's routes are multiplied together, in units of
# 16, 32 or 64 rows (by the average, and 256 workgroups): (E, N, K, M, R,
# x_bcast, skew); skew sends that share of the routes to expert 1.  Column
# remainders (N 100, 257), one and several 256-column chunks, rows per route
# that straddle tiles, an expert above 1024 routes, index arrays beyond the
# 4096 entries kept in registers, experts without a route.
ROWS = [(4, 100, 256, 1, 5, 1, 0.0), (16, 257, 768, 1, 40, 8, 0.0), (6, 96, 512, 3, 33, 3, 0.5),
        (3, 64, 256, 8, 60, 1, 0.9), (5, 288, 512, 1, 200, 4, 0.3), (2, 32, 256, 1, 2500, 1, 0.99),
        (4, 40, 256, 1, 20011, 1, 0.25), (9, 256, 2048, 1, 300, 1, 0.0)]
# ... 16 rows a unit over 8 chunks, even and all but one route to one expert;
# 32 rows over 3 chunks; 64 rows over 8, 3 and 2 chunks with 1, 2 and 3 rows a
# route; more experts than threads, and the most there are counters for
ROWS += [(8, 1536, 2048, 1, 160, 8, 0.0), (16, 1200, 2048, 1, 200, 1, 0.99), (32, 1000, 768, 1, 1200, 8, 0.3),
         (3, 1500, 2048, 1, 1500, 1, 0.3), (4, 1030, 768, 2, 1000, 1, 0.6), (4, 1030, 512, 3, 700, 1, 0.3),
         (600, 64, 256, 1, 1500, 1, 0.1), (4096, 32, 256, 1, 9000, 1, 0.05)]


@pytest.mark.parametrize("E,N,K,M,R,x_bcast,skew", ROWS)
def test_gather_qmm_by_expert(gpu, orc, E, N, K, M, R, x_bcast, skew):
    import torch

    print(f"gather_qmm by expert E={E} N={N} K={K} M={M} R={R} x_bcast={x_bcast} skew={skew}", flush=True)
    (w, s, b), (wq, sq, bq) = _experts(gpu, orc, 5000 + K, E, N, K)
    rng = np.random.default_rng(R + E)
    rhs = rng.integers(0, max(E - 1, 1), R).astype(np.uint32)  # the last expert gets no route
    rhs[rng.random(R) < skew] = 1
    x = gpu.fill_normal_bf16(5100 + M, (R // x_bcast, M, K))
    y = gpu.gather_qmm(x, w, s, b, torch.from_numpy(rhs.view(np.int32)).cuda(), x_bcast)
    # the same routes through lhs_indices, permuted, with ids past the end
    perm = rng.permutation(R).astype(np.uint32)
    lhs = (perm // x_bcast).astype(np.uint32)
    rhs2 = rhs[perm]
    rhs2[0] = E + 7
    z = gpu.gather_qmm_indexed(x, w, s, b, torch.from_numpy(lhs.view(np.int32)).cuda(),
                               torch.from_numpy(rhs2.view(np.int32)).cuda())
    torch.cuda.synchronize()
    ref = orc.gather_qmm(torch_bf16_bits(x), wq, sq, bq, rhs, x_bcast)
    assert _close(torch_bf16_bits(y), ref) > 0.999
    # a route's bits do not depend on where it stands among its expert's
    np.testing.assert_array_equal(torch_bf16_bits(z)[1:], torch_bf16_bits(y)[perm[1:]])
    last = orc.gather_qmm(torch_bf16_bits(x)[lhs[:1]], wq, sq, bq, np.array([E - 1], np.uint32), 1)
    assert _close(torch_bf16_bits(z)[:1], last) > 0.999


@pytest.mark.parametrize("E,N,K,M,R", [(8, 1536, 2048, 1, 16), (1, 2048, 768, 1, 2), (4, 512, 512, 2, 8)])
def test_gather_qmm_few_routes_stay_apart(gpu, orc, E, N, K, M, R):
    """Few routes over few experts leave CUs idle when taken by expert, so
    they have the bits of the per-route kernel: those of the same routes among
    enough further experts that no expert could get two."""
    import torch

    (w, s, b), _ = _experts(gpu, orc, 6000 + K, E, N, K)
    more = [torch.cat([t] + [t[:1]] * (2 * R)).contiguous() for t in (w, s, b)]
    rhs = torch.from_numpy(np.random.default_rng(K).integers(0, E, R).astype(np.int32)).cuda()
    x = gpu.fill_normal_bf16(6100 + M, (R, M, K))
    y = torch_bf16_bits(gpu.gather_qmm(x, w, s, b, rhs))
    np.testing.assert_array_equal(y, torch_bf16_bits(gpu.gather_qmm(x, *more, rhs)))
