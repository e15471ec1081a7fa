"""GPU parity of the ops around the matmul and of the MFMA qmm against the
CPU oracle on identical inputs (bf16 out; tolerances in each test)."""
import numpy as np
import pytest

from _util import bf16_to_f32, bf16_ulp_diff, max_rel_err, to_torch_bf16, torch_bf16_bits, u32_of

pytestmark = pytest.mark.gpu


def _close(y_bits, ref_bits, ulps=2, floor=1e-3):
    y = bf16_to_f32(y_bits).astype(np.float64)
    r = bf16_to_f32(ref_bits).astype(np.float64)
    ok = np.abs(y - r) <= np.maximum(ulps * np.abs(r) * 2.0 ** -7, floor * np.max(np.abs(r)))
    return ok.mean()


def test_rms_norm(gpu, orc):
    x = gpu.fill_normal_bf16(1, (37, 2560), sigma=2.0)
    w = gpu.fill_normal_bf16(2, (2560,), sigma=0.5)
    y = gpu.rms_norm(x, w, 1e-6)
    ref = orc.rms_norm(torch_bf16_bits(x), torch_bf16_bits(w), 1e-6)
    assert _close(torch_bf16_bits(y), ref) == 1.0


@pytest.mark.parametrize("offset", [0, 1, 4095])
def test_rope(gpu, orc, offset):
    x = gpu.fill_normal_bf16(3, (8, 5, 128))
    y = gpu.rope(x, 1e6, offset)
    ref = orc.rope(torch_bf16_bits(x), 1e6, offset)
    assert _close(torch_bf16_bits(y), ref) == 1.0


def test_slice_update(gpu, orc):
    import torch

    src = gpu.fill_normal_bf16(4, (8, 64, 128))
    upd = gpu.fill_normal_bf16(5, (4, 3, 32))
    ref = torch_bf16_bits(src).copy()
    gpu.slice_update(src, upd, [1, 2, 0], [8, 9, 128], [2, 3, 4])
    ref[1:8:2, 2:9:3, 0:128:4] = torch_bf16_bits(upd)
    np.testing.assert_array_equal(torch_bf16_bits(src), ref)
    with pytest.raises(gpu.BmxError):
        gpu.slice_update(src, upd, [1, 2, 0], [8, 9, 129], [2, 3, 4])
    torch.cuda.synchronize()


# (the kernel takes heads in groups of 8: 12 / 4 and 20 / 10 leave partial groups)
@pytest.mark.parametrize("M,offset,Hq,Hkv", [(1, 0, 32, 8), (1, 100, 32, 8), (5, 60, 32, 8), (20, 0, 32, 8),
                                             (20, 13, 32, 8), (20, 13, 12, 4), (3, 5, 20, 10)])
def test_qk_norm_rope_kv(gpu, orc, M, offset, Hq, Hkv):
    import torch

    cap = 128
    q = gpu.fill_normal_bf16(6, (M, Hq * 128), sigma=3.0)
    k = gpu.fill_normal_bf16(7, (M, Hkv * 128), sigma=3.0)
    v = gpu.fill_normal_bf16(8, (M, Hkv * 128))
    qn = gpu.fill_normal_bf16(9, (128,), sigma=0.3)
    kn = gpu.fill_normal_bf16(10, (128,), sigma=0.3)
    kc = torch.zeros(Hkv, cap, 128, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros_like(kc)
    qo = gpu.qk_norm_rope_kv(q, k, v, qn, kn, kc, vc, offset, 1e-6, 1e6)
    torch.cuda.synchronize()
    # oracle: per-head norm, [H, M, 128] transpose, rope, slice write
    qb = orc.rms_norm(torch_bf16_bits(q).reshape(M * Hq, 128), torch_bf16_bits(qn)).reshape(M, Hq, 128)
    kb = orc.rms_norm(torch_bf16_bits(k).reshape(M * Hkv, 128), torch_bf16_bits(kn)).reshape(M, Hkv, 128)
    qr = orc.rope(np.ascontiguousarray(qb.transpose(1, 0, 2)), 1e6, offset)
    kr = orc.rope(np.ascontiguousarray(kb.transpose(1, 0, 2)), 1e6, offset)
    assert _close(torch_bf16_bits(qo), qr) == 1.0
    kcg, vcg = torch_bf16_bits(kc), torch_bf16_bits(vc)
    assert _close(kcg[:, offset:offset + M], kr) == 1.0
    np.testing.assert_array_equal(vcg[:, offset:offset + M], torch_bf16_bits(v).reshape(M, Hkv, 128).transpose(1, 0, 2))
    # nothing outside the written rows
    assert not kcg[:, :offset].any() and not kcg[:, offset + M:].any()
    with pytest.raises(gpu.BmxError) as ei:
        gpu.qk_norm_rope_kv(q, k, v, qn, kn, kc, vc, cap - M + 1)
    assert ei.value.code == gpu.BMX_E_KV_CAPACITY


@pytest.mark.parametrize("Hq,Hkv,M,offset", [(32, 8, 1, 0), (32, 8, 1, 4095), (32, 8, 1, 777), (16, 8, 1, 31),
                                             (32, 8, 5, 2043), (64, 8, 5, 300), (32, 8, 3, 100), (64, 8, 8, 1000),
                                             (32, 8, 37, 0), (32, 8, 40, 100), (32, 8, 200, 0), (16, 8, 130, 70),
                                             (32, 8, 513, 3), (8, 8, 100, 0), (24, 8, 90, 3), (64, 8, 300, 17)])
def test_attention(gpu, orc, Hq, Hkv, M, offset):
    cap = offset + M + 5
    q = gpu.fill_normal_bf16(11, (Hq, M, 128))
    kc = gpu.fill_normal_bf16(12, (Hkv, cap, 128))
    vc = gpu.fill_normal_bf16(13, (Hkv, cap, 128))
    scale = 1 / np.sqrt(128)
    ref = orc.sdpa(torch_bf16_bits(q), torch_bf16_bits(kc), torch_bf16_bits(vc), offset + M, offset, M > 1,
                   np.float32(scale))
    for ws in (True, False):
        y = gpu.attention(q, kc, vc, offset, scale, use_workspace=ws)
        yb = torch_bf16_bits(y)
        assert max_rel_err(bf16_to_f32(yb), bf16_to_f32(ref)) < 1e-2
        assert _close(yb, ref, ulps=2, floor=2e-3) > 0.999


@pytest.mark.parametrize("M,offset", [(130, 70), (300, 0)])
def test_attention_prefill_v_beyond_fp16_range(gpu, orc, M, offset):
    """The prefill kernel multiplies p by an fp16 copy of V; a key block with
    a V value beyond fp16's range (here keys 64..127 scaled by 2^17, about
    1.3e5) must take the two-term bf16 product instead, or those keys'
    contributions would saturate at 65504."""
    Hq, Hkv = 32, 8
    cap = offset + M + 5
    q = gpu.fill_normal_bf16(21, (Hq, M, 128))
    kc = gpu.fill_normal_bf16(22, (Hkv, cap, 128))
    vc = gpu.fill_normal_bf16(23, (Hkv, cap, 128))
    vc[:, 64:128] *= 2.0 ** 17  # exact in bf16
    assert float(vc.float().abs().max()) > 65504.0
    scale = 1 / np.sqrt(128)
    ref = orc.sdpa(torch_bf16_bits(q), torch_bf16_bits(kc), torch_bf16_bits(vc), offset + M, offset, True,
                   np.float32(scale))
    yb = torch_bf16_bits(gpu.attention(q, kc, vc, offset, scale))
    assert max_rel_err(bf16_to_f32(yb), bf16_to_f32(ref)) < 1e-2
    assert _close(yb, ref, ulps=2, floor=2e-3) > 0.999


# (Hq, Hkv, M, offset): few query tiles over many keys, where the flash kernel
# splits the keys given a workspace: 4, 2, 8 and 1 q heads per kv head, a last
# tile of 1 token, key counts around a block, splits whose keys the first
# rows of a tile do not see
@pytest.mark.parametrize("Hq,Hkv,M,offset", [(32, 8, 70, 3000), (16, 8, 129, 700), (64, 8, 17, 943), (8, 8, 257, 1000),
                                             (32, 8, 513, 1111), (32, 8, 65, 448)])
def test_attention_flash_key_split(gpu, orc, Hq, Hkv, M, offset):
    import torch

    cap = offset + M + 5
    q = gpu.fill_normal_bf16(61, (Hq, M, 128))
    kc = gpu.fill_normal_bf16(62, (Hkv, cap, 128))
    vc = gpu.fill_normal_bf16(63, (Hkv, cap, 128))
    vc[:, offset - 64:offset] *= 2.0 ** 17  # one block or two beyond fp16's range
    scale = 1 / np.sqrt(128)
    ref = orc.sdpa(torch_bf16_bits(q), torch_bf16_bits(kc), torch_bf16_bits(vc), offset + M, offset, True,
                   np.float32(scale))
    ws = gpu.attention_workspace(Hq, 16)
    one = torch_bf16_bits(gpu.attention(q, kc, vc, offset, scale, use_workspace=False))
    for _ in range(2):  # the workspace reused as it was left
        yb = torch_bf16_bits(gpu.attention(q, kc, vc, offset, scale, workspace=ws))
        assert max_rel_err(bf16_to_f32(yb), bf16_to_f32(ref)) < 1e-2
        assert _close(yb, ref, ulps=2, floor=2e-3) > 0.999
    assert not ws[:8192].any()  # the decode kernel's counters untouched
    # a workspace with no room for two splits: the unsplit kernel's bits
    small = torch.zeros(8192 + 100, dtype=torch.float32, device="cuda")
    np.testing.assert_array_equal(torch_bf16_bits(gpu.attention(q, kc, vc, offset, scale, workspace=small)), one)


@pytest.mark.parametrize("Hq,Hkv,M,offset", [(32, 8, 70, 3000), (8, 8, 257, 1000)])
def test_attention_flash_key_split_nan_and_inf(gpu, Hq, Hkv, M, offset):
    """NaN and infinite scores come out of the split kernel where the unsplit
    one has them, also where every score that a row has in a split is NaN (or
    -inf: weight zero)."""
    import torch

    print(f"key split, NaN and inf: Hq={Hq} Hkv={Hkv} M={M} offset={offset}", flush=True)
    nan, inf, rep, cap = float("nan"), float("inf"), Hq // Hkv, offset + M + 5
    q = gpu.fill_normal_bf16(64, (Hq, M, 128))
    kc = gpu.fill_normal_bf16(65, (Hkv, cap, 128))
    vc = gpu.fill_normal_bf16(66, (Hkv, cap, 128))
    q[0, 3, 17] = nan                        # a query: all its scores
    kc[1, :offset // 2, 5] = nan             # half the keys of a head: whole splits
    kc[2, offset // 2:offset, 5] = nan       # ... the other half
    kc[3, offset - 1, 9] = nan               # one key
    q[4 * rep:5 * rep] = q[4 * rep:5 * rep].abs().clamp(min=0.01)
    kc[4, :offset // 2] = -inf               # scores of -inf over whole splits
    q[5 * rep:6 * rep] = q[5 * rep:6 * rep].abs().clamp(min=0.01)
    kc[5, offset // 2] = inf                 # a score of +inf
    q[6 * rep:7 * rep] = q[6 * rep:7 * rep].abs().clamp(min=0.01)
    kc[6] = -inf                             # nothing but -inf: zeros
    one = gpu.attention(q, kc, vc, offset, use_workspace=False).float()
    two = gpu.attention(q, kc, vc, offset, workspace=gpu.attention_workspace(Hq, 16)).float()
    assert torch.equal(one.isnan(), two.isnan())
    heads = one.isnan().view(M, Hq, 128)
    assert heads[3, 0].all() and heads[:, rep:4 * rep].all() and heads[:, 5 * rep:6 * rep].all()
    assert not heads[4:].any(dim=2)[:, :rep].any() and not heads[:, 4 * rep:5 * rep].any()
    assert not one.view(M, Hq, 128)[:, 6 * rep:7 * rep].any()
    # finite values: sums in another order, two bf16 roundings (2^-8 each) apart
    fin = ~one.isnan()
    assert ((one - two).abs()[fin] <= 2.0 ** -7 * one.abs()[fin] + 2e-3 * one[fin].abs().max()).all()


def test_attention_flash_key_split_not_into_two_rounds(gpu):
    """176 workgroups of about 134 key blocks: halved they are 352 nearly equal
    ones for 256 CUs, no faster than whole, so the call has the unsplit bits."""
    Hq, Hkv, M, offset = 64, 8, 700, 8192
    q = gpu.fill_normal_bf16(67, (Hq, M, 128))
    kc = gpu.fill_normal_bf16(68, (Hkv, offset + M, 128))
    vc = gpu.fill_normal_bf16(69, (Hkv, offset + M, 128))
    one = gpu.attention(q, kc, vc, offset, use_workspace=False)
    two = gpu.attention(q, kc, vc, offset, workspace=gpu.attention_workspace(Hq, 16))
    np.testing.assert_array_equal(torch_bf16_bits(one), torch_bf16_bits(two))


def test_attention_workspace_reuse(gpu, orc):
    """One zero-filled workspace over calls of different split counts and row
    tilings: the arrival counters come back to zero after every call."""
    import torch

    scale = 1 / np.sqrt(128)
    ws = gpu.attention_workspace(64, 8)
    for i, (Hq, M, offset) in enumerate([(32, 1, 4000), (32, 1, 10), (64, 5, 700), (64, 8, 1000), (32, 1, 3)]):
        cap = offset + M + 1
        q = gpu.fill_normal_bf16(40 + i, (Hq, M, 128))
        kc = gpu.fill_normal_bf16(50 + i, (8, cap, 128))
        vc = gpu.fill_normal_bf16(60 + i, (8, cap, 128))
        y = gpu.attention(q, kc, vc, offset, scale, workspace=ws)
        ref = orc.sdpa(torch_bf16_bits(q), torch_bf16_bits(kc), torch_bf16_bits(vc), offset + M, offset, M > 1,
                       np.float32(scale))
        assert _close(torch_bf16_bits(y), ref, ulps=2, floor=2e-3) > 0.999, (Hq, M, offset)
    torch.cuda.synchronize()
    assert not ws[:1024].any()  # counters


# (Hq, Hkv, M, offset): decode at several context lengths, new keys straddling
# a 256-key split boundary (253 + 5), 16 new tokens with 4 q heads per kv head
# (64 rows, four row tiles), rep 8 verify
@pytest.mark.parametrize("Hq,Hkv,M,offset", [(32, 8, 1, 0), (32, 8, 1, 4095), (32, 8, 1, 300), (64, 8, 5, 2043),
                                             (32, 8, 5, 253), (32, 8, 16, 100), (16, 8, 3, 511)])
def test_qk_norm_rope_kv_attention_fused(gpu, orc, Hq, Hkv, M, offset):
    """The fused kernel against the two-call sequence (bit-identical out and
    cache rows), twice in a row on one workspace, and against the oracle."""
    import torch

    cap = offset + 2 * M + 3
    kc0 = gpu.fill_normal_bf16(20, (Hkv, cap, 128))
    vc0 = gpu.fill_normal_bf16(21, (Hkv, cap, 128))
    qn = gpu.fill_normal_bf16(22, (128,), sigma=0.3)
    kn = gpu.fill_normal_bf16(23, (128,), sigma=0.3)
    kc_a, vc_a = kc0.clone(), vc0.clone()
    kc_b, vc_b = kc0.clone(), vc0.clone()
    ws = gpu.attention_workspace(Hq, M)
    for step in range(2):
        off = offset + step * M
        q = gpu.fill_normal_bf16(24 + step, (M, Hq * 128), sigma=3.0)
        k = gpu.fill_normal_bf16(26 + step, (M, Hkv * 128), sigma=3.0)
        v = gpu.fill_normal_bf16(28 + step, (M, Hkv * 128))
        qr = gpu.qk_norm_rope_kv(q, k, v, qn, kn, kc_a, vc_a, off)
        y_a = gpu.attention(qr, kc_a, vc_a, off)
        y_b = gpu.qk_norm_rope_kv_attention(q, k, v, qn, kn, kc_b, vc_b, off, workspace=ws)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(torch_bf16_bits(y_b), torch_bf16_bits(y_a))
        np.testing.assert_array_equal(torch_bf16_bits(kc_b), torch_bf16_bits(kc_a))
        np.testing.assert_array_equal(torch_bf16_bits(vc_b), torch_bf16_bits(vc_a))
        ref = orc.sdpa(torch_bf16_bits(qr), torch_bf16_bits(kc_a), torch_bf16_bits(vc_a), off + M, off, M > 1,
                       np.float32(1 / np.sqrt(128)))
        assert _close(torch_bf16_bits(y_b), ref, ulps=2, floor=2e-3) > 0.999
    assert not ws[:1024].any()  # counters back at zero


@pytest.mark.parametrize("M,offset", [(1, 300), (5, 253), (3, 0)])
def test_qk_norm_rope_kv_attention_stale_nan_rows(gpu, M, offset):
    """Cache rows from the new positions on hold NaN (never written memory):
    the fused kernel reads those rows before it writes them, and positions past
    the context are clamped onto them; neither may leak into the output."""
    import torch

    Hq, Hkv = 32, 8
    cap = offset + M + 40
    kc = gpu.fill_normal_bf16(60, (Hkv, cap, 128))
    vc = gpu.fill_normal_bf16(61, (Hkv, cap, 128))
    kc[:, offset:] = float("nan")
    vc[:, offset:] = float("nan")
    kc_a, vc_a = kc.clone(), vc.clone()
    q = gpu.fill_normal_bf16(62, (M, Hq * 128), sigma=3.0)
    k = gpu.fill_normal_bf16(63, (M, Hkv * 128), sigma=3.0)
    v = gpu.fill_normal_bf16(64, (M, Hkv * 128))
    n = gpu.fill_normal_bf16(65, (128,), sigma=0.3)
    y_a = gpu.attention(gpu.qk_norm_rope_kv(q, k, v, n, n, kc_a, vc_a, offset), kc_a, vc_a, offset)
    y_b = gpu.qk_norm_rope_kv_attention(q, k, v, n, n, kc, vc, offset)
    torch.cuda.synchronize()
    assert not torch.isnan(y_b.float()).any()
    np.testing.assert_array_equal(torch_bf16_bits(y_b), torch_bf16_bits(y_a))


def test_qk_norm_rope_kv_attention_limits(gpu):
    import torch

    q = gpu.fill_normal_bf16(30, (17, 32 * 128))
    k = gpu.fill_normal_bf16(31, (17, 8 * 128))
    kc = torch.zeros(8, 64, 128, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros_like(kc)
    n = gpu.fill_normal_bf16(32, (128,))
    with pytest.raises(gpu.BmxError) as ei:  # 17 new tokens: more than the fused prologue takes
        gpu.qk_norm_rope_kv_attention(q, k, k, n, n, kc, vc, 0)
    assert ei.value.code == gpu.BMX_E_UNSUPPORTED
    with pytest.raises(gpu.BmxError) as ei:
        gpu.qk_norm_rope_kv_attention(q[:4], k[:4], k[:4], n, n, kc, vc, 61)
    assert ei.value.code == gpu.BMX_E_KV_CAPACITY
    torch.cuda.synchronize()
    assert not kc.any() and not vc.any()


@pytest.mark.parametrize("n", [151936, 1001])
def test_argmax(gpu, orc, n):
    """16-byte vector path (rows of a multiple of 8) and the scalar path."""
    x = gpu.fill_normal_bf16(14, (6, n))
    xb = torch_bf16_bits(x).copy()
    xb[1, 7] = xb[1, n - 936] = orc.f32_to_bf16(np.array([30.0], np.float32))[0]
    xb[2, :] = 0x3F80
    xb[3, :] = 0xFF80  # -inf row: index 0
    got = gpu.argmax_rows(to_torch_bf16(xb)).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), orc.argmax_rows(xb))
    assert got[1] == 7 and got[2] == 0 and got[3] == 0


@pytest.mark.parametrize("n", [8, 8200, 81928])
def test_argmax_ties_nan_and_inf(gpu, orc, n):
    """The 16-byte path's bookkeeping by unit: ties inside a unit and across
    threads, -0 before +0, NaN anywhere, rows of NaN and -inf alone (first
    -inf, else 0), the last unit, a row of +inf."""
    nan, ninf = 0x7FC1, 0xFF80
    rng = np.random.default_rng(n)
    x = np.repeat(torch_bf16_bits(gpu.fill_normal_bf16(17, (1, n))), 9, axis=0).copy()
    x[1, n - 1] = x[1, n - 3] = 0x4200  # 32.0 twice in the last unit
    x[2, :] = np.where(rng.random(n) < 0.5, 0x8000, 0)
    x[3, rng.random(n) < 0.3] = nan
    x[4, :] = nan
    x[4, n - 2:] = ninf
    x[5, :] = nan
    x[6, n // 2:] = 0x7F80
    x[7, :] = ninf
    x[7, 5] = nan
    x[8, 3] = x[8, n - 8] = 0x4200
    x[8, 0] = 0x7F81  # a signalling NaN beside them
    f = bf16_to_f32(x)
    want = np.where(np.isnan(f).all(axis=1), 0, np.argmax(np.where(np.isnan(f), -np.inf, f), axis=1))
    for r in range(9):  # NaN counts as nothing, not as -inf
        if not np.isnan(f[r]).all() and np.nanmax(f[r]) == -np.inf:
            want[r] = int(np.flatnonzero(f[r] == -np.inf)[0])
    np.testing.assert_array_equal(gpu.argmax_rows(to_torch_bf16(x)).cpu().numpy(), want)


@pytest.mark.parametrize("n", [8, 8200, 8201, 81928])
def test_argmax_more_rows_than_cus(gpu, n):
    """Above 256 rows, other loads in flight per thread: ties, NaN and
    infinities as one row at a time."""
    x = np.repeat(torch_bf16_bits(gpu.fill_normal_bf16(22, (1, n))), 257, axis=0).copy()
    x[1, n - 1] = x[1, n - 3] = 0x4200
    x[2, :] = 0x7FC1
    x[3, :n - 1] = 0x7FC1
    x[3, n - 1] = 0xFF80
    x[4, n // 2:] = 0x7F80
    for r in range(5, 257):
        x[r, (r * 7919) % n] = 0x4200
    x = to_torch_bf16(x)
    want = [int(gpu.argmax_rows(x[r:r + 1])[0]) for r in range(257)]
    np.testing.assert_array_equal(gpu.argmax_rows(x).cpu().numpy(), want)


@pytest.mark.parametrize("n", [131072, 131080, 131064, 131073, 655352, 655360, 655361, 655368, 1048568, 1048576, 1048577,
                               1048584])
def test_elementwise_vector_path(gpu, n):
    """Either side of the 8-values-per-thread rules (add from 655360 values,
    silu_mul from 1048576), and operands 2 bytes off a 16-byte address: the
    same bits each way; add in place."""
    import torch

    a = gpu.fill_normal_bf16(18, (n + 1,), sigma=3.0)
    b = gpu.fill_normal_bf16(19, (n + 1,))
    for op in (gpu.silu_mul, gpu.add):
        one = torch_bf16_bits(op(a[1:], b[1:]))
        two = torch_bf16_bits(op(a[1:].clone(), b[1:].clone()))
        np.testing.assert_array_equal(one, two)
    c = a[1:].clone()
    gpu.call("bmx_add", c.data_ptr(), b[1:].data_ptr(), c.data_ptr(), n, gpu._stream())
    torch.cuda.synchronize()
    np.testing.assert_array_equal(torch_bf16_bits(c), torch_bf16_bits(a[1:] + b[1:]))


@pytest.mark.parametrize("dim", [4096, 4104, 5120, 8192, 8200])
def test_rms_norm_row_lengths(gpu, orc, dim):
    x = gpu.fill_normal_bf16(20, (5, dim))
    w = gpu.fill_normal_bf16(21, (dim,))
    y = torch_bf16_bits(gpu.rms_norm(x, w))
    # the sums' order may move bf16(x / rms) by one ulp, at most 2^-7 of it,
    # which after the product with w is under two ulps of the result
    assert np.max(bf16_ulp_diff(y, orc.rms_norm(torch_bf16_bits(x), torch_bf16_bits(w)))) <= 2


def test_silu_mul_and_add(gpu, orc):
    g = gpu.fill_normal_bf16(15, (3, 9728), sigma=3.0)
    u = gpu.fill_normal_bf16(16, (3, 9728))
    y = torch_bf16_bits(gpu.silu_mul(g, u))
    ref = orc.silu_mul(torch_bf16_bits(g), torch_bf16_bits(u))
    assert np.max(bf16_ulp_diff(y, ref)) <= 1
    s = torch_bf16_bits(gpu.add(g, u))
    np.testing.assert_array_equal(s, orc.f32_to_bf16(bf16_to_f32(torch_bf16_bits(g)) + bf16_to_f32(torch_bf16_bits(u))))


@pytest.mark.parametrize("M,N,K", [(9, 256, 2560), (16, 1024, 2560), (64, 4096, 2560), (128, 2560, 9728),
                                   (300, 1000, 1024), (37, 151936, 2560), (520, 768, 1536), (24, 512, 320),
                                   (130, 300, 576), (1100, 1024, 1536)])
def test_qmm_vs_oracle(gpu, orc, M, N, K):
    import torch

    print(f"qmm M={M} N={N} K={K}", flush=True)
    w, s, b = gpu.init_qlinear(7000 + M, N, K)
    x = gpu.fill_normal_bf16(8000 + M, (M, K))
    y = gpu.quantized_matmul(x, w, s, b)
    torch.cuda.synchronize()
    xb, wq, sb, bb = torch_bf16_bits(x), u32_of(w), torch_bf16_bits(s), torch_bf16_bits(b)
    ref64 = orc.qmatmul_f64(xb, wq, sb, bb)
    yb = torch_bf16_bits(y)
    assert max_rel_err(bf16_to_f32(yb), ref64) < 1e-2
    # the matrix path of the oracle (bf16-dequantized weights, fp32
    # accumulation): within 2 bf16 ulps of it
    assert _close(yb, orc.qmm_dequant(xb, wq, sb, bb), ulps=2, floor=1e-4) == 1.0


# The few-rows GEMM: one row past the GEMV, edges of the 16-row tiles and of
# their heights (48 | 49: 16 or 8 waves; 128 | 129: a second row tile), column
# remainders of 64- and 128-column tiles, K of one slab, a broken last slab (2,
# 6 and 18 groups), K split over workgroups, several rounds of workgroups
SLAB = [(9, 64, 128), (16, 65, 384), (17, 100, 1152), (32, 1, 256), (33, 257, 2560), (48, 640, 9728), (49, 130, 640),
        (65, 1000, 896), (80, 512, 5120), (112, 2560, 2560), (128, 192, 12288), (129, 96, 1152), (250, 520, 2560),
        (300, 256, 4096), (24, 34000, 128), (57, 17000, 384), (130, 16390, 256)]


@pytest.mark.parametrize("M,N,K", SLAB)
def test_qmm_few_rows(gpu, orc, M, N, K):
    import torch

    print(f"qmm few rows M={M} N={N} K={K}", flush=True)
    w, s, b = gpu.init_qlinear(7100 + M, N, K)
    # the last row of x is the end of its allocation, y has guard rows
    x = gpu.fill_normal_bf16(8100 + M, (M, K))
    out = torch.full((M + 2, N), 7.0, dtype=torch.bfloat16, device="cuda")
    gpu.quantized_matmul(x, w, s, b, out=out[1:-1])
    torch.cuda.synchronize()
    assert (out[0] == 7.0).all() and (out[-1] == 7.0).all()
    xb, wq, sb, bb = torch_bf16_bits(x), u32_of(w), torch_bf16_bits(s), torch_bf16_bits(b)
    yb = torch_bf16_bits(out[1:-1])
    assert _close(yb, orc.qmm_dequant(xb, wq, sb, bb), ulps=2, floor=1e-4) == 1.0
    # scales and biases two bytes off a word take the tile kernel
    if N * K <= 1 << 20:
        so, bo = (torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].view(t.shape) for t in (s, b))
        so.copy_(s)
        bo.copy_(b)
        yo = torch_bf16_bits(gpu.quantized_matmul(x, w, so, bo))
        assert _close(yo, orc.qmm_dequant(xb, wq, sb, bb), ulps=2, floor=1e-4) == 1.0


@pytest.mark.parametrize("M,N,K", [(64, 1024, 2560), (24, 768, 2048), (16, 2048, 4096), (5, 5120, 8192),
                                   (1, 4096, 2560)])
def test_qmatmul_ws_matches_qmatmul(gpu, M, N, K):
    """bmx_qmatmul_affine_ws with a workspace of exactly
    bmx_qmatmul_workspace_bytes(M, N, K) bytes gives the bits of
    bmx_qmatmul_affine (same kernels, caller-owned partials), and also when
    captured into a graph and replayed."""
    import torch

    print(f"qmatmul_ws M={M} N={N} K={K}", flush=True)
    w, s, b = gpu.init_qlinear(310 + M, N, K)
    x = gpu.fill_normal_bf16(410 + M, (M, K))
    need = gpu.qmatmul_workspace_bytes(M, N, K)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda") if need else None
    ref = gpu.quantized_matmul(x, w, s, b)
    got = gpu.quantized_matmul_ws(x, w, s, b, ws)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(torch_bf16_bits(got), torch_bf16_bits(ref))
    st = torch.cuda.Stream()
    out = torch.empty_like(ref)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st):
        with torch.cuda.graph(g, stream=st):
            gpu.quantized_matmul_ws(x, w, s, b, ws, out=out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(torch_bf16_bits(out), torch_bf16_bits(ref))
