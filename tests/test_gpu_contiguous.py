"""GPU parity of the standalone (contiguous) entry points against the oracle:
per-channel decode and prefill (reference kernels/kv_dequant_kernels.cuh:113-502),
per-token decode (:528-655) and the per-channel quantizer on the GPU
(reference host code kernels/benchmark/benchmark.py:26-56, bit-exact)."""
from pathlib import Path

import numpy as np
import pytest
import torch

from common import assert_close, kv_values
from oracle import attention as oa
from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GOLDEN = Path(__file__).resolve().parent / "golden" / "per_channel_quant.npz"


def _kd():
    from kernels import kv_dequant
    return kv_dequant


def _outliers(x: torch.Tensor, gen, frac=0.01, factor=8.0):
    KV, S, D = x.shape
    n = max(1, int(np.ceil(frac * KV * D)))
    for c in torch.randperm(KV * D, generator=gen)[:n].tolist():
        x[c // D, :, c % D] *= factor
    return x


# ------------------------------------------------------------------ quantizer
def _same_fp16(got, ref):
    """Bit-exact fp16, except that any NaN matches any NaN (the sign and
    payload of a NaN produced by 0/0 differ between x86 and the GPU)."""
    same = (got.view(np.uint16) == ref.view(np.uint16)) | (np.isnan(got) & np.isnan(ref))
    assert same.all(), f"{int((~same).sum())} values differ, first at {np.argwhere(~same)[:3].tolist()}"


@pytest.mark.parametrize("name", sorted({k.split("__")[0] for k in np.load(GOLDEN).files}))
def test_quantize_per_channel_matches_reference_golden(name):
    z = np.load(GOLDEN)
    x = torch.from_numpy(z[f"{name}__x"].view(np.float16).copy())
    packed, scale, zero = _kd().quantize_per_channel(x.to(DEV))
    torch.cuda.synchronize()
    _same_fp16(scale.cpu().numpy(), z[f"{name}__scale"].view(np.float16))
    _same_fp16(zero.cpu().numpy(), z[f"{name}__zero"].view(np.float16))
    assert np.array_equal(packed.cpu().numpy(), z[f"{name}__packed"])


@pytest.mark.parametrize("name", sorted({k.split("__")[0] for k in np.load(GOLDEN).files}))
def test_quantize_tensor_with_rulers_matches_reference_golden(name):
    """The fixed-ruler append packs the reference quantizer's own (x, scale,
    zero) into exactly the reference's bytes."""
    z = np.load(GOLDEN)
    x = torch.from_numpy(z[f"{name}__x"].view(np.float16).copy()).to(DEV)
    scale = torch.from_numpy(z[f"{name}__scale"].view(np.float16).copy()).to(DEV)
    zero = torch.from_numpy(z[f"{name}__zero"].view(np.float16).copy()).to(DEV)
    packed = _kd().quantize_tensor(x, scale, zero)
    torch.cuda.synchronize()
    assert np.array_equal(packed.cpu().numpy(), z[f"{name}__packed"])


@pytest.mark.parametrize("KV,S0,S1,D", [(2, 64, 1, 128), (4, 512, 37, 64), (2, 100, 300, 80), (1, 16, 8, 128)])
def test_quantize_tensor_appends_with_frozen_rulers(KV, S0, S1, D):
    """The reference's model-harness append (kernels/benchmark/benchmark.py:
    205-216): rulers from the first S0 tokens, new tokens (some outside the
    rulers' range, so the clamp acts) packed into a slice of a preallocated
    [KV, capacity, D/2] cache; bytes outside the slice stay as they were."""
    g = torch.Generator().manual_seed(S0 + S1 + D)
    x0 = _outliers(torch.randn(KV, S0, D, generator=g), g).half()
    x1 = (3.0 * torch.randn(KV, S1, D, generator=g)).half()
    _, scale, zero = _kd().quantize_per_channel(x0.to(DEV))
    cap = S0 + S1 + 9
    cache = torch.full((KV, cap, D // 2), 0xA5, dtype=torch.uint8, device=DEV)
    # a token-strided source, as a slice of a longer [KV, L, D] tensor
    src = torch.cat([x0, x1], dim=1).to(DEV)[:, S0:, :]
    _kd().quantize_tensor(src, scale, zero, out=cache[:, S0:S0 + S1])
    torch.cuda.synchronize()
    ref = oq.quantize_tensor(x1.numpy(), scale.cpu().numpy(), zero.cpu().numpy())
    got = cache.cpu().numpy()
    assert np.array_equal(got[:, S0:S0 + S1], ref)
    assert (got[:, :S0] == 0xA5).all() and (got[:, S0 + S1:] == 0xA5).all()
    codes = np.stack([ref & 15, ref >> 4], axis=-1)
    assert (codes == 0).any() and (codes == 15).any()      # both clamps were exercised


def test_quantize_tensor_special_values():
    """NaN, +-inf, +-0, +-65504 and subnormal inputs against tiny, unit and
    huge rulers, bit-exact with the oracle (NaN codes become 0 on both)."""
    D, KV = 64, 2
    vals = np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 65504.0, -65504.0, 6e-8, -6e-8, 1.0, -1.0,
                     0.5, 1.5, 2.5, 7.49, 7.51], dtype=np.float16)
    x = np.resize(vals, (KV, 8, D)).astype(np.float16)
    scale = np.resize(np.array([6e-8, 1.0, 4096.0, 0.0133], dtype=np.float16), (KV, D)).astype(np.float16)
    zero = np.resize(np.array([0.0, 8.0, 15.0, 3.0], dtype=np.float16), (KV, D)).astype(np.float16)
    got = _kd().quantize_tensor(torch.from_numpy(x).to(DEV), torch.from_numpy(scale).to(DEV),
                                torch.from_numpy(zero).to(DEV))
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), oq.quantize_tensor(x, scale, zero))


@pytest.mark.parametrize("KV,S,D", [(4, 512, 64), (2, 2048, 128), (2, 333, 80), (8, 1, 128)])
def test_quantize_per_channel_matches_oracle(KV, S, D):
    g = torch.Generator().manual_seed(S + D)
    x = _outliers(torch.randn(KV, S, D, generator=g), g).half()
    packed, scale, zero = _kd().quantize_per_channel(x.to(DEV))
    torch.cuda.synchronize()
    s_ref, z_ref = oq.compute_scale_zero(x.numpy())
    p_ref = oq.quantize_tensor(x.numpy(), s_ref, z_ref)
    _same_fp16(scale.cpu().numpy(), s_ref)
    _same_fp16(zero.cpu().numpy(), z_ref)
    assert np.array_equal(packed.cpu().numpy(), p_ref)


# ------------------------------------------------------------------ per-channel decode
def _pc_inputs(seed, H, KV, S, D, outliers=False):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(H, 1, D, generator=g).half()
    k = torch.randn(KV, S, D, generator=g)
    v = torch.randn(KV, S, D, generator=g)
    if outliers:
        k, v = _outliers(k, g), _outliers(v, g)
    kp, ks, kz, vp, vs, vz = oq.quantize_kv(k.half().numpy(), v.half().numpy())
    return q, [torch.from_numpy(a) for a in (kp, ks, kz, vp, vs, vz)]


@pytest.mark.parametrize("H,KV,D,S,outl", [(4, 4, 64, 512, False),            # config 1
                                           (12, 2, 128, 512, True),            # config 2
                                           (12, 2, 128, 1024, True),
                                           (12, 2, 128, 2048, True),
                                           (32, 4, 64, 1024, False), (32, 8, 128, 700, False),
                                           (14, 2, 64, 333, False), (8, 8, 80, 97, False)])
def test_decode_per_channel(H, KV, D, S, outl):
    q, t = _pc_inputs(H * 7 + S, H, KV, S, D, outl)
    out = _kd().kv_dequant_decode_attention(q.to(DEV), *[x.to(DEV) for x in t], num_kv_heads=KV)
    torch.cuda.synchronize()
    assert out.shape == (H, 1, D) and out.dtype == torch.float32
    ref = oa.decode_per_channel(q.numpy(), *[x.numpy() for x in t])
    assert_close(out.cpu().numpy(), ref, what="per-channel decode")
    # The reference benchmark's own check rounds the dequantized KV to fp16
    # before attending (kernels/benchmark/benchmark.py:112).  Against that
    # oracle the bar widens by the two oracles' own difference.
    ref16 = oa.decode_per_channel(q.numpy(), *[x.numpy() for x in t], round_fp16=True)
    gap = np.abs(ref16 - ref).max()
    assert_close(out.cpu().numpy(), ref16, atol=2e-3 + gap, what="vs fp16-rounded dequant")


def test_decode_per_channel_raw_nibbles_and_block_n():
    q, t = _pc_inputs(5, 8, 2, 300, 128)
    kd = _kd()
    raw = kd.kv_dequant_decode_attention(q.to(DEV), *[x.to(DEV) for x in t], BLOCK_N=32,
                                         use_quant=False, num_kv_heads=2)
    torch.cuda.synchronize()
    ref = oa.decode_per_channel(q.numpy(), *[x.numpy() for x in t], use_quant=False)
    assert_close(raw.cpu().numpy(), ref, what="use_quant=False")


def test_decode_per_channel_fewer_kv_heads_than_tensor():
    """num_kv_heads < k_packed.shape[0]: only the first heads are attended."""
    q, t = _pc_inputs(6, 8, 4, 200, 64)
    out = _kd().kv_dequant_decode_attention(q.to(DEV), *[x.to(DEV) for x in t], num_kv_heads=2)
    torch.cuda.synchronize()
    kp, ks, kz, vp, vs, vz = [x.numpy() for x in t]
    ref = oa.decode_per_channel(q.numpy(), kp[:2], ks[:2], kz[:2], vp[:2], vs[:2], vz[:2])
    assert_close(out.cpu().numpy(), ref)


# ------------------------------------------------------------------ prefill
@pytest.mark.parametrize("H,KV,D,M,S,causal", [(32, 4, 64, 256, 256, True), (14, 2, 64, 100, 100, True),
                                               (8, 2, 128, 64, 64, True), (8, 8, 80, 50, 50, False),
                                               (4, 4, 64, 40, 70, True), (4, 2, 64, 70, 40, True)])
def test_prefill_per_channel(H, KV, D, M, S, causal):
    g = torch.Generator().manual_seed(M * 3 + S)
    q = torch.randn(H, M, D, generator=g).half()
    k = torch.randn(KV, S, D, generator=g).half()
    v = torch.randn(KV, S, D, generator=g).half()
    kp, ks, kz, vp, vs, vz = [torch.from_numpy(a) for a in oq.quantize_kv(k.numpy(), v.numpy())]
    kw = {} if D == 64 else {"BLOCK_M": 16, "BLOCK_N": 32}
    out = _kd().kv_dequant_prefill_attention(q.to(DEV), kp.to(DEV), ks.to(DEV), kz.to(DEV), vp.to(DEV),
                                             vs.to(DEV), vz.to(DEV), causal=causal, num_kv_heads=KV, **kw)
    torch.cuda.synchronize()
    ref = oa.prefill_per_channel(q.numpy(), kp.numpy(), ks.numpy(), kz.numpy(), vp.numpy(), vs.numpy(),
                                 vz.numpy(), causal=causal)
    assert out.shape == (H, M, D)
    assert_close(out.cpu().numpy(), ref, what="prefill")


def _pf_inputs(seed, H, KV, M, S, D, outliers=False, t3=False):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(H, M, D, generator=g).half()
    if t3:
        k, v = kv_values(g, (KV, S, D), "t3"), kv_values(g, (KV, S, D), "t3")
    else:
        k, v = torch.randn(KV, S, D, generator=g), torch.randn(KV, S, D, generator=g)
    if outliers:
        k, v = _outliers(k, g), _outliers(v, g)
    kp, ks, kz, vp, vs, vz = oq.quantize_kv(k.half().numpy(), v.half().numpy())
    return q, [torch.from_numpy(a) for a in (kp, ks, kz, vp, vs, vz)]


def _prefill(q, t, **kw):
    out = _kd().kv_dequant_prefill_attention(q.to(DEV), *[x.to(DEV) for x in t], **kw)
    torch.cuda.synchronize()
    return out.cpu().numpy()


# head_dim 64 and 128 run on the matrix-core kernel: query blocks of 64 rows,
# key tiles of 64, so these cover partial blocks and tiles, M > S and M < S
@pytest.mark.parametrize("H,KV,D,M,S,causal,outl,t3", [
    (32, 4, 64, 512, 512, True, False, False),     # the reference's op-level prefill shapes
    (14, 2, 64, 1024, 1024, True, False, False),
    (12, 2, 128, 300, 300, True, True, False),      # config-2 heads, 1 % outlier channels x8
    (8, 2, 128, 129, 1000, False, False, True),     # Student-t K/V, non-causal
    (8, 8, 64, 65, 63, True, True, False),          # M > S
    (4, 1, 128, 1, 777, True, False, False),        # a single row
    (16, 2, 64, 200, 1500, True, False, True)])     # M < S
def test_prefill_matrix_cores(H, KV, D, M, S, causal, outl, t3):
    q, t = _pf_inputs(H + M + S, H, KV, M, S, D, outl, t3)
    out = _prefill(q, t, causal=causal, num_kv_heads=KV)
    ref = oa.prefill_per_channel(q.numpy(), *[x.numpy() for x in t], causal=causal)
    assert_close(out, ref, what=f"prefill H={H} KV={KV} D={D} M={M} S={S}")


# head_dim 80: one row, edges of the 64-row blocks and 64-key tiles, one and two
# heads per workgroup (the second needs over 256 of them), raw codes, rulers that
# are not 8-byte aligned.
@pytest.mark.parametrize("H,KV,M,S,causal,quant,shift", [
    (2, 2, 1, 1, True, True, 0), (4, 2, 63, 64, True, True, 1), (4, 2, 64, 65, False, True, 0),
    (8, 2, 65, 63, True, False, 0), (6, 2, 200, 129, False, True, 1), (3, 3, 130, 500, True, True, 0),
    (16, 2, 2100, 2100, True, True, 0)])
def test_prefill_matrix_cores_head_dim_80(H, KV, M, S, causal, quant, shift):
    q, t = _pf_inputs(H + 3 * M + S, H, KV, M, S, 80, outliers=M == 200)
    dev = []
    for x in t:
        if x.dtype == torch.float16 and shift:
            buf = torch.zeros(x.numel() + shift, dtype=torch.float16, device=DEV)
            buf[shift:] = x.to(DEV).flatten()
            dev.append(buf[shift:].view(x.shape))
        else:
            dev.append(x.to(DEV))
    kw = dict(causal=causal, use_quant=quant, num_kv_heads=KV)
    out = _kd().kv_dequant_prefill_attention(q.to(DEV), *dev, **kw)
    torch.cuda.synchronize()
    ref = oa.prefill_per_channel(q.numpy(), *[x.numpy() for x in t], causal=causal, use_quant=quant)
    assert_close(out.cpu().numpy(), ref, what=f"prefill D=80 H={H} M={M} S={S}")
    assert torch.equal(out, _kd().kv_dequant_prefill_attention(q.to(DEV), *dev, **kw))


# Long causal prefills (up to 32 query blocks): one and two query heads per
# workgroup, both head dims, outliers and Student-t K/V, and S > M with a partial
# last block; a second call gives the same bits.
@pytest.mark.parametrize("H,KV,D,M,S,outl,t3", [
    (4, 2, 128, 2048, 2048, False, False),
    (8, 2, 64, 2048, 2048, True, False),
    (24, 2, 128, 1536, 1536, False, True),
    (32, 4, 64, 1536, 1536, False, False),
    (8, 4, 64, 1000, 1300, False, False)])
def test_prefill_matrix_cores_long(H, KV, D, M, S, outl, t3):
    q, t = _pf_inputs(H * 7 + M, H, KV, M, S, D, outl, t3)
    out = _prefill(q, t, causal=True, num_kv_heads=KV)
    ref = oa.prefill_per_channel(q.numpy(), *[x.numpy() for x in t], causal=True)
    assert_close(out, ref, what=f"long prefill H={H} KV={KV} D={D} M={M} S={S}")
    assert np.array_equal(out, _prefill(q, t, causal=True, num_kv_heads=KV))


# The two 4096-query causal prefills that bench.py --op-level times (two query
# heads per workgroup, every query block from 1 to 64 key tiles): heads spread
# over every KV head checked against the oracle head by head, and a second call
# gives the same bits.
@pytest.mark.parametrize("H,KV,D,heads", [
    (32, 4, 64, (0, 9, 18, 31)),
    (12, 2, 128, (0, 5, 6, 11))])
def test_prefill_matrix_cores_bench_shapes(H, KV, D, heads):
    S = 4096
    q, t = _pf_inputs(H + D, H, KV, S, S, D)
    out = _prefill(q, t, causal=True, num_kv_heads=KV)
    G = H // KV
    for h in heads:
        kv = h // G
        kvt = [x[kv:kv + 1].numpy() for x in t]
        ref = oa.prefill_per_channel(q[h:h + 1].numpy(), *kvt, causal=True)
        assert_close(out[h:h + 1], ref, what=f"bench-shape prefill H={H} KV={KV} D={D} head {h}")
    assert np.array_equal(out, _prefill(q, t, causal=True, num_kv_heads=KV))


def test_prefill_matrix_cores_unaligned_rulers():
    """V scale / zero point views that start 2 bytes into their storage (the
    epilogue's 8-byte ruler loads then take the 2-byte path)."""
    q, t = _pf_inputs(12, 8, 2, 200, 400, 64)
    qd = q.to(DEV)
    dev_t = [x.to(DEV) for x in t]
    for i in (4, 5):                                 # v_scale, v_zero
        big = torch.empty((t[i].numel() + 1,), dtype=t[i].dtype, device=DEV)
        big[1:] = dev_t[i].reshape(-1)
        dev_t[i] = big[1:].view(t[i].shape)
        assert dev_t[i].data_ptr() % 8 != 0
    out = _kd().kv_dequant_prefill_attention(qd, *dev_t, causal=True, num_kv_heads=2)
    torch.cuda.synchronize()
    ref = oa.prefill_per_channel(q.numpy(), *[x.numpy() for x in t], causal=True)
    assert_close(out.cpu().numpy(), ref, what="unaligned V rulers")


def test_prefill_matrix_cores_raw_nibbles_and_tensor_heads():
    """use_quant=False (raw codes), and num_kv_heads < k_packed.shape[0]."""
    q, t = _pf_inputs(9, 8, 4, 100, 300, 64)
    out = _prefill(q, t, causal=True, use_quant=False, num_kv_heads=4)
    ref = oa.prefill_per_channel(q.numpy(), *[x.numpy() for x in t], causal=True, use_quant=False)
    assert_close(out, ref, what="use_quant=False")
    out = _prefill(q, t, causal=True, num_kv_heads=2)
    kp, ks, kz, vp, vs, vz = [x.numpy() for x in t]
    ref = oa.prefill_per_channel(q.numpy(), kp[:2], ks[:2], kz[:2], vp[:2], vs[:2], vz[:2], causal=True)
    assert_close(out, ref, what="num_kv_heads=2 of 4")


def test_prefill_matrix_cores_fractional_zero_points():
    """Zero points need not be integers: the kernel takes the integer part into
    the operand and the rest in fp32."""
    q, t = _pf_inputs(10, 8, 2, 130, 200, 128)
    g = torch.Generator().manual_seed(3)
    t[2] = (t[2].float() + torch.rand(t[2].shape, generator=g) * 3 - 1.5).half()   # k_zero
    t[5] = (t[5].float() + torch.rand(t[5].shape, generator=g) * 3 - 1.5).half()   # v_zero
    out = _prefill(q, t, causal=True, num_kv_heads=2)
    ref = oa.prefill_per_channel(q.numpy(), *[x.numpy() for x in t], causal=True)
    assert_close(out, ref, what="fractional zero points")


# ------------------------------------------------------------------ per-token contiguous decode
@pytest.mark.parametrize("H,KV,D,S", [(32, 8, 128, 1000), (4, 4, 64, 17), (12, 2, 80, 333)])
def test_decode_per_token_contiguous(H, KV, D, S):
    g = torch.Generator().manual_seed(S)
    q = torch.randn(H, 1, D, generator=g).half()
    k = kv_values(g, (S, KV, D))
    v = kv_values(g, (S, KV, D))
    # quantize rows with the oracle store into a scratch cache, then unpack to the contiguous layout
    cache = np.zeros((S, 1, KV, D + 8), dtype=np.uint8)
    oq.quantize_store(k.numpy(), v.numpy(), cache, np.arange(S, dtype=np.int64), 1)
    slots = cache[:, 0].transpose(1, 0, 2)                              # [KV, S, D+8]
    kp, vp = slots[..., : D // 2].copy(), slots[..., D // 2: D].copy()
    rul = np.ascontiguousarray(slots[..., D:]).view(np.float16)         # [KV, S, 4]
    kmin, kstep, vmin, vstep = (np.ascontiguousarray(rul[..., i]) for i in range(4))
    tens = [torch.from_numpy(a).to(DEV) for a in (kp, kmin, kstep, vp, vmin, vstep)]
    out = _kd().kv_dequant_decode_per_token_attention(q.to(DEV), *tens, num_kv_heads=KV)
    torch.cuda.synchronize()
    ref = oa.decode_per_token(q.numpy(), kp, kmin, kstep, vp, vmin, vstep)
    assert_close(out.cpu().numpy(), ref, what="per-token decode")


# One sequence, head_dim 64 / 128, up to 8 query heads per KV head and 16384
# keys: the split (KV head, key chunk) kernel; 20000 keys take the general path.
@pytest.mark.parametrize("H,KV,D,S,outl", [(8, 8, 64, 1, False), (6, 2, 128, 17, True), (24, 8, 64, 5000, False),
                                           (16, 2, 128, 9000, True), (4, 4, 128, 20000, False),
                                           (8, 1, 64, 3333, False)])
def test_decode_per_channel_split_chunks(H, KV, D, S, outl):
    q, t = _pc_inputs(H + S, H, KV, S, D, outl)
    kd = _kd()
    for _ in range(2):                        # the arrival counters must be left at zero
        out = kd.kv_dequant_decode_attention(q.to(DEV), *[x.to(DEV) for x in t], num_kv_heads=KV)
        torch.cuda.synchronize()
        ref = oa.decode_per_channel(q.numpy(), *[x.numpy() for x in t])
        assert_close(out.cpu().numpy(), ref, what=f"H={H} KV={KV} D={D} S={S}")


# The register kernel's thread and row counts (up to 8192 rows), the three launches
# past it (test_quantize_kv_long has more of these), inputs at odd multiples of 4
# bytes, NaN and infinities, constant channels: each byte against the oracle, K and
# V together as one by one.
@pytest.mark.parametrize("KV,S,D", [(1, 1, 64), (2, 31, 80), (3, 32, 128), (2, 33, 64), (1, 511, 80), (2, 513, 128),
                                    (2, 1025, 64), (1, 2049, 80), (2, 4096, 64), (2, 4097, 80), (3, 4999, 128),
                                    (1, 9001, 64)])
def test_quantize_kv_row_counts(KV, S, D):
    g = torch.Generator().manual_seed(S + D)
    k, v = torch.randn(KV, S, D, generator=g).half(), (3 * torch.randn(KV, S, D, generator=g)).half()
    k[0, S // 2, 1] = float("nan")
    k[0, S - 1, 2] = float("inf")
    k[KV - 1, 0, 3] = -60000.0
    v[:, :, 4] = 0.25
    v[0, S - 1, D - 1] = 100.0
    buf = torch.zeros(k.numel() + 2, dtype=torch.float16, device=DEV)
    kd_ = buf[2:].view(k.shape)
    kd_.copy_(k)
    got = _kd().quantize_kv(kd_, v.to(DEV))
    alone = _kd().quantize_per_channel(kd_)
    torch.cuda.synchronize()
    ref = oq.quantize_kv(k.numpy(), v.numpy())
    for i, (a, b) in enumerate(zip(got, ref)):
        if a.dtype == torch.uint8:
            assert np.array_equal(a.cpu().numpy(), b), f"codes {i}: {int((a.cpu().numpy() != b).sum())} differ"
        else:
            _same_fp16(a.cpu().numpy(), b)
    for a, b in zip(alone, got):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


# The last register case and the three launches: every head_dim (80: 25 rows a pass and 6
# idle threads), several KV heads (whose minima and maxima wait in their own codes), chunk
# counts held down by the KV heads, remainders, and special values in the last row of the
# last chunk of the last KV head.
@pytest.mark.parametrize("KV,S,D", [(1, 8192, 64), (2, 8193, 64), (2, 8193, 80), (3, 9001, 128), (2, 20011, 80),
                                    (40, 8200, 80), (1, 70001, 128)])
def test_quantize_kv_long(KV, S, D):
    g = torch.Generator().manual_seed(S + D)
    k, v = torch.randn(KV, S, D, generator=g).half(), (3 * torch.randn(KV, S, D, generator=g)).half()
    k[KV - 1, S - 1, D - 1] = float("nan")
    k[KV - 1, S - 1, D - 2] = float("inf")
    k[KV - 1, S - 1, 0] = -60000.0
    k[0, 0, 1] = 500.0
    v[KV - 1, :, 4] = 0.25
    v[KV - 1, S - 1, D - 1] = 100.0
    v[KV - 1, S // 2, 3] = -float("inf")
    got = _kd().quantize_kv(k.to(DEV), v.to(DEV))
    alone = _kd().quantize_per_channel(k.to(DEV))
    ref = oq.quantize_kv(k.numpy(), v.numpy())
    for i, (a, b) in enumerate(zip(got, ref)):
        if a.dtype == torch.uint8:
            assert np.array_equal(a.cpu().numpy(), b), f"codes {i}: {int((a.cpu().numpy() != b).sum())} differ"
        else:
            _same_fp16(a.cpu().numpy(), b)
    for a, b in zip(alone, got):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


# Chunks of 64, 128 and 256 keys with remainders, one chunk, waves without keys, every
# head-slot count, and head_dim 80 of both layouts; 20000 keys take the general path.
@pytest.mark.gpu
@pytest.mark.parametrize("H,KV,D,S", [(1, 1, 64, 1), (8, 8, 128, 64), (8, 8, 80, 65), (14, 2, 64, 1025), (8, 4, 80, 2049),
                                      (24, 6, 128, 3000), (32, 8, 80, 8000), (4, 2, 128, 16384), (4, 2, 64, 20000)])
def test_decode_split_per_token_and_head_dim_80(H, KV, D, S):
    """Weights and sums are fp32: 1e-5 of the output's size, against 64 bits."""
    kd = _kd()
    g = torch.Generator().manual_seed(S + D)
    q = torch.randn(H, 1, D, generator=g).half()
    kv = torch.randn(2, KV, S, D, generator=g).half()
    packed = torch.randint(0, 256, (2, KV, S, D // 2), generator=g, dtype=torch.uint8)
    mins, steps = kv.amin(-1), (torch.rand(2, KV, S, generator=g) * 0.4 + 0.05).half()
    ref = oa.decode_per_token(q.numpy(), packed[0].numpy(), mins[0].numpy(), steps[0].numpy(), packed[1].numpy(),
                                mins[1].numpy(), steps[1].numpy())
    dev = "cuda:0"
    t = [x.to(dev) for x in (packed[0], mins[0], steps[0], packed[1], mins[1], steps[1])]
    atol = (1e-5 if S <= 16384 else 1e-3) * np.abs(ref).max()
    for _ in range(2):
        out = kd.kv_dequant_decode_per_token_attention(q.to(dev), *t)
        assert_close(out.cpu().numpy(), ref, atol=atol, rtol=0, what="per-token split")
    if D == 80:
        scale, zero = (torch.rand(2, KV, D, generator=g) * 0.4 + 0.05).half(), torch.randint(0, 16, (2, KV, D), generator=g).half()
        ref = oa.decode_per_channel(q.numpy(), packed[0].numpy(), scale[0].numpy(), zero[0].numpy(), packed[1].numpy(),
                                      scale[1].numpy(), zero[1].numpy())
        c = [x.to(dev) for x in (packed[0], scale[0], zero[0], packed[1], scale[1], zero[1])]
        out = kd.kv_dequant_decode_attention(q.to(dev), *c)
        assert_close(out.cpu().numpy(), ref, atol=1e-5 * np.abs(ref).max(), rtol=0, what="per-channel split, head_dim 80")


# Columns of q * k_scale past fp16's largest number beside ordinary ones of the same
# 16-row block: the pairs that hold a column carry a power of two of its own.
@pytest.mark.parametrize("H,KV,D", [(4, 2, 64), (4, 2, 80), (4, 2, 128), (3, 3, 80)])
@pytest.mark.parametrize("M,S,causal,quant", [(150, 150, True, True), (17, 70, False, True), (33, 33, True, False)])
def test_prefill_wide_range_queries(H, KV, D, M, S, causal, quant):
    g = torch.Generator().manual_seed(D + M)
    q = torch.randn(H, M, D, generator=g)
    q[:, ::3] *= 100.0 if quant else 6000.0
    q[:, 1::3] *= 1e-3 if quant else 1.0
    q[0, M - 1] = 65504.0
    q = q.clamp(-65504, 65504).half()
    packed = torch.randint(0, 256, (2, KV, S, D // 2), generator=g, dtype=torch.uint8)
    scale = (torch.rand(2, KV, D, generator=g) * 0.4 + 0.05).half()
    scale[0, 0] = 5000.0 * (1 + scale[0, 0])
    zero = torch.randint(0, 16, (2, KV, D), generator=g).half()
    t = (packed[0], scale[0], zero[0], packed[1], scale[1], zero[1])
    out = _kd().kv_dequant_prefill_attention(q.to(DEV), *[x.to(DEV) for x in t], causal=causal, use_quant=quant)
    ref = oa.prefill_per_channel(q.numpy(), *[x.numpy() for x in t], causal=causal, use_quant=quant)
    assert np.isfinite(ref).all()
    assert_close(out.cpu().numpy(), ref, what=f"D={D} causal={causal} quant={quant}")


# Head_dim 80 holds the query column in 22 bits and its weights too, so what is left is
# fp32 rounding: logits of up to about 10 (0.5 for the small column) that are off by a
# few 2^-24 of their size, 4 * 10 * 2^-24 = 2.4e-6 at the most and less on average.
@pytest.mark.parametrize("ks,qf,bound", [(0.47, 1.0, 1e-6), (0.05, 0.05, 5e-7)])
def test_prefill_head_dim_80_precision(ks, qf, bound):
    g = torch.Generator().manual_seed(5)
    H, KV, D, S = 8, 2, 80, 600
    q = (torch.randn(H, S, D, generator=g) * qf).half()
    packed = torch.randint(0, 256, (2, KV, S, D // 2), generator=g, dtype=torch.uint8)
    scale = (torch.rand(2, KV, D, generator=g) * 0.4 + 0.05).half()
    scale[0] *= ks / 0.25
    zero = torch.randint(0, 16, (2, KV, D), generator=g).half()
    t = (packed[0], scale[0], zero[0], packed[1], scale[1], zero[1])
    out = _kd().kv_dequant_prefill_attention(q.to(DEV), *[x.to(DEV) for x in t]).cpu().numpy().astype(np.float64)
    ref = oa.prefill_per_channel(q.numpy(), *[x.numpy() for x in t])
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    assert err <= bound, err


# A channel whose scale underflows to 0 with the minimum 0 has the zero point NaN
# (0 / 0), and the formula makes every output of its KV head NaN, as head_dim 80 does.
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_head_dim_80_zero_points_that_are_no_numbers(bad):
    H, KV, D, S = 4, 2, 80, 130
    q, t = _pc_inputs(5, H, KV, S, D, False)
    t[2][0, 77] = bad                                                    # the K zero point of the first KV head
    dev = [x.to(DEV) for x in t]
    qs = torch.randn(H, 40, D, generator=torch.Generator().manual_seed(1)).half()
    for out, ref in [(_kd().kv_dequant_decode_attention(q.to(DEV), *dev), oa.decode_per_channel(q.numpy(), *[x.numpy() for x in t])),
                     (_kd().kv_dequant_prefill_attention(qs.to(DEV), *dev), oa.prefill_per_channel(qs.numpy(), *[x.numpy() for x in t]))]:
        out = out.cpu().numpy()
        assert np.isnan(out[:H // KV]).all() and np.isnan(ref[:H // KV]).all()
        assert_close(out[H // KV:], ref[H // KV:], what=f"zero point {bad}, the other KV head")
    raw = _kd().kv_dequant_decode_attention(q.to(DEV), *dev, use_quant=False)
    assert torch.isfinite(raw).all()                                     # the raw codes need no ruler


def test_prefill_codes_past_four_gib():
    """A KV head's codes pass 2^32 bytes: the last keys, which take all of the weight, are
    read where they lie and not from the start."""
    D, S = 80, 2**32 // 40 + 300
    q = torch.ones(1, 1, D, dtype=torch.float16, device=DEV)
    one, zero = torch.ones(1, D, dtype=torch.float16, device=DEV), torch.zeros(1, D, dtype=torch.float16, device=DEV)
    k = torch.zeros(1, S, D // 2, dtype=torch.uint8, device=DEV)
    v = torch.zeros_like(k)
    k[:, -100:] = 0xFF
    v[:, -100:] = 0x33
    out = _kd().kv_dequant_prefill_attention(q, k, one, zero, v, one, zero, causal=False)
    assert (out - 3.0).abs().max() <= 1e-5                                   # exp(-134) for every other key


@pytest.mark.parametrize("H,KV,D", [(32, 8, 64), (32, 4, 80), (32, 8, 128)])
def test_prefill_wide_range_queries_two_heads_per_workgroup(H, KV, D):
    """The long prefills' form (more than 256 workgroups of two heads): waves with and
    without such columns, staging and not, walk different loops through the same barriers."""
    M = 1100
    g = torch.Generator().manual_seed(D)
    q = torch.randn(H, M, D, generator=g)
    q[:, 5::97] *= 1e4
    q[1::2, 200:300] *= 1e4
    q = q.clamp(-65504, 65504).half()
    packed = torch.randint(0, 256, (2, KV, M, D // 2), generator=g, dtype=torch.uint8)
    scale = (torch.rand(2, KV, D, generator=g) * 0.4 + 0.05).half()
    scale[0, 0] *= 500
    zero = torch.randint(0, 16, (2, KV, D), generator=g).half()
    t = (packed[0], scale[0], zero[0], packed[1], scale[1], zero[1])
    out = _kd().kv_dequant_prefill_attention(q.to(DEV), *[x.to(DEV) for x in t]).cpu()
    G, heads = H // KV, [0, 1, H // KV, H - 1]
    for h in heads:
        one = [x[h // G: h // G + 1].numpy() for x in t]
        assert_close(out[h:h + 1].numpy(), oa.prefill_per_channel(q[h:h + 1].numpy(), *one), what=f"D={D} head {h}")
    assert torch.isfinite(out).all()
