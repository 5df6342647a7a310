"""GPU parity of flash-attention forward against the brute-force CPU oracle, through the C ABI.

Tolerance: fp16 / bf16 inputs: max-abs <= 2e-2 (outputs are convex combinations of V rows, |o| <~ 4; the
probabilities are rounded to the 16-bit input type before P V as in the reference's linalg form,
test/python/mlir/hexkl_attention/input.mlir:140-145); fp32 inputs: rel-err 1e-5.
"""
import math

import numpy as np
import pytest
import torch

from util import from_np, rel_err, to_np

pytestmark = pytest.mark.gpu


def _gen(seed):
    return torch.Generator().manual_seed(seed)


def _qkv(Z, H, S, D, dtype, seed=0, rand=False):
    g = _gen(seed)
    f = torch.rand if rand else torch.randn
    return tuple(f(Z, H, S, D, generator=g).to(dtype) for _ in range(3))


def _oracle(oracle, q, k, v, scale, causal, out_dtype=None):
    qn, tag = to_np(q)
    kn, _ = to_np(k)
    vn, _ = to_np(v)
    o = oracle.attention(qn, kn, vn, scale, causal, out_dtype=np.float32, dtype=tag)
    return torch.from_numpy(o)


CASES = [(1, 1, 1024, 64), (2, 3, 256, 128), (1, 2, 128, 128), (1, 2, 64, 64), (1, 1, 200, 128), (2, 1, 77, 64),
         (1, 1, 1, 128), (1, 3, 129, 128), (1, 1, 640, 128)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
def test_attention_parity_half(hexmi, oracle, case, dtype, causal):
    Z, H, S, D = case
    q, k, v = _qkv(Z, H, S, D, dtype)
    scale = 1.0 / math.sqrt(D)
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal).cpu()
    want = _oracle(oracle, q, k, v, scale, causal)
    assert got.dtype == dtype
    tol = 2e-2 if dtype == torch.float16 else 4e-2
    assert (got.float() - want).abs().max() <= tol
    got32 = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out_dtype=torch.float32).cpu()
    assert (got32 - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [(1, 2, 300, 80), (2, 1, 129, 96), (1, 3, 64, 32), (1, 1, 513, 8), (2, 8, 200, 48),
                                  (1, 1, 1000, 120), (1, 2, 77, 16), (1, 1, 260, 112), (1, 16, 384, 40), (1, 1, 1, 72)])
def test_attention_other_head_sizes(hexmi, oracle, case, dtype, causal):
    # head sizes below 128 in multiples of 8 run on tiles for 64 or 128 padded with zero columns (up to 64 keys the
    # 128-query kernel, these few heads beyond that the key-group kernel; the former with more: MANY_UNIT_CASES); the output buffer starts as NaN and has one row more than the result, which must stay as it is
    Z, H, S, D = case
    q, k, v = _qkv(Z, H, S, D, dtype, seed=D + S)
    scale = 1.0 / math.sqrt(D)
    buf = torch.full((Z * H * S + 1, D), float("nan"), dtype=dtype, device="cuda")
    out = buf[:Z * H * S].view(Z, H, S, D)
    hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out=out)
    want = _oracle(oracle, q, k, v, scale, causal)
    tol = 2e-2 if dtype == torch.float16 else 4e-2
    assert (out.cpu().float() - want).abs().max() <= tol
    assert torch.isnan(buf[-1]).all()
    got32 = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out_dtype=torch.float32).cpu()
    assert (got32 - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [(1, 2, 300, 256), (2, 1, 129, 192), (1, 3, 64, 136), (1, 8, 200, 160), (1, 1, 1000, 200),
                                  (1, 1, 1, 256), (2, 8, 515, 144)])
def test_attention_head_sizes_up_to_256(hexmi, oracle, case, dtype, causal):
    # head sizes above 128 run the kernel for 128 on two halves of the head: the scores sum over both halves' K
    # tiles, the second half is padded like a narrow head
    Z, H, S, D = case
    q, k, v = _qkv(Z, H, S, D, dtype, seed=D + S)
    scale = 1.0 / math.sqrt(D)
    buf = torch.full((Z * H * S + 1, D), float("nan"), dtype=dtype, device="cuda")
    out = buf[:Z * H * S].view(Z, H, S, D)
    hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out=out)
    want = _oracle(oracle, q, k, v, scale, causal)
    tol = 2e-2 if dtype == torch.float16 else 4e-2
    assert (out.cpu().float() - want).abs().max() <= tol
    assert torch.isnan(buf[-1]).all()
    got32 = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out_dtype=torch.float32).cpu()
    assert (got32 - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


# widths on both sides of 80 and 96 columns (the instances that leave the rest of 128 out), both kernels, heads where they stand
@pytest.mark.parametrize("D", [72, 80, 88, 96, 104])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Z,H,S", [(1, 2, 33), (2, 8, 700), (4, 35, 260)])
def test_attention_narrow_heads_equal_the_zero_padded_problem(hexmi, D, dtype, Z, H, S):
    q, k, v = (t.cuda() for t in _qkv(Z, H, S, D, dtype, seed=D))
    scale = 1.0 / math.sqrt(D)
    for causal in (False, True):
        qp, kp, vp = (torch.nn.functional.pad(t, (0, 128 - D)) for t in (q, k, v))
        want = hexmi.flash_attention(qp, kp, vp, scale, causal)[..., :D]
        assert torch.equal(hexmi.flash_attention(q, k, v, scale, causal), want)
        wide = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
        assert torch.equal(hexmi.flash_attention(*wide, scale, causal), want)


def test_attention_padded_head_equals_the_zero_padded_problem(hexmi):
    # head size 80 on the kernel for 128 is the 128-wide problem with 48 zero columns in Q, K and V (and 1/sqrt(80)):
    # the same kernel, the same arithmetic -- bit for bit
    D = 80                                               # 176 units of 64 queries: key groups; 700: the 128-query kernel
    for Z, H, S in ((2, 8, 700), (4, 35, 260)):
        q, k, v = _qkv(Z, H, S, D, torch.float16, seed=31)
        scale = 1.0 / math.sqrt(D)
        for causal in (False, True):
            got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal).cpu()
            qp, kp, vp = (torch.nn.functional.pad(t, (0, 48)) for t in (q, k, v))
            want = hexmi.flash_attention(qp.cuda(), kp.cuda(), vp.cuda(), scale, causal).cpu()
            assert torch.equal(got, want[..., :D])
            assert (want[..., D:] == 0).all()
    # and head size 192 is the 256-wide problem with 64 zero columns (both on the two-halves form)
    q, k, v = _qkv(1, 8, 400, 192, torch.float16, seed=32)
    scale = 1.0 / math.sqrt(192)
    for causal in (False, True):
        got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal).cpu()
        qp, kp, vp = (torch.nn.functional.pad(t, (0, 64)) for t in (q, k, v))
        want = hexmi.flash_attention(qp.cuda(), kp.cuda(), vp.cuda(), scale, causal).cpu()
        assert torch.equal(got, want[..., :192])
        assert (want[..., 192:] == 0).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("case", [(1, 1, 1024, 64), (1, 2, 100, 128), (2, 2, 65, 32), (1, 1, 130, 80),
                                  # head sizes 64 and 128 run on the fp32 matrix cores: ragged query and key blocks,
                                  # several workgroups per head, a single row
                                  (2, 3, 333, 64), (1, 2, 515, 128), (1, 1, 1, 64), (3, 1, 129, 128),
                                  # narrower heads in multiples of 4: the same kernels on padded tiles
                                  (1, 2, 300, 4), (2, 1, 257, 36), (1, 3, 200, 100), (1, 1, 640, 124), (2, 2, 129, 72)])
def test_attention_parity_fp32(hexmi, oracle, case, causal):
    # (1,1,1024,64) rand inputs, scale 0.5, non-causal is test_flash_attention.py:20-34,171-213
    Z, H, S, D = case
    q, k, v = _qkv(Z, H, S, D, torch.float32, rand=True)
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), 0.5, causal).cpu()
    want = _oracle(oracle, q, k, v, 0.5, causal)
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("case", [(2, 8, 2048, 64), (1, 4, 1536 + 40, 128)])
def test_attention_fp32_larger_and_randn(hexmi, case, causal):
    # N(0,1) operands (scores of both signs, running maxima that move) at sizes with many key blocks. Oracle: the
    # PyTorch CPU call the reference's test uses (test/python/triton/test_flash_attention.py:212), in float64.
    Z, H, S, D = case
    q, k, v = _qkv(Z, H, S, D, torch.float32, seed=11)
    scale = 1.0 / math.sqrt(D)
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal).cpu()
    want = torch.nn.functional.scaled_dot_product_attention(q.double(), k.double(), v.double(), is_causal=causal,
                                                            scale=scale)
    assert got.dtype == torch.float32
    assert torch.allclose(got.double(), want, rtol=1e-5, atol=2e-6)


def test_reference_call_site(hexmi, oracle):
    Z, H, N_CTX, D_HEAD = 1, 1, 1024, 64
    q, k, v = _qkv(Z, H, N_CTX, D_HEAD, torch.float32, rand=True, seed=1)
    out = torch.zeros_like(q)
    hexmi.kernels.attention_fwd_kernel[(4,)](
        pid1=0, Q=q, K=k, V=v, sm_scale=0.5, Out=out, H=H, N_CTX=N_CTX, BLOCK_M=N_CTX // 4, BLOCK_DMODEL=D_HEAD,
        BLOCK_N=64, STAGE=1, stride_0=H * N_CTX * D_HEAD, stride_1=N_CTX * D_HEAD, stride_2=D_HEAD, stride_3=1,
        enableVectorization=True, enableSplitReduceGeneric=True, enableHVXInlining=True, enableSCFLoopUnroll=True,
        enableMultiThreading=True, enableHexKL=False, enableVTCMTiling=False, enableConvertToHexagonmem=False,
        enableHexagonmemCopyToDMA=False)
    assert torch.allclose(out, _oracle(oracle, q, k, v, 0.5, False), rtol=1e-5, atol=1e-6)


def test_reference_call_site_one_head_per_launch(hexmi, oracle):
    # pid1 = off_hz picks the (z, h) pair a launch computes (test_flash_attention.py:102-105): a loop over Z * H
    # fills the output head by head, and a single launch leaves the other heads untouched
    Z, H, N_CTX, D_HEAD = 2, 3, 256, 64
    q, k, v = _qkv(Z, H, N_CTX, D_HEAD, torch.float32, rand=True, seed=4)
    want = _oracle(oracle, q, k, v, 0.5, False)
    out = torch.full_like(q, -7.0)
    kw = dict(Q=q, K=k, V=v, sm_scale=0.5, Out=out, H=H, N_CTX=N_CTX, BLOCK_M=64, BLOCK_DMODEL=D_HEAD, BLOCK_N=64,
              STAGE=1, stride_0=H * N_CTX * D_HEAD, stride_1=N_CTX * D_HEAD, stride_2=D_HEAD, stride_3=1)
    hexmi.kernels.attention_fwd_kernel[(4,)](pid1=4, **kw)              # z = 1, h = 1
    assert torch.allclose(out[1, 1], want[1, 1], rtol=1e-5, atol=1e-6)
    untouched = torch.ones(Z, H, dtype=torch.bool)
    untouched[1, 1] = False
    assert (out[untouched] == -7.0).all()
    for pid1 in range(Z * H):
        hexmi.kernels.attention_fwd_kernel[(4,)](pid1=pid1, **kw)
    assert torch.allclose(out, want, rtol=1e-5, atol=1e-6)
    with pytest.raises(ValueError):
        hexmi.kernels.attention_fwd_kernel[(4,)](pid1=Z * H, **kw)
    all_heads = torch.zeros_like(q)
    hexmi.kernels.attention_fwd_kernel[(4,)](pid1=None, **{**kw, "Out": all_heads})
    assert torch.equal(all_heads, out)


def test_hexkl_attention_fixture_types(hexmi, oracle):
    # test/python/mlir/hexkl_attention: fp16 Q/K/V ~ N(0, 0.5) rounded to 4 decimals, fp32 output, MAX_DIFF 1e-3
    g = _gen(2)
    q, k, v = ((torch.randn(1, 1, 1024, 64, generator=g) * 0.5 * 10000).round() / 10000 for _ in range(3))
    q, k, v = q.half(), k.half(), v.half()
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), 0.5, False, out_dtype=torch.float32).cpu()
    assert (got - _oracle(oracle, q, k, v, 0.5, False)).abs().max() <= 1e-3


def test_causal_invariants(hexmi):
    q, k, v = _qkv(2, 2, 512, 128, torch.float16, seed=3)
    o = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), None, True).cpu()
    assert torch.equal(o[:, :, 0], v[:, :, 0])                            # row 0 attends to key 0 only
    k2, v2 = k.clone(), v.clone()
    k2[:, :, 300:] = 9.0
    v2[:, :, 300:] = -7.0
    o2 = hexmi.flash_attention(q.cuda(), k2.cuda(), v2.cuda(), None, True).cpu()
    assert torch.equal(o2[:, :, :300], o[:, :, :300])                      # later keys never reach earlier rows
    # constant V: any softmax weights give back the constant
    vc = torch.full_like(v, 0.75)
    oc = hexmi.flash_attention(q.cuda(), k.cuda(), vc.cuda(), None, False).cpu()
    assert (oc.float() - 0.75).abs().max() <= 1e-3


@pytest.mark.parametrize("shape", [(4, 32, 4096, 128), (1, 32, 16384, 128)])
def test_attention_config_sizes(hexmi, oracle, shape):
    """Measured configurations (causal fp16). The oracle runs on 3 heads x 48 query rows spread over the
    sequence (all keys each); the whole output is covered by properties: heads are independent (running one
    head alone gives the same bits) and row 0 of every head equals V[0]."""
    from hexmi.workloads import attention_inputs
    Z, H, S, D = shape
    inp = attention_inputs(Z, H, S, D)
    q, k, v, scale = inp["q"], inp["k"], inp["v"], inp["sm_scale"]
    o = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, True).cpu()
    assert torch.equal(o[:, :, 0], v[:, :, 0])
    rows = torch.cat([torch.arange(0, 16), torch.arange(S // 2 - 8, S // 2 + 8), torch.arange(S - 16, S)])
    for (z, h) in [(0, 0), (Z - 1, H - 1), (0, 17)]:
        qh, kh, vh = q[z, h], k[z, h], v[z, h]
        s = (qh[rows].double() @ kh.double().t()) * scale
        mask = torch.arange(S)[None, :] > rows[:, None]
        s = s.masked_fill(mask, float("-inf"))
        want = torch.softmax(s, -1) @ vh.double()
        assert (o[z, h, rows].double() - want).abs().max() <= 2e-2
        one = hexmi.flash_attention(qh[None, None].cuda(), kh[None, None].cuda(), vh[None, None].cuda(), scale, True).cpu()
        assert torch.equal(one[0, 0], o[z, h])
    # cross-check the in-test closed form against the oracle on a short prefix (causal rows see only keys <= row)
    z, h = 0, 0
    P = 192
    want_o = _oracle(oracle, q[z, h, :P][None, None], k[z, h, :P][None, None], v[z, h, :P][None, None], scale, True)
    assert (o[z, h, :P].float() - want_o[0, 0]).abs().max() <= 2e-2


def test_attention_errors(hexmi):
    q = torch.zeros(1, 1, 8, 16, dtype=torch.float16)
    with pytest.raises(ValueError):
        hexmi.flash_attention(q, q[:, :, :4], q)
    with pytest.raises(TypeError):
        hexmi.flash_attention(q, q.float(), q)
    assert hexmi.flash_attention(torch.empty(1, 2, 0, 64, device="cuda", dtype=torch.float16),
                                 torch.empty(1, 2, 0, 64, device="cuda", dtype=torch.float16),
                                 torch.empty(1, 2, 0, 64, device="cuda", dtype=torch.float16)).shape == (1, 2, 0, 64)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("scale", [0.0, -0.3])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_attention_zero_and_negative_scale(hexmi, oracle, dtype, scale, causal):
    # the matrix-core kernels take the row maximum before scaling, which is right for a positive scale only: other
    # scales must still give softmax(scale * Q K^T) V (scale 0: the mean of the visible V rows)
    q, k, v = _qkv(1, 2, 200, 128, dtype, seed=11)
    o = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out_dtype=torch.float32).cpu()
    want = _oracle(oracle, q, k, v, scale, causal)
    assert torch.isfinite(o).all()
    assert (o - want).abs().max() <= (2e-2 if dtype == torch.float16 else 1e-5 * want.abs().max())
    if scale == 0.0 and not causal:
        assert (o - v.float().mean(2, keepdim=True)).abs().max() <= 2e-3


def test_attention_head_size_256(hexmi, oracle):
    q, k, v = _qkv(1, 2, 70, 256, torch.float16, seed=12)
    o = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), 1 / 16.0, True, out_dtype=torch.float32).cpu()
    assert (o - _oracle(oracle, q, k, v, 1 / 16.0, True)).abs().max() <= 2e-2


# ---- tm_tensor.attention: [B, S, D] operands, rectangular scores, additive mask -----------------------------
def _oracle_masked(oracle, q, k, v, mask, scale):
    qn, tag = to_np(q)
    kn, _ = to_np(k)
    vn, _ = to_np(v)
    mn = None if mask is None else to_np(mask)[0]
    return torch.from_numpy(oracle.attention_masked(qn, kn, vn, mn, scale, out_dtype=np.float32, dtype=tag))


def _mask(B, Sq, Skv, dtype, seed, drop=0.3):
    g = _gen(seed)
    m = torch.randn(B, Sq, Skv, generator=g)
    m[torch.rand(B, Sq, Skv, generator=g) < drop] = float("-inf")
    m[:, :, 0] = 0.0                                   # every row keeps a key
    return m.to(dtype)


MASKED_CASES = [(2, 128, 128, 128), (3, 200, 72, 64), (1, 1, 64, 128), (2, 77, 516, 128), (1, 300, 4, 64),
                (1, 130, 1024, 128), (2, 65, 66, 64), (1, 40, 100, 80),   # the last two: Skv % 4 != 0 / other D
                # more than 128 queries and Skv % 8 == 0 in few units of 64 queries: the key-group kernel (the mask tiles
                # that 256-row workgroups stage through LDS: MANY_UNIT_CASES)
                (3, 300, 520, 128), (2, 513, 72, 64), (1, 257, 2048 + 8, 128), (40, 129, 136, 64),
                # head sizes below 128 in multiples of 8: tiles padded with zero columns
                (2, 200, 72, 80), (1, 300, 520, 96), (3, 129, 136, 32), (1, 77, 516, 40), (2, 64, 64, 112),
                # key counts that are not multiples of 4
                (4, 1024, 77, 64), (2, 300, 1, 128), (1, 129, 515, 80)]


@pytest.mark.parametrize("with_mask", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", MASKED_CASES)
def test_masked_attention_parity_half(hexmi, oracle, case, dtype, with_mask):
    B, Sq, Skv, D = case
    g = _gen(21)
    q = torch.randn(B, Sq, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    mask = _mask(B, Sq, Skv, dtype, 22) if with_mask else None
    scale = 1.0 / math.sqrt(D)
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), None if mask is None else mask.cuda()).cpu()
    want = _oracle_masked(oracle, q, k, v, mask, scale)
    assert got.dtype == dtype and got.shape == (B, Sq, D)
    assert (got.float() - want).abs().max() <= (2e-2 if dtype == torch.float16 else 4e-2)
    got32 = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), None if mask is None else mask.cuda(),
                            out_dtype=torch.float32).cpu()
    assert (got32 - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


# more units of 64 queries than the key-group kernel takes, so the 128-query kernels: masks staged through LDS (several key
# blocks, a ragged last one, ragged rows), read in runs of four keys, no mask with an odd key count; heads of 64 and 128
# and padded ones
MANY_UNIT_CASES = [(100, 200, 520, 128, True), (150, 260, 712, 64, True), (100, 200, 516, 128, True), (150, 260, 524, 64, True),
                   (100, 200, 520, 80, True), (150, 260, 516, 40, True), (100, 200, 515, 128, False), (150, 260, 77, 64, False),
                   (100, 200, 333, 96, False), (150, 260, 515, 24, False)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", MANY_UNIT_CASES)
def test_attention_of_many_units(hexmi, case, dtype):
    # the bound of the parity tests (fp32 output, probabilities rounded to 16 bits)
    B, Sq, Skv, D, with_mask = case
    g = _gen(67)
    q = torch.randn(B, Sq, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    mask = _mask(B, Sq, Skv, dtype, 68) if with_mask else None
    scores = q.float() @ k.float().transpose(1, 2) / math.sqrt(D)
    if with_mask:
        scores = scores + mask.float()
    want = torch.softmax(scores, dim=-1) @ v.float()
    buf = torch.full((B * Sq + 1, D), float("nan"), dtype=torch.float32, device="cuda")
    hexmi.attention(q.cuda(), k.cuda(), v.cuda(), None if mask is None else mask.cuda(), out=buf[:B * Sq].view(B, Sq, D))
    got = buf.cpu()
    assert (got[:B * Sq].view(B, Sq, D) - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)
    assert torch.isnan(got[B * Sq]).all()


@pytest.mark.parametrize("H,S,D,dtype,same_bits", [(40, 4100, 64, torch.bfloat16, True), (12, 4608, 96, torch.float16, True),
                                                   (20, 5000, 128, torch.float16, True), (17, 2048, 128, torch.float16, False),
                                                   (120, 300, 64, torch.float16, False)])
def test_causal_head_beside_others(hexmi, H, S, D, dtype, same_bits):
    # one head alone against the same head among H: the same bits from 4096 queries on; below, another kernel may run it,
    # whose 16-bit probabilities and result round apart (fp16: a result below 4 in units of 2^-9 at most, so 2^-8)
    q, k, v = _qkv(1, H, S, D, dtype, seed=69)
    many = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), None, True).cpu()
    for h in (0, H // 2, H - 1):
        one = hexmi.flash_attention(*(t[:, h:h + 1].contiguous().cuda() for t in (q, k, v)), None, True).cpu()
        if same_bits:
            assert torch.equal(one[0, 0], many[0, h])
        else:
            assert (one[0, 0].float() - many[0, h].float()).abs().max() <= 2.0 ** -8


def test_attention_workspace_under_capture_and_on_two_streams(hexmi):
    # few queries over many keys: hexmi.attention hands the library scratch for the chunks' sums. Captured, the scratch is
    # the graph's own and every replay must match the eager call; on two streams at once each call has its own
    B, Skv, D = 4, 4096, 128
    g = _gen(70)
    k, v = (torch.randn(B, Skv, D, generator=g).half().cuda() for _ in range(2))
    mask = torch.zeros(B, 2, Skv, dtype=torch.float16, device="cuda")
    mask[:, :, :700] = float("-inf")
    q = torch.randn(B, 2, D, generator=g).half().cuda()
    out = torch.zeros(B, 2, D, dtype=torch.float16, device="cuda")
    hexmi.attention(q, k, v, mask, out=out)                              # warm-up outside the capture
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            hexmi.attention(q, k, v, mask, out=out)
    for _ in range(3):
        q.copy_(torch.randn(B, 2, D, generator=g).half().cuda())
        eager = hexmi.attention(q, k, v, mask)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    qs = [torch.randn(B, 2, D, generator=g).half().cuda() for _ in range(2)]
    want = [hexmi.attention(x, k, v, mask) for x in qs]
    streams, outs = [torch.cuda.Stream(), torch.cuda.Stream()], [[], []]
    torch.cuda.synchronize()
    for _ in range(20):
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                outs[i].append(hexmi.attention(qs[i], k, v, mask))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(o, want[i]) for o in outs[i])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [(2, 5, 1, 64), (1, 33, 3, 128), (3, 129, 63, 64), (2, 130, 65, 128), (2, 64, 127, 80),
                                  (3, 128, 130, 128), (1, 300, 1023, 96), (2, 257, 2051, 128)])
def test_masked_attention_mask_rows_of_any_length_and_alignment(hexmi, oracle, case, dtype):
    # mask rows of an odd number of keys on the matrix cores, the mask itself one element off its allocation; the
    # tolerances are those of test_masked_attention_parity_half (the test below holds these masks to fp32 sums)
    B, Sq, Skv, D = case
    g = _gen(27)
    q = torch.randn(B, Sq, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    mask = _mask(B, Sq, Skv, dtype, 28)
    shifted = torch.empty(mask.numel() + 1, dtype=dtype, device="cuda")[1:].view(B, Sq, Skv)
    shifted.copy_(mask)
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), shifted, out_dtype=torch.float32).cpu()
    want = _oracle_masked(oracle, q, k, v, mask, 1.0 / math.sqrt(D))
    assert (got - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


@pytest.mark.parametrize("case", [(2, 50, 70, 32), (1, 64, 64, 128), (1, 33, 129, 64),
                                  # Skv % 4 == 0 with head size 64 / 128: the fp32 matrix-core kernel with a mask
                                  (2, 200, 72, 64), (1, 130, 516, 128), (3, 129, 1028, 64),
                                  # ... and narrower heads on padded tiles
                                  (2, 200, 72, 80), (1, 130, 516, 36), (2, 129, 132, 100)])
def test_masked_attention_parity_fp32(hexmi, oracle, case):
    B, Sq, Skv, D = case
    g = _gen(23)
    q, k, v = torch.rand(B, Sq, D, generator=g), torch.rand(B, Skv, D, generator=g), torch.rand(B, Skv, D, generator=g)
    mask = _mask(B, Sq, Skv, torch.float32, 24)
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), mask.cuda()).cpu()
    want = _oracle_masked(oracle, q, k, v, mask, 1.0 / math.sqrt(D))
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-6)


def test_masked_attention_properties(hexmi):
    # a causal additive mask reproduces the causal kernel; a constant added to the mask changes nothing;
    # host tensors are staged and `out` is filled in place
    B, S, D = 2, 256, 128
    g = _gen(25)
    q, k, v = (torch.randn(B, S, D, generator=g).half() for _ in range(3))
    tri = torch.full((S, S), float("-inf")).triu(1).half().expand(B, S, S).contiguous()
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), tri.cuda()).cpu()
    causal = hexmi.flash_attention(q.view(B, 1, S, D).cuda(), k.view(B, 1, S, D).cuda(), v.view(B, 1, S, D).cuda(),
                                   None, True).cpu().view(B, S, D)
    assert (got.float() - causal.float()).abs().max() <= 2e-3
    shifted = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), (tri + 2.0).cuda()).cpu()
    assert (shifted.float() - got.float()).abs().max() <= 2e-3
    out = torch.empty(B, S, D, dtype=torch.float16)
    ret = hexmi.attention(q, k, v, tri, out=out)
    assert ret is out and torch.equal(out, got)
    with pytest.raises(ValueError):
        hexmi.attention(q, k, v, tri[:, :, :-4])


def test_masked_attention_fully_masked_row_is_nan(hexmi):
    # LowerTmTensor.cpp:164-222: max = -inf, x - max = nan, exp / sum / div propagate it
    B, S, D = 1, 64, 64
    g = _gen(26)
    q, k, v = (torch.randn(B, S, D, generator=g).half() for _ in range(3))
    mask = torch.zeros(B, S, S).half()
    mask[0, 5, :] = float("-inf")
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), mask.cuda()).cpu()
    assert torch.isnan(got[0, 5]).all() and not torch.isnan(got[0, :5]).any() and not torch.isnan(got[0, 6:]).any()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [(2, 200, 320, 128, 40), (1, 130, 260, 64, 70)])
def test_masked_attention_window_mask(hexmi, oracle, case, dtype):
    # a band mask (-inf outside a window that ends past the row index): most rows have every key of their first
    # 64-key blocks masked out, so the running maximum is still -inf when the first finite score arrives
    B, Sq, Skv, D, width = case
    g = _gen(31)
    q = torch.randn(B, Sq, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    rows, cols = torch.arange(Sq)[:, None], torch.arange(Skv)[None, :]
    keep = (cols > rows + 60 - width) & (cols <= rows + 60)
    mask = torch.zeros(Sq, Skv).masked_fill(~keep, float("-inf")).to(dtype).expand(B, Sq, Skv).contiguous()
    scale = 1.0 / math.sqrt(D)
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), mask.cuda()).cpu()
    want = _oracle_masked(oracle, q, k, v, mask, scale)
    assert not torch.isnan(got).any()
    assert (got.float() - want).abs().max() <= (2e-2 if dtype == torch.float16 else 4e-2)


@pytest.mark.parametrize("case", [(1, 1, 8200, 64, True), (1, 1, 8192, 128, False), (1, 2, 8192 + 130, 128, True)])
def test_attention_long_sequences(hexmi, oracle, case):
    # long sequences, few heads (too few 256-row workgroups to fill the chip: 128-row workgroups)
    Z, H, S, D, causal = case
    q, k, v = _qkv(Z, H, S, D, torch.float16, seed=7)
    scale = 1.0 / math.sqrt(D)
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal).cpu()
    want = _oracle(oracle, q, k, v, scale, causal)
    assert (got.float() - want).abs().max() <= 2e-2
    # rows of different 256-row blocks do not interact: the first 300 rows of a causal run equal a 300-row run
    if causal:
        short = hexmi.flash_attention(q[:, :, :300].contiguous().cuda(), k[:, :, :300].contiguous().cuda(),
                                      v[:, :, :300].contiguous().cuda(), scale, True).cpu()
        assert (short.float() - got[:, :, :300].float()).abs().max() <= 2e-3


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("case", [(2, 16, 2048 + 70, 128, torch.float16), (1, 40, 2048, 64, torch.float16),
                                  (4, 8, 2304, 128, torch.bfloat16), (1, 8, 8192 + 130, 128, torch.float16)])
def test_attention_256_row_workgroups(hexmi, case, causal):
    # from 2048 keys on, grids with at least one 256-row block per CU run 8-wave workgroups (256 query rows per
    # K/V tile copy): ragged lengths, head counts off the XCD multiple, both dtypes. Oracle: the PyTorch CPU call
    # the reference's test uses (test/python/triton/test_flash_attention.py:212).
    Z, H, S, D, dtype = case
    q, k, v = _qkv(Z, H, S, D, dtype, seed=9)
    scale = 1.0 / math.sqrt(D)
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out_dtype=torch.float32).cpu()
    want = torch.nn.functional.scaled_dot_product_attention(q.float(), k.float(), v.float(), is_causal=causal,
                                                            scale=scale)
    assert (got - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("case", [(2, 52, 2048, torch.float16), (1, 100, 2048 + 40, torch.bfloat16)])
def test_attention_three_workgroups_per_cu(hexmi, case, causal):
    # D = 64 between 2048 and 4095 keys with six or more 128-row units per CU runs three 128-row workgroups per CU
    # (a persistent grid of 768): head counts off the XCD multiple, a ragged length, both dtypes. Oracle: the
    # PyTorch CPU call the reference's test uses (test/python/triton/test_flash_attention.py:212).
    Z, H, S, dtype = case
    q, k, v = _qkv(Z, H, S, 64, dtype, seed=13)
    scale = 1.0 / math.sqrt(64)
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out_dtype=torch.float32).cpu()
    want = torch.nn.functional.scaled_dot_product_attention(q.float(), k.float(), v.float(), is_causal=causal,
                                                            scale=scale)
    assert (got - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("case", [(2, 36, 1280, 64), (1, 72, 1024, 128), (5, 13, 777, 128)])
def test_attention_more_units_than_resident_workgroups(hexmi, case, causal):
    # more (head, query block) units than the persistent grid holds, head counts that are and are not multiples of
    # the 8 XCDs, ragged lengths: every unit must be visited exactly once. Oracle: the PyTorch CPU call the
    # reference's test uses (test/python/triton/test_flash_attention.py:212).
    Z, H, S, D = case
    q, k, v = _qkv(Z, H, S, D, torch.float16, seed=5)
    scale = 1.0 / math.sqrt(D)
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, causal, out_dtype=torch.float32).cpu()
    want = torch.nn.functional.scaled_dot_product_attention(q.float(), k.float(), v.float(), is_causal=causal,
                                                            scale=scale)
    assert (got - want).abs().max() <= 5e-3


@pytest.mark.parametrize("case", [(1, 32, 3840, 128), (1, 32, 2176, 128), (1, 24, 5120, 128), (1, 64, 2176, 64)])
def test_causal_attention_block_counts_off_the_power_of_two(hexmi, case):
    # causal units of unequal length are dealt to the persistent workgroups in groups of heads, longest first and
    # padded to whole passes (15, 9, 20 query blocks of 256 rows on 32 workgroups per XCD; 17 blocks of 128 rows on
    # 96): every unit must be visited exactly once, so the output starts as NaN. Oracle: the PyTorch CPU call the
    # reference's test uses (test/python/triton/test_flash_attention.py:212).
    Z, H, S, D = case
    q, k, v = _qkv(Z, H, S, D, torch.float16, seed=21)
    scale = 1.0 / math.sqrt(D)
    out = torch.full((Z, H, S, D), float("nan"), dtype=torch.float32, device="cuda")
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), scale, True, out=out).cpu()
    assert not torch.isnan(got).any()
    want = torch.nn.functional.scaled_dot_product_attention(q.float(), k.float(), v.float(), is_causal=True, scale=scale)
    assert (got - want).abs().max() <= 5e-3


# units of 64 queries whose keys four groups of waves share (flash_attn_keys.hip): one step of 128 keys and its edges,
# groups left without a tile, ragged row tiles; and few enough queries that the key range is cut over workgroups
KEY_GROUP_CASES = [(1, 1, 65, 64), (2, 33, 96, 128), (3, 64, 97, 64), (1, 65, 127, 128), (8, 31, 128, 64), (2, 32, 129, 128),
                   (2, 96, 160, 64), (1, 200, 257, 128), (16, 127, 385, 64), (8, 1, 4096, 128), (3, 2, 8191, 64), (24, 70, 1000, 128)]


@pytest.mark.parametrize("with_mask", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", KEY_GROUP_CASES)
def test_attention_keys_shared_by_wave_groups(hexmi, case, dtype, with_mask):
    # against the same sums in fp32; fp32 output, so what differs is the rounding of the probabilities to the 16-bit
    # type (relative 2^-11 / 2^-8 each, averaged over V of unit variance): the bounds of the parity tests above
    B, Sq, Skv, D = case
    g = _gen(61)
    q = torch.randn(B, Sq, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    mask = _mask(B, Sq, Skv, dtype, 62) if with_mask else None
    scores = q.float() @ k.float().transpose(1, 2) / math.sqrt(D)
    if mask is not None:
        scores = scores + mask.float()
    want = torch.softmax(scores, dim=-1) @ v.float()
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), None if mask is None else mask.cuda(), out_dtype=torch.float32).cpu()
    assert (got - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [(1, 1, 65, 64), (1, 3, 127, 128), (2, 4, 128, 64), (1, 8, 129, 128), (1, 24, 300, 64),
                                  (1, 16, 257, 128), (2, 12, 1000, 64), (1, 2, 2049, 128), (1, 1, 4095, 64), (1, 1, 4100, 64)])
def test_causal_attention_keys_shared_by_wave_groups(hexmi, case, dtype):
    Z, H, S, D = case
    q, k, v = _qkv(Z, H, S, D, dtype, seed=63)
    scores = (q.float() @ k.float().transpose(2, 3) / math.sqrt(D)).masked_fill(torch.ones(S, S).triu(1).bool(), float("-inf"))
    want = torch.softmax(scores, dim=-1) @ v.float()
    got = hexmi.flash_attention(q.cuda(), k.cuda(), v.cuda(), None, True, out_dtype=torch.float32).cpu()
    assert (got - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


# one query of each of many heads (flash_decode.hip): the shortest key range, tiles of 32 (heads of 128) and 64 keys and
# their edges, waves left without a tile, a second tile of some waves
DECODE_CASES = [(130, 65, 64), (129, 66, 128), (131, 95, 128), (130, 128, 64), (129, 255, 128), (300, 257, 128),
                (130, 511, 64), (129, 2051, 128), (513, 577, 64)]


@pytest.mark.parametrize("with_mask", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", DECODE_CASES)
def test_attention_one_query_of_many_heads(hexmi, case, dtype, with_mask):
    # everything is summed in fp32 and the output is fp32: a score is off by about D * 2^-24 * |score| < 5e-5, so is a
    # probability by that share, and the result by no more of |V| < 6 (the errors average): 1e-4. Mask rows start one
    # element off the allocation; a head with every key masked out gives NaN
    B, Skv, D = case
    g = _gen(65)
    q = torch.randn(B, 1, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    scores = (q.float() @ k.float().transpose(1, 2)) / math.sqrt(D)
    shifted = None
    if with_mask:
        mask = _mask(B, 1, Skv, dtype, 66)
        mask[1, :, :Skv - 1] = float("-inf")
        mask[1, :, Skv - 1] = 0.0
        mask[2, :, Skv // 2:] = float("-inf")
        mask[B - 1] = float("-inf")
        scores = scores + mask.float()
        shifted = torch.empty(mask.numel() + 1, dtype=dtype, device="cuda")[1:].view(B, 1, Skv)
        shifted.copy_(mask)
    want = torch.softmax(scores, dim=-1) @ v.float()
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), shifted, out_dtype=torch.float32).cpu()
    if with_mask:
        assert torch.isnan(got[B - 1]).all()
        got, want = got[:B - 1], want[:B - 1]
    assert (got - want).abs().max() <= 1e-4


def test_attention_workspace(hexmi):
    # the size asked for is enough and needed; without one the same problem runs in one launch, to the same rounding;
    # rows with every key masked out stay NaN through the merge
    from hexmi import _lib
    lib = _lib.lib()
    B, Sq, Skv, D = 4, 1, 4096, 128
    g = _gen(64)
    q, k, v = (torch.randn(B, n, D, generator=g).half().cuda() for n in (Sq, Skv, Skv))
    mask = torch.zeros(B, Sq, Skv, dtype=torch.float16, device="cuda")
    mask[:, :, :2000] = float("-inf")
    mask[2] = float("-inf")
    need = lib.hexmi_attention_workspace(B, Sq, Skv, D, 1, _lib.F16)
    assert need > 0 and lib.hexmi_attention_workspace(4096, 2048, 2048, 128, 1, _lib.F16) == 0
    assert lib.hexmi_attention_workspace(1, 1, _lib.ATTENTION_ONE_LAUNCH_KEYS, 128, 1, _lib.F16) == 0
    assert lib.hexmi_attention_workspace(B, Sq, Skv, D, 1, _lib.F32) == 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    outs = [torch.zeros(B, Sq, D, dtype=torch.float16, device="cuda") for _ in range(2)]

    def call(out, workspace, size):
        return lib.hexmi_attention_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), mask.data_ptr(), out.data_ptr(), B, Sq, Skv,
                                      D, D ** -0.5, _lib.F16, _lib.F16, workspace, size, None)
    torch.cuda.synchronize()
    assert call(outs[0], ws.data_ptr(), need - 1) == _lib.EINVAL
    assert call(outs[0], ws.data_ptr(), need) == _lib.OK
    assert call(outs[1], None, 0) == _lib.OK
    torch.cuda.synchronize()
    assert torch.isnan(outs[0][2]).all() and torch.isnan(outs[1][2]).all()
    keep = [0, 1, 3]
    assert (outs[0][keep].float() - outs[1][keep].float()).abs().max() <= 1e-3


# one case for each kernel that takes a mask, at key counts with and without whole runs of four: the key-group kernel (one
# workgroup's keys, padded heads, keys cut into chunks), the decode kernel, and, from 360 units of 64 queries on, the
# 128-query kernel (mask staged through LDS, read in runs, padded heads)
FINITE_MASK_CASES = [(2, 40, 256, 128), (2, 40, 255, 128), (3, 70, 60, 64), (2, 33, 130, 80), (4, 3, 4096, 128), (4, 3, 4095, 64),
                     (130, 1, 300, 128), (130, 1, 301, 64), (90, 200, 72, 128), (90, 200, 72, 64), (90, 200, 76, 128),
                     (90, 200, 76, 80), (90, 200, 75, 128), (90, 200, 75, 64)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", FINITE_MASK_CASES)
def test_masked_attention_rows_of_one_large_finite_value(hexmi, case, dtype):
    # a row whose keys all carry the same value: the value drowns the scores in fp32 and the result is the average of V
    # (torch's own fp32 softmax gives it), whatever the value; beside ordinary keys such a value is no weight at all.
    # fp16's lowest leaves the scores a spacing of 2^-8, which a probability may be off by, and the result by that share
    # of an average of |V| (below 1): 1e-2 covers it with the 16-bit rounding of the probabilities (5e-3)
    B, Sq, Skv, D = case
    g = _gen(71)
    q = torch.randn(B, Sq, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    values = [-65504.0, -3e4] if dtype == torch.float16 else [-1e38, -1e30, -2e9, torch.finfo(dtype).min, 1e30]
    mask = _mask(B, Sq, Skv, dtype, 72)
    rows = mask.view(B * Sq, Skv)
    for i, value in enumerate(values):
        rows[i] = value                                                  # the whole row
        rows[-1 - i, Skv // 3:] = value                                  # all but a few keys
    if dtype == torch.bfloat16:
        rows[-1 - values.index(1e30), :] = 1e30
    scores = q.float() @ k.float().transpose(1, 2) / math.sqrt(D) + mask.float()
    want = torch.softmax(scores, dim=-1) @ v.float()
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), mask.cuda(), out_dtype=torch.float32).cpu()
    assert torch.isfinite(got).all()
    assert (got - want).abs().max() <= (1e-2 if dtype == torch.float16 else 3e-2)


# masks that are not whole aligned runs of four keys: few keys, one step and its edges, key chunks, far more units than
# compute units, padded heads; the last two have whole runs in a mask that starts one element off its allocation
ANY_MASK_CASES = [(2, 5, 1, 64), (1, 33, 3, 128), (3, 129, 63, 64), (2, 130, 65, 128), (2, 64, 127, 80), (3, 2, 4095, 128),
                  (90, 200, 75, 128), (150, 200, 129, 64), (90, 200, 76, 24), (3, 70, 512, 128)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", ANY_MASK_CASES)
def test_masked_attention_any_mask_in_fp32(hexmi, case, dtype):
    # these masks keep fp32 probabilities (in 16-bit parts on the matrix cores). A raw score adds up D <= 128 products
    # whose partial sums stay below about 60: 128 roundings of 60 * 2^-24 at random signs are 4e-5, scaled by 1/sqrt(D)
    # 4e-6; the exponent adds its own 2^-23 * |t| < 3e-6. A probability is off by that share, the result by no more of an
    # average of |V|: 2e-5. (16-bit probabilities alone are off by up to 5e-4 and 4e-3.)
    B, Sq, Skv, D = case
    g = _gen(73)
    q = torch.randn(B, Sq, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    mask = _mask(B, Sq, Skv, dtype, 74)
    shifted = torch.empty(mask.numel() + 1, dtype=dtype, device="cuda")[1:].view(B, Sq, Skv)
    shifted.copy_(mask)
    scores = q.double() @ k.double().transpose(1, 2) / math.sqrt(D) + mask.double()
    want = torch.softmax(scores, dim=-1) @ v.double()
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), shifted, out_dtype=torch.float32).cpu()
    assert (got.double() - want).abs().max() <= 2e-5


@pytest.mark.parametrize("with_mask", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [(2, 40, 65, 128), (3, 20, 79, 64), (2, 33, 130, 80), (2, 1, 4095, 128), (130, 1, 301, 64),
                                  (130, 1, 70, 128)])
def test_attention_infinities_in_the_last_row_of_v(hexmi, case, dtype, with_mask):
    # odd columns of the last key are +inf or -inf: they come out infinite or NaN (a tile repeats the last row past the end
    # at weight 0, and probabilities in parts have negative ones), the even columns as without them; and a head's
    # NaN stays in that head. Bound: the parity tests'
    B, Sq, Skv, D = case
    g = _gen(75)
    q = torch.randn(B, Sq, D, generator=g).to(dtype)
    k, v = torch.randn(B, Skv, D, generator=g).to(dtype), torch.randn(B, Skv, D, generator=g).to(dtype)
    v[:, -1, 1::4] = float("inf")
    v[:, -1, 3::4] = -float("inf")
    k[1, 0], v[1, 0] = float("nan"), float("nan")
    mask = torch.randn(B, Sq, Skv, generator=g).to(dtype) if with_mask else None
    got = hexmi.attention(q.cuda(), k.cuda(), v.cuda(), None if mask is None else mask.cuda(), out_dtype=torch.float32).cpu()
    assert torch.isnan(got[1]).all()
    heads = [h for h in range(B) if h != 1]
    got = got[heads]
    assert not torch.isfinite(got[:, :, 1::2]).any()
    scores = q.float() @ k.float().transpose(1, 2) / math.sqrt(D) + (0.0 if mask is None else mask.float())
    want = torch.softmax(scores[heads], dim=-1) @ v[heads][:, :, ::2].float()
    assert (got[:, :, ::2] - want).abs().max() <= (5e-3 if dtype == torch.float16 else 3e-2)


@pytest.mark.parametrize("with_mask", [False, True])
def test_attention_more_heads_than_a_grid_of_512_threads_holds(hexmi, with_mask):
    # 2^23 workgroups of 512 threads are more than a launch takes: the persistent kernel (without a mask) and the row-wise
    # one (with this one, rows of 65 keys) do. K is V here; four heads against the fp32 sums, bound as in the parity tests
    B, Skv, D = (1 << 23) + 3, 65, 8
    g = torch.Generator(device="cuda").manual_seed(77)
    q = torch.randn(B, 1, D, generator=g, device="cuda", dtype=torch.float16)
    k = torch.randn(B, Skv, D, generator=g, device="cuda", dtype=torch.float16)
    mask = torch.randn(B, 1, Skv, generator=g, device="cuda", dtype=torch.float16) if with_mask else None
    out = torch.full_like(q, float("nan"))
    hexmi.attention(q, k, k, mask, out=out)
    assert torch.isfinite(out).all()
    pick = [0, 1, 1 << 22, B - 1]
    scores = q[pick].float() @ k[pick].float().transpose(1, 2).contiguous() / math.sqrt(D)
    if with_mask:
        scores = scores + mask[pick].float()
    want = torch.softmax(scores, dim=-1) @ k[pick].float()
    assert (out[pick].float() - want).abs().max() <= 2e-2


@pytest.mark.parametrize("case", [(9, 130, 300, 64, False), (11, 3, 4000, 128, False), (63, 300, 520, 64, False), (1, 700, 700, 64, True),
                                  (9, 260, 260, 128, True), (35, 800, 800, 64, True), (16, 200, 200, 128, True)])
def test_attention_head_counts_off_the_multiple_of_eight(hexmi, case):
    # units are dealt to the 8 XCDs in parts of the list of all of them (causal: the last ZH % 8 heads apart): each must be
    # visited exactly once, so the output starts as NaN. Bound: the parity tests'
    B, Sq, Skv, D, causal = case
    g = _gen(79)
    q, k, v = (torch.randn(B, n, D, generator=g).half() for n in (Sq, Skv, Skv))
    out = torch.full((B, Sq, D), float("nan"), dtype=torch.float32, device="cuda")
    if causal:
        hexmi.flash_attention(q[None].cuda(), k[None].cuda(), v[None].cuda(), None, True, out=out[None])
    else:
        hexmi.attention(q.cuda(), k.cuda(), v.cuda(), out=out)
    scores = q.float() @ k.float().transpose(1, 2) / math.sqrt(D)
    if causal:
        scores = scores.masked_fill(torch.ones(Sq, Skv).triu(1).bool(), float("-inf"))
    want = torch.softmax(scores, dim=-1) @ v.float()
    assert (out.cpu() - want).abs().max() <= 5e-3


def _standing(form, Z, H, S, D, dtype, g):
    """q, k, v of one shape that are not contiguous, as programs have them."""
    def r(*shape):
        return torch.randn(*shape, generator=g).to(dtype).cuda()
    if form == "slices":                                     # one projection [Z, S, 3 H D]
        return tuple(t.view(Z, S, H, D).transpose(1, 2) for t in r(Z, S, 3 * H * D).split(H * D, dim=-1))
    if form == "rows first":                                 # q [Z, S, H, D], k [S, Z, H, D], v contiguous
        return r(Z, S, H, D).transpose(1, 2), r(S, Z, H, D).permute(1, 2, 0, 3), r(Z, H, S, D)
    if form == "expanded":                                   # one key and value head for all, batches apart
        return r(H, Z, S, D).transpose(0, 1), r(Z, 1, S, D).expand(Z, H, S, D), r(Z, S, 1, D).transpose(1, 2).expand(Z, H, S, D)
    if form == "padded rows":
        return tuple(r(Z, H, S, D + 8)[..., :D] for _ in range(3))
    if form == "odd rows":                                   # rows off the 16-byte boundaries
        return tuple(r(Z, H, S, D + 3)[..., :D] for _ in range(3))
    if form == "off base":
        return tuple(r(Z, H, S, D + 8)[..., 1:D + 1] for _ in range(3))
    return tuple(r(Z, H, D, S).transpose(2, 3) for _ in range(3))        # "columns apart"


# the key-group and the persistent kernels (128 and 256 queries a workgroup), padded and two-half heads, one query; the last
# three forms, one query of many heads, a zero scale and fp32 are copied first
@pytest.mark.parametrize("form", ["slices", "rows first", "expanded", "padded rows", "odd rows", "off base", "columns apart"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("case", [(2, 3, 200, 64, torch.bfloat16), (2, 4, 129, 128, torch.float16), (3, 40, 300, 64, torch.float16),
                                  (2, 70, 130, 128, torch.bfloat16), (1, 64, 2100, 64, torch.float16), (2, 32, 1100, 128, torch.float16),
                                  (2, 16, 2049, 128, torch.bfloat16), (2, 5, 100, 80, torch.float16), (2, 24, 515, 40, torch.bfloat16),
                                  (1, 3, 70, 256, torch.float16), (2, 3, 1, 64, torch.float16), (2, 300, 1, 128, torch.float16),
                                  (1, 2, 65, 64, torch.float32)])
def test_attention_of_heads_where_they_stand(hexmi, form, causal, case):
    Z, H, S, D, dtype = case
    q, k, v = _standing(form, Z, H, S, D, dtype, _gen(S + D + H))
    want = hexmi.flash_attention(q.contiguous(), k.contiguous(), v.contiguous(), 0.11, causal)
    got = hexmi.flash_attention(q, k, v, 0.11, causal)
    assert got.is_contiguous() and torch.equal(got, want)
    out = torch.full_like(want, float("nan"))
    assert hexmi.flash_attention(q, k, v, 0.11, causal, out=out) is out and torch.equal(out, want)
    if S == 200:
        zero = hexmi.flash_attention(q, k, v, 0.0, causal)
        assert torch.equal(zero, hexmi.flash_attention(q.contiguous(), k.contiguous(), v.contiguous(), 0.0, causal))


def test_attention_of_heads_where_they_stand_into_their_own_memory(hexmi):
    # out lies in the storage of the operands: they are copied before anything is written
    g = _gen(5)
    Z, H, S, D = 1, 4, 300, 64
    buf = torch.randn(4, Z * H * S * D, generator=g).half().cuda()
    q, k, v = (buf[i].view(Z, S, H, D).transpose(1, 2) for i in range(3))
    want = hexmi.flash_attention(q.contiguous(), k.contiguous(), v.contiguous(), 0.125, True)
    keep = buf.clone()
    for i in range(4):                                       # of q, k, v and of none of them
        for alias in (buf[i], torch.from_dlpack(buf[i]), torch.from_dlpack(buf.view(-1)[i * Z * H * S * D - (i > 0) * 64:][:Z * H * S * D])):
            got = hexmi.flash_attention(q, k, v, 0.125, True, out=alias.view(Z, H, S, D))
            assert torch.equal(got, want) and got.data_ptr() == alias.data_ptr()
            buf.copy_(keep)
    assert hexmi.ops._overlaps(buf[1], k) and not hexmi.ops._overlaps(buf[3], q, k, v)
    assert hexmi.ops._overlaps(torch.from_dlpack(buf[2])[-1:], v) and not hexmi.ops._overlaps(buf[0], k, v)


def test_strided_entry_refuses_what_it_cannot_read(hexmi):
    import ctypes
    from hexmi import _lib
    lib = _lib.lib()
    x = torch.zeros(1, 2, 64, 64, dtype=torch.float16, device="cuda")
    out = torch.full_like(x, 7.0)
    s = torch.cuda.current_stream().cuda_stream

    def call(strides, dtype=_lib.F16, scale=0.1, S=64):
        a = (ctypes.c_int64 * 9)(*strides)
        p = x.data_ptr()
        return lib.hexmi_flash_attn_fwd_strided(p, p, p, out.data_ptr(), 1, 2, S, 64, a, scale, 0, dtype, dtype, s)
    good = [8192, 4096, 64] * 3
    assert call([8192, 4096, 60] + good[3:]) == _lib.ENOTSUP
    assert call(good[:3] + [8192, 4092, 64] + good[6:]) == _lib.ENOTSUP
    assert call(good[:6] + [8192, 4096, -64]) == _lib.ENOTSUP
    assert call(good[:3] + [8192, 4096, 1 << 28] + good[6:]) == _lib.ENOTSUP
    assert call(good, _lib.F32) == _lib.ENOTSUP
    assert call(good, scale=0.0) == _lib.ENOTSUP
    p = x.data_ptr()
    assert lib.hexmi_flash_attn_fwd_strided(p, p, p, p, 1, 2, 64, 64, None, 0.1, 0, _lib.F16, _lib.F16, s) == _lib.EINVAL
    assert lib.hexmi_flash_attn_fwd_strided(None, None, None, None, 1, 0, 64, 64, None, 0.1, 0, _lib.F16, _lib.F16, s) == _lib.OK
    torch.cuda.synchronize()
    assert (out == 7.0).all()
    assert call([3, 4096, 64] * 3) == _lib.OK                # a single batch has no stride
