"""GPU parity of the dense GEMM against the CPU oracle, through the C ABI.

Tolerances. The kernel accumulates in fp32 on the matrix cores; the oracle accumulates in double.
  fp32 output: |got - want| <= 1e-5 * sum_k |a_ik b_kj| (rel-err 1e-5 of the magnitude actually summed; the
    plain rel-err of max|C| is reported by the config-size test and must be <= 1e-5 as well);
  fp16 / bf16 output: within one unit in the last place of the oracle's rounded value, or within 1e-5 of the
    summed magnitude where the value is a cancellation residue. (A flat 2e-2 max-abs is
    also asserted after scaling by 1/sqrt(K), the scale attention-sized outputs have; at |c| ~ 100 one fp16 ulp
    is 0.06, so the raw bound cannot hold for any implementation.)
"""
import math

import numpy as np
import pytest
import torch

from util import close16, from_np, rel_err, to_np

pytestmark = pytest.mark.gpu


def _gen(seed):
    return torch.Generator().manual_seed(seed)


def _inputs(M, N, K, dtype, trans_b, seed=0):
    g = _gen(seed)
    a = (2 * torch.rand(M, K, generator=g) - 1).to(dtype)
    b = (2 * torch.rand(*((N, K) if trans_b else (K, N)), generator=g) - 1).to(dtype)
    return a, b


def _oracle_mm(oracle, a, b, out_dtype, trans_b):
    an, tag = to_np(a)
    bn, _ = to_np(b)
    if out_dtype == torch.float32:
        return torch.from_numpy(oracle.matmul(an, bn, out_dtype=np.float32, trans_b=trans_b, dtype=tag))
    od = "bf16" if out_dtype == torch.bfloat16 else np.float16
    return from_np(oracle.matmul(an, bn, out_dtype=od, trans_b=trans_b, dtype=tag), out_dtype)


SHAPES = [
    (1024, 512, 64),      # test_matmul.py:26-28
    (256, 256, 64), (512, 768, 128), (256, 512, 192),
    (100, 72, 64), (300, 264, 128),          # ragged M / N on the tiled path
    (256, 256, 96), (300, 264, 160),         # K % 64 == 32: the four-stage 32-wide-slab kernel
    (384, 256, 320),                         # odd number of 64-wide slabs
    (33, 17, 40), (1, 8, 8), (65, 130, 24), (7, 5, 3),   # any-shape kernel (and, [N,K] weights, the ragged-K one)
    (300, 264, 1000), (130, 136, 72),        # K % 8 == 0 only: the 32-wide-slab kernel with a masked last slab
    (200, 257, 96), (260, 1003, 72),         # ... with an odd N: rows leave through LDS ([N,K]); any-shape ([K,N])
    (300, 1001, 256), (129, 70, 64),         # odd N, whole 64-wide slabs: the paired-slab kernel, element stores
    (130, 136, 2049), (257, 129, 333),       # K % 8 != 0: unaligned rows, the any-shape kernel
]


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
def test_gemm_parity(hexmi, oracle, shape, dtype, trans_b):
    M, N, K = shape
    a, b = _inputs(M, N, K, dtype, trans_b)
    got32 = hexmi.matmul(a.cuda(), b.cuda(), out_dtype=torch.float32, trans_b=trans_b).cpu()
    want32 = _oracle_mm(oracle, a, b, torch.float32, trans_b)
    bb = b.float().t() if trans_b else b.float()
    mag = a.float().abs() @ bb.abs()
    assert ((got32 - want32).abs() <= 1e-5 * mag + 1e-30).all()
    got = hexmi.matmul(a.cuda(), b.cuda(), trans_b=trans_b).cpu()
    want = _oracle_mm(oracle, a, b, dtype, trans_b)
    # values that are cancellation residues (|c| << sum |a b|) carry the fp32 rounding of the larger partial sums
    assert got.dtype == dtype and close16(got, want, max_ulp=1, atol=1e-5 * float(mag.max()))
    assert ((got.float() - want.float()).abs().max() / math.sqrt(K)) <= 2e-2


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 12, 13, 16, 17, 32, 33, 48, 64])
@pytest.mark.parametrize("N,K", [(64, 8), (100, 64), (4096, 2048), (1000, 2056), (257, 4096), (130, 11008)])
def test_gemm_few_rows_against_transposed_weights(hexmi, oracle, dtype, M, N, K):
    # up to 64 rows with B as [N,K]: a wave per output channel up to four rows, a workgroup per 16 channels or the tiles of
    # gemm_few.hip beyond, with and without the epilogue operands, 16-bit and fp32 results
    a, b = _inputs(M, N, K, dtype, True, seed=M + N)
    got32 = hexmi.matmul(a.cuda(), b.cuda(), out_dtype=torch.float32, trans_b=True).cpu()
    want32 = _oracle_mm(oracle, a, b, torch.float32, True)
    mag = a.float().abs() @ b.float().t().abs()
    assert ((got32 - want32).abs() <= 1e-5 * mag + 1e-30).all()
    got = hexmi.matmul(a.cuda(), b.cuda(), trans_b=True).cpu()
    want = _oracle_mm(oracle, a, b, dtype, True)
    assert got.dtype == dtype and close16(got, want, max_ulp=1, atol=1e-5 * float(mag.max()))
    g = _gen(K)
    bias, resid = torch.randn(N, generator=g).to(dtype), torch.randn(M, N, generator=g).to(dtype)
    fused = hexmi.matmul(a.cuda(), b.cuda(), trans_b=True, bias=bias.cuda(), residual=resid.cuda()).cpu()
    ref = (want32.double() + bias.double() + resid.double()).to(dtype)
    assert close16(fused, ref, max_ulp=1, atol=2e-5 * float(mag.max()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [
    (9, 50257, 96), (16, 33001, 1120),              # 16 rows: 32 channels a workgroup
    (17, 5121, 544), (32, 11001, 4128),             # 32 rows: 32 and 64 channels, the larger weights read non-temporally
    (33, 5121, 2080), (64, 11007, 2048), (40, 8200, 32), (64, 77, 480)])     # 64 rows; fewer rounds of K than waves
def test_gemm_few_rows_wide_workgroups(hexmi, dtype, M, N, K):
    a, b = _inputs(M, N, K, dtype, True, seed=M + K)
    want, mag = a.double() @ b.double().t(), a.double().abs() @ b.double().t().abs()
    got = hexmi.matmul(a.cuda(), b.cuda(), out_dtype=torch.float32, trans_b=True).cpu()
    # fp32 products summed in parts: K roundings of at most 2^-24 of the magnitude, far fewer in effect
    assert ((got.double() - want).abs() <= 1e-5 * mag + 1e-30).all()
    g = _gen(K)
    bias, resid = torch.randn(N, generator=g).to(dtype), torch.randn(M, N, generator=g).to(dtype)
    fused = hexmi.matmul(a.cuda(), b.cuda(), trans_b=True, bias=bias.cuda(), residual=resid.cuda()).cpu()
    assert close16(fused, (want + bias.double() + resid.double()).to(dtype), max_ulp=1, atol=2e-5 * float(mag.max()))


# every (channels, waves) that plan_gemm_skinny picks on 256 CUs, at widths off the workgroup's, with K of a few rounds of 64,
# fewer rounds than waves, and the last 32 of K on its own: 16x2, 16x8, 32x4 (16 rows); 16x2, 16x8, 32x2, 32x4 (32
# rows); 16x4, 16x2, 32x2, 64x4 and the tiles (64 rows) -- where plan_gemm_few leaves the product to it
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(5, 401, 160), (16, 8195, 480), (16, 401, 736), (3, 33001, 800), (12, 16501, 3104),
                                   (17, 10003, 96), (32, 8999, 992), (25, 77, 1056), (32, 14007, 544), (20, 5003, 800),
                                   (31, 14005, 4128), (32, 33003, 800),
                                   (33, 100, 480), (64, 333, 1056), (47, 9001, 160), (64, 17003, 224), (50, 7001, 544),
                                   (64, 12005, 544), (64, 20500, 96), (33, 20501, 800)])
def test_gemm_few_rows_every_workgroup_shape(hexmi, dtype, M, N, K):
    a, b = _inputs(M, N, K, dtype, True, seed=M + N)
    want, mag = a.double() @ b.double().t(), a.double().abs() @ b.double().t().abs()
    out = torch.full((M + 1, N), float("nan"), dtype=torch.float32, device="cuda")
    hexmi.matmul(a.cuda(), b.cuda(), out=out[:M], trans_b=True)
    got = out.cpu()
    # fp32 products summed in parts: K roundings of at most 2^-24 of the magnitude, far fewer in effect
    assert ((got[:M].double() - want).abs() <= 1e-5 * mag + 1e-30).all()
    assert torch.isnan(got[M]).all()
    # with a residual the widths here, off whole runs of four columns, keep the widest products from the tiles
    resid = torch.randn(M, N, generator=_gen(K)).to(dtype)
    fused = hexmi.matmul(a.cuda(), b.cuda(), trans_b=True, residual=resid.cuda()).cpu()
    assert close16(fused, (want + resid.double()).to(dtype), max_ulp=1, atol=2e-5 * float(mag.max()))


# both sides of the lines of plan_gemm_few on 256 CUs: three and four rows on tiles and, where the weights are large or the tiles few,
# by dot products; five to eight rows by dot products of sixteen waves where there are more tiles than CUs; half a tile of 32 x 64 and
# two of 16 x 32 where K keeps the weight stream from the call or does not
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(3, 4094, 3080), (4, 5200, 2424), (3, 16380, 1032), (3, 4099, 3104), (4, 9001, 1408), (4, 6151, 8192),
                                   (5, 16401, 2056), (8, 50257, 2048), (6, 17001, 2112), (7, 20011, 2048), (16, 9001, 1408), (9, 16380, 1032),
                                   (4, 16384, 1984), (4, 16392, 1984), (3, 20001, 2048), (20, 3001, 2816), (20, 3001, 2808), (25, 3001, 2816), (24, 4090, 8256),
                                   (11, 2030, 6400), (30, 4090, 12352), (16, 16401, 544), (24, 20001, 288), (25, 20001, 288)])
def test_gemm_few_rows_at_the_lines_between_kernels(hexmi, dtype, M, N, K):
    for out_dtype in (dtype, torch.float32):
        _against_double(hexmi, dtype, out_dtype, True, M, N, K, False, False, M + N)
        _against_double(hexmi, dtype, out_dtype, True, M, N, K, True, True, M + K)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(64, 8), (104, 64), (4096, 2048), (1000, 2056), (256, 4096), (136, 11008)])
def test_gemm_few_rows_against_row_major_weights(hexmi, oracle, dtype, M, N, K):
    # a few rows with B as [K,N] (these run on the tiles: a kernel that streams B in 64-byte pieces measured slower)
    a, b = _inputs(M, N, K, dtype, False, seed=M + N)
    got32 = hexmi.matmul(a.cuda(), b.cuda(), out_dtype=torch.float32).cpu()
    want32 = _oracle_mm(oracle, a, b, torch.float32, False)
    mag = a.float().abs() @ b.float().abs()
    assert ((got32 - want32).abs() <= 1e-5 * mag + 1e-30).all()
    got = hexmi.matmul(a.cuda(), b.cuda()).cpu()
    want = _oracle_mm(oracle, a, b, dtype, False)
    assert got.dtype == dtype and close16(got, want, max_ulp=1, atol=1e-5 * float(mag.max()))
    g = _gen(K)
    bias, resid = torch.randn(N, generator=g).to(dtype), torch.randn(M, N, generator=g).to(dtype)
    fused = hexmi.matmul(a.cuda(), b.cuda(), bias=bias.cuda(), residual=resid.cuda()).cpu()
    ref = (want32.double() + bias.double() + resid.double()).to(dtype)
    assert close16(fused, ref, max_ulp=1, atol=2e-5 * float(mag.max()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("K", [64, 128, 192, 448])
def test_gemm_two_small_tiles_per_cu(hexmi, dtype, trans_b, K):
    # 16 x 17 tiles of 128 x 128, more than there are CUs: one slab, whole and guarded last passes; rows of the output on
    # and (B as [N,K]) off the boundaries; the epilogue operands; fp32 results
    M = 2040
    for N in ((2104, 2101) if trans_b else (2104,)):
        a, b = _inputs(M, N, K, dtype, trans_b, seed=K + N)
        ad, bd = a.cuda(), b.cuda()
        bt = b.double().t() if trans_b else b.double()
        want, mag = a.double() @ bt, float((a.double().abs() @ bt.abs()).max())
        got32 = hexmi.matmul(ad, bd, out_dtype=torch.float32, trans_b=trans_b).cpu()
        assert ((got32.double() - want).abs().max()) <= 1e-5 * mag
        assert close16(hexmi.matmul(ad, bd, trans_b=trans_b).cpu(), want.to(dtype), max_ulp=1, atol=1e-5 * mag)
        g = _gen(K)
        bias, resid = torch.randn(N, generator=g).to(dtype), torch.randn(M, N, generator=g).to(dtype)
        fused = hexmi.matmul(ad, bd, trans_b=trans_b, bias=bias.cuda(), residual=resid.cuda()).cpu()
        assert close16(fused, (want + bias.double() + resid.double()).to(dtype), max_ulp=1, atol=2e-5 * mag)


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("K", [1472, 1536, 1600])
def test_gemm_tiles_left_over_after_a_round_of_two_per_cu(hexmi, trans_b, K):
    # 8 x 70 tiles of 128 x 128 with epilogue operands: two stages below K = 1536, four from there on
    M, N, dtype = 1000, 8896, torch.float16
    a, b = _inputs(M, N, K, dtype, trans_b, seed=K)
    bt = b.double().t() if trans_b else b.double()
    g = _gen(K)
    bias = torch.randn(N, generator=g).to(dtype)
    want, mag = a.double() @ bt + bias.double(), float((a.double().abs() @ bt.abs()).max())
    got = hexmi.matmul(a.cuda(), b.cuda(), trans_b=trans_b, bias=bias.cuda()).cpu()
    assert close16(got, want.to(dtype), max_ulp=1, atol=2e-5 * mag)


def _against_double(hexmi, dtype, out_dtype, trans_b, M, N, K, bias, residual, seed, out=None):
    g = _gen(seed)
    a, b = _inputs(M, N, K, dtype, trans_b, seed=seed)
    bi = torch.randn(N, generator=g).to(out_dtype) if bias else None
    r = torch.randn(M, N, generator=g).to(out_dtype) if residual else None
    ref = a.cuda().double() @ (b.cuda().double().t() if trans_b else b.cuda().double())
    mag = a.cuda().double().abs() @ (b.cuda().double().abs().t() if trans_b else b.cuda().double().abs())
    for t in (bi, r):
        if t is not None:
            ref, mag = ref + t.cuda().double(), mag + t.cuda().double().abs()
    got = hexmi.matmul(a.cuda(), b.cuda(), trans_b=trans_b, bias=None if bi is None else bi.cuda(),
                       residual=None if r is None else r.cuda(), out_dtype=out_dtype, out=out)
    # sums in fp32 in another order: 1e-5 of the summed magnitudes; one rounding to the output type: half an ulp
    eps = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[out_dtype]
    assert ((got.double() - ref).abs() <= 1e-5 * mag + eps * ref.abs() + 1e-7).all(), (M, N, K)


# every tile of plan_gemm_few on 256 CUs: its edges (one row or column over, one short), slabs of K that are whole, short or
# one chunk over, fewer slabs than stages and more; outputs that leave in runs of eight and that do not
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                             (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("M,N,K", [
    (64, 1024, 256), (33, 40, 2056), (49, 16, 136), (64, 24, 1280),      # 16 x 16 ([N,K]), 16 x 32
    (33, 4104, 2048), (65, 4072, 264), (500, 500 // 8 * 8, 1288),        # 16 x 32 and 32 x 32 and their edges
    (17, 16328, 520), (129, 4096, 776), (500, 1016, 896),                # 32 x 64
    (1000, 1024, 136), (1025, 960, 640), (257, 3264, 72),                # 64 x 64
    (1921, 1024, 392), (2000, 768, 1032), (129, 8128, 8), (2048, 1024, 128),     # 128 x 64; the last of a round
    (1345, 1536, 264), (1343, 1544, 520), (70, 17752, 72), (193, 8056, 136),     # 96 x 96
    (640, 3456, 128), (640, 3456, 192), (640, 3456, 256), (640, 3456, 320), (544, 3484, 512), (544, 3484, 576),      # ... and not
    (130, 4096, 1784), (130, 4096, 1792), (130, 4096, 2040), (130, 4096, 2048), (129, 8192, 1032), (282, 5248, 1600),   # 128 x 64 half empty
    (1985, 760, 136), (1983, 776, 520), (65, 12296, 264), (2017, 672, 1288),     # 64 x 96, 96 x 64
    (2305, 264, 1032), (47, 8200, 1160), (145, 2008, 2056), (95, 4088, 1024),    # 48 x 32
    (113, 304, 1000), (197, 408, 264), (511, 256, 72), (65, 1592, 2056)])        # sixteen rows a tile, many rows
def test_gemm_one_round_of_tiles(hexmi, dtype, out_dtype, trans_b, M, N, K):
    _against_double(hexmi, dtype, out_dtype, trans_b, M, N, K, True, True, M + N + K)
    _against_double(hexmi, dtype, out_dtype, trans_b, M, N, K, False, False, M + N + K + 1)
    if trans_b:                                                          # rows of the output off the boundaries
        _against_double(hexmi, dtype, out_dtype, True, M, N + 1, K, True, True, M + N + K + 2)
    # a strided output one element off, the residual the output itself, nothing written around it
    g = _gen(3)
    a, b = _inputs(M, N, K, dtype, trans_b, seed=5)
    a, b = a.cuda(), b.cuda()
    from hexmi import _lib
    code = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16, torch.float32: _lib.F32}
    for ldc, off in ((N + 8, 0), (N + 3, 1)):
        c = torch.randn(M * ldc + 16, generator=g).to(out_dtype).cuda()
        view = c[off:off + M * ldc].view(M, ldc)
        want = a.double() @ (b.double().t() if trans_b else b.double()) + view[:, :N].double()
        keep = view[:, N:].clone()
        s = torch.cuda.current_stream().cuda_stream
        assert _lib.lib().hexmi_gemm_ex(M, N, K, a.data_ptr(), K, b.data_ptr(), b.stride(0), view.data_ptr(), ldc, None,
                                        view.data_ptr(), ldc, code[dtype], code[out_dtype], int(trans_b), s) == _lib.OK
        eps = torch.finfo(out_dtype).eps
        assert ((view[:, :N].double() - want).abs() <= eps * want.abs() + 2e-5 * K).all()
        assert torch.equal(view[:, N:], keep)


# parts of K through a workspace (plan_gemm_parts on 256 CUs): each tile, three parts and many, a short last part, K off whole slabs, a
# column run and a row over and short of a tile; beside them shapes that go as a whole. Without a workspace every shape does.
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                             (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("M,N,K,trans_b,parts", [
    (1, 8, 4608, False, True), (16, 1024, 4104, False, True), (3, 1000, 11376, False, True),                        # 16 x 64
    (1, 8, 3072, False, False),                                     # (in parts before: 1 x 16 x 3088 7.0 us, as a whole 5.9)
    (1, 1032, 4096, False, True), (16, 4096, 4096, False, True), (15, 8200, 9000, False, True),                     # 16 x 128
    (17, 72, 3080, False, True), (32, 2048, 11008, False, True), (29, 2560, 5128, False, True),                     # 32 x 64
    (33, 56, 4608, False, True), (113, 304, 11968, False, True), (513, 512, 8192, False, True),                     # 64 x 64
    (17, 2047, 11008, True, True), (64, 4097, 11008, True, True), (255, 1030, 11016, True, True),
    (16, 4104, 4096, False, False), (16, 11008, 11376, False, False), (64, 768, 4096, False, False), (16, 1024, 11008, True, False),
    (64, 4096, 8192, True, False), (32, 4096, 11008, True, False),
    (128, 1032, 9216, True, True), (128, 1032, 9208, True, False), (64, 700, 12800, True, True), (64, 700, 12792, True, False),
    (24, 1000, 9728, True, True), (24, 1000, 9720, True, False), (1536, 96, 9216, True, True), (1537, 96, 9216, True, False),
    (1537, 97, 9216, True, True),                                                                            # the lines of [N,K]
    (16, 32, 4608, False, True), (16, 32, 4600, False, False), (17, 24, 5632, False, True), (17, 24, 5624, False, False),
    (1025, 32, 7168, False, True), (1025, 32, 7160, False, False), (2049, 16, 8192, False, False), (128, 40, 4608, False, True),
    (16, 64, 4096, False, True), (16, 64, 4088, False, False), (129, 40, 5632, False, True), (129, 40, 5624, False, False),
    (16, 1032, 4096, False, True), (16, 1032, 4088, False, False), (16, 1024, 3072, False, True),            # ... of [K,N]
    (8, 1001, 4096, False, True), (16, 4097, 4100, False, True), (1, 3, 3075, False, True), (31, 2049, 5001, False, True),   # rows off the
    (128, 531, 9736, False, True), (64, 1024, 4611, False, True), (64, 2047, 11009, True, False)])                          # boundaries
def test_gemm_parts_of_a_long_k(hexmi, dtype, out_dtype, M, N, K, trans_b, parts):
    from hexmi import _lib
    lib, code = _lib.lib(), {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16, torch.float32: _lib.F32}
    need = lib.hexmi_gemm_workspace(M, N, K, code[dtype], int(trans_b))
    assert (need > 0) == parts
    a, b = _inputs(M, N, K, dtype, trans_b, seed=M + N + K)
    a, b = a.cuda(), b.cuda()
    bias = torch.randn(N, generator=_gen(4)).to(out_dtype).cuda()
    # rows of the output three longer, the residual the output itself, nothing written around it; the scratch starts as garbage
    view = torch.randn(M, N + 3, generator=_gen(3)).to(out_dtype).cuda()
    keep, wide = view.clone(), b.double().t() if trans_b else b.double()
    want = a.double() @ wide + bias.double() + view[:, :N].double()
    mag = a.double().abs() @ wide.abs() + bias.double().abs() + view[:, :N].double().abs()
    ws = torch.full((need + 64,), 0xFF, dtype=torch.uint8, device="cuda")
    s = torch.cuda.current_stream().cuda_stream

    def call(ws_ptr, ws_bytes):
        view.copy_(keep)
        return lib.hexmi_gemm_ws(M, N, K, a.data_ptr(), K, b.data_ptr(), b.stride(0), view.data_ptr(), N + 3, bias.data_ptr(), view.data_ptr(),
                                 N + 3, code[dtype], code[out_dtype], int(trans_b), ws_ptr, ws_bytes, s)
    for ptr, size in ((ws.data_ptr(), need), (None, 0)):
        assert call(ptr, size) == _lib.OK
        # fp32 sums in another order, then one rounding to the output type
        assert ((view[:, :N].double() - want).abs() <= 1e-5 * mag + torch.finfo(out_dtype).eps / 2 * want.abs() + 1e-7).all()
        assert torch.equal(view[:, N:], keep[:, N:])
    assert (ws[need:] == 0xFF).all()
    if parts:
        assert call(ws.data_ptr(), need - 1) == _lib.EINVAL and call(ws.data_ptr() + 4, need) == _lib.EINVAL
        assert torch.equal(view, keep)
    if parts and K % 8 == 0 and (trans_b or N % 8 == 0):
        # a base off the boundaries where the sizes are not: as a whole, and the scratch is not touched
        ab, ws[:] = torch.zeros(M * K + 8, dtype=dtype, device="cuda"), 0xFF
        ab[1:1 + M * K] = a.reshape(-1)
        view.copy_(keep)
        assert lib.hexmi_gemm_ws(M, N, K, ab.data_ptr() + 2, K, b.data_ptr(), b.stride(0), view.data_ptr(), N + 3, bias.data_ptr(),
                                 view.data_ptr(), N + 3, code[dtype], code[out_dtype], int(trans_b), ws.data_ptr(), need, s) == _lib.OK
        assert ((view[:, :N].double() - want).abs() <= 1e-5 * mag + torch.finfo(out_dtype).eps / 2 * want.abs() + 1e-7).all()
        assert (ws == 0xFF).all()
    # the operator gives the same with an output of its own and with one it is handed, and under capture
    if dtype == out_dtype:
        y = hexmi.matmul(a, b, trans_b=trans_b, bias=bias)
        assert torch.equal(y, hexmi.matmul(a, b, trans_b=trans_b, bias=bias, out=torch.empty_like(y)))
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            z = hexmi.matmul(a, b, trans_b=trans_b, bias=bias)
        for _ in range(3):
            z.fill_(7.0)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(z, y)


# the tiles of plan_gemm_mid on 256 CUs: one row and one run of columns over and short of them, K of fewer slabs than stages, of whole slabs
# and chunks over, slabs that the stages do not divide
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,bias,residual", [
    (1025, 4096, 8, False, False), (2049, 1096, 72, False, False), (1153, 4104, 200, True, True), (2047, 4088, 120, False, True),
    (2049, 1096, 1000, True, False),                                              # 128 x 128, two and one to a CU
    (1345, 6216, 1608, False, True), (1291, 3096, 2552, True, False), (2177, 2056, 640, False, False),           # 192 x 128
    (4097, 4104, 1016, False, False), (1300, 6400, 1600, True, False), (1345, 6344, 1600, True, True),           # 192 x 192
    (700, 9000, 1000, False, True), (511, 16376, 1160, True, False),                                          # 256 x 128
    (645, 12456, 704, True, False), (1009, 24000, 328, True, False), (3073, 3080, 128, True, False),           # 256 x 192
    (301, 16392, 64, False, False), (339, 28864, 64, False, False), (192, 12800, 64, False, True), (130, 16120, 128, False, True),
    (384, 30464, 768, False, False), (384, 30464, 832, False, False),                                         # ... and not 192 x 128
    (16, 32776, 264, False, False), (3, 40000, 600, True, True), (17, 32776, 264, False, False), (16, 32776, 256, True, False),    # few rows
    (4088, 4104, 40, False, False), (4089, 4104, 40, True, False), (4088, 4112, 136, True, False), (4088, 4128, 40, False, False),
    (3001, 8200, 64, False, False), (2100, 8008, 200, False, True)])                                          # 32 MiB and more, rows off the lines
def test_gemm_tiles_between_128_and_256(hexmi, dtype, trans_b, M, N, K, bias, residual):
    _against_double(hexmi, dtype, dtype, trans_b, M, N, K, bias, residual, M + N + K)
    # a strided output, the residual the output itself, nothing written around it
    from hexmi import _lib
    a, b = _inputs(M, N, K, dtype, trans_b, seed=5)
    a, b = a.cuda(), b.cuda()
    view = torch.randn(M, N + 8, generator=_gen(3)).to(dtype).cuda()
    want, mag = a.double() @ (b.double().t() if trans_b else b.double()), a.double().abs() @ (b.double().abs().t() if trans_b else b.double().abs())
    if residual:
        want, mag = want + view[:, :N].double(), mag + view[:, :N].double().abs()
    keep = view[:, N:].clone()
    code = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}[dtype]
    assert _lib.lib().hexmi_gemm_ex(M, N, K, a.data_ptr(), K, b.data_ptr(), b.stride(0), view.data_ptr(), N + 8, None,
                                    view.data_ptr() if residual else None, N + 8 if residual else 0, code, code, int(trans_b),
                                    torch.cuda.current_stream().cuda_stream) == _lib.OK
    # fp32 sums in another order, then one rounding to the output type
    assert ((view[:, :N].double() - want).abs() <= 1e-5 * mag + torch.finfo(dtype).eps / 2 * want.abs() + 1e-7).all()
    assert torch.equal(view[:, N:], keep)


# ... and output rows of any length at any place, which take bias and residual by elements
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,bias,residual", [
    (1025, 4097, 8, False, False), (2049, 1097, 72, True, True), (482, 4069, 1024, True, True), (2177, 1033, 136, False, True),   # 128 x 128
    (2049, 1095, 1000, True, False), (1345, 6215, 1608, False, True), (1300, 6401, 1600, True, False), (1300, 6401, 1600, False, True),
    (700, 9001, 1000, False, True), (645, 12457, 704, True, False), (1009, 24001, 328, True, False),
    (2049, 1097, 312, False, False), (2049, 1097, 328, False, False), (1345, 6215, 1016, False, False), (1345, 6215, 1032, False, False),
    (2049, 1100, 120, True, False), (2049, 1100, 136, True, False), (2049, 1100, 40, False, True)])    # the lines of K; runs of four
def test_gemm_tiles_between_128_and_256_odd_rows(hexmi, dtype, M, N, K, bias, residual):
    _against_double(hexmi, dtype, dtype, True, M, N, K, bias, residual, M + N + K)
    # an output one element off in rows three longer, the residual the output itself, nothing written around it
    from hexmi import _lib
    a, b = _inputs(M, N, K, dtype, True, seed=5)
    a, b = a.cuda(), b.cuda()
    bi = torch.randn(N + 1, generator=_gen(4)).to(dtype).cuda()[1:]
    buf = torch.randn(M * (N + 3) + 8, generator=_gen(3)).to(dtype).cuda()
    view = buf[1:1 + M * (N + 3)].view(M, N + 3)
    want, mag = a.double() @ b.double().t() + bi.double(), a.double().abs() @ b.double().abs().t() + bi.double().abs()
    if residual:
        want, mag = want + view[:, :N].double(), mag + view[:, :N].double().abs()
    keep, ends = view[:, N:].clone(), torch.cat([buf[:1], buf[1 + M * (N + 3):]]).clone()
    code = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}[dtype]
    assert _lib.lib().hexmi_gemm_ex(M, N, K, a.data_ptr(), K, b.data_ptr(), K, view.data_ptr(), N + 3, bi.data_ptr(),
                                    view.data_ptr() if residual else None, N + 3 if residual else 0, code, code, 1,
                                    torch.cuda.current_stream().cuda_stream) == _lib.OK
    # fp32 sums in another order, then one rounding to the output type
    assert ((view[:, :N].double() - want).abs() <= 1e-5 * mag + torch.finfo(dtype).eps / 2 * want.abs() + 1e-7).all()
    assert torch.equal(view[:, N:], keep) and torch.equal(torch.cat([buf[:1], buf[1 + M * (N + 3):]]), ends)


# up to 64 rows against [N,K] weights that the weight stream does not take: K off whole 32s, fewer than 64 channels
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(3, 64, 8), (8, 700, 1000), (9, 65, 40), (16, 272, 4264), (17, 257, 1128), (32, 384, 856), (33, 2000, 72),
                                   (64, 513, 2056), (3, 63, 1056), (40, 50, 2048), (64, 1, 256), (16, 4097, 776)])
def test_gemm_few_rows_the_weight_stream_leaves(hexmi, dtype, M, N, K):
    for out_dtype in (dtype, torch.float32):
        _against_double(hexmi, dtype, out_dtype, True, M, N, K, False, False, M + N)
        _against_double(hexmi, dtype, out_dtype, True, M, N, K, True, True, M + K)


# operand rows off the boundaries: every tile of plan_gemm_any on 256 CUs and its edges, K of fewer slabs than are on their way, of whole
# slabs and one element over and short, rows of fewer columns than a chunk
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("M,N,K", [
    (1, 1, 1), (3, 5, 7), (5, 9, 300), (2, 7, 1000), (16, 4097, 257), (17, 33, 2049), (64, 2047, 255), (33, 1025, 1281),    # 16 x 32
    (65, 2049, 513), (200, 501, 767), (97, 1999, 264), (500, 993, 1024),                                        # 32 x 32, 32 x 64
    (300, 3001, 129), (1000, 1001, 1000), (1900, 1023, 333),                                                    # 64 x 64, 128 x 64
    (2100, 2049, 63), (2049, 2050, 193), (2177, 2191, 256), (70, 33001, 65), (33025, 129, 127),                 # 128 x 128
    (300, 7, 8), (64, 1, 9), (8, 6, 15), (200, 2, 4096), (1000, 3, 511), (9000, 1, 1030), (33000, 4, 130),      # fewer than eight columns,
    (4096, 5, 64), (16, 300, 2), (300, 300, 1), (3000, 100, 6), (33000, 130, 7), (70000, 1, 5),                 # or of K
    (40, 65, 511), (40, 65, 513), (40, 65, 769), (40, 65, 1023), (40, 65, 1025), (33025, 5, 129), (33025, 5, 257)])    # one to five slabs
def test_gemm_operand_rows_off_the_boundaries(hexmi, dtype, out_dtype, trans_b, M, N, K):
    _against_double(hexmi, dtype, out_dtype, trans_b, M, N, K, False, False, M + N + K)
    _against_double(hexmi, dtype, out_dtype, trans_b, M, N, K, True, True, M + N + K + 1)
    # views one and three elements into larger buffers of infinities: nothing outside the operands reaches a sum
    from hexmi import _lib
    code = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16, torch.float32: _lib.F32}
    a, b = _inputs(M, N, K, dtype, trans_b, seed=7)
    br, bc = b.shape
    lda, ldb = K + 3, bc + 5
    ab, bb = torch.full((M * lda + 8,), math.inf, dtype=dtype), torch.full((br * ldb + 8,), math.inf, dtype=dtype)
    ab[1:1 + M * lda].view(M, lda)[:, :K] = a
    bb[3:3 + br * ldb].view(br, ldb)[:, :bc] = b
    ab, bb = ab.cuda(), bb.cuda()
    c = torch.full((M, N), math.nan, dtype=out_dtype, device="cuda")
    assert _lib.lib().hexmi_gemm_ex(M, N, K, ab.data_ptr() + 2, lda, bb.data_ptr() + 6, ldb, c.data_ptr(), N, None, None, 0, code[dtype],
                                    code[out_dtype], int(trans_b), torch.cuda.current_stream().cuda_stream) == _lib.OK
    a, b = a.cuda().double(), b.cuda().double()
    b = b.t() if trans_b else b
    # sums in fp32 in another order: 1e-5 of the summed magnitudes; one rounding to the output type: half an ulp
    eps = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[out_dtype]
    assert ((c.double() - a @ b).abs() <= 1e-5 * (a.abs() @ b.abs()) + eps * (a @ b).abs() + 1e-7).all()


def test_gemm_longest_inner_dimension(hexmi):
    # one workgroup walks all of K: the slabs asked for past the last one lie past 2^31 elements
    K = 0x7fffffff - 64
    a, b = (torch.zeros(1, K, dtype=torch.float16, device="cuda") for _ in range(2))
    at = torch.tensor([0, 1, K // 2, 1 << 30, K - 600, K - 257, K - 9, K - 8, K - 1], device="cuda")
    a[0, at] = 2.0 ** torch.arange(9, device="cuda").half()
    b[0, at] = 1.0
    assert float(hexmi.matmul(a, b, trans_b=True)) == 511.0


# more tiles than a grid of 512 threads each holds: rows of eight on the tiles of 16-bit results, single columns through registers
@pytest.mark.parametrize("N", [1, 8])
def test_gemm_more_tiles_than_a_grid_holds(hexmi, N):
    M = (0xffffffff // 512 + 1) * 128 + 3
    a = torch.randint(-2048, 2049, (M, N), dtype=torch.float16, device="cuda", generator=torch.Generator("cuda").manual_seed(5))
    assert torch.equal(hexmi.matmul(a, torch.eye(N, dtype=torch.float16, device="cuda")), a)


# more tiles than one round of them: the 128 x 128 and 256 x 256 kernels and the slabs, widths and outputs each is for
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,bias,residual", [
    (2049, 1096, 64, False, False), (2049, 1096, 96, False, False), (2049, 1096, 160, True, True),   # whole slabs of 64 and 32
    (2049, 1096, 72, False, False), (2049, 1096, 1000, True, False), (2100, 1096, 448, True, True),  # chunks past K masked
    (2049, 1033, 256, False, False), (2049, 1033, 72, False, True), (2049, 1033, 96, True, False),   # odd widths
    (2049, 1096, 77, False, False), (2049, 1033, 333, True, True)])                                  # unaligned rows
def test_gemm_more_than_a_round_of_tiles(hexmi, dtype, trans_b, M, N, K, bias, residual):
    _against_double(hexmi, dtype, dtype, trans_b, M, N, K, bias, residual, M + N + K)


def test_gemm_closed_forms(hexmi):
    g = _gen(1)
    a = torch.randn(256, 128, generator=g).half()
    eye = torch.eye(128).half()
    assert torch.equal(hexmi.matmul(a.cuda(), eye.cuda()).cpu(), a)
    ones = torch.ones(128, 256).half()
    got = hexmi.matmul(a.cuda(), ones.cuda(), out_dtype=torch.float32).cpu()
    assert torch.allclose(got, a.double().sum(-1, keepdim=True).float().expand(256, 256), rtol=1e-5, atol=1e-5)
    onehot = torch.zeros(128, 256).half()
    onehot[5, 200] = 1
    c = hexmi.matmul(a.cuda(), onehot.cuda()).cpu()
    assert torch.equal(c[:, 200], a[:, 5]) and c.abs().sum() == a[:, 5].abs().sum()
    # transposed operand: a row-index / column-index swap in either loader changes this
    b = torch.randn(128, 264, generator=g).half()
    c1 = hexmi.matmul(a.cuda(), b.cuda(), out_dtype=torch.float32).cpu()
    c2 = hexmi.matmul(a.cuda(), b.t().contiguous().cuda(), out_dtype=torch.float32, trans_b=True).cpu()
    assert torch.equal(c1, c2)


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gemm_large_ragged_tiles(hexmi, dtype, trans_b):
    # enough 256x256 tiles for the large-tile kernel, ragged in M and N, odd slab count; checked on sampled rows
    # against a float64 product of the same rounded inputs
    M, N, K = 2900, 2904, 192
    a, b = _inputs(M, N, K, dtype, trans_b, seed=11)
    got = hexmi.matmul(a.cuda(), b.cuda(), out_dtype=torch.float32, trans_b=trans_b).cpu()
    rows = torch.cat([torch.arange(0, M, 37), torch.arange(M - 50, M)])
    bb = b.double().t() if trans_b else b.double()
    want = a[rows].double() @ bb
    mag = a[rows].double().abs() @ bb.abs()
    assert ((got[rows].double() - want).abs() <= 1e-5 * mag + 1e-30).all()
    got16 = hexmi.matmul(a.cuda(), b.cuda(), trans_b=trans_b).cpu()
    assert torch.equal(got16, got.to(dtype))          # the 16-bit result is the rounded fp32 result, staged or not


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gemm_odd_width_on_large_tiles(hexmi, dtype):
    # [N,K] weights with an odd N and enough tiles for the 256x256 form (a vocabulary-sized projection): the same
    # kernel as with the weight padded to a multiple of 8 rows, only the way out differs -- bit for bit
    M, N, K = 4096, 8193, 128
    a, b = _inputs(M, N, K, dtype, True, seed=13)
    got = hexmi.matmul(a.cuda(), b.cuda(), trans_b=True)
    b_pad = torch.cat([b, torch.zeros(7, K, dtype=dtype)])
    want = hexmi.matmul(a.cuda(), b_pad.cuda(), trans_b=True)
    assert torch.equal(got, want[:, :N])
    rows = torch.arange(0, M, 97)
    ref = a[rows].double() @ b.double().t()
    assert (got.cpu()[rows].double() - ref).abs().max() <= 2e-2 * math.sqrt(K)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gemm_output_rows_off_the_boundaries(hexmi, dtype):
    # [N,K] weights, whole 64-wide slabs, output rows that start anywhere (odd widths, leading dimensions wider than
    # the rows, a base 2 or 6 bytes into its buffer; C ABI): the staged tile leaves in the aligned 16-byte pieces of
    # each row and its ends by elements. Bit for bit the dense call's values, nothing outside the window written.
    from hexmi import _lib
    L = _lib.lib()
    st = torch.cuda.current_stream().cuda_stream
    dt = _lib.F16 if dtype == torch.float16 else _lib.BF16
    for M, N, K, pad, lead in ((300, 1001, 256, 0, 0), (300, 1001, 256, 3, 1), (129, 70, 64, 1, 3), (520, 777, 128, 6, 0),
                               (4096, 2049, 128, 0, 1), (64, 5, 64, 2, 1), (257, 263, 192, 4, 3)):
        a, b = _inputs(M, N, K, dtype, True, seed=M + N + pad)
        ldc = N + pad
        c_buf = torch.full((M * ldc + lead + 9,), 7.0, dtype=dtype, device="cuda")
        ad, bd = a.cuda(), b.cuda()
        rc = L.hexmi_gemm(M, N, K, ad.data_ptr(), K, bd.data_ptr(), K, c_buf.data_ptr() + 2 * lead, ldc, dt, dt, 1, st)
        assert rc == 0
        b_pad = torch.cat([b, torch.zeros((-N) % 8, K, dtype=dtype)])
        want = hexmi.matmul(ad, b_pad.cuda(), trans_b=True)[:, :N]
        c = c_buf[lead:lead + M * ldc].view(M, ldc)
        assert torch.equal(c[:, :N], want), (M, N, K, pad, lead)
        assert (c_buf[:lead] == 7.0).all() and (c[:, N:] == 7.0).all() and (c_buf[lead + M * ldc:] == 7.0).all()


# A few 256 x 256 tiles more than whole rounds over 256 CUs: the columns past the rounds go as a product of their own. One column,
# eight, less and more than a tile's width; rows of the output on and off the boundaries; just under and over the line.
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("trans_b,M,N,K", [
    (True, 4096, 8193, 128), (True, 4096, 8200, 192), (False, 4096, 8200, 128), (True, 4090, 8451, 128), (False, 4090, 8704, 96),
    (True, 1021, 33025, 128), (False, 1021, 33280, 64), (True, 4096, 9984, 64), (True, 4096, 9985, 128),
    (True, 3762, 4721, 768), (False, 3762, 4720, 832), (True, 3700, 4720, 704)])      # 1.1 rounds; half a tile of padded rows
def test_gemm_columns_past_whole_rounds(hexmi, out_dtype, trans_b, M, N, K):
    _against_double(hexmi, torch.bfloat16, out_dtype, trans_b, M, N, K, False, False, N)


# The ends of a ragged row: the last tile holds 1 to 8 columns, ends just before, on and behind the seam between two waves' halves
# (128 columns on 256 x 256 tiles, 64 on 128 x 128), with rows starting at every offset from a 16-byte boundary.
@pytest.mark.parametrize("M,N", [(4096, 2049), (4096, 2054), (4096, 2175), (4096, 2177), (4096, 2183), (4096, 2303),
                                 (300, 1025), (300, 1087), (300, 1089), (300, 1095)])
@pytest.mark.parametrize("pad,lead", [(0, 0), (1, 5)])
def test_gemm_ragged_row_ends(hexmi, M, N, pad, lead):
    from hexmi import _lib
    K, ldc = 128, N + pad
    a, b = _inputs(M, N, K, torch.bfloat16, True, seed=N)
    ad, bd = a.cuda(), b.cuda()
    c_buf = torch.full((M * ldc + lead + 9,), 7.0, dtype=torch.bfloat16, device="cuda")
    rc = _lib.lib().hexmi_gemm(M, N, K, ad.data_ptr(), K, bd.data_ptr(), K, c_buf.data_ptr() + 2 * lead, ldc, _lib.BF16, _lib.BF16,
                               1, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    # the dense call of the padded weight leaves in whole pieces; the sums are the same, bit for bit
    want = hexmi.matmul(ad, torch.cat([b, torch.zeros((-N) % 8, K, dtype=b.dtype)]).cuda(), trans_b=True)[:, :N]
    c = c_buf[lead:lead + M * ldc].view(M, ldc)
    assert torch.equal(c[:, :N], want)
    assert (c_buf[:lead] == 7.0).all() and (c[:, N:] == 7.0).all() and (c_buf[lead + M * ldc:] == 7.0).all()


def test_gemm_unaligned_views(hexmi):
    # operands and result that start 2 bytes into their buffers, odd leading dimensions (C ABI only): the any-shape
    # kernel; nothing outside the result's window is written
    from hexmi import _lib
    L = _lib.lib()
    st = torch.cuda.current_stream().cuda_stream
    g = _gen(14)
    for trans_b in (0, 1):
        for M, N, K in ((200, 136, 264), (130, 77, 100), (64, 64, 64)):
            lda, ldb, ldc = K + 3, (K if trans_b else N) + 5, N + 1
            a_buf = (2 * torch.rand(M * lda + 1, generator=g) - 1).half().cuda()
            b_buf = (2 * torch.rand((N if trans_b else K) * ldb + 1, generator=g) - 1).half().cuda()
            c_buf = torch.full((M * ldc + 1,), 7.0, dtype=torch.float16, device="cuda")
            rc = L.hexmi_gemm(M, N, K, a_buf.data_ptr() + 2, lda, b_buf.data_ptr() + 2, ldb, c_buf.data_ptr() + 2, ldc,
                              1, 1, trans_b, st)
            assert rc == 0
            a = a_buf[1:].view(M, lda)[:, :K].contiguous()
            b = b_buf[1:].view(-1, ldb)[:, :(K if trans_b else N)].contiguous()
            want = hexmi.matmul(a, b, trans_b=bool(trans_b))
            c = c_buf[1:].view(M, ldc)
            assert close16(c[:, :N].contiguous(), want, max_ulp=1, atol=1e-4)
            assert float(c_buf[0]) == 7.0 and (c[:, N:] == 7.0).all()


def test_gemm_strided_operands(hexmi):
    # leading dimensions larger than the rows (C ABI only): same arithmetic as the dense call, bit for bit; ldc % 8 != 0
    # takes the direct (unstaged) 16-bit stores
    from hexmi import _lib
    L = _lib.lib()
    M, N, K = 300, 264, 128
    lda, ldb, ldc = K + 8, N + 16, N + 4
    g = _gen(12)
    a_big = (2 * torch.rand(M, lda, generator=g) - 1).half().cuda()
    b_big = (2 * torch.rand(K, ldb, generator=g) - 1).half().cuda()
    c_big = torch.full((M, ldc), 7.0, dtype=torch.float16, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    rc = L.hexmi_gemm(M, N, K, a_big.data_ptr(), lda, b_big.data_ptr(), ldb, c_big.data_ptr(), ldc, 1, 1, 0, st)
    assert rc == 0
    dense = hexmi.matmul(a_big[:, :K].contiguous(), b_big[:, :N].contiguous())
    assert torch.equal(c_big[:, :N], dense)
    assert (c_big[:, N:] == 7.0).all()                # nothing written past the N columns


def test_hexkl_entry_point(hexmi, oracle):
    # hexmi_matmul_f16f16_f32(n_row, n_col, n_inner, out, act, w): the fixture's sizes
    # (test/python/mlir/hexkl_linalg_matmul/wrapper.cpp:31-33: N=1024, K=64, M=512) and its MAX_DIFF 1e-2
    from hexmi import _lib
    g = _gen(2)
    act = (torch.randn(1024, 64, generator=g) * 0.5).half()
    w = (torch.randn(64, 512, generator=g) * 0.5).half()
    out = torch.empty(1024, 512, device="cuda")
    ad, wd = act.cuda(), w.cuda()
    rc = _lib.lib().hexmi_matmul_f16f16_f32(1024, 512, 64, out.data_ptr(), ad.data_ptr(), wd.data_ptr(),
                                            torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want = torch.from_numpy(oracle.matmul(act.numpy(), w.numpy(), out_dtype=np.float32))
    assert (out.cpu() - want).abs().max() < 1e-2
    assert rel_err(out, want) <= 1e-5


def test_reference_matmul_call_site(hexmi, oracle):
    # test_matmul.py:72-91: host tensors, C zero-initialised and filled in place, atol 2e-1
    g = _gen(3)
    A = torch.rand((1024, 64), generator=g).half()
    B = torch.rand((64, 512), generator=g).half()
    C = torch.zeros((1024, 512), dtype=torch.float16)
    hexmi.kernels.matmul[(1,)](A, B, C, 1024, 512, 64, enableMultiThreading=True, enableVTCMTiling=True,
                               enableConvertToHexagonmem=True, enableHexagonmemCopyToDMA=True)
    want = from_np(oracle.matmul(A.numpy(), B.numpy()), torch.float16)
    assert torch.allclose(C, want, atol=2e-1) and close16(C, want, 1, atol=1e-4)
    # matmul_hexkl.md:100-111: fp32 C, rtol 1e-2
    C32 = torch.zeros((1024, 512), dtype=torch.float32)
    hexmi.kernels.matmul_hexkl[(1,)](A, B, C32, 1024, 512, 64, enableHexKL=True)
    assert torch.allclose(C32, torch.from_numpy(oracle.matmul(A.numpy(), B.numpy(), out_dtype=np.float32)), rtol=1e-5)


def test_macro_matmul_shapes(hexmi, oracle):
    # test_hexkl_macro_matmul.py:31-68: 1024^3 and x[1024,512] @ W[256,512].T, randn seed 42, rtol/atol 1e-2
    torch.manual_seed(42)
    x = torch.randn(512, 1024).half()
    w = torch.randn(1024, 1024).half()
    got = hexmi.matmul(x.cuda(), w.cuda()).cpu()
    assert close16(got, from_np(oracle.matmul(x.numpy(), w.numpy()), torch.float16), 1, atol=1e-4)
    x2 = torch.randn(1024, 512).half()
    w2 = torch.randn(256, 512).half()
    got2 = hexmi.matmul(x2.cuda(), w2.cuda(), trans_b=True).cpu()
    want2 = from_np(oracle.matmul(x2.numpy(), w2.numpy(), trans_b=True), torch.float16)
    assert close16(got2, want2, 1, atol=1e-4) and torch.allclose(got2.float(), want2.float(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("dtype,size", [(torch.float16, 4096), (torch.bfloat16, 8192)])
def test_gemm_config_sizes(hexmi, oracle, dtype, size):
    """Measured configurations. The oracle is run on a deterministic subset of rows (every 61st row, all
    columns); the full result is covered by a size-independent property: linearity in A,
    (A + A') B == A B + A' B exactly in fp32 output when A' is a row permutation of A scaled by 0 or 1 --
    here checked as: C computed from a row-shuffled A equals the row-shuffled C, bit for bit."""
    from hexmi.workloads import gemm_inputs
    inp = gemm_inputs(size, size, size, dtype)
    a, b = inp["a"], inp["b"]
    ad, bd = a.cuda(), b.cuda()
    c = hexmi.matmul(ad, bd)
    c32 = hexmi.matmul(ad, bd, out_dtype=torch.float32)
    rows = torch.arange(0, size, 61)
    an, tag = to_np(a[rows])
    bn, _ = to_np(b)
    want32 = torch.from_numpy(oracle.matmul(an, bn, out_dtype=np.float32, dtype=tag))
    got32 = c32[rows.cuda()].cpu()
    assert rel_err(got32, want32) <= 1e-5
    od = "bf16" if dtype == torch.bfloat16 else np.float16
    want = from_np(oracle.matmul(an, bn, out_dtype=od, dtype=tag), dtype)
    assert close16(c[rows.cuda()].cpu(), want, 1, atol=1e-4)
    perm = torch.randperm(size, generator=_gen(7)).cuda()
    c_perm = hexmi.matmul(ad[perm].contiguous(), bd)
    assert torch.equal(c_perm, c[perm])
    # the same product through the transposed-weight loader must agree exactly (same fp32 sums, same order in k)
    c_t = hexmi.matmul(ad, bd.t().contiguous(), trans_b=True)
    assert torch.equal(c_t, c)


def test_gemm_empty_inner_dimension_is_zero(hexmi):
    # a product over K = 0 is all zeros (torch.matmul gives the same), for every output type, with a leading dimension
    for dt, odt in ((torch.float16, torch.float16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)):
        buf = torch.full((5, 12), 3.0, dtype=odt, device="cuda")
        out = buf[:, :7]
        from hexmi import _lib
        code = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16, torch.float32: _lib.F32}
        rc = _lib.lib().hexmi_gemm(5, 7, 0, None, 0, None, 7, out.data_ptr(), 12, code[dt], code[odt], 0, None)
        assert rc == _lib.OK
        torch.cuda.synchronize()
        assert torch.equal(buf[:, :7].cpu(), torch.zeros(5, 7, dtype=odt))
        assert torch.equal(buf[:, 7:].cpu(), torch.full((5, 5), 3.0, dtype=odt))       # past N: untouched
    assert hexmi.matmul(torch.zeros(4, 0, dtype=torch.float16, device="cuda"),
                        torch.zeros(0, 8, dtype=torch.float16, device="cuda")).abs().sum().item() == 0


def test_gemm_argument_errors(hexmi):
    from hexmi import _lib
    a = torch.zeros(8, 8, device="cuda", dtype=torch.float16)
    lib = _lib.lib()
    assert lib.hexmi_gemm(8, 8, 8, a.data_ptr(), 4, a.data_ptr(), 8, a.data_ptr(), 8, _lib.F16, _lib.F16, 0, None) == _lib.EINVAL
    assert lib.hexmi_gemm(8, 8, 8, a.data_ptr(), 8, a.data_ptr(), 8, a.data_ptr(), 8, _lib.F32, _lib.F16, 0, None) == _lib.ENOTSUP
    assert lib.hexmi_gemm(8, 8, 8, a.data_ptr(), 8, a.data_ptr(), 8, a.data_ptr(), 8, _lib.F16, _lib.BF16, 0, None) == _lib.ENOTSUP
    with pytest.raises(TypeError):
        hexmi.matmul(torch.zeros(4, 4, device="cuda", dtype=torch.float64), torch.zeros(4, 4, device="cuda", dtype=torch.float64))
    with pytest.raises(ValueError):
        hexmi.matmul(a, torch.zeros(4, 4, device="cuda", dtype=torch.float16))


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("shape", [(32, 32, 32), (1, 1, 1), (65, 130, 17), (200, 77, 300), (512, 512, 512),
                                   # K % 32 == 0 (and N % 4 == 0 for [K,N] operands): the matrix-core kernel; ragged
                                   # tiles on both sides, fewer rows than a fragment, several slabs, odd slab counts
                                   (128, 128, 32), (5, 4, 64), (300, 264, 160), (129, 1028, 96), (1000, 520, 1024),
                                   (2048, 384, 224), (64, 132, 4096)])
def test_matmul_fp32(hexmi, oracle, shape, trans_b):
    M, N, K = shape
    g = torch.Generator().manual_seed(40)
    a = torch.randn(M, K, generator=g)
    b = torch.randn(N, K, generator=g) if trans_b else torch.randn(K, N, generator=g)
    got = hexmi.matmul(a.cuda(), b.cuda(), trans_b=trans_b).cpu()
    want = a.double() @ (b.double().t() if trans_b else b.double())
    assert got.dtype == torch.float32
    assert torch.allclose(got.double(), want, rtol=1e-5, atol=1e-5 * (K ** 0.5))
    with pytest.raises(TypeError):
        hexmi.matmul(a.cuda(), b.cuda(), trans_b=trans_b, out_dtype=torch.float16)


@pytest.mark.parametrize("trans_b", [False, True])
def test_matmul_fp32_strided_and_exact(hexmi, trans_b):
    # operands that are views into wider buffers (leading dimensions larger than the rows), an output view, and
    # small-integer operands whose products and sums are exact in fp32: the result must be exact, whatever the order
    M, N, K = 200, 136, 96
    g = torch.Generator().manual_seed(45)
    abuf = torch.randint(-8, 9, (M, K + 32), generator=g).float().cuda()
    bbuf = (torch.randint(-8, 9, (N, K + 64), generator=g) if trans_b else torch.randint(-8, 9, (K, N + 24), generator=g)).float().cuda()
    cbuf = torch.full((M, N + 8), -1.0, device="cuda")
    a, b, c = abuf[:, :K], (bbuf[:, :K] if trans_b else bbuf[:, :N]), cbuf[:, :N]
    lib, st = hexmi.lib(), torch.cuda.current_stream().cuda_stream
    from hexmi import _lib
    rc = lib.hexmi_gemm(M, N, K, a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), c.data_ptr(), c.stride(0),
                        _lib.F32, _lib.F32, int(trans_b), st)
    assert rc == 0
    torch.cuda.synchronize()
    want = a.double().cpu() @ (b.double().cpu().t() if trans_b else b.double().cpu())
    assert torch.equal(c.cpu().double(), want)
    assert (cbuf[:, N:] == -1.0).all()                       # nothing written past the N columns


def test_add_matmul_softmax_reference_graph(hexmi):
    # test/python/torch-mlir/test_add_matmul_softmax.py:32-60: three 32x32 fp32 randn, rtol 1e-5, atol 1e-6
    g = torch.Generator().manual_seed(41)
    x, y, z = (torch.randn(32, 32, generator=g) for _ in range(3))
    got = hexmi.add_matmul_softmax(x, y, z)
    want = torch.nn.functional.softmax(torch.matmul(x + y, z), dim=-1)
    assert got.device.type == "cuda"
    assert torch.allclose(got.cpu(), want, rtol=1e-5, atol=1e-6)
    # fp16 operands run the matrix-core GEMM
    got16 = hexmi.add_matmul_softmax(x.half(), y.half(), z.half()).cpu()
    want16 = torch.nn.functional.softmax(torch.matmul((x.half() + y.half()).float(), z.half().float()), dim=-1)
    assert torch.allclose(got16.float(), want16, atol=2e-2)


# ---- hexmi_gemm_ex: bias and residual in the GEMM epilogue ------------------------------------------------------
def _linear_ref(a, b, bias, resid, trans_b):
    c = a.double() @ (b.double().T if trans_b else b.double())
    if bias is not None:
        c = c + bias.double()
    if resid is not None:
        c = c + resid.double()
    return c


@pytest.mark.parametrize("dtype,out_dtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16),
                                             (torch.float16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("shape", [(512, 2304, 768), (512, 768, 3072),      # GPT-2 small layers (64-k tiled kernel)
                                   (256, 256, 96),                           # 32-k tiled kernel
                                   (100, 72, 40), (33, 50, 17),              # any-shape kernel (ragged, unaligned)
                                   (260, 1003, 72), (130, 136, 1000),        # ragged-K kernel: rows through LDS / runs
                                   (1024, 1024, 1024)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_gemm_ex_bias_and_residual(hexmi, dtype, out_dtype, shape, trans_b):
    M, N, K = shape
    g = torch.Generator().manual_seed(M * 7 + N * 3 + K + trans_b)
    a = (torch.randn(M, K, generator=g) * 0.5).to(dtype)
    b = (torch.randn((N, K) if trans_b else (K, N), generator=g) * 0.5).to(dtype)
    bias = torch.randn(N, generator=g).to(out_dtype)
    resid = torch.randn(M, N, generator=g).to(out_dtype)
    tol = {torch.float16: 2e-2, torch.bfloat16: 1.5e-1, torch.float32: 2e-3 if dtype != torch.float32 else 2e-4}[out_dtype]
    for use_bias, use_resid in ((True, True), (True, False), (False, True)):
        got = hexmi.matmul(a.cuda(), b.cuda(), out_dtype=out_dtype, trans_b=trans_b,
                           bias=bias.cuda() if use_bias else None, residual=resid.cuda() if use_resid else None)
        want = _linear_ref(a, b, bias if use_bias else None, resid if use_resid else None, trans_b)
        err = (got.cpu().double() - want).abs().max().item()
        assert err <= tol * max(1.0, want.abs().max().item() / 16), (use_bias, use_resid, err)


def test_gemm_ex_rounds_once(hexmi):
    # fp16: A B + bias + residual rounded once from fp32 == the correctly rounded fp64 result on all but ties; the
    # separate kernels (round the product, round the sum, round again) are measurably further away.
    g = torch.Generator().manual_seed(11)
    M, N, K = 256, 512, 256
    a = torch.randn(M, K, generator=g).half()
    b = torch.randn(K, N, generator=g).half()
    bias = torch.randn(N, generator=g).half()
    resid = torch.randn(M, N, generator=g).half()
    want = _linear_ref(a, b, bias, resid, False)
    fused = hexmi.matmul(a.cuda(), b.cuda(), bias=bias.cuda(), residual=resid.cuda()).cpu().double()
    parts = hexmi.binary("add", hexmi.binary("add", hexmi.matmul(a.cuda(), b.cuda()),
                                             bias.cuda().expand(M, N).contiguous()), resid.cuda()).cpu().double()
    e_fused = (fused - want).abs().mean().item()
    e_parts = (parts - want).abs().mean().item()
    assert e_fused < e_parts
    assert (fused - want.half().double()).abs().max().item() <= 2 * torch.finfo(torch.float16).eps * want.abs().max().item()


# one shape per kernel that takes a residual: paired 64-k slabs, 32-k slabs (K % 64 != 0), the any-shape kernel
# (odd N), the fp32 matrix-core kernel and the fp32 vector-ALU kernel (K % 32 != 0)
@pytest.mark.parametrize("dtype,M,N,K", [(torch.float16, 384, 768, 768), (torch.float16, 256, 512, 96),
                                         (torch.bfloat16, 200, 333, 64), (torch.float32, 256, 512, 128),
                                         (torch.float32, 130, 77, 50)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_gemm_ex_residual_may_alias_output(hexmi, dtype, M, N, K, trans_b):
    g = torch.Generator().manual_seed(12)
    a = (torch.randn(M, K, generator=g) * 0.1).to(dtype).cuda()
    b = (torch.randn(*((N, K) if trans_b else (K, N)), generator=g) * 0.1).to(dtype).cuda()
    x = torch.randn(M, N, generator=g).to(dtype).cuda()
    want = hexmi.matmul(a, b, residual=x, trans_b=trans_b)
    acc = x.clone()
    hexmi.matmul(a, b, residual=acc, out=acc, trans_b=trans_b)      # x += a @ b, in place
    assert torch.equal(acc, want)


def test_gemm_ex_strided_residual_and_bad_arguments(hexmi):
    from hexmi import _lib
    lib = _lib.lib()
    g = torch.Generator().manual_seed(13)
    M, N, K = 128, 256, 128
    a = torch.randn(M, K, generator=g).half().cuda()
    b = torch.randn(K, N, generator=g).half().cuda()
    wide = torch.randn(M, N + 64, generator=g).half().cuda()       # residual with a leading dimension of N + 64
    c = torch.empty(M, N, dtype=torch.float16, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    st = lib.hexmi_gemm_ex(M, N, K, a.data_ptr(), K, b.data_ptr(), N, c.data_ptr(), N, None, wide.data_ptr(), N + 64,
                           _lib.F16, _lib.F16, 0, s)
    assert st == 0
    want = _linear_ref(a.cpu(), b.cpu(), None, wide[:, :N].cpu(), False)
    assert (c.cpu().double() - want).abs().max().item() <= 2e-2 * max(1.0, want.abs().max().item() / 16)
    # a residual narrower than the result is refused
    assert lib.hexmi_gemm_ex(M, N, K, a.data_ptr(), K, b.data_ptr(), N, c.data_ptr(), N, None, wide.data_ptr(), N - 8,
                             _lib.F16, _lib.F16, 0, s) == _lib.EINVAL
    with pytest.raises(ValueError):
        hexmi.matmul(a, b, bias=torch.zeros(N + 1, dtype=torch.float16, device="cuda"))
    with pytest.raises(ValueError):
        hexmi.matmul(a, b, residual=torch.zeros(M, N, dtype=torch.float32, device="cuda"))


# ---- hexmi_add_matmul_softmax: the fused graph in one launch ----------------------------------------------------
def _ams_ref(x, y, z):
    total = (x + y)                                                  # torch.add rounds the sum to the dtype
    return torch.softmax(total.double() @ z.double(), dim=-1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(32, 32, 32),                     # test_add_matmul_softmax.py:32-60
                                   (1, 1, 1), (7, 5, 3), (100, 130, 70), (33, 257, 100), (64, 512, 48),
                                   (50, 1000, 37), (96, 1024, 64), (512, 768, 768)])
def test_add_matmul_softmax_one_launch(hexmi, dtype, shape):
    M, N, K = shape
    g = torch.Generator().manual_seed(M + N * 5 + K * 11)
    x = torch.randn(M, K, generator=g).to(dtype)
    y = torch.randn(M, K, generator=g).to(dtype)
    z = (torch.randn(K, N, generator=g) * (1.0 if K <= 64 else 0.2)).to(dtype)
    got = hexmi.add_matmul_softmax(x.cuda(), y.cuda(), z.cuda(), fused=True).cpu()
    want = _ams_ref(x, y, z)
    assert got.dtype == dtype and got.shape == (M, N)
    if dtype == torch.float32:
        # the reference test's own bounds at its size; longer fp32 sums carry their rounding into the exponent
        torch.testing.assert_close(got.double(), want, rtol=1e-5 if K <= 64 else 2e-4, atol=1e-6)
    else:
        eps = torch.finfo(dtype).eps
        torch.testing.assert_close(got.double(), want, rtol=2 * eps, atol=eps * 0.25)
    sums = got.double().sum(-1)
    assert (sums - 1).abs().max().item() <= (1e-5 if dtype == torch.float32 else N ** 0.5 * torch.finfo(dtype).eps)
    # the three-launch route agrees (it rounds the product to the dtype before the softmax, so only to that rounding)
    three = hexmi.add_matmul_softmax(x.cuda(), y.cuda(), z.cuda(), fused=False).cpu()
    tol = 1e-5 if dtype == torch.float32 else 0.02 if dtype == torch.float16 else 0.15
    assert (three.double() - got.double()).abs().max().item() <= tol


def test_add_matmul_softmax_limits_and_layouts(hexmi):
    from hexmi import _lib
    lib = _lib.lib()
    assert lib.hexmi_add_matmul_softmax_max_n() == 1024
    g = torch.Generator().manual_seed(3)
    M, N, K = 40, 96, 24
    s = torch.cuda.current_stream().cuda_stream
    # leading dimensions wider than the rows, output at an odd element offset (no 4-element runs)
    xw = torch.randn(M, K + 3, generator=g).cuda()
    yw = torch.randn(M, K + 5, generator=g).cuda()
    zw = torch.randn(K, N + 7, generator=g).cuda()
    ow = torch.full((M * (N + 1) + 1,), -7.0, device="cuda")
    st = lib.hexmi_add_matmul_softmax(M, N, K, xw.data_ptr(), K + 3, yw.data_ptr(), K + 5, zw.data_ptr(), N + 7,
                                      ow.data_ptr() + 4, N + 1, _lib.F32, s)
    assert st == 0
    got = ow[1:].reshape(M, N + 1).cpu()
    want = _ams_ref(xw[:, :K].cpu(), yw[:, :K].cpu(), zw[:, :N].cpu())
    torch.testing.assert_close(got[:, :N].double(), want, rtol=1e-5, atol=1e-6)
    assert (got[:, N] == -7.0).all() and ow[0].item() == -7.0       # nothing written outside the result
    # too wide, and nonsense sizes
    big = torch.zeros(8, 1025, device="cuda")
    assert lib.hexmi_add_matmul_softmax(8, 1025, 8, big.data_ptr(), 8, big.data_ptr(), 8, big.data_ptr(), 1025,
                                        big.data_ptr(), 1025, _lib.F32, s) == _lib.ETOOBIG
    assert lib.hexmi_add_matmul_softmax(8, 16, 8, big.data_ptr(), 4, big.data_ptr(), 8, big.data_ptr(), 16,
                                        big.data_ptr(), 16, _lib.F32, s) == _lib.EINVAL
    assert lib.hexmi_add_matmul_softmax(0, 16, 8, None, 8, None, 8, None, 16, None, 16, _lib.F32, s) == 0
    # K == 0: every score is an empty sum, every row uniform
    out = torch.empty(5, 10, device="cuda")
    assert lib.hexmi_add_matmul_softmax(5, 10, 0, None, 0, None, 0, None, 10, out.data_ptr(), 10, _lib.F32, s) == 0
    torch.testing.assert_close(out.cpu(), torch.full((5, 10), 0.1))
    with pytest.raises(ValueError):
        hexmi.add_matmul_softmax(big, big, torch.zeros(1025, 2048, device="cuda"), fused=True)


# ---- hexmi_transpose16: one-time weight re-layout ----------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 1), (3, 70), (64, 64), (65, 129), (768, 3072), (1000, 37), (4096, 4096)])
def test_pack_weight_is_the_transpose(hexmi, dtype, shape):
    g = torch.Generator().manual_seed(shape[0] * 3 + shape[1])
    w = torch.randn(*shape, generator=g).to(dtype)
    w[0, 0] = float("inf")                                          # bit patterns are moved, whatever they are
    got = hexmi.pack_weight(w.cuda())
    assert got.shape == (shape[1], shape[0]) and got.dtype == dtype and got.is_contiguous()
    assert torch.equal(got.cpu().view(torch.int16), w.t().contiguous().view(torch.int16))


def test_packed_weight_product_is_the_same_product(hexmi):
    # A . B and A . pack(B)^T multiply the same numbers: equal to the last bit in the fp32-output mode
    g = torch.Generator().manual_seed(5)
    a = torch.randn(256, 512, generator=g).half().cuda()
    b = torch.randn(512, 384, generator=g).half().cuda()
    bt = hexmi.pack_weight(b)
    c1 = hexmi.matmul(a, b, out_dtype=torch.float32)
    c2 = hexmi.matmul(a, bt, out_dtype=torch.float32, trans_b=True)
    assert torch.equal(c1, c2)


def test_transpose16_strides_and_bad_arguments(hexmi):
    from hexmi import _lib
    lib = _lib.lib()
    s = torch.cuda.current_stream().cuda_stream
    src = torch.arange(20 * 12, dtype=torch.int16, device="cuda").reshape(20, 12)        # rows 20, ld 12, cols 10 used
    dst = torch.full((10, 24), -1, dtype=torch.int16, device="cuda")
    assert lib.hexmi_transpose16(20, 10, src.data_ptr(), 12, dst.data_ptr(), 24, s) == 0
    assert torch.equal(dst[:, :20].cpu(), src[:, :10].t().cpu())
    assert (dst[:, 20:] == -1).all()
    assert lib.hexmi_transpose16(20, 10, src.data_ptr(), 8, dst.data_ptr(), 24, s) == _lib.EINVAL
    assert lib.hexmi_transpose16(20, 10, src.data_ptr(), 12, dst.data_ptr(), 16, s) == _lib.EINVAL
    assert lib.hexmi_transpose16(0, 10, None, 12, None, 24, s) == 0
    with pytest.raises(TypeError):
        hexmi.pack_weight(torch.zeros(4, 4, device="cuda"))


def test_gemm_ex_and_fused_graph_against_the_oracle(hexmi, oracle):
    # the C oracle's product with its numpy epilogue / softmax (oracle.linear, oracle.add_matmul_softmax), fp16 and fp32
    g = torch.Generator().manual_seed(31)
    a = torch.randn(192, 320, generator=g).half()
    b = (torch.randn(320, 136, generator=g) * 0.2).half()
    bias = torch.randn(136, generator=g).half()
    res = torch.randn(192, 136, generator=g).half()
    got = hexmi.matmul(a.cuda(), b.cuda(), bias=bias.cuda(), residual=res.cuda()).cpu()
    want = torch.from_numpy(oracle.linear(a.numpy(), b.numpy(), bias.numpy(), res.numpy()))
    assert close16(got, want, max_ulp=1, atol=2e-4)
    got32 = hexmi.matmul(a.cuda(), b.cuda(), out_dtype=torch.float32, bias=bias.float().cuda(),
                         residual=res.float().cuda()).cpu()
    want32 = torch.from_numpy(oracle.linear(a.numpy(), b.numpy(), bias.float().numpy(), res.float().numpy(),
                                            out_dtype=np.float32))
    assert torch.allclose(got32, want32, rtol=1e-5, atol=1e-4)
    for dtype in (torch.float32, torch.float16):
        x, y = (torch.randn(70, 48, generator=g).to(dtype) for _ in range(2))
        z = torch.randn(48, 200, generator=g).to(dtype)
        gf = hexmi.add_matmul_softmax(x.cuda(), y.cuda(), z.cuda(), fused=True).cpu()
        wf = torch.from_numpy(oracle.add_matmul_softmax(x.numpy(), y.numpy(), z.numpy()))
        if dtype == torch.float32:
            assert torch.allclose(gf, wf, rtol=1e-5, atol=1e-6)
        else:
            assert close16(gf, wf, max_ulp=1, atol=1e-5)
