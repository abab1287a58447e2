"""GPU parity of quantized_matmul for the compute dtypes and code widths
outside the bf16 2/4-bit kernels (lisaq_quantized_matmul_typed): f16 and f32
with 2/4/8-bit codes, bf16 with 8-bit codes, on both sides of the matvec /
matmul split, against the oracle's typed restatements (oracle.qmv_typed,
oracle.qmm_typed).  Tolerances are per output dtype: one rounding of the
output plus f32 summation-order differences."""
import numpy as np
import pytest

from lisa_amd import ops
from lisa_amd.synth import bf16_bits_to_f32, np_linear
from tests._util import to_dev_u32

pytestmark = pytest.mark.gpu

# (atol, rtol) per output dtype
TOL = {"bf16": (2e-2, 1e-2), "f16": (2e-3, 2e-3), "f32": (1e-4, 1e-5)}


def _tensor(a, dtype, dev):
    import torch

    t = torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(dev)
    return t.to({"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype])


def _close(got, ref, dtype, what):
    atol, rtol = TOL[dtype]
    err = np.abs(got - ref)
    bound = atol + rtol * np.abs(ref)
    assert (err <= bound).all(), f"{what}: {int((err > bound).sum())} outside, max err {err.max():.3g}"


@pytest.mark.parametrize("dtype,bits", [("f16", 2), ("f16", 4), ("f16", 8), ("f32", 2), ("f32", 4), ("f32", 8),
                                        ("bf16", 8)])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("M", [1, 5, 40, 130])
def test_quantized_matmul_typed(dev, oracle, dtype, bits, gs, M):
    import torch

    rng = np.random.default_rng(M * 100 + bits * 10 + gs)
    N, K = 200, 384
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits < 8 else 0.002)
    # values of the compute dtype: round once through it on the host
    sf = oracle._round_to(bf16_bits_to_f32(s), dtype)
    bf = oracle._round_to(bf16_bits_to_f32(b), dtype)
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), dtype)
    y = ops.quantized_matmul(_tensor(xf, dtype, dev), to_dev_u32(w, dev), _tensor(sf, dtype, dev),
                             _tensor(bf, dtype, dev), True, gs, bits)
    assert y.dtype == _tensor(xf, dtype, dev).dtype
    got = y.float().cpu().numpy()
    if M < ops.qmv_batch_limit(K, N):
        ref = oracle.qmv_typed(xf, w, sf, bf, gs, bits)
    else:
        ref = oracle.qmm_typed(xf, w, sf, bf, gs, bits, dtype)
    _close(got, ref, dtype, f"{dtype} bits={bits} gs={gs} M={M}")
    torch.cuda.synchronize()


def test_promotion_bf16_x_f32_scales(dev, oracle):
    """x in bf16 with f32 scales/biases computes in f32 (AO:398-404) and
    returns f32."""
    import torch

    rng = np.random.default_rng(3)
    N, K, gs, bits = 64, 256, 64, 4
    w, s, b = np_linear(rng, N, K, bits, gs)
    x = oracle._round_to(rng.standard_normal((2, K)).astype(np.float32), "bf16")
    sf, bf = bf16_bits_to_f32(s), bf16_bits_to_f32(b)
    y = ops.quantized_matmul(_tensor(x, "bf16", dev), to_dev_u32(w, dev), _tensor(sf, "f32", dev),
                             _tensor(bf, "f32", dev), True, gs, bits)
    assert y.dtype == torch.float32
    _close(y.cpu().numpy(), oracle.qmv_typed(x, w, sf, bf, gs, bits), "f32", "promoted")


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("M", [1, 3, 64])
def test_quantized_matmul_typed_long_k(dev, oracle, dtype, M):
    """K = 5120: the matvec's lanes take several 32-code chunks each (K/32 =
    160 chunks over 64 lanes; f16 with three rows: the dot-instruction
    matvec) and the matmul's K loop runs 80 steps over 16 column tiles."""
    import torch

    rng = np.random.default_rng(5120 + M)
    N, K, gs, bits = 1000, 5120, 64, 4
    w, s, b = np_linear(rng, N, K, bits, gs)
    sf = oracle._round_to(bf16_bits_to_f32(s), dtype)
    bf = oracle._round_to(bf16_bits_to_f32(b), dtype)
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), dtype)
    y = ops.quantized_matmul(_tensor(xf, dtype, dev), to_dev_u32(w, dev), _tensor(sf, dtype, dev),
                             _tensor(bf, dtype, dev), True, gs, bits)
    got = y.float().cpu().numpy()
    assert (M < ops.qmv_batch_limit(K, N)) == (M < 64)  # both sides of the split
    if M < 64:
        ref = oracle.qmv_typed(xf, w, sf, bf, gs, bits)
    else:
        ref = oracle.qmm_typed(xf, w, sf, bf, gs, bits, dtype)
    _close(got, ref, dtype, f"{dtype} K={K} M={M}")
    torch.cuda.synchronize()


@pytest.mark.parametrize("K", [256, 320])
@pytest.mark.parametrize("dtype,bits", [("f16", 4), ("bf16", 8), ("f16", 2)])
def test_quantized_matmul_typed_wide_tiles(dev, oracle, dtype, bits, K):
    """M, N ragged and large: rows of an odd number of groups (K = 320) take the matrix-core tiles of 128 x 128 (at
    least 512 of them: 16 x 33 here), the others the bf16 matmul's kernel; against the oracle's matmul semantics."""
    import torch

    rng = np.random.default_rng(2000 + bits)
    M, N, gs = 2000, 4200, 64
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits < 8 else 0.002)
    sf = oracle._round_to(bf16_bits_to_f32(s), dtype)
    bf = oracle._round_to(bf16_bits_to_f32(b), dtype)
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), dtype)
    y = ops._mm_typed(_tensor(xf, dtype, dev), to_dev_u32(w, dev), _tensor(sf, dtype, dev), _tensor(bf, dtype, dev),
                      True, gs, bits, _tensor(xf[:1], dtype, dev).dtype)
    got = y.float().cpu().numpy()
    _close(got, oracle.qmm_typed(xf, w, sf, bf, gs, bits, dtype), dtype, f"{dtype} bits={bits} wide tiles")
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype,bits", [("f16", 4), ("f16", 2), ("f16", 8), ("bf16", 8)])
@pytest.mark.parametrize("M,N,K,gs", [
    (25, 8, 2176, 64),       # the matmul's first row count, one 8-column tile edge, 34 K-steps (34 groups a row)
    (33, 777, 64, 32),       # one K-step, odd N (single stores)
    (130, 300, 1024, 128),   # two row tiles, N a multiple of 4 only; split over K
    (257, 1000, 4608, 64),   # rows past 256, split over K
    (2100, 8200, 64, 32),    # one K-step, too many tiles for the 64 x 64 ones
    (700, 4100, 512, 64),    # several column tiles, the last partial
    (700, 12288, 128, 64),   # 4 x 48 tiles of 192 rows
    (1300, 12288, 1152, 64), # more than one round of tiles: 256-row tiles with the last round split (2 and 4 bits)
])
def test_typed_matmul_matrix_core_tiles(dev, oracle, dtype, bits, M, N, K, gs):
    """The 16-bit typed matmuls on the bf16 matmul's kernel: every tile height and split, at the edges of tiles,
    against float64 products of the weights rounded to the compute dtype; the same bits on a repeat."""
    import torch

    rng = np.random.default_rng(M + N + K + bits)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits < 8 else 0.002)
    sf = oracle._round_to(bf16_bits_to_f32(s), dtype)
    bf = oracle._round_to(bf16_bits_to_f32(b), dtype)
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), dtype)
    args = (_tensor(xf, dtype, dev), to_dev_u32(w, dev), _tensor(sf, dtype, dev), _tensor(bf, dtype, dev))
    assert M >= ops.qmv_batch_limit(K, N)
    run = lambda: ops._mm_typed(*args, True, gs, bits, args[0].dtype)
    got = run()
    q = np.stack([(w >> np.uint32(bits * j)) & np.uint32(2**bits - 1) for j in range(32 // bits)], -1).reshape(N, K)
    wd = oracle._round_to(np.repeat(sf, gs, 1) * q.astype(np.float32) + np.repeat(bf, gs, 1), dtype)
    rows = np.unique(np.concatenate([np.arange(min(M, 5)), rng.integers(0, M, 40), [M - 1]]))
    ref = xf[rows].astype(np.float64) @ wd.astype(np.float64).T
    _close(got.float().cpu().numpy()[rows], ref, dtype, f"{dtype} bits={bits} {M}x{N}x{K}")
    for _ in range(2):
        assert torch.equal(got, run())


@pytest.mark.parametrize("dtype,bits", [("bf16", 4), ("bf16", 2), ("bf16", 8), ("f16", 4), ("f16", 2), ("f16", 8)])
@pytest.mark.parametrize("M,N,K,gs", [
    (33, 8, 128, 64),        # one chunk, a part of a column group
    (34, 40, 192, 32),       # a chunk that ends partway (three K-steps of 64), 6 groups a row
    (32, 2051, 1408, 64),    # all 32 rows, odd N (single stores), 22 K-steps: parts ending partway
    (64, 260, 4224, 64),     # all 64 rows, K parts, 66 groups a row (scale blocks past the last row's end)
    (40, 5120, 2560, 128),   # 20 scale groups of 128 a row
    (13, 4100, 5120, 64),    # the fewest rows, several column tiles
    (17, 33000, 512, 64),    # more column tiles than half the compute units: no split
    (13, 4100, 5120, 32),    # at most 32 rows, groups of 32: every chunk starts a scale block, K parts
    (25, 100, 2176, 32),     # the same with a chunk that ends partway
    (32, 300, 2304, 128),    # at most 32 rows, groups of 128 (18 a row)
    (33, 8, 640, 64),        # past 32 rows: five chunks, a part of a column group
    (64, 40, 704, 32),       # a chunk that ends partway (eleven K-steps), 22 groups a row
    (40, 300, 512, 64),      # the last K on 64 x 64 tiles (typed)
    (130, 4100, 768, 64),    # (past 64 rows) 195 tiles of 64 x 64 at their last K but one
    (128, 3072, 1024, 128),  # 96 of them at their last K
])
def test_few_rows_matmul(dev, oracle, dtype, bits, M, N, K, gs):
    """The matmul of at most 64 rows at the edges of its chunks, column groups, scale blocks and K parts, against
    float64 products of the rounded weights; the same bits on a repeat."""
    import torch

    rng = np.random.default_rng(M + N + K + bits)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits < 8 else 0.002)
    sf = oracle._round_to(bf16_bits_to_f32(s), dtype)
    bf = oracle._round_to(bf16_bits_to_f32(b), dtype)
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), dtype)
    args = (_tensor(xf, dtype, dev), to_dev_u32(w, dev), _tensor(sf, dtype, dev), _tensor(bf, dtype, dev))
    assert M >= ops.qmv_batch_limit(K, N)
    run = lambda: ops.quantized_matmul(*args, True, gs, bits)
    got = run()
    q = np.stack([(w >> np.uint32(bits * j)) & np.uint32(2**bits - 1) for j in range(32 // bits)], -1).reshape(N, K)
    wd = oracle._round_to(np.repeat(sf, gs, 1) * q.astype(np.float32) + np.repeat(bf, gs, 1), dtype)
    ref = xf.astype(np.float64) @ wd.astype(np.float64).T
    _close(got.float().cpu().numpy(), ref, dtype, f"{dtype} bits={bits} {M}x{N}x{K}")
    assert torch.equal(got, run())


@pytest.mark.parametrize("dtype,bits", [("bf16", 8), ("f16", 2), ("f16", 4), ("f16", 8), ("f32", 2), ("f32", 4), ("f32", 8)])
@pytest.mark.parametrize("M,N,K,gs", [
    (1, 3, 32, 32),         # one piece (two of 8 bits), fewer rows than a wave takes
    (1, 4097, 2080, 32),    # two rows of W per wave, a tail row, 65 pieces of 32 (one past a wave's pass)
    (2, 70, 4224, 128),     # two rows of x, few workgroups
    (3, 4100, 2560, 64),    # a group of two and one, four rows of W per wave
    (5, 17408, 2560, 64),   # (8 bits: groups of four rows of x, one in the second)
    (7, 500, 17408, 64),    # long rows: one row of x per workgroup
    (12, 1001, 1024, 64),   # the most rows here, N odd
])
def test_typed_matvec_rows(dev, oracle, dtype, bits, M, N, K, gs):
    """The matvec with x in LDS at the edges of its pieces, row groups and rows per wave, against the oracle; the
    same rows from an x that is not 16-byte aligned (a wave per output row) within the output's rounding of them."""
    import torch

    rng = np.random.default_rng(M * 31 + N + K + bits)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits < 8 else 0.002)
    sf = oracle._round_to(bf16_bits_to_f32(s), dtype)
    bf = oracle._round_to(bf16_bits_to_f32(b), dtype)
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), dtype)
    assert M < ops.qmv_batch_limit(K, N)
    x, wd, sd, bd = _tensor(xf, dtype, dev), to_dev_u32(w, dev), _tensor(sf, dtype, dev), _tensor(bf, dtype, dev)
    ref = oracle.qmv_typed(xf, w, sf, bf, gs, bits)
    _close(ops.quantized_matmul(x, wd, sd, bd, True, gs, bits).float().cpu().numpy(), ref, dtype, "rows kernel")
    off = torch.empty(M * K + 1, dtype=x.dtype, device=dev)[1:].view(M, K)
    off.copy_(x)
    _close(ops.quantized_matmul(off, wd, sd, bd, True, gs, bits).float().cpu().numpy(), ref, dtype, "unaligned x")


@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("M,N,K,gs", [
    (33, 5, 32, 32),         # one K-step, a quarter of a 128-value step; fewer columns than a tile
    (70, 100, 416, 32),      # 32 x 32 tiles, row and column tails, K ends inside a step
    (25, 2100, 3072, 128),   # the fewest rows
    (1500, 1470, 320, 64),   # 64 x 64 tiles (24 x 23), row and column tails
])
def test_f32_matmul_matrix_cores(dev, oracle, bits, M, N, K, gs):
    """The f32 matmul on the matrix cores: relative error of the whole result against float64 at most that of f32
    sums of K products (K 2^-24 bounds every order; the square root is typical)."""
    import torch

    rng = np.random.default_rng(M + N + K + bits)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits < 8 else 0.002)
    sf, bf = bf16_bits_to_f32(s), bf16_bits_to_f32(b)
    xf = rng.standard_normal((M, K)).astype(np.float32)
    assert M >= ops.qmv_batch_limit(K, N)
    y = ops.quantized_matmul(_tensor(xf, "f32", dev), to_dev_u32(w, dev), _tensor(sf, "f32", dev),
                             _tensor(bf, "f32", dev), True, gs, bits).cpu().numpy()
    q = np.stack([(w >> np.uint32(bits * j)) & np.uint32(2**bits - 1) for j in range(32 // bits)], -1).reshape(N, K)
    wd = np.repeat(sf, gs, 1).astype(np.float64) * q + np.repeat(bf, gs, 1)
    ref = xf.astype(np.float64) @ wd.T
    bound = 2.0**-24 * (K * np.abs(xf).astype(np.float64) @ np.abs(wd).T / np.sqrt(K) + np.abs(ref))
    assert (np.abs(y - ref) <= 4 * bound).all()
    assert np.linalg.norm(y - ref) <= 1e-6 * np.linalg.norm(ref) * max(1.0, np.sqrt(K / 1024))


@pytest.mark.parametrize("M,N,K,gs", [(25, 264, 2176, 64), (40, 100, 640, 64), (150, 300, 1280, 128), (700, 264, 1280, 32)])
def test_bf16_8bit_matmul_scale_range(dev, oracle, M, N, K, gs):
    """bf16 scales over their whole range (2^104 and more among them) with 8-bit codes: every weight is
    bf16(fma(scale, q, bias)), finite wherever that is, for code 0 too."""
    import torch

    rng = np.random.default_rng(M + N + K)
    w, s, b = np_linear(rng, N, K, 8, gs, s_std=0.002)
    w[:, ::3] &= np.uint32(0xFFFF00FF)  # zeros among the codes
    sf, bf = bf16_bits_to_f32(s).copy(), bf16_bits_to_f32(b)
    sf[3], sf[N // 2], sf[N - 1] = 2.0**104, -(2.0**108), 1.5 * 2.0**106
    sf[5], bf = 2.0**-120, bf.copy()
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), "bf16")
    assert M >= ops.qmv_batch_limit(K, N)
    y = ops.quantized_matmul(_tensor(xf, "bf16", dev), to_dev_u32(w, dev), _tensor(sf, "bf16", dev),
                             _tensor(bf, "bf16", dev), True, gs, 8).float().cpu().numpy().astype(np.float64)
    ref = oracle.qmm_typed(xf, w, sf, bf, gs, 8, "bf16")
    # one rounding to bf16 (2^-9 relative) and f32 sums of K products (K 2^-24 of the sum of magnitudes)
    q = oracle.unpack(w, K, 8).astype(np.float64)
    wt = np.abs(np.repeat(sf.astype(np.float64), gs, 1) * q + np.repeat(bf.astype(np.float64), gs, 1))
    bound = 2.0**-8 * np.abs(ref) + K * 2.0**-24 * (np.abs(xf).astype(np.float64) @ wt.T)
    assert np.isfinite(y).all() and (np.abs(y - ref) <= bound).all()


@pytest.mark.parametrize("dtype,bits", [("f32", 2), ("f32", 4), ("f32", 8), ("f16", 2), ("f16", 4), ("f16", 8), ("bf16", 8)])
@pytest.mark.parametrize("M,N,K,gs", [(40, 70, 96, 32), (130, 200, 384, 64), (65, 1, 128, 128)])
def test_typed_matmul_unaligned_x(dev, oracle, dtype, bits, M, N, K, gs):
    """The typed matmul with x off 16 bytes (64 x 64 FMA tiles; row, column and K tails), and with the other tensors
    off the alignment of the faster kernels, against the oracle."""
    import torch

    rng = np.random.default_rng(M + N + K + bits)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits < 8 else 0.002)
    sf = oracle._round_to(bf16_bits_to_f32(s), dtype)
    bf = oracle._round_to(bf16_bits_to_f32(b), dtype)
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), dtype)
    assert M >= ops.qmv_batch_limit(K, N)
    ref = oracle.qmm_typed(xf, w, sf, bf, gs, bits, dtype)

    def off(t):  # the same values one element past a 16-byte boundary
        o = torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)[1:].view(t.shape)
        return o.copy_(t)

    x, wd, sd, bd = _tensor(xf, dtype, dev), to_dev_u32(w, dev), _tensor(sf, dtype, dev), _tensor(bf, dtype, dev)
    run = lambda *a: ops.quantized_matmul(*a, True, gs, bits).float().cpu().numpy()
    _close(run(off(x), wd, sd, bd), ref, dtype, "unaligned x")
    _close(run(x, off(wd), sd, bd), ref, dtype, "unaligned w")
    _close(run(x, wd, off(sd), off(bd)), ref, dtype, "unaligned scales")


@pytest.mark.parametrize("scale", [1.0, 2.0**-21])
@pytest.mark.parametrize("N,K,gs", [(1, 32, 32), (7, 128, 128), (4095, 2080, 32), (4096, 1024, 64), (2560, 9728, 128)])
def test_f16_one_row_dot(dev, oracle, N, K, gs, scale):
    """One f16 row and 4-bit codes of at most 4096 rows (dot instructions) at the edges of its pieces and rows, against
    the oracle; scale 2^-21: values of x below the smallest normal f16, which count like any other."""
    rng = np.random.default_rng(N + K)
    w, s, b = np_linear(rng, N, K, 4, gs)
    up = np.float32(2.0**10 if scale < 1 else 1.0)
    sf = oracle._round_to(bf16_bits_to_f32(s) * up, "f16")
    bf = oracle._round_to(bf16_bits_to_f32(b) * up, "f16")
    xf = oracle._round_to(rng.standard_normal((1, K)).astype(np.float32) * np.float32(scale), "f16")
    y = ops.quantized_matmul(_tensor(xf, "f16", dev), to_dev_u32(w, dev), _tensor(sf, "f16", dev),
                             _tensor(bf, "f16", dev), True, gs, 4).float().cpu().numpy()
    ref = oracle.qmv_typed(xf, w, sf, bf, gs, 4)
    # one rounding to f16 (2^-11 relative, 2^-25 below its normal range) and f32 sums
    mag = oracle.qmv_typed(np.abs(xf), w, np.abs(sf), np.abs(bf), gs, 4)
    assert (np.abs(y - ref) <= 2.0**-10 * np.abs(ref) + 2.0**-24 + K * 2.0**-24 * mag).all()


@pytest.mark.parametrize("dtype,bits", [("bf16", 8), ("f16", 2), ("f16", 4), ("f16", 8), ("f32", 4), ("f32", 8)])
@pytest.mark.parametrize("M,N,K,gs", [
    (2, 9, 2048, 64),        # pairs of rows of x, one row of W per wave, most workgroups' waves without rows
    (2, 3001, 1056, 32),     # a wave's stream of several rows, its last piece's lanes partly past the row
    (4, 700, 17408, 64),     # 16 bits: pairs of long rows (80 KB); f32: one at a time, one row of W per wave
    (3, 2600, 12288, 128),   # three long rows one at a time, four rows of W
    (1, 33000, 96, 32),      # short rows: every step ends one, more rows than the chip holds at once
    (12, 33000, 64, 64),
])
def test_typed_matvec_streams(dev, oracle, dtype, bits, M, N, K, gs):
    """The matvec's streams of rows: steps that cross from one row to the next, clamped ends, long and short rows."""
    rng = np.random.default_rng(M + N + K + bits)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits < 8 else 0.002)
    sf = oracle._round_to(bf16_bits_to_f32(s), dtype)
    bf = oracle._round_to(bf16_bits_to_f32(b), dtype)
    xf = oracle._round_to(rng.standard_normal((M, K)).astype(np.float32), dtype)
    assert M < ops.qmv_batch_limit(K, N)
    y = ops.quantized_matmul(_tensor(xf, dtype, dev), to_dev_u32(w, dev), _tensor(sf, dtype, dev),
                             _tensor(bf, dtype, dev), True, gs, bits).float().cpu().numpy()
    q = oracle.unpack(w, K, bits).astype(np.float64)
    wd = np.repeat(sf.astype(np.float64), gs, 1) * q + np.repeat(bf.astype(np.float64), gs, 1)
    _close(y, xf.astype(np.float64) @ wd.T, dtype, f"{dtype} bits={bits} {M}x{N}x{K}")
