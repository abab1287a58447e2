"""GPU parity of quantized_matmul (matvec and matmul paths), dequantize and
quantize against the CPU oracle, through the C ABI (lisa_amd.ops -> liblisaq).

Tolerance for outputs: |got - ref| <= 2e-2 + 1e-2*|ref| per element (the
north-star bound; see tests/_util.py).  Integer work (codes, quantize output,
dequantize bits) is compared bit-exactly."""
import numpy as np
import pytest

from lisa_amd import ops
from lisa_amd.synth import bf16_bits_to_f32, np_linear, np_x
from tests._util import assert_close_bf16, from_dev_bf16, to_dev, to_dev_bf16, to_dev_u32

pytestmark = pytest.mark.gpu


def _run(fn, dev, x, w, s, b, gs, bits):
    y = fn(to_dev_bf16(x, dev), to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev),
           group_size=gs, bits=bits)
    return from_dev_bf16(y)


QMV_CASES = [
    # (M, N, K, bits, gs)
    (1, 3072, 1024, 4, 64),      # configs[0]
    (1, 256, 512, 4, 64),
    (3, 64, 512, 4, 64),         # array_ops.rs:650-710 shape
    (1, 100, 512, 4, 64),        # N tail (not a multiple of 32)
    (5, 77, 320, 4, 64),         # K/gs = 5 groups (U = 1 path), N tail
    (1, 9728, 2560, 4, 64),      # configs[1] up
    (2, 9728, 2560, 4, 64),
    (4, 9728, 2560, 4, 64),
    (8, 9728, 2560, 4, 64),
    (1, 2560, 9728, 4, 64),      # configs[1] down
    (2, 2560, 9728, 4, 64),
    (8, 2560, 9728, 4, 64),      # (split over K)
    (4, 2560, 9728, 4, 64),
    (1, 512, 1024, 2, 64),
    (8, 640, 2048, 2, 64),
    (1, 256, 1024, 4, 32),
    (3, 256, 1024, 4, 128),
    (1, 256, 1024, 2, 32),
    (2, 256, 1024, 2, 128),
    (12, 1024, 1024, 4, 64),     # MQ = 2
    (20, 512, 2048, 4, 64),      # MQ = 3
    (32, 512, 1024, 4, 64),      # MQ = 4 (forced qmv)
]


@pytest.mark.parametrize("M,N,K,bits,gs", QMV_CASES)
def test_qmv_parity(dev, oracle, M, N, K, bits, gs):
    rng = np.random.default_rng(M * 7 + N + K + bits + gs)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits == 4 else 0.05,
                        b_std=0.01 if bits == 4 else 0.02)
    x = np_x(rng, M, K)
    ref = oracle.qmv(x, w, s, b, gs, bits)
    got = _run(ops.qmv, dev, x, w, s, b, gs, bits)
    assert_close_bf16(got, ref, what=f"qmv M={M} N={N} K={K} bits={bits} gs={gs}")
    if M < ops.qmv_batch_limit(K, N):
        got2 = _run(ops.quantized_matmul, dev, x, w, s, b, gs, bits)
        assert np.array_equal(got, got2)


@pytest.mark.parametrize("kernel", ["w", "p", "s", "d", "t", "16", "32"])
@pytest.mark.parametrize("M,N,K,bits,gs", [
    (1, 100, 1024, 4, 64),      # fewer rows than waves (persistent kernel), J = 1
    (1, 4099, 2560, 4, 64),     # J = 2, N tail
    (1, 17408, 5120, 4, 64),    # north star, J = 3
    (1, 3000, 5120, 2, 64),
    (1, 1000, 4096, 4, 32),
    (1, 1000, 6144, 4, 128),
    (1, 777, 2048, 2, 128),
    (2, 3001, 5120, 4, 64),
    (2, 640, 2048, 2, 64),
    (2, 4097, 2560, 4, 32),     # four rows a step (K = 2560), ragged last step, two rows of x
    (1, 1001, 5120, 4, 128),    # two rows a step (K = 5120), odd N
])
def test_qmv_every_kernel(dev, oracle, force_path, kernel, M, N, K, bits, gs):
    """Each matvec kernel (forced through LISAQ_QMV_KERNEL; a shape it does not
    take falls through to the next one) against the oracle."""
    force_path("LISAQ_QMV_KERNEL", kernel)
    rng = np.random.default_rng(N * 3 + K + bits + gs + M)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits == 4 else 0.05,
                        b_std=0.01 if bits == 4 else 0.02)
    x = np_x(rng, M, K)
    ref = oracle.qmv(x, w, s, b, gs, bits)
    got = _run(ops.qmv, dev, x, w, s, b, gs, bits)
    assert_close_bf16(got, ref, what=f"qmv[{kernel}] M={M} N={N} K={K} bits={bits} gs={gs}")


@pytest.mark.parametrize("M,N,K,bits,gs", [
    (33, 256, 512, 4, 64), (64, 256, 1024, 4, 64), (130, 300, 512, 4, 64), (128, 512, 2048, 2, 64),
    (96, 256, 1024, 4, 32), (50, 256, 1024, 4, 128), (200, 1024, 768, 4, 64), (13, 256, 4096, 2, 128),
])
def test_qmm_parity(dev, oracle, M, N, K, bits, gs):
    rng = np.random.default_rng(M + N + K + bits * 3 + gs)
    w, s, b = np_linear(rng, N, K, bits, gs)
    x = np_x(rng, M, K)
    ref = oracle.qmm(x, w, s, b, gs, bits)
    got = _run(ops.qmm, dev, x, w, s, b, gs, bits)
    assert_close_bf16(got, ref, what=f"qmm M={M} N={N} K={K} bits={bits} gs={gs}")
    if M >= ops.qmv_batch_limit(K, N):
        got2 = _run(ops.quantized_matmul, dev, x, w, s, b, gs, bits)
        assert np.array_equal(got, got2)


@pytest.mark.parametrize("split", ["1", "2", "3", "7"])
def test_qmm_split_k(dev, oracle, force_path, split):
    """The matmul split over K (f32 partials in the workspace, summed in split
    order): every split count against the oracle, and the same bits on a repeat."""
    force_path("LISAQ_QMM_SPLIT", split)
    rng = np.random.default_rng(77)
    M, N, K = 70, 300, 1024
    w, s, b = np_linear(rng, N, K, 4, 64)
    x = np_x(rng, M, K)
    ref = oracle.qmm(x, w, s, b, 64, 4)
    got = _run(ops.qmm, dev, x, w, s, b, 64, 4)
    assert_close_bf16(got, ref, what=f"qmm split={split}")
    assert np.array_equal(_run(ops.qmm, dev, x, w, s, b, 64, 4), got)


@pytest.mark.parametrize("M,N,K,bits", [(128, 17408, 5120, 4), (128, 5120, 17408, 4), (512, 17408, 5120, 4),
                                        (512, 5120, 17408, 4), (2048, 17408, 5120, 4), (2048, 5120, 17408, 4),
                                        (512, 17408, 5120, 2), (512, 5120, 17408, 2)])
def test_qmm_prefill_shapes_sampled_rows(dev, oracle, M, N, K, bits):
    """configs[2]/[3] prefill shapes; the oracle checks 8 sampled rows (every column)."""
    import torch

    rng = np.random.default_rng(M + N)
    w, s, b = np_linear(rng, N, K, bits, 64, s_std=0.02 if bits == 4 else 0.05, b_std=0.01 if bits == 4 else 0.02)
    x = np_x(rng, M, K)
    y = ops.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev),
                             group_size=64, bits=bits)
    torch.cuda.synchronize()
    rows = np.sort(rng.choice(M, 8, replace=False))
    rows[0], rows[-1] = 0, M - 1
    ref = oracle.qmm(x[rows], w, s, b, 64, bits)
    got = from_dev_bf16(y)[rows]
    assert_close_bf16(got, ref, what=f"prefill M={M} N={N} K={K}")


@pytest.mark.parametrize("M", [4, 8])
def test_qmv_split_k_and_its_fallback(dev, oracle, force_path, M):
    """Few row tiles (N = 2560): the streaming matvec splits K over workgroups when the workspace holds
    the parts; given none, the same call runs unsplit. Both against the oracle, and close to each other."""
    import torch

    force_path("LISAQ_QMV_KERNEL", "t")

    from lisa_amd import _lib

    N, K, gs, bits = 2560, 9728, 64, 4
    rng = np.random.default_rng(2560 + M)
    w, s, b = np_linear(rng, N, K, bits, gs)
    x = np_x(rng, M, K)
    ref = oracle.qmv(x, w, s, b, gs, bits)
    lib = _lib.load()
    need = lib.lisaq_quantized_matmul_workspace(M, N, K, gs, bits)
    assert need > 0  # the split is on for this shape
    xd, wd, sd, bd = to_dev_bf16(x, dev), to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev)
    outs = []
    for with_ws in (True, False):
        y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        ws = ops.workspace(dev, need) if with_ws else None
        _lib.call("lisaq_quantized_matmul", torch.cuda.current_stream().cuda_stream, xd.data_ptr(), wd.data_ptr(),
                  sd.data_ptr(), bd.data_ptr(), y.data_ptr(), M, N, K, 1, gs, bits,
                  ws.data_ptr() if with_ws else None, need if with_ws else 0)
        got = from_dev_bf16(y)
        assert_close_bf16(got, ref, what=f"qmv M={M} {'split' if with_ws else 'unsplit (no workspace)'}")
        if with_ws:  # parts summed in part order: the same bits on a repeat
            y2 = torch.empty_like(y)
            _lib.call("lisaq_quantized_matmul", torch.cuda.current_stream().cuda_stream, xd.data_ptr(),
                      wd.data_ptr(), sd.data_ptr(), bd.data_ptr(), y2.data_ptr(), M, N, K, 1, gs, bits,
                      ws.data_ptr(), need)
            assert np.array_equal(from_dev_bf16(y2), got)
        outs.append(bf16_bits_to_f32(got))
    # same tolerance between the two as against the oracle (they differ in summation order only)
    assert (np.abs(outs[0] - outs[1]) <= 2e-2 + 1e-2 * np.abs(outs[1])).all()


@pytest.mark.parametrize("bits", [2, 4])
def test_north_star_qmv_shape(dev, oracle, bits):
    rng = np.random.default_rng(17408 + bits)
    N, K = 17408, 5120
    w, s, b = np_linear(rng, N, K, bits, 64, s_std=0.02 if bits == 4 else 0.05, b_std=0.01 if bits == 4 else 0.02)
    for M in (1, 5, 8):  # 5 and 8: two 16-row tiles per workgroup share the staged x
        x = np_x(rng, M, K)
        ref = oracle.qmv(x, w, s, b, 64, bits)
        got = _run(ops.quantized_matmul, dev, x, w, s, b, 64, bits)
        assert_close_bf16(got, ref, what=f"north-star qmv M={M} bits={bits}")
        assert np.array_equal(_run(ops.quantized_matmul, dev, x, w, s, b, 64, bits), got)


@pytest.mark.parametrize("bits", [2, 4])
def test_down_shape_qmv(dev, oracle, bits):
    """configs[3] (2-bit) and configs[2] (4-bit) down shape at decode: N = 5120, K = 17408 (272 groups a
    row), M = 1 over every row, with the config's scale/bias distributions."""
    rng = np.random.default_rng(5120 + bits)
    N, K = 5120, 17408
    w, s, b = np_linear(rng, N, K, bits, 64, s_std=0.02 if bits == 4 else 0.05, b_std=0.01 if bits == 4 else 0.02)
    for M in (1, 4):
        x = np_x(rng, M, K)
        ref = oracle.qmv(x, w, s, b, 64, bits)
        got = _run(ops.quantized_matmul, dev, x, w, s, b, 64, bits)
        assert_close_bf16(got, ref, what=f"down-shape qmv M={M} bits={bits}")


@pytest.mark.parametrize("N,K,gs", [(17408, 5120, 64), (9728, 2560, 64), (2560, 9728, 64), (5120, 17408, 64), (5120, 17408, 128), (1000, 1024, 64),
                                    (777, 2048, 128), (5, 512, 64)])
def test_one_stream_rows_bitwise(dev, oracle, force_path, N, K, gs):
    """The one-stream matvec (1..8 rows of x on one pass over W): every row of an M-row call is bitwise
    equal to the same kernel's one-row call (the matrix-core column of a row never mixes other rows), for
    every M; every row within tolerance of the oracle.  Eight rows at K = 9728 and four at K = 17408
    stage x in two passes over K, eight at K = 17408 in four (all of it does not fit the LDS): bitwise
    equal to the one-pass one-row call as well."""
    force_path("LISAQ_QMV_KERNEL", "w")
    rng = np.random.default_rng(N + K + gs)
    w, s, b = np_linear(rng, N, K, 4, gs)
    x = np_x(rng, 8, K)
    ref = oracle.qmv(x, w, s, b, gs, 4)
    ones = np.concatenate([_run(ops.qmv, dev, x[r:r + 1], w, s, b, gs, 4) for r in range(8)])
    assert_close_bf16(ones, ref, what=f"one-stream M=1 N={N} K={K}")
    for M in range(2, 9):
        got = _run(ops.qmv, dev, x[:M], w, s, b, gs, 4)
        assert_close_bf16(got, ref[:M], what=f"one-stream M={M} N={N} K={K}")
        if _one_stream_fits(M, N, K):
            assert np.array_equal(got, ones[:M]), (N, K, M)


def _one_stream_fits(M, N, K):
    """LDS bytes of the one-stream matvec at its default grid (256 workgroups) within 160 KB, with x
    staged in one pass over K, or (four or eight staged rows) two or four: staged rows of x (each padded by
    256 bytes), block sums, per-unit partials (qmvw.hip, qmvw_lds)."""
    MP = 1 if M == 1 else 2 if M == 2 else 4 if M <= 4 else 8
    RP = min(MP, 4)
    T = (-(-N // 256) + 15) // 16
    segs = K // 512
    for passes in ((1, 2, 4) if MP >= 4 else (1,)):
        KP = -(-segs // passes) * 512
        if MP * (2 * KP + 256) + (K // 64) * MP * 4 + T * segs * 64 * RP * 4 <= 160 * 1024:
            return True
    return False


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("M", [2, 3, 4, 5, 6, 8])
def test_serial_rows_bitwise_equal_to_single_rows(dev, force_path, bits, M):
    """array_ops.rs:650-710 / jit::affine_verify_qmm (matmul.rs:579-664): batched rows == independent
    M=1 calls, bitwise.  Eight or four rows at a time run on one weight stream (fours where eight rows
    of x do not fit the LDS: K = 9728), the rest in a pair and/or a single row; long rows (K = 17408) in
    pairs; the pair path forced for comparison."""
    rng = np.random.default_rng(99 + bits + 10 * M)
    for N, K in ((64, 512), (2560, 9728), (9728, 2560), (17408, 5120), (1000, 17408), (77, 2048)):
        w, s, b = np_linear(rng, N, K, bits, 64)
        x = np_x(rng, M, K)
        batched = _run(ops.quantized_matmul_serial_rows, dev, x, w, s, b, 64, bits)
        for r in range(M):
            one = _run(ops.quantized_matmul, dev, x[r:r + 1], w, s, b, 64, bits)
            assert np.array_equal(batched[r:r + 1], one), (N, K, M, r)
        force_path("LISAQ_SERIAL_ROWS", "0")
        assert np.array_equal(_run(ops.quantized_matmul_serial_rows, dev, x, w, s, b, 64, bits), batched), (N, K, M)
        force_path("LISAQ_SERIAL_ROWS", None)


@pytest.mark.parametrize("M,N,K,bits", [(5, 100, 512, 4), (7, 33, 2560, 4), (6, 2051, 4096, 2), (5, 300, 6400, 4),
                                        (6, 40, 9728, 4), (7, 40, 9728, 2), (7, 16, 10240, 4)])
def test_serial_rows_five_to_seven_in_one_launch(dev, M, N, K, bits):
    """Five to seven verify rows in one launch of six or eight (one to five passes over K, row tails; K = 9728 and
    10240: six or fours, by what fits the LDS): every row bitwise the one-row call's."""
    rng = np.random.default_rng(M + N + K)
    w, s, b = np_linear(rng, N, K, bits, 64)
    x = np_x(rng, M, K)
    batched = _run(ops.quantized_matmul_serial_rows, dev, x, w, s, b, 64, bits)
    for r in range(M):
        one = _run(ops.quantized_matmul, dev, x[r:r + 1], w, s, b, 64, bits)
        assert np.array_equal(batched[r:r + 1], one), r


def test_repeated_calls_deterministic(dev):
    """Split-K partials are summed in slab order: identical bits every call."""
    rng = np.random.default_rng(5)
    w, s, b = np_linear(rng, 2560, 9728)
    x = np_x(rng, 4, 9728)
    first = _run(ops.quantized_matmul, dev, x, w, s, b, 64, 4)
    for _ in range(3):
        assert np.array_equal(_run(ops.quantized_matmul, dev, x, w, s, b, 64, 4), first)


@pytest.mark.parametrize("bits,gs", [(4, 64), (2, 64), (4, 32), (2, 128), (8, 64)])
def test_dequantize_bit_exact(dev, oracle, bits, gs):
    rng = np.random.default_rng(bits * gs)
    N, K = 300, 1024
    w, s, b = np_linear(rng, N, K, bits, gs)
    got = from_dev_bf16(ops.dequantize(to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev), gs, bits))
    ref = oracle.f32_to_bf16(oracle.dequantize(w, s, b, gs, bits))
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("bits", [2, 4, 8])
def test_quantize_bit_exact_f32(dev, oracle, bits):
    import torch

    from lisa_amd.synth import lcg_array

    N, K, gs = 64, 512, 64
    wf = lcg_array(0x2F1D4A73, N * K).reshape(N, K)
    wf[0, :64] = 0.0  # all-zero group
    wf[1, :64] = -np.abs(wf[1, :64]) - 0.1  # all-negative group
    wq, sc, bi = ops.quantize(to_dev(wf, dev), gs, bits)
    rq, rs, rb = oracle.quantize_f32(wf, gs, bits)
    assert np.array_equal(wq.cpu().numpy().view(np.uint32), rq)
    assert np.array_equal(sc.cpu().numpy(), rs) and np.array_equal(bi.cpu().numpy(), rb)
    # bf16 input: scales/biases rounded to bf16 like to_dtype(wdt)
    wb = torch.from_numpy(wf).to(torch.bfloat16)
    wbf = wb.float().numpy()
    wq2, sc2, bi2 = ops.quantize(wb.to(dev), gs, bits)
    rq2, rs2, rb2 = oracle.quantize_f32(wbf, gs, bits)
    assert np.array_equal(wq2.cpu().numpy().view(np.uint32), rq2)
    assert np.array_equal(from_dev_bf16(sc2), oracle.f32_to_bf16(rs2))
    assert np.array_equal(from_dev_bf16(bi2), oracle.f32_to_bf16(rb2))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bits", [2, 4, 8])
def test_quantize_edges_bit_exact(dev, oracle, dtype, bits, gs):
    """Groups that decide a code on a half step, constant, tiny (the scale's floor), huge and one-sided groups, over
    a count of 16-value chunks that ends inside a workgroup: codes, scales and biases equal the oracle's.  The same
    values with NaN and infinities among them, from an address that the wide loads cannot take, equal the aligned
    call's bits."""
    import torch

    rng = np.random.default_rng(bits * gs + len(dtype))
    N, K = 37, 3 * 128
    wf = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    wf[0:4] = np.round(rng.uniform(-7, 8, (4, K))) * 0.5  # multiples of half a step
    wf[0:4, ::gs] = 2.0**bits - 1.0
    wf[4] = 0.0
    wf[5] = 0.25
    wf[6] = -0.25
    wf[7] *= 1e-9
    wf[8] *= 1e34
    wf[9] = np.abs(wf[9]) + 0.1
    wf[10] = -np.abs(wf[10]) - 0.1
    wt = torch.from_numpy(wf).to(torch.bfloat16 if dtype == "bf16" else torch.float32)
    wq, sc, bi = ops.quantize(wt.to(dev), gs, bits)
    rq, rs, rb = oracle.quantize_f32(wt.float().numpy(), gs, bits)
    assert np.array_equal(wq.cpu().numpy().view(np.uint32), rq)
    assert torch.equal(sc.cpu(), torch.from_numpy(rs).to(wt.dtype))
    assert torch.equal(bi.cpu(), torch.from_numpy(rb).to(wt.dtype))
    wt[11, 5], wt[12, 9], wt[13, 70] = float("nan"), float("inf"), float("-inf")
    buf = torch.empty(N * K + 1, dtype=wt.dtype, device=dev)
    off = buf[1:].view(N, K)  # one element past a 16-byte boundary
    off.copy_(wt)
    for a, b in zip(ops.quantize(wt.to(dev), gs, bits), ops.quantize(off, gs, bits)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_quantize_then_matmul_smoke(dev):
    """smoke.rs:19-40 with our ops: quantize -> quantized_matmul vs dequantize -> matmul (max |d| < 0.1)."""
    import torch

    from lisa_amd.synth import lcg_array

    w = torch.from_numpy(lcg_array(42, 64 * 256).reshape(64, 256)).to(dev)
    x = torch.from_numpy(lcg_array(7, 256).reshape(1, 256)).to(dev).to(torch.bfloat16)
    wq, sc, bi = ops.quantize(w, 32, 4)
    y1 = ops.quantized_matmul(x, wq, sc.to(torch.bfloat16), bi.to(torch.bfloat16), True, 32, 4)
    wd = ops.dequantize(wq, sc.to(torch.bfloat16), bi.to(torch.bfloat16), 32, 4)
    y2 = (x.float() @ wd.float().T)
    assert (y1.float() - y2).abs().max().item() < 0.1


def test_rejections_raise(dev):
    rng = np.random.default_rng(0)
    w, s, b = np_linear(rng, 64, 128)
    x = np_x(rng, 1, 128)
    with pytest.raises(ops.LisaqError, match="biases"):
        ops.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(w, dev), to_dev_bf16(s, dev), None)
    with pytest.raises(ops.LisaqError, match="transpose"):
        ops.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev),
                             transpose=False)
    import torch
    with pytest.raises(ops.LisaqError, match="dtype"):  # (f16/f32 are supported; f64 is not)
        ops.quantized_matmul(torch.zeros(1, 128, device=dev, dtype=torch.float64), to_dev_u32(w, dev),
                             to_dev_bf16(s, dev), to_dev_bf16(b, dev))


@pytest.mark.parametrize("N,K", [(264, 5120), (1000, 9728), (17408, 5120), (16384, 4608), (5120, 5120)])
def test_qmv_addnorm(dev, oracle, N, K):
    """Residual add + RMSNorm + matvec (jit::affine_qmv_fast_addnorm, matmul.rs:315-443): the sum row
    bit-exact; the normed row within one bf16 step of the oracle (the f32 sum of squares may differ in
    its last bit from the float64 one); y bitwise equal to the matvec on the kernel's own normed row and
    within tolerance of the oracle's matvec on the oracle's normed row.  Every shape here is one launch: the
    persistent matvec (N >= 16384, K <= 6144) or the wave-rows matvec, each with the add + RMSNorm folded in."""
    import torch

    rng = np.random.default_rng(N + K)
    w, s, b = np_linear(rng, N, K, 4, 64)
    x = np_x(rng, 1, K)
    r = np_x(rng, 1, K)
    from lisa_amd.synth import f32_to_bf16_bits
    nw = f32_to_bf16_bits((1.0 + 0.1 * rng.standard_normal(K)).astype(np.float32))
    dw = (to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev))
    y, sm, nm = ops.qmv_addnorm(to_dev_bf16(x, dev), to_dev_bf16(r, dev), to_dev_bf16(nw, dev), *dw, 1e-6)
    torch.cuda.synchronize()
    s_ref, n_ref = oracle.add_rms_norm(x, r, nw, 1e-6)
    assert np.array_equal(from_dev_bf16(sm), s_ref)
    got_n = bf16_bits_to_f32(from_dev_bf16(nm))
    ref_n = bf16_bits_to_f32(n_ref)
    step = np.abs(ref_n) * 2.0**-7 + 1e-30
    assert (np.abs(got_n - ref_n) <= step).all()
    assert (got_n != ref_n).mean() < 0.01
    chain = from_dev_bf16(ops.quantized_matmul(nm, *dw, True, 64, 4))
    assert np.array_equal(from_dev_bf16(y), chain)
    assert_close_bf16(from_dev_bf16(y), oracle.qmv(n_ref, w, s, b, 64, 4), what=f"qmv_addnorm N={N} K={K}")
    _, _, none = ops.qmv_addnorm(to_dev_bf16(x, dev), to_dev_bf16(r, dev), to_dev_bf16(nw, dev), *dw, 1e-6,
                                 write_norm=False)
    assert none is None


@pytest.mark.parametrize("M,N,K,bits", [(1, 17408, 5120, 4), (2, 17408, 5120, 4), (1, 9728, 2560, 4), (1, 2560, 9728, 4),
                                        (8, 2560, 9728, 4), (1, 17408, 5120, 2)])
def test_null_workspace_when_none_needed(dev, M, N, K, bits):
    """A caller that passes NULL/0 where lisaq_quantized_matmul_workspace() is 0 gets the same bits as
    one that passes a workspace (the header's contract)."""
    import torch

    from lisa_amd import _lib

    lib = _lib.load()
    if lib.lisaq_quantized_matmul_workspace(M, N, K, 64, bits) != 0:
        pytest.skip("this shape uses a workspace")
    rng = np.random.default_rng(N + K + M)
    w, s, b = np_linear(rng, N, K, bits, 64)
    x = np_x(rng, M, K)
    xd, wd, sd, bd = to_dev_bf16(x, dev), to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    _lib.call("lisaq_quantized_matmul", torch.cuda.current_stream().cuda_stream, xd.data_ptr(), wd.data_ptr(),
              sd.data_ptr(), bd.data_ptr(), y.data_ptr(), M, N, K, 1, 64, bits, None, 0)
    ref = ops.quantized_matmul(xd, wd, sd, bd, True, 64, bits)
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))



@pytest.mark.parametrize("M,N,K,bits", [(1, 17408, 5120, 4), (1, 3000, 5120, 2), (2, 3001, 5120, 4), (1, 9728, 2560, 4),
                                        (2, 640, 2048, 2), (1, 100, 1024, 4), (2, 777, 6144, 4)])
def test_wave_rows_equal_persistent(dev, force_path, M, N, K, bits):
    """The wave-rows matvec and the persistent matvec share the one-row arithmetic (lane l chains the chunks
    l, l+64, ... and the same 64-lane sum): every shape both take gives bitwise equal rows, so
    serial_rows may pair rows in either kernel."""
    rng = np.random.default_rng(N * 5 + K + M + bits)
    w, s, b = np_linear(rng, N, K, bits, 64)
    x = np_x(rng, M, K)
    force_path("LISAQ_QMV_KERNEL", "s")
    got_s = _run(ops.qmv, dev, x, w, s, b, 64, bits)
    force_path("LISAQ_QMV_KERNEL", "p")
    got_p = _run(ops.qmv, dev, x, w, s, b, 64, bits)
    assert np.array_equal(got_s, got_p)


@pytest.mark.parametrize("N,K", [(264, 5120), (2000, 6144)])
def test_addnorm_folded_kernels_agree(dev, force_path, N, K):
    """The add + RMSNorm prologue folded into the wave-rows matvec and into the persistent matvec: the same
    sum row, normed row and outputs bit for bit (same sum-of-squares order, same matvec arithmetic)."""
    import torch

    rng = np.random.default_rng(N + 7 * K)
    w, s, b = np_linear(rng, N, K, 4, 64)
    from lisa_amd.synth import f32_to_bf16_bits
    x, r = np_x(rng, 1, K), np_x(rng, 1, K)
    nw = f32_to_bf16_bits((1.0 + 0.1 * rng.standard_normal(K)).astype(np.float32))
    dw = (to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev))
    outs = []
    for k in ("s", "p"):
        force_path("LISAQ_QMV_KERNEL", k)
        y, sm, nm = ops.qmv_addnorm(to_dev_bf16(x, dev), to_dev_bf16(r, dev), to_dev_bf16(nw, dev), *dw, 1e-6)
        torch.cuda.synchronize()
        outs.append([from_dev_bf16(t) for t in (y, sm, nm)])
    for a, c in zip(*outs):
        assert np.array_equal(a, c)


@pytest.mark.parametrize("dtype,bits,M", [("bf16", 4, 1), ("bf16", 4, 40), ("bf16", 8, 3), ("f16", 4, 30), ("f32", 2, 2)])
def test_native_call_path(dev, dtype, bits, M):
    """quantized_matmul's native call path against the Python path on every form of the arguments that one of them
    takes: leading dimensions, Parameters, uint32 codes, non-contiguous views, mixed dtypes, a side stream; what
    the Python path refuses is refused with the same error."""
    import torch

    from lisa_amd import _lib

    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    g = torch.Generator(device=dev)
    g.manual_seed(M + bits)
    N, K, gs = 264, 1024, 64
    w = torch.randint(-(2**31), 2**31, (N, K * bits // 32), dtype=torch.int32, device=dev, generator=g)
    s, b = ((torch.randn(N, K // gs, device=dev, generator=g) * 0.02).to(dt) for _ in range(2))
    x = torch.randn(M, K, device=dev, generator=g).to(dt)
    python = lambda *a: (ops._mm_typed(*a, True, gs, bits, torch.promote_types(a[0].dtype, a[2].dtype))
                         if dtype != "bf16" or bits == 8 or a[0].dtype != a[2].dtype
                         else ops._mm("lisaq_quantized_matmul", *a, True, gs, bits))
    native = _lib.native().linear
    ref = python(x, w, s, b)
    plain = [(x, w, s, b), (x.view(M, 1, K), w, s, b), (torch.nn.Parameter(x), w, s, b), (x, w.view(torch.uint32), s, b)]
    for a in plain:
        y = native(*a, gs, bits, 0)
        assert y is not None and y.dtype == ref.dtype and tuple(y.shape) == (*a[0].shape[:-1], N) and not y.requires_grad
        assert torch.equal(y.view(M, N), ref) and torch.equal(ops.quantized_matmul(*a, True, gs, bits).view(M, N), ref)
    wide = torch.stack([x, x], -1)[..., 0]  # strided
    other = torch.float32 if dtype != "f32" else torch.float16
    for a in [(wide, w, s, b), (x, w, s.t().contiguous().t(), b), (x.to(other), w, s, b)]:
        assert native(*a, gs, bits, 0) is None
        assert torch.equal(ops.quantized_matmul(*a, True, gs, bits), python(*a))
    for a in [(x, w, s, None), (x[:, :512], w, s, b), (x, w[:, :8], s, b), (x, w, s[:5], b), (x, w.float(), s, b),
              (x.cpu(), w, s, b)]:
        assert native(*a, gs, bits, 0) is None
        with pytest.raises(ops.LisaqError):
            ops.quantized_matmul(*a, True, gs, bits)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = ops.quantized_matmul(x, w, s, b, True, gs, bits)
    side.synchronize()
    assert torch.equal(y, ref)


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("M,N,K,gs", [
    (40, 1, 64, 64),         # one group in all
    (40, 264, 64, 64),       # one group a row
    (20, 264, 320, 64),      # five groups a row: one scale/bias block
    (100, 77, 384, 128),     # three groups of 128
    (300, 260, 960, 64),     # fifteen: the last block holds seven
    (33, 300, 576, 64),      # nine: the last block holds one
    (100, 513, 2880, 64),    # 45 groups, split over K
    (300, 100, 1152, 128),   # nine groups of 128
    (700, 516, 320, 64),     # several row tiles
    (4352, 4352, 1088, 64),  # 17 groups, 17 x 17 tiles: 256-row tiles, the last round split over K
])
def test_matmul_odd_group_counts(dev, oracle, M, N, K, gs, bits):
    """Rows of an odd number of groups: the scales of the matrix's last row end off a dword, and its last group counts
    like any other -- every column against the oracle's arithmetic in float64, with and without a workspace."""
    import torch

    from lisa_amd import _lib

    rng = np.random.default_rng(M + N + K + bits)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits == 4 else 0.05, s_floor=0.01)
    x = np_x(rng, M, K)
    xd, wd, sd, bd = to_dev_bf16(x, dev), to_dev_u32(w, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev)
    cols = np.unique(np.r_[np.arange(min(N, 40)), np.arange(max(N - 40, 0), N), rng.integers(0, N, 40)])
    ref = oracle.qmm_typed(bf16_bits_to_f32(x), w[cols], bf16_bits_to_f32(s)[cols], bf16_bits_to_f32(b)[cols], gs,
                           bits, "bf16").astype(np.float32)
    got = from_dev_bf16(ops.qmm(xd, wd, sd, bd, gs, bits))
    assert_close_bf16(got[:, cols], ref, what=f"qmm M={M} N={N} K={K} bits={bits} gs={gs}")
    y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    _lib.call("lisaq_qmm", torch.cuda.current_stream().cuda_stream, xd.data_ptr(), wd.data_ptr(), sd.data_ptr(),
              bd.data_ptr(), y.data_ptr(), M, N, K, gs, bits, None, 0)
    assert_close_bf16(from_dev_bf16(y)[:, cols], ref, what=f"unsplit M={M} N={N} K={K} bits={bits} gs={gs}")
    if M >= ops.qmv_batch_limit(K, N):
        assert np.array_equal(from_dev_bf16(ops.quantized_matmul(xd, wd, sd, bd, True, gs, bits)), got)


@pytest.mark.parametrize("dtype,bits,strided", [("bf16", 4, False), ("f16", 4, False), ("bf16", 8, True)])
def test_scratch_of_a_capture_begun_outside_torch(dev, dtype, bits, strided):
    """A stream capture that torch did not begin has no memory pool of its own: the split-K scratch of a captured call
    stays allocated as long as its output, and replays leave other tensors alone.  (strided: the Python call path)"""
    import ctypes

    import torch

    path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
    hip = ctypes.CDLL(path)
    M, N, K, gs = 30, 1024, 5120, 64
    dt = torch.float16 if dtype == "f16" else torch.bfloat16
    g = torch.Generator(device=dev)
    g.manual_seed(bits)
    w = torch.randint(-(2**31), 2**31, (N, K * bits // 32), dtype=torch.int32, device=dev, generator=g)
    s, b = ((torch.randn(N, K // gs, device=dev, generator=g) * 0.01).to(dt) for _ in range(2))
    x = torch.randn(M, K, device=dev, generator=g).to(dt)
    arg = torch.stack([x, x], -1)[..., 0] if strided else x
    from lisa_amd import _lib
    need = _lib.load().lisaq_quantized_matmul_workspace(M, N, K, gs, bits)
    assert need > M * N * 4 and M >= ops.qmv_batch_limit(K, N)
    ref = ops.quantized_matmul(x, w, s, b, True, gs, bits)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
    with torch.cuda.stream(st):
        for _ in range(2):
            ops.quantized_matmul(arg, w, s, b, True, gs, bits)
        torch.cuda.synchronize()
        held = torch.cuda.memory_allocated(dev)
        assert hip.hipStreamBeginCapture(ctypes.c_void_p(st.cuda_stream), 1) == 0
        y = ops.quantized_matmul(arg, w, s, b, True, gs, bits)
        assert hip.hipStreamEndCapture(ctypes.c_void_p(st.cuda_stream), ctypes.byref(graph)) == 0
        assert torch.cuda.memory_allocated(dev) - held >= M * N * 2 + need
        assert y.is_contiguous() and y.storage_offset() == 0 and tuple(y.shape) == (M, N)
        others = [torch.full((need,), 7, dtype=torch.uint8, device=dev) for _ in range(4)]
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0) == 0
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        assert hip.hipGraphLaunch(exe, ctypes.c_void_p(st.cuda_stream)) == 0
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
        assert all(bool((o == 7).all()) for o in others)
        assert torch.equal(ops.quantized_matmul(x, w, s, b, True, gs, bits), ref)
    assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0


def test_native_calls_leave_other_threads_running(dev):
    """A call that waits for room in a full queue does not stop the process's other Python threads."""
    import threading
    import time

    import torch

    g, u = (torch.randn(8, 64, device=dev).to(torch.bfloat16) for _ in range(2))
    ref = ops.swiglu(g, u)
    cycles, busy = 100_000, 0.0
    while busy < 0.7:  # (a spin of about a second, whatever its clock)
        cycles = int(cycles * (min(10.0, 0.9 / busy) if busy > 1e-4 else 10.0))
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        torch.cuda._sleep(cycles)
        torch.cuda.synchronize()
        busy = time.perf_counter() - t0
    gap, stop = [0.0], threading.Event()

    def watch():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.0005)
            now = time.perf_counter()
            gap[0], last = max(gap[0], now - last), now

    th = threading.Thread(target=watch)
    th.start()
    done = torch.cuda.Event()
    torch.cuda._sleep(cycles)
    done.record()
    slowest, calls, t0 = 0.0, 0, time.perf_counter()
    while not done.query() and time.perf_counter() - t0 < 5 * busy:
        t = time.perf_counter()
        y = ops.swiglu(g, u)
        slowest, calls = max(slowest, time.perf_counter() - t), calls + 1
    stop.set()
    th.join()
    torch.cuda.synchronize()
    print(f"busy {busy:.2f} s, {calls} calls, slowest {slowest:.3f} s, longest gap of the other thread {gap[0]:.3f} s")
    assert torch.equal(y, ref)
    assert gap[0] < 0.25 * busy


def _native_ops(dev):
    """name -> (native call, Python op, arguments, positions of the tensors among them)"""
    import torch

    from lisa_amd import _lib

    n = _lib.native()
    g = torch.Generator(device=dev)
    g.manual_seed(7)
    E, k, H, I, gs, bits = 8, 2, 256, 128, 64, 4

    def packed(*lead, K):
        w = torch.randint(-(2**31), 2**31, (*lead, K * bits // 32), dtype=torch.int32, device=dev, generator=g)
        s, b = ((torch.randn(*lead, K // gs, device=dev, generator=g) * 0.02).to(torch.bfloat16) for _ in range(2))
        return w, s, b

    bf = lambda *sh: torch.randn(*sh, device=dev, generator=g).to(torch.bfloat16)
    x, q = bf(3, H), packed(40, K=H)
    gate, up, down = packed(E, I, K=H), packed(E, I, K=H), packed(E, H, K=I)
    xt, lg = bf(5, H), torch.randn(5, E, device=dev, generator=g)
    ops.moe_forward(xt, lg, gate, up, down, k, gs, bits)  # (makes the workspace)
    ws = ops.workspace(dev, 0, "moe_forward")
    moe = lambda *a: ops.moe_forward(a[0], a[1], a[2:5], a[5:8], a[8:11], *a[11:14])
    return {
        "linear": (n.linear, lambda *a: ops.quantized_matmul(*a[:4], True, *a[4:6]), (x, *q, gs, bits, 0), range(4)),
        "addnorm": (n.addnorm, ops.qmv_addnorm, (bf(1, 4608), bf(1, 4608), bf(4608), *packed(40, K=4608), 1e-6, gs, bits),
                    range(6)),
        "swiglu": (n.swiglu, ops.swiglu, (bf(3, 40), bf(3, 40)), range(2)),
        "dequantize": (n.dequantize, ops.dequantize, (*q, gs, bits), range(3)),
        "quantize": (n.quantize, ops.quantize, (bf(6, H), gs, bits), range(1)),
        "moe": (n.moe, moe, (xt, lg, *gate, *up, *down, k, gs, bits, ws), range(11)),
    }


_NATIVE = ["linear", "addnorm", "swiglu", "dequantize", "quantize", "moe"]


def _same(a, b):
    import torch

    a, b = (t if isinstance(t, tuple) else (t,) for t in (a, b))
    return len(a) == len(b) and all(p.dtype == q.dtype and p.shape == q.shape and
                                    torch.equal(p.contiguous().view(torch.uint8), q.contiguous().view(torch.uint8))
                                    for p, q in zip(a, b))


@pytest.mark.parametrize("name", _NATIVE)
def test_native_call_accepts_and_declines(dev, name):
    """Each native call gives what its op's Python path gives (forced by a strided view of one argument at a time), and
    declines views, other dtypes, host tensors, missing arguments, tensor subclasses, vmap, dispatch and function
    modes, leaving those to the Python path."""
    import torch
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    native, op, args, tensors = _native_ops(dev)[name]
    ref = native(*args)
    assert ref is not None and _same(ref, op(*args))
    put = lambda i, t: (*args[:i], t, *args[i + 1:])

    class Sub(torch.Tensor):
        pass

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, a=(), kw=None):
            return func(*a, **(kw or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, a=(), kw=None):
            return func(*a, **(kw or {}))

    for i in tensors:
        t = args[i]
        strided = torch.stack([t, t], -1)[..., 0]
        assert native(*put(i, torch.nn.Parameter(t, requires_grad=False))) is not None
        if t.dim() > 1 or t.numel() > 1:
            assert not strided.is_contiguous() and native(*put(i, strided)) is None
            assert _same(ref, op(*put(i, strided)))
        for other in (None, t.cpu(), t.double(), t.as_subclass(Sub), t.to_sparse() if t.dim() == 2 else None):
            assert native(*put(i, other)) is None
        seen = []
        torch.func.vmap(lambda v: (seen.append(native(*put(i, v))), v)[1])(torch.stack([t, t]))
        assert seen == [None]
    assert native(*args[:-1]) is None and native(*args, 0) is None
    for mode in (Dispatch(), Function()):
        with mode:
            declined = native(*args)
        assert declined is None
    assert _same(ref, native(*args))


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("M,N,K,gs", [(20, 8, 64, 32), (13, 40, 192, 32), (32, 300, 128, 64), (1, 77, 256, 128),
                                      (32, 515, 256, 32), (33, 300, 256, 64), (64, 100, 128, 64), (64, 260, 320, 32)])
def test_few_rows_short_rows(dev, oracle, M, N, K, gs, bits):
    """The matmul of few rows forced on rows of one chunk and less, and past 32 rows on both sides of the K from which
    it is chosen."""
    rng = np.random.default_rng(M + N + K + bits)
    w, s, b = np_linear(rng, N, K, bits, gs, s_std=0.02 if bits == 4 else 0.05)
    x = np_x(rng, M, K)
    got = _run(ops.qmm, dev, x, w, s, b, gs, bits)
    assert_close_bf16(got, oracle.qmm(x, w, s, b, gs, bits), what=f"M={M} N={N} K={K} bits={bits} gs={gs}")
