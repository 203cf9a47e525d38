"""GPU quantisers and device shuffles: bit-exact against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from gcnasm_amd import f4gemm, ops

pytestmark = pytest.mark.gpu


def edge_values():
    """Ties, subnormal boundaries, saturation, zeros of both signs, infinities
    (NaNs: test_quant_nan_blocks)."""
    vals = [0.0, -0.0, 448.0, -448.0, 464.0, 480.0, 1e30, -1e30, np.inf, -np.inf,
            2.0 ** -6, 2.0 ** -7, 2.0 ** -9, 2.0 ** -10, 1.5 * 2.0 ** -10, 1.0625, 1.1875,
            1.0 + 2.0 ** -4, 1.0 + 3 * 2.0 ** -4, 3.0e-45]
    # midpoints between consecutive E4M3 values (exact ties)
    t = oracle.e4m3_decode_table()
    pos = np.sort(t[np.isfinite(t) & (t > 0)])
    mids = (pos[:-1] + pos[1:]) / 2
    return np.concatenate([np.array(vals, dtype=np.float32), mids.astype(np.float32),
                           -mids.astype(np.float32)])


@pytest.mark.parametrize("rule", [0, 1, 2])
@pytest.mark.parametrize("in_bf16", [False, True])
def test_quant_mx(dev, rule, in_bf16):
    rows, K = 96, 1024
    x = oracle.gen_mx_input(rows, K, 100 + rule, 1.0, 6)
    e = edge_values()
    x.reshape(-1)[: e.size] = e
    if in_bf16:
        xb = oracle.to_bf16_bits(x)
        x = oracle.bf16_bits_to_f32(xb)
        xt = torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16)
    else:
        xt = torch.from_numpy(x).to(dev)
    q, s = ops.quant_mxfp8(xt, rule)
    torch.cuda.synchronize()
    qo, so = oracle.quant_mxfp8(x, rule)
    np.testing.assert_array_equal(s.cpu().numpy(), so)
    np.testing.assert_array_equal(q.cpu().numpy(), qo)


@pytest.mark.parametrize("in_bf16", [False, True])
def test_quant_1x128_128x128_per_tensor(dev, in_bf16):
    rows, K = 300, 1024
    x = oracle.randn(rows * K, 7).reshape(rows, K) * np.float32(3.0)
    x[5, :128] = 0.0  # an all-zero group
    x.reshape(-1)[1000:1000 + 40] = edge_values()[:40]
    x[np.isinf(x)] = 1000.0
    if in_bf16:
        xb = oracle.to_bf16_bits(x)
        x = oracle.bf16_bits_to_f32(xb)
        xt = torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16)
    else:
        xt = torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    q1, s1 = ops.quant_fp8_1x128(xt)
    q2, s2 = ops.quant_fp8_128x128(xt)
    q3, s3 = ops.quant_fp8_per_tensor(xt)
    torch.cuda.synchronize()
    o1, os1 = oracle.quant_fp8_1x128(x)
    o2, os2 = oracle.quant_fp8_128x128(x)
    o3, os3 = oracle.quant_fp8_per_tensor(x)
    np.testing.assert_array_equal(s1.cpu().numpy().view(np.uint32), os1.view(np.uint32))
    np.testing.assert_array_equal(q1.cpu().numpy(), o1)
    np.testing.assert_array_equal(s2.cpu().numpy().view(np.uint32), os2.view(np.uint32))
    np.testing.assert_array_equal(q2.cpu().numpy(), o2)
    np.testing.assert_array_equal(s3.cpu().numpy().view(np.uint32), os3.view(np.uint32))
    np.testing.assert_array_equal(q3.cpu().numpy(), o3)


@pytest.mark.parametrize("in_bf16", [False, True])
def test_quant_strided_rows_and_tails(dev, in_bf16):
    """Rows whose stride is a multiple of 4 but not 8 elements (bf16 takes the
    8-byte load path), a block count that leaves a partial last workgroup, and a
    per-tensor size with n % 4 != 0."""
    rows, K = 97, 1152
    base = oracle.gen_mx_input(rows, K + 4, 55, 1.0, 6)
    x = np.ascontiguousarray(base[:, :K])
    if in_bf16:
        bb = oracle.to_bf16_bits(base)
        x = oracle.bf16_bits_to_f32(np.ascontiguousarray(bb[:, :K]))
        xt = torch.from_numpy(bb.view(np.int16)).to(dev).view(torch.bfloat16)[:, :K]
    else:
        xt = torch.from_numpy(base).to(dev)[:, :K]
    assert xt.stride(0) == K + 4
    q, s = ops.quant_mxfp8(xt, 0)
    q4, s4 = ops.quant_mxfp4(xt, 2)
    q1, s1 = ops.quant_fp8_1x128(xt)
    q2, s2 = ops.quant_fp8_128x128(xt)
    torch.cuda.synchronize()
    qo, so = oracle.quant_mxfp8(x, 0)
    np.testing.assert_array_equal(s.cpu().numpy(), so)
    np.testing.assert_array_equal(q.cpu().numpy(), qo)
    q4o, s4o = oracle.quant_mxfp4(x, 2)
    np.testing.assert_array_equal(s4.cpu().numpy(), s4o)
    np.testing.assert_array_equal(q4.cpu().numpy(), q4o)
    o1, os1 = oracle.quant_fp8_1x128(x)
    np.testing.assert_array_equal(s1.cpu().numpy().view(np.uint32), os1.view(np.uint32))
    np.testing.assert_array_equal(q1.cpu().numpy(), o1)
    o2, os2 = oracle.quant_fp8_128x128(x)
    np.testing.assert_array_equal(s2.cpu().numpy().view(np.uint32), os2.view(np.uint32))
    np.testing.assert_array_equal(q2.cpu().numpy(), o2)
    flat = x.reshape(-1)[:12345]
    ft = xt.contiguous().reshape(-1)[:12345]
    q3, s3 = ops.quant_fp8_per_tensor(ft)
    torch.cuda.synchronize()
    o3, os3 = oracle.quant_fp8_per_tensor(flat)
    np.testing.assert_array_equal(s3.cpu().numpy().view(np.uint32), os3.view(np.uint32))
    np.testing.assert_array_equal(q3.cpu().numpy(), o3)


def test_e4m3_encoder_every_bf16_value(dev):
    """Per-tensor quantisation with amax = 448 has scale 1, so q = e4m3(x): every
    bf16 bit pattern of magnitude <= 448 (and every NaN) goes through the
    device encoder and is compared with the oracle's."""
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    vals = oracle.bf16_bits_to_f32(bits)
    keep = np.isnan(vals) | (np.abs(vals) <= 448.0)
    xb = bits[keep]
    xb = np.concatenate([xb, oracle.to_bf16_bits(np.array([448.0], np.float32))])
    x = oracle.bf16_bits_to_f32(xb)
    for t in (torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16),
              torch.from_numpy(np.ascontiguousarray(x)).to(dev)):
        q, s = ops.quant_fp8_per_tensor(t)
        torch.cuda.synchronize()
        assert s.cpu().numpy()[0] == np.float32(1.0)
        np.testing.assert_array_equal(q.cpu().numpy(), oracle.e4m3_encode(x))


@pytest.mark.parametrize("in_bf16", [False, True])
def test_quant_nan_blocks(dev, in_bf16):
    """Block maxima ignore NaNs (the CPU reference's `a > amax` scan): NaNs,
    quiet, signalling and negative, as the first or last element of a 1x32
    block, next to the block's largest value, filling a whole 1x32 / 1x128
    block, and in one 128x128 tile only, among blocks without NaNs in the same
    wave; every quantiser against the oracle, codes and scales."""
    rows, K = 256, 1024
    x = oracle.gen_mx_input(rows, K, 91, 1.0, 6)
    nans = np.array([0x7FC00000, 0x7F800001, 0xFFC00000, 0xFFBFFFFF], np.uint32).view(np.float32)
    x[0, 0] = nans[0]                  # first of its 1x32 block
    x[1, 31] = nans[1]                 # last of its block (signalling)
    x[2, 40] = nans[2]                 # negative
    x[2, 41] = 300.0                   # beside the block's maximum
    x[3, 64:96] = nans[3]              # a whole 1x32 block
    x[4, 128:256] = nans[0]            # a whole 1x128 block
    x[200, 900] = nans[1]              # one NaN in tile (1, 7)
    if in_bf16:
        xb = oracle.to_bf16_bits(x)
        x = oracle.bf16_bits_to_f32(xb)
        xt = torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16)
    else:
        xt = torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    assert np.isnan(x).sum() == 3 + 32 + 128 + 1
    for rule in (0, 1, 2):
        q, sc = ops.quant_mxfp8(xt, rule)
        q4, s4 = ops.quant_mxfp4(xt, rule)
        torch.cuda.synchronize()
        qo, so = oracle.quant_mxfp8(x, rule)
        np.testing.assert_array_equal(sc.cpu().numpy(), so)
        np.testing.assert_array_equal(q.cpu().numpy(), qo)
        q4o, s4o = oracle.quant_mxfp4(x, rule)
        np.testing.assert_array_equal(s4.cpu().numpy(), s4o)
        np.testing.assert_array_equal(q4.cpu().numpy(), q4o)
    q1, s1 = ops.quant_fp8_1x128(xt)
    q2, s2 = ops.quant_fp8_128x128(xt)
    torch.cuda.synchronize()
    o1, os1 = oracle.quant_fp8_1x128(x)
    o2, os2 = oracle.quant_fp8_128x128(x)
    np.testing.assert_array_equal(s1.cpu().numpy().view(np.uint32), os1.view(np.uint32))
    np.testing.assert_array_equal(q1.cpu().numpy(), o1)
    np.testing.assert_array_equal(s2.cpu().numpy().view(np.uint32), os2.view(np.uint32))
    np.testing.assert_array_equal(q2.cpu().numpy(), o2)


@pytest.mark.parametrize("narrow", [False, True])
@pytest.mark.parametrize("in_bf16", [False, True])
def test_quant_nan_quotients(dev, in_bf16, narrow):
    """Quotients that are NaN where no input is: an infinity over the infinite
    scale it makes, and a zero over a scale that rounds to 0 (an fp32 maximum
    of at most 224 * 2^-149). Infinities of both signs as the first, last and
    every element of a 1x128 group, beside a NaN, and in groups whose wave
    holds no NaN; groups of the smallest subnormals. Codes and scales of the
    three divided formats against the oracle. narrow: rows that take the
    8-byte bf16 loads."""
    rows, K, pad = 384, 1152, 4 if narrow else 0
    x = oracle.randn(rows * (K + pad), 17).reshape(rows, K + pad) * np.float32(3.0)
    inf, tiny = np.float32(np.inf), np.float32(2.0 ** -149)
    x[0, 0] = inf                       # first of its group
    x[1, 255] = -inf                    # last of its group
    x[2, 256:384] = inf                 # a whole group
    x[3, 384:512:2] = -inf
    x[3, 385:512:2] = inf
    x[4, 5], x[4, 6] = np.nan, -inf     # beside a NaN
    x[290, 1100] = inf                  # the only one of its 128x128 tile
    if not in_bf16:                     # 128x128 tiles (1, 2) and (1, 3) hold nothing larger
        x[128:256, 256:512] = 0.0
        x[130, 260], x[131, 270] = tiny, -tiny
        x[140, 400], x[141, 401] = 223 * tiny, -200 * tiny
        x[150, 300], x[151, 310] = 224 * tiny, 224 * tiny
    x = np.ascontiguousarray(x)
    if in_bf16:
        xb = oracle.to_bf16_bits(x)
        xt = torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16)[:, :K]
        x = oracle.bf16_bits_to_f32(xb)
    else:
        xt = torch.from_numpy(x).to(dev)[:, :K]
    x = np.ascontiguousarray(x[:, :K])
    got = [ops.quant_fp8_1x128(xt), ops.quant_fp8_128x128(xt), ops.quant_fp8_per_tensor(xt)]
    torch.cuda.synchronize()
    want = [oracle.quant_fp8_1x128(x), oracle.quant_fp8_128x128(x), oracle.quant_fp8_per_tensor(x)]
    assert (want[0][0][2, 256:384] == 0x7F).all() and np.isinf(want[0][1]).sum() == 6
    assert in_bf16 or (want[0][1] == 0).any() and (want[1][1] == 0).any()
    for (q, s), (qo, so) in zip(got, want):
        np.testing.assert_array_equal(s.cpu().numpy().view(np.uint32), so.view(np.uint32))
        np.testing.assert_array_equal(q.cpu().numpy(), qo)


@pytest.mark.parametrize("amax", [1000.5, 3.7e-5, 1.7 * 2.0 ** -50, 2.0 ** -60, 3.0e38])
def test_quant_division_every_bf16_value(dev, amax):
    """The 1x128, 128x128 and per-tensor quantisers divide by s = amax/448,
    which is not a power of two: blocks whose first element is the maximum
    and whose other elements run through every bf16 value of magnitude <=
    amax (both signs, zeros included), at scales on both sides of the 2^-64
    bound of the shared-reciprocal division (1.7 * 2^-50 / 448 above it,
    2^-60 / 448 below), checked bit for bit against the oracle's fp32 division
    for fp32 and bf16 input."""
    top = oracle.bf16_bits_to_f32(oracle.to_bf16_bits(np.array([amax], np.float32)))[0]
    allv = oracle.bf16_bits_to_f32(np.arange(0x7F80, dtype=np.uint32).astype(np.uint16))
    vals = allv[allv <= top]
    vals = np.concatenate([vals, -vals]).astype(np.float32)
    nblk = -(-len(vals) // 127)
    nblk = -(-nblk // 8) * 8  # whole rows of K = 1024
    body = np.zeros(nblk * 127, np.float32)
    body[:len(vals)] = vals
    x = np.concatenate([np.full((nblk, 1), top, np.float32), body.reshape(nblk, 127)], axis=1)
    x = np.ascontiguousarray(x.reshape(-1, 1024))
    xb = oracle.to_bf16_bits(x)
    assert np.array_equal(oracle.bf16_bits_to_f32(xb), x)
    o1, os1 = oracle.quant_fp8_1x128(x)
    o2, os2 = oracle.quant_fp8_128x128(x)
    o3, os3 = oracle.quant_fp8_per_tensor(x)
    for t in (torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16),
              torch.from_numpy(x).to(dev)):
        q1, s1 = ops.quant_fp8_1x128(t)
        q2, s2 = ops.quant_fp8_128x128(t)
        q3, s3 = ops.quant_fp8_per_tensor(t)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(s1.cpu().numpy().view(np.uint32), os1.view(np.uint32))
        np.testing.assert_array_equal(q1.cpu().numpy(), o1)
        np.testing.assert_array_equal(s2.cpu().numpy().view(np.uint32), os2.view(np.uint32))
        np.testing.assert_array_equal(q2.cpu().numpy(), o2)
        np.testing.assert_array_equal(s3.cpu().numpy().view(np.uint32), os3.view(np.uint32))
        np.testing.assert_array_equal(q3.cpu().numpy(), o3)


@pytest.mark.parametrize("NK", [(16, 32), (256, 512), (272, 4096)])
def test_device_shuffle_weight(dev, NK):
    N, Kp = NK
    rng = np.random.default_rng(N + Kp)
    w = rng.integers(0, 256, size=(N, Kp), dtype=np.uint8)
    got = ops.shuffle_weight_16x16(torch.from_numpy(w).to(dev)).cpu().numpy().reshape(-1)
    np.testing.assert_array_equal(got, oracle.shuffle_weight_16x16(w, N, Kp))


@pytest.mark.parametrize("shape", [(1, 8, 256, 8), (300, 32, 512, 32), (17, 5, 32, 8)])
def test_device_shuffle_scale(dev, shape):
    rows, cols, sm, sn = shape
    rng = np.random.default_rng(rows)
    s = rng.integers(100, 140, size=(rows, cols), dtype=np.uint8)
    got = ops.shuffle_scale(torch.from_numpy(s).to(dev), sm, sn).cpu().numpy()
    np.testing.assert_array_equal(got, oracle.shuffle_scale(s, rows, cols, sm, sn))


def test_prepare_matches_host_path(dev):
    """prepare_mx_b on the GPU == oracle quantiser + host shuffles."""
    N, K = 256, 768
    x = oracle.gen_mx_input(N, K, 5, 0.02, 4)
    b = ops.prepare_mx_b(torch.from_numpy(x).to(dev))
    q, s = oracle.quant_mxfp8(x)
    sh = f4gemm.Shape(1, N, K)
    np.testing.assert_array_equal(b.codes.cpu().numpy().reshape(-1),
                                  oracle.shuffle_weight_16x16(q, N, K))
    np.testing.assert_array_equal(b.scales.cpu().numpy(),
                                  oracle.shuffle_scale(s, N, K // 32, sh.scale_b_rows(),
                                                       sh.scale_cols()))


@pytest.mark.parametrize("rule", [0, 1, 2])
@pytest.mark.parametrize("in_bf16", [False, True])
def test_quant_mx8_e5m2(dev, rule, in_bf16):
    """MX 1x32 with E5M2 elements (ga_quant_mx8 fmt 1) byte for byte against
    the oracle, codes and scales, fp32 and bf16 inputs, a partial 16-byte tail
    of rows; fmt 0 equals the E4M3 quantiser."""
    rows, K = 77, 1056
    x = oracle.gen_mx_input(rows, K, 55 + rule, 1.0, 6)
    x[0, :32] = 0.0
    x[1, 5] = np.nan
    x[2, :32] = 57344.0
    if in_bf16:
        xb = oracle.to_bf16_bits(x)
        t = torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16)
        x = oracle.bf16_bits_to_f32(xb)
    else:
        t = torch.from_numpy(x).to(dev)
    q, s = ops.quant_mx8(t, 1, rule)
    q8, s8 = ops.quant_mx8(t, 0, rule)
    q0, s0 = ops.quant_mxfp8(t, rule)
    torch.cuda.synchronize()
    qo, so = oracle.quant_mx8(x, 1, rule)
    np.testing.assert_array_equal(s.cpu().numpy(), so)
    np.testing.assert_array_equal(q.cpu().numpy(), qo)
    np.testing.assert_array_equal(q8.cpu().numpy(), q0.cpu().numpy())
    np.testing.assert_array_equal(s8.cpu().numpy(), s0.cpu().numpy())


def test_e5m2_encoder_every_bf16_value(dev):
    """Every bf16 bit pattern of magnitude <= 57344 (and every NaN) through the
    device E5M2 encoder at scale 1: each 32-block holds 57344 first, so the
    floor rule gives exponent 0, then 31 of the test values."""
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    vals = oracle.bf16_bits_to_f32(bits)
    keep = np.isnan(vals) | (np.abs(vals) <= 57344.0)
    v = vals[keep]
    per = 31
    nblk = (len(v) + per - 1) // per
    pad = np.zeros(nblk * per, np.float32)
    pad[:len(v)] = v
    blocks = np.concatenate([np.full((nblk, 1), 57344.0, np.float32), pad.reshape(nblk, per)],
                            axis=1)
    rows = (nblk + 31) // 32
    x = np.zeros((rows * 32, 32), np.float32)
    x[:nblk] = blocks
    x = x.reshape(rows, 32 * 32)
    xb = oracle.to_bf16_bits(x)
    assert np.array_equal(oracle.bf16_bits_to_f32(xb)[np.isfinite(x)], x[np.isfinite(x)])
    t = torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16)
    q, s = ops.quant_mx8(t, 1, 0)
    torch.cuda.synchronize()
    xf = oracle.bf16_bits_to_f32(xb)
    sc = s.cpu().numpy()[:, :]
    assert np.all(sc.reshape(-1)[:nblk] == 127)
    np.testing.assert_array_equal(q.cpu().numpy(), oracle.quant_mx8(xf, 1, 0)[0])
    np.testing.assert_array_equal(q.cpu().numpy().reshape(-1, 32)[:nblk, 1:].reshape(-1)[:len(v)],
                                  oracle.e5m2_encode(v))


@pytest.mark.parametrize("in_bf16", [False, True])
@pytest.mark.parametrize("n", [1, 3, 7, 8, 2047, 2049, 262147, 9000011])
def test_quant_per_tensor_scratch_sizes(dev, n, in_bf16):
    """One word of scratch (atomics), partial maxima, and pointers that do not
    allow 16-byte loads write the same bytes; the scratch starts dirty. The
    maximum sits in the last element (the scalar tail where there is one)."""
    import ctypes

    from gcnasm_amd import _lib
    x = oracle.randn(n + 1, 11)
    x[n // 2] = np.float32("nan")
    x[n - 1] = -37.5
    if in_bf16:
        xb = oracle.to_bf16_bits(x)
        x = oracle.bf16_bits_to_f32(xb)
        xt = torch.from_numpy(xb.view(np.int16)).to(dev).view(torch.bfloat16)
    else:
        xt = torch.from_numpy(x).to(dev)
    for first in (0, 1):
        src = xt[first:first + n]
        want, scale = oracle.quant_fp8_per_tensor(x[first:first + n])
        for words in (1, 1024):
            q = torch.full((n,), 0xAA, dtype=torch.uint8, device=dev)
            s = torch.zeros(1, dtype=torch.float32, device=dev)
            ws = torch.full((words,), -1, dtype=torch.int32, device=dev)
            _lib.check(_lib.lib().ga_quant_fp8_per_tensor_ws(
                src.data_ptr(), 1 if in_bf16 else 0, n, q.data_ptr(), s.data_ptr(),
                ws.data_ptr(), words * 4, ctypes.c_void_p(0)))
            torch.cuda.synchronize()
            np.testing.assert_array_equal(s.cpu().numpy().view(np.uint32),
                                          np.asarray(scale, np.float32).reshape(1).view(np.uint32))
            np.testing.assert_array_equal(q.cpu().numpy(), want.reshape(-1))


@pytest.mark.parametrize("rule", [0, 1, 2])
@pytest.mark.parametrize("in_bf16", [False, True])
@pytest.mark.parametrize("M,K", [(1, 32), (17, 288), (32, 256), (33, 1056), (256, 512), (300, 384)])
def test_prepare_activations_one_pass(dev, M, K, in_bf16, rule):
    """prepare_mx_a / prepare_mx4_a and the E5M2 form write the bytes of the
    oracle's quantiser, zero rows and the oracle's scale shuffle, from rows
    with a stride and from a base that does not allow 16-byte loads; NaN,
    infinities and an all-zero block among the values."""
    from gcnasm_amd import _lib
    buf = oracle.gen_mx_input(M, K + 64, 9 + rule, 1.0, 6)
    buf[0, 4:8] = [np.nan, np.inf, -np.inf, -np.nan]
    buf[M - 1, K - 28:K] = 0.0
    if in_bf16:
        bits = oracle.to_bf16_bits(buf)
        buf = oracle.bf16_bits_to_f32(bits)
        t = torch.from_numpy(bits.view(np.int16)).to(dev).view(torch.bfloat16)
    else:
        t = torch.from_numpy(buf).to(dev)
    sh = f4gemm.Shape(M, 1, K)
    rows, cols = sh.scale_a_rows(), sh.scale_cols()
    for off in (0, 4):
        x, xt = np.ascontiguousarray(buf[:, off:off + K]), t[:, off:off + K]
        for elem in (0, 1, 2):
            q, s = (oracle.quant_mxfp8(x, rule) if elem == 0 else
                    oracle.quant_mx8(x, 1, rule) if elem == 1 else oracle.quant_mxfp4(x, rule))
            want = np.zeros((rows, q.shape[1]), np.uint8)
            want[:M] = q
            if elem == 1:
                codes = torch.full(want.shape, 0xAA, dtype=torch.uint8, device=dev)
                scales = torch.full((rows * cols,), 0xAA, dtype=torch.uint8, device=dev)
                _lib.check(_lib.lib().ga_prepare_mx_a(
                    xt.data_ptr(), 1 if in_bf16 else 0, M, K, xt.stride(0), 1, codes.data_ptr(),
                    scales.data_ptr(), rule, None))
            else:
                a = (ops.prepare_mx_a if elem == 0 else ops.prepare_mx4_a)(xt, rule)
                codes, scales = a.codes, a.scales
            torch.cuda.synchronize()
            np.testing.assert_array_equal(codes.cpu().numpy(), want)
            np.testing.assert_array_equal(scales.cpu().numpy(),
                                          oracle.shuffle_scale(s, M, K // 32, rows, cols))
