"""The kernels of the fp32-scaled FP8 GEMMs that a call's shape picks: the K-split
kernel (few rows; every wave tile and slice count of its plan) and the tiles of
128x128, 128x256 and 256x256, at the edges of rows, columns and K, with padded
strides and batches, against the CPU oracle in the K slices the library
reports."""
import numpy as np
import pytest
import torch

import oracle
from gcnasm_amd import _lib, opus_gemm
from helpers import assert_parity, bf16_compare, f32_compare

pytestmark = pytest.mark.gpu

# rows: one block of 16 or 32, two to four of 32, blocks of 64 with a short
# last one; columns below, at and past a 16-column group and a 128-column
# block, few and many groups; K of one group, fewer groups than slices, a
# number that no slice count divides, and long.
SHAPES = [(1, 16, 128), (1, 37, 256), (15, 4112, 384), (16, 8200, 1152), (17, 130, 640),
          (32, 2100, 1152), (33, 1000, 2048), (63, 4097, 384), (64, 24576, 256), (65, 300, 128),
          (127, 2112, 896), (128, 1024, 3456), (129, 515, 1152), (200, 6000, 640),
          (300, 2113, 1792), (513, 1032, 1024), (700, 4096, 512), (1024, 200, 1280),
          (8, 64, 8192), (24, 80, 7168), (64, 96, 7168)]


def problem(batch, M, N, K, group_n, seed):
    rng = np.random.default_rng(seed)
    G = K // 128

    def codes(rows):
        x = rng.standard_normal((batch, rows, K)).astype(np.float32)
        return np.stack([oracle.quant_fp8_per_tensor(v)[0] for v in x])

    sfa = rng.uniform(0.5, 2.0, (batch, G, M)).astype(np.float32)
    shape = (batch, -(-N // 128), G) if group_n == 128 else (batch, G, N)
    return codes(M), codes(N), sfa, rng.uniform(0.5, 2.0, shape).astype(np.float32)


def padded(x, ld, dev):
    """x [batch, rows, K] on the device with rows of ld bytes, the pad 0x7F (NaN codes)."""
    out = np.full(x.shape[:-1] + (ld,), 0x7F, x.dtype)
    out[..., :x.shape[-1]] = x
    return torch.from_numpy(out).to(dev)


def strided(x, pad, dev):
    """x [batch, rows, cols] on the device as a view whose rows are `pad` NaNs
    apart and whose storage ends with its last element; the strides with it."""
    b, r, c = x.shape
    flat = torch.full((b * r * (c + pad) - pad,), float("nan"), dtype=torch.float32, device=dev)
    view = flat.as_strided((b, r, c), (r * (c + pad), c + pad, 1))
    view.copy_(torch.from_numpy(x))
    return view


def run(dev, shape, group_n, batch, pad_a, pad_b, pad_c, whole_k=False, pad_s=0):
    M, N, K = shape
    qa, qb, sfa, sfb = problem(batch, M, N, K, group_n or 128, M + N + K)
    gps = opus_gemm.k_slices(M, N, K, batch)
    assert not whole_k or gps == K // 128
    A, B = padded(qa, K + pad_a, dev), padded(qb, K + pad_b, dev)
    SA, SB = strided(sfa, pad_s, dev), strided(sfb, pad_s, dev)
    rows = np.unique(np.r_[np.arange(min(M, 48)), np.arange(max(0, M - 20), M)])
    want, absdot = [], []
    for b in range(batch):
        a = np.ascontiguousarray(qa[b][rows])
        if group_n:
            s = np.ascontiguousarray(sfa[b][:, rows])
            want.append(oracle.gemm_blockscale_mfma(a, qb[b], s, sfb[b], group_n, gps))
            absdot.append(oracle.blockscale_absdot(a, qb[b], s, sfb[b], group_n))
        else:
            sa, sb = sfa[0].reshape(-1)[:1], sfb[0].reshape(-1)[:1]
            want.append(oracle.gemm_per_tensor_mfma(a, qb[b], sa, sb, gps))
            absdot.append(oracle.fp8_absdot(a, qb[b]) * float(sa[0]) * float(sb[0]))
    want, absdot = np.stack(want), np.stack(absdot)
    for dtype in (torch.float32, torch.bfloat16):
        C = torch.full((batch, M, N + pad_c), float("nan"), dtype=dtype, device=dev)
        ka = opus_gemm.make_kargs(A, B, C, SA, SB, M, N, K, batch, group_n)
        ka.stride_a, ka.stride_b, ka.stride_c = K + pad_a, K + pad_b, N + pad_c
        ka.stride_a_batch, ka.stride_b_batch = M * ka.stride_a, N * ka.stride_b
        ka.stride_c_batch = M * ka.stride_c
        if group_n:
            (ka.stride_sfa_batch, ka.stride_sfa), (ka.stride_sfb_batch, ka.stride_sfb) = (
                SA.stride()[:2], SB.stride()[:2])
        out = _lib.GA_DTYPE_F32 if dtype == torch.float32 else _lib.GA_DTYPE_BF16
        print("fp32 scales", shape, group_n, dtype, "groups per slice", gps, flush=True)
        if group_n:
            opus_gemm.gemm_a8w8_blockscale(ka, out, group_n)
        else:
            opus_gemm.fp8_gemm(ka, out)
        torch.cuda.synchronize()
        assert torch.isnan(C[:, :, N:]).all() and not torch.isnan(C[:, :, :N]).any()
        got = C[:, rows, :N].contiguous()
        if dtype == torch.float32:
            ok, st = f32_compare(got.cpu().numpy(), want, absdot=absdot)
        else:
            ok, st = bf16_compare(got.view(torch.int16).cpu().numpy().view(np.uint16),
                                  oracle.to_bf16_bits(want), absdot)
        assert_parity(st, "fp32 scales %s g%d %s" % (shape, group_n, dtype))


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("group_n", [128, 1, 0])
def test_k_split_kernel(dev, shape, group_n):
    M, N, K = shape
    run(dev, shape, group_n, *((2, 16, 48, 3) if M <= 129 and N <= 1100 else (1, 0, 32, 4)))


# More rows than the K-split kernel takes. 128x128 tiles: whole and ragged, one
# group to nine (LDS slots wrap at 4, scale slots at 8). 128x256: one to seven
# (3 and 4), the last round full. 256x256: odd and even numbers of groups.
QUARTER = [(1100, 2000, 128), (1100, 1024, 256), (1152, 2049, 384), (1026, 128, 512),
           (2048, 2048, 640), (1280, 770, 1152), (4100, 520, 1024)]
HALF = [(1100, 6900, 128), (1152, 4096, 256), (2048, 4096, 384), (2000, 3600, 512),
        (1280, 4098, 640), (1152, 6400, 896)]
FULL = [(1100, 7700, 128), (2304, 4096, 256), (2100, 4360, 384), (2304, 4100, 640)]


@pytest.mark.parametrize("shape", QUARTER + HALF + FULL)
@pytest.mark.parametrize("group_n", [128, 1, 0])
def test_tiles(dev, shape, group_n):
    M, N, K = shape
    run(dev, shape, group_n, 1, 0, 32 if M % 128 else 0, -N % 4 + 4 if N % 8 else 8, True)


# 33-64 rows with 64x256 tiles for three quarters of 256 CUs and more: one
# group, an odd number, even; ragged columns; batches of few tiles each.
@pytest.mark.parametrize("batch,shape", [(1, (33, 49157, 128)), (1, (64, 49152, 640)),
                                         (1, (48, 65538, 256)), (24, (40, 2049, 384)),
                                         (64, (63, 640, 512))])
@pytest.mark.parametrize("group_n", [128, 1, 0])
def test_rows64_tile(dev, batch, shape, group_n):
    M, N, K = shape
    run(dev, shape, group_n, batch, 16, 48, -N % 4 + 4 if N % 8 else 8, True)
    # one tile fewer than that, and 32 rows: the K-split kernel
    assert opus_gemm.k_slices(64, 256 * 191, 1024) < 8 == opus_gemm.k_slices(64, 256 * 192, 1024)
    assert opus_gemm.k_slices(32, 256 * 192, 1024) < 8


@pytest.mark.parametrize("shape,batch", [((5, 40, 256), 2), ((30, 1000, 384), 1), ((64, 2113, 1152), 1),
                                         ((40, 49157, 128), 1), ((1026, 200, 256), 1),
                                         ((1030, 2100, 384), 3), ((1100, 7700, 128), 1)])
@pytest.mark.parametrize("group_n", [128, 1])
def test_strided_scales(dev, shape, batch, group_n):
    """Scale matrices with NaNs between their rows and nothing behind the last
    one: the K-split kernel's wave tiles, the 64x256, 128x128, 128x256 and 256x256
    tiles (the copies of the groups past K and the columns past N are not used)."""
    run(dev, shape, group_n, batch, 0, 16, 0, pad_s=5)


# Batches: the K-split kernel only against the 128x128 tile, and only where it
# wins by half the time of the operands' bytes.
@pytest.mark.parametrize("batch,M,N,K,split", [(4, 96, 4096, 7168, True), (2, 128, 7168, 2048, True),
                                               (16, 128, 1024, 4096, False),
                                               (200, 128, 512, 512, False),
                                               (16, 300, 7168, 512, False)])
def test_batches_route(dev, batch, M, N, K, split):
    assert (opus_gemm.k_slices(M, N, K, batch) < K // 128) == split


@pytest.mark.parametrize("shape", [(1030, 384, 384), (1030, 2100, 384)])
@pytest.mark.parametrize("group_n", [128, 1, 0])
def test_tiles_batched_unaligned(dev, shape, group_n):
    """128x128 and 128x256 tiles, three batches, padded A and B rows, C rows
    that no 16-byte store fits."""
    run(dev, shape, group_n, 3, 16, 48, 3, True)
