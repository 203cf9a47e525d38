"""The MX kernels that a launch's shape picks (the K-split kernel, the 128x256
and 128x128 tiles, the entry's own kernel), each at the edges of its tiles and
of the rule that picks it, against the CPU oracle: formats, B layouts, splits,
alpha and beta, a strided D."""
import numpy as np
import pytest
import torch

import oracle
from gcnasm_amd import _lib, f4gemm
from helpers import assert_parity, bf16_compare

pytestmark = pytest.mark.gpu

NAMES = {(8, 1): "ga_mxfp8_bf16_BpreShuffle_256x256", (8, 0): "ga_mxfp8_bf16_noBpreShuffle_256x256",
         (4, 1): "ga_mxfp4_bf16_BpreShuffle_256x256", (4, 0): "ga_mxfp4_bf16_noBpreShuffle_256x256"}


def padded(q, pad, dev):
    """Codes q [rows, bytes] on the device with rows `pad` bytes of 0x7F (an E4M3
    NaN) apart, in storage that ends with the last one; the tensor and its stride."""
    rows, n = q.shape
    flat = torch.full((rows * (n + pad) - pad,), 0x7F, dtype=torch.uint8, device=dev)
    flat.as_strided((rows, n), (n + pad, 1)).copy_(torch.from_numpy(np.ascontiguousarray(q)))
    return flat, n + pad


def run(dev, M, N, K, elem, bps, fa=0, fb=0, l2=0, alpha=1.0, beta=0.0, pad_d=0, seed=1, pad_a=0,
        pad_b=0):
    xa = oracle.gen_mx_input(M, K, seed, 1.0, 4)
    xb = oracle.gen_mx_input(N, K, seed + 1, 1.0, 4)
    if elem == 4:
        (qa, sa), (qb, sb) = oracle.quant_mxfp4(xa), oracle.quant_mxfp4(xb)
    else:
        (qa, sa), (qb, sb) = oracle.quant_mx8(xa, fa), oracle.quant_mx8(xb, fb)
    sh = f4gemm.Shape(M, N, K, elem_bits=elem)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)  # noqa: E731
    A, lda = padded(qa, pad_a, dev)
    B, ldb = (t(f4gemm.shuffle_weight_16x16(qb, N, sh.Kp())), sh.Kp()) if bps else padded(
        qb, pad_b, dev)
    SA = t(f4gemm.shuffle_scale(sa, M, K // 32, sh.scale_a_rows(), sh.scale_cols()))
    SB = t(f4gemm.shuffle_scale(sb, N, K // 32, sh.scale_b_rows(), sh.scale_cols()))
    ldd = N + pad_d
    D = torch.full((M, ldd), float("nan"), dtype=torch.bfloat16, device=dev)
    C = torch.randn((M, ldd), generator=torch.Generator(device=dev).manual_seed(seed),
                    device=dev).to(torch.bfloat16) if beta else None
    name = NAMES[(elem, bps)] + ("_splitK" if l2 else "")
    cfg = [c for c in f4gemm.manifest() + f4gemm.manifest_fp4() if c.knl_name == name][0]
    ld = f4gemm.make_launch(cfg, M, N, K, l2)
    args = f4gemm.fill_args(D, C, A, B, SA, SB, M, N, K, ldd, sh.scale_cols(),
                            sh.scale_cols(), alpha, beta, ld.log2_k_split)
    args.stride_A0, args.stride_B0 = lda * 8 // elem, ldb * 8 // elem
    kern = f4gemm.Kernel().load(None, cfg)
    need = kern.workspace_bytes(ld, M, N) // 4
    # past the bytes the call may use: two slices that no kernel writes
    ws = torch.full((need + 2 * M * N,), float("nan"), dtype=torch.float32, device=dev)
    plan = kern.plan(args, ld.gdz, fmt_a=fa, fmt_b=fb)
    print("mx route", M, N, K, elem, bps, fa, fb, l2, flush=True)
    kern.launch(args, ld.gdx, ld.gdy, ld.gdz, workspace=ws, fmt_a=fa, fmt_b=fb)
    torch.cuda.synchronize()
    assert torch.isnan(D[:, N:]).all() and not torch.isnan(D[:, :N]).any()
    assert torch.isnan(ws[need:]).all()
    rows = np.unique(np.r_[np.arange(min(M, 24)), np.arange(max(0, M - 40), M),
                           np.arange(0, M, 97)])
    qr, sr = np.ascontiguousarray(qa[rows]), np.ascontiguousarray(sa[rows])
    if elem == 4:
        want = oracle.gemm_mx_fp32acc(qr, sr, qb, sb, 4, l2)
        dot = oracle.mx4_absdot(qr, sr, qb, sb)
    else:
        want = oracle.gemm_mx8_mfma(qr, sr, qb, sb, fa, fb, l2)
        dot = oracle.mx_absdot(qr, sr, qb, sb, fa, fb)
    want = (np.float32(alpha) * want).astype(np.float32)
    dot = abs(alpha) * dot
    if beta:
        c = C[:, :N].float().cpu().numpy()[rows]
        want, dot = want + np.float32(beta) * c, dot + abs(beta) * np.abs(c)
    got = D[:, :N].contiguous().view(torch.int16).cpu().numpy().view(np.uint16)[rows]
    ok, st = bf16_compare(got, oracle.to_bf16_bits(want), dot)
    assert_parity(st, "mx %dx%dx%d e%d bps%d f%d%d l%d" % (M, N, K, elem, bps, fa, fb, l2))
    return plan


# K-split: rows at the 32- and 64-row blocks, an odd number of 16-column groups,
# one group, more shares than CUs; K of one 256-K unit, an odd number of steps
# (MXFP8), fewer units than slices and long.
KSPLIT = [(1, 16, 256), (16, 48, 1280), (17, 1040, 512), (31, 528, 768), (33, 2064, 1024),
          (64, 144, 8192), (65, 16, 512), (96, 4112, 768), (129, 1040, 2304), (200, 3088, 1024),
          (300, 784, 1536), (500, 2064, 512), (1000, 272, 1024)]


@pytest.mark.parametrize("shape", KSPLIT)
@pytest.mark.parametrize("elem,bps", [(8, 1), (8, 0), (4, 1), (4, 0)])
def test_k_split(dev, shape, elem, bps):
    run(dev, *shape, elem, bps, pad_d=4, seed=sum(shape))


@pytest.mark.parametrize("M,N,K", [(40, 272, 128), (70, 144, 384), (150, 528, 1152)])
@pytest.mark.parametrize("bps", [1, 0])
def test_k_split_odd_steps(dev, M, N, K, bps):
    """MXFP8 K that is not a multiple of 256: the last slice ends in half a
    scale block; alpha, beta and C."""
    run(dev, M, N, K, 8, bps, alpha=0.5, beta=2.0, pad_d=8, seed=K)


@pytest.mark.parametrize("fa,fb", [(1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K,bps", [(48, 1040, 1024, 1), (130, 528, 768, 1),
                                       (130, 528, 768, 0), (900, 8192, 512, 1)])
def test_formats(dev, M, N, K, bps, fa, fb):
    run(dev, M, N, K, 8, bps, fa, fb, seed=M)


@pytest.mark.parametrize("l2", [1, 2, 3])
@pytest.mark.parametrize("M,N,K", [(17, 1040, 2048), (64, 2064, 4096), (48, 528, 2304)])
def test_k_split_keeps_a_callers_slices(dev, M, N, K, l2):
    """17-64 rows with a split: the caller's slices as the kernel's (a short
    last one among them), MXFP8 and MXFP4."""
    run(dev, M, N, K, 8, 1, l2=l2, seed=l2)
    run(dev, M, N, K, 4, 1, l2=l2, seed=l2)


# 17-64 rows, the slices over fewer workgroups along K than slices: 7 over 4,
# 5 over 3, 6 over 3 and 4 over 2, the last with one slice or two.
@pytest.mark.parametrize("M,N,K,l2,gdz,groups_k", [(20, 6000, 5120, 3, 7, 4), (64, 8192, 1280, 3, 5, 3),
                                                   (33, 7168, 1536, 3, 6, 3),
                                                   (17, 12288, 8448, 2, 4, 2)])
def test_slices_over_fewer_workgroups(dev, M, N, K, l2, gdz, groups_k):
    p = run(dev, M, N, K, 8, 1, l2=l2, pad_d=4, seed=gdz)
    assert (p.kernel, p.k_slices, p.k_workgroups) == (_lib.GA_MX_RUNS_FEW_ROWS_SPLIT, gdz, groups_k)


# The 128x256 tile: whole and ragged tiles, one K step to seven (its slots and
# scale ring wrap at 3 and 6), alpha / beta (the unstaged stores), and one
# round of tiles on the CUs exactly full.
HALF = [(1000, 8192, 128), (1024, 8192, 256), (900, 8208, 384), (1000, 8192, 640),
        (2048, 4096, 768), (1990, 4080, 896)]


@pytest.mark.parametrize("shape", HALF)
@pytest.mark.parametrize("bps", [1, 0])
def test_half_tile(dev, shape, bps):
    M, N, K = shape
    run(dev, M, N, K, 8, bps, seed=K)
    if K % 256 == 0:
        run(dev, M, N, 2 * K, 4, bps, seed=K)


# The 128x128 tile where its tiles fill one round: the same edges, its slots and
# scale ring wrapping at 4 and 6 steps, and the unstaged stores.
QUARTER = [(1000, 4096, 384), (2048, 2048, 128), (1990, 2064, 512), (512, 8192, 640),
           (500, 8192, 768), (1024, 4096, 896), (2048, 2048, 1152)]


@pytest.mark.parametrize("shape", QUARTER)
@pytest.mark.parametrize("bps", [1, 0])
def test_quarter_tile(dev, shape, bps):
    M, N, K = shape
    run(dev, M, N, K, 8, bps, seed=K)
    run(dev, M, N, 2 * K, 4, bps, seed=K)


def test_quarter_tile_formats_alpha_beta(dev):
    run(dev, 1000, 4096, 2048, 8, 1, 1, 0, alpha=-1.5, beta=0.25, pad_d=12, seed=5)
    run(dev, 1000, 4096, 2048, 8, 0, 0, 1, pad_d=4, seed=6)
    run(dev, 1000, 4096, 2048, 8, 1, 1, 1, seed=7)


def test_half_tile_alpha_beta(dev):
    run(dev, 1000, 8192, 512, 8, 1, alpha=-1.5, beta=0.25, pad_d=12, seed=3)


# More than 1024 rows whose 128x128 tiles leave half the CUs idle: the four-wave
# tile of the shape, whichever entry is named, whole and ragged.
@pytest.mark.parametrize("M,N,K", [(5290, 368, 1024), (4096, 512, 1152), (4090, 496, 1536)])
def test_shape_tile(dev, M, N, K):
    assert run(dev, M, N, K, 8, 1, pad_d=4, seed=K).kernel == _lib.GA_MX_RUNS_SHAPE_TILE
    if K % 256 == 0:
        p = run(dev, M, N, 2 * K, 4, 1, alpha=0.5, beta=2.0, seed=K)
        assert p.kernel == _lib.GA_MX_RUNS_SHAPE_TILE


@pytest.mark.parametrize("M,N,K,kernel", [
    (12, 8208, 5120, _lib.GA_MX_RUNS_FEW_ROWS), (24, 12288, 8448, _lib.GA_MX_RUNS_FEW_ROWS),
    (48, 20496, 5120, _lib.GA_MX_RUNS_FEW_ROWS_SHARED_A), (40, 272, 768, _lib.GA_MX_RUNS_K_SPLIT),
    (300, 784, 1536, _lib.GA_MX_RUNS_K_SPLIT), (1000, 2064, 2048, _lib.GA_MX_RUNS_TILE128),
    (1000, 8192, 512, _lib.GA_MX_RUNS_TILE128), (5290, 368, 1024, _lib.GA_MX_RUNS_SHAPE_TILE),
    (2100, 4368, 512, _lib.GA_MX_RUNS_ENTRY)])
@pytest.mark.parametrize("elem,bps", [(8, 1), (8, 0), (4, 1), (4, 0)])
def test_strided_operands(dev, M, N, K, kernel, elem, bps):
    """A and row-major B with NaN codes between their rows and nothing behind the
    last one, every kernel (row-major B runs some of the shapes on another)."""
    p = run(dev, M, N, K, elem, bps, seed=K, pad_a=16, pad_b=48)
    assert elem == 4 or bps == 0 or p.kernel == kernel


@pytest.mark.parametrize("elem", [8, 4])
def test_more_tiles_than_cus(dev, elem):
    """Past one round of 128x256 tiles: the entry's own kernel, ragged."""
    run(dev, 2100, 4368, 512, elem, 1, seed=elem)
    run(dev, 2100, 4368, 256, elem, 0, seed=elem + 1)
