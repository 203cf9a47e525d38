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
        pad_b=0, entry=None):
    """One launch of the 256x256 entry (or `entry`) against the oracle, on a
    sample of rows and, of large weights, of columns; the plan it ran."""
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
    name = entry or NAMES[(elem, bps)] + ("_splitK" if l2 else "")
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
    cols = np.arange(N)
    if N * K > 3e7:  # the first and last, and every 53rd 16-column group
        cols = np.unique(np.r_[np.arange(300), np.arange(N - 300, N),
                               np.flatnonzero(np.arange(N) // 16 % 53 == 0)])
        qb, sb = np.ascontiguousarray(qb[cols]), np.ascontiguousarray(sb[cols])
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
        c = C[:, :N].float().cpu().numpy()[np.ix_(rows, cols)]
        want, dot = want + np.float32(beta) * c, dot + abs(beta) * np.abs(c)
    got = D[:, :N].contiguous().view(torch.int16).cpu().numpy().view(np.uint16)[np.ix_(rows, cols)]
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
    p = run(dev, *shape, elem, bps, pad_d=4, seed=sum(shape))
    assert p.kernel == _lib.GA_MX_RUNS_K_SPLIT


# Its larger wave tiles, with each number of slices: a short last row block, an odd
# number of 16-column groups, more column shares than row blocks and fewer.
@pytest.mark.parametrize("elem,shape,cut", [
    (8, (513, 2064, 512), (64, 32, 2)), (8, (100, 2064, 2048), (64, 32, 4)),
    (8, (100, 2064, 4096), (64, 32, 8)), (8, (450, 4112, 512), (64, 64, 2)),
    (8, (100, 6160, 2048), (64, 64, 4)), (8, (100, 4112, 4096), (64, 64, 8)),
    (4, (100, 2064, 4096), (64, 32, 4)), (4, (100, 2064, 6144), (64, 32, 8)),
    (4, (450, 4112, 512), (64, 64, 2)), (4, (100, 6160, 3072), (64, 64, 4)),
    (4, (100, 4112, 8192), (64, 64, 8)), (8, (70, 272, 6144), (32, 32, 8))])
@pytest.mark.parametrize("bps", [1, 0])
def test_k_split_cuts(dev, elem, shape, cut, bps):
    p = run(dev, *shape, elem, bps, pad_d=4, seed=sum(shape))
    assert (p.kernel, p.rows, p.cols, p.k_slices) == (_lib.GA_MX_RUNS_K_SPLIT,) + cut


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
HALF = [(1000, 8192, 128), (1024, 8192, 256), (1990, 2064, 384), (1000, 8192, 640),
        (2048, 4096, 768), (1990, 4080, 896)]


@pytest.mark.parametrize("shape", HALF)
@pytest.mark.parametrize("bps", [1, 0])
def test_half_tile(dev, shape, bps):
    M, N, K = shape
    half = (_lib.GA_MX_RUNS_TILE128, 128, 256)
    p = run(dev, M, N, K, 8, bps, seed=K)
    assert (p.kernel, p.rows, p.cols) == half
    p = run(dev, M, N, 2 * K, 4, bps, seed=K)
    assert (p.kernel, p.rows, p.cols) == half


# The 128x128 tile where its tiles fill one round: the same edges, its slots and
# scale ring wrapping at 4 and 6 steps, and the unstaged stores.
QUARTER = [(8, 1000, 4096, 384), (8, 2048, 2048, 128), (8, 1900, 2064, 512), (8, 512, 8192, 640),
           (8, 500, 8192, 768), (8, 1024, 4096, 896), (8, 2048, 2048, 1152), (8, 1000, 2064, 2048),
           (4, 1500, 2576, 1536), (4, 1900, 2064, 2048), (4, 2048, 2048, 2304),
           (4, 1990, 1936, 2304), (4, 1000, 2064, 4096)]


@pytest.mark.parametrize("shape", QUARTER)
@pytest.mark.parametrize("bps", [1, 0])
def test_quarter_tile(dev, shape, bps):
    elem, M, N, K = shape
    p = run(dev, M, N, K, elem, bps, seed=K)
    assert (p.kernel, p.rows, p.cols) == (_lib.GA_MX_RUNS_TILE128, 128, 128)


def test_quarter_tile_formats_alpha_beta(dev):
    """Ragged tiles and formats; alpha and beta take the unstaged stores."""
    run(dev, 1000, 2064, 4096, 4, 1, alpha=-1.5, beta=0.25, pad_d=12, seed=4)
    run(dev, 1000, 2064, 2048, 8, 1, 1, 0, alpha=-1.5, beta=0.25, pad_d=12, seed=4)
    run(dev, 1000, 4096, 2048, 8, 1, 1, 0, alpha=-1.5, beta=0.25, pad_d=12, seed=5)
    run(dev, 1000, 4096, 2048, 8, 0, 0, 1, pad_d=4, seed=6)
    run(dev, 1000, 4096, 2048, 8, 1, 1, 1, seed=7)


def test_half_tile_alpha_beta(dev):
    run(dev, 1000, 8192, 512, 8, 1, alpha=-1.5, beta=0.25, pad_d=12, seed=3)


# More than 1024 rows whose 128x128 tiles leave half the CUs idle: the four-wave
# tile of the shape, whichever entry is named, whole and ragged.
@pytest.mark.parametrize("M,N,K", [(3000, 368, 3328), (4096, 512, 3200), (4090, 496, 3072)])
def test_shape_tile(dev, M, N, K):
    assert run(dev, M, N, K, 8, 1, pad_d=4, seed=K).kernel == _lib.GA_MX_RUNS_SHAPE_TILE
    if K % 256 == 0:
        p = run(dev, M, N, 2 * K, 4, 1, alpha=0.5, beta=2.0, seed=K)
        assert p.kernel == _lib.GA_MX_RUNS_SHAPE_TILE


@pytest.mark.parametrize("M,N,K,kernel", [
    (12, 8208, 5120, _lib.GA_MX_RUNS_FEW_ROWS), (24, 12288, 8448, _lib.GA_MX_RUNS_FEW_ROWS),
    (48, 20496, 5120, _lib.GA_MX_RUNS_FEW_ROWS_SHARED_A), (40, 272, 768, _lib.GA_MX_RUNS_K_SPLIT),
    (300, 784, 1536, _lib.GA_MX_RUNS_K_SPLIT), (1000, 2064, 2048, _lib.GA_MX_RUNS_TILE128),
    (1000, 8192, 512, _lib.GA_MX_RUNS_TILE128), (3000, 368, 3328, _lib.GA_MX_RUNS_SHAPE_TILE),
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
    for shape, bps in (((2100, 4368, 512), 1), ((2100, 4368, 256), 0), ((900, 8208, 768), 1)):
        p = run(dev, *shape, elem, bps, seed=elem)
        assert p.kernel == _lib.GA_MX_RUNS_ENTRY


@pytest.mark.parametrize("name", [c.knl_name for c in f4gemm.manifest() + f4gemm.manifest_fp4()])
@pytest.mark.parametrize("steps", [1, 3, 6])
def test_every_entry_past_one_round(dev, name, steps):
    """Each manifest entry's own tile on one slice, which the shape rule leaves to
    it past one round of 128x256 tiles: rows and columns that end in 8 and 16 of
    every tile, one to six K steps."""
    elem = 4 if "mxfp4" in name else 8
    p = run(dev, 520, 13328, steps * (128 if elem == 8 else 256), elem, int("noBpre" not in name),
            pad_d=4, seed=steps, entry=name)
    assert p.kernel == _lib.GA_MX_RUNS_ENTRY


# The few-row kernels where the rule leaves calls to them (names: test_route).
# One slice, B from memory: a wave per group for one and eight rows; A through LDS
# for 9-16 rows of many columns, two groups per wave of fewer; 17-32 and 33-64 rows
# with more steps in flight for one two-group task per CU, eight waves of two
# groups, a wave per group; five to seven groups per wave, the last wave short; A
# shared by eight waves of one group (5-7 per workgroup, a ring that wraps within
# a slice) and four of four.
FEW, SPLIT, SHARED = (_lib.GA_MX_RUNS_FEW_ROWS, _lib.GA_MX_RUNS_FEW_ROWS_SPLIT,
                      _lib.GA_MX_RUNS_FEW_ROWS_SHARED_A)
FEW_ROWS = [(1, 8208, 5120, 1, FEW, 0), (8, 20496, 2048, 1, FEW, 0), (9, 16448, 3200, 1, FEW, 0),
            (16, 8208, 6272, 1, FEW, 0), (24, 8192, 12544, 1, FEW, 0), (31, 12304, 8448, 0, FEW, 0),
            (64, 8192, 12544, 1, FEW, 0), (40, 8192, 12416, 0, FEW, 0), (48, 16384, 6272, 1, FEW, 0),
            (33, 4080, 25088, 1, FEW, 0), (20, 19216, 5376, 1, SPLIT, 80),
            (24, 22400, 4608, 1, SPLIT, 96), (32, 28656, 3584, 1, SPLIT, 112),
            (20, 22400, 4608, 0, SPLIT, 96), (33, 24576, 4224, 1, SHARED, 96),
            (33, 24576, 4224, 0, SHARED, 96), (40, 20496, 5120, 1, SHARED, 96),
            (64, 28672, 3712, 1, SHARED, 112), (64, 32784, 3328, 1, SHARED, 80),
            (64, 32784, 3200, 0, SHARED, 80)]


@pytest.mark.parametrize("M,N,K,bps,kernel,cols", FEW_ROWS)
def test_few_rows_one_slice(dev, M, N, K, bps, kernel, cols):
    p = run(dev, M, N, K, 8, bps, pad_d=4, seed=M + K)
    assert (p.kernel, p.cols, p.k_slices) == (kernel, cols, 1)


@pytest.mark.parametrize("M,N,K,kernel", [(12, 16448, 8192, FEW), (16, 8208, 12800, FEW),
                                          (24, 8192, 25088, FEW), (24, 22400, 9216, SPLIT),
                                          (64, 28672, 7680, SHARED)])
def test_few_rows_one_slice_fp4(dev, M, N, K, kernel):
    assert run(dev, M, N, K, 4, 1, pad_d=4, seed=M).kernel == kernel


# A caller's slices over workgroups: three of 512, 512 and 128 K with each number of
# groups per wave (16-column groups: 65 a last wave of one; 515 and 1025 ragged), the
# second workgroup with one slice where there are two; and all in one workgroup for
# N of five groups per CU and more, 17-32 rows and, A shared, 33-64.
SPLITS = [(N, 1152, 2, M, SPLIT, 16 * g, 3, kw)
          for N, g, kw in ((1040, 2, 3), (5440, 4, 3), (6800, 5, 3), (8192, 6, 3), (8240, 7, 3),
                           (10240, 8, 3), (16400, 5, 2), (19216, 5, 2))
          for M in (20, 64)]
SPLITS += [(28656, 2048, 3, 24, SPLIT, 112, 8, 1), (22400, 1152, 2, 17, SPLIT, 96, 3, 1),
           (28656, 2048, 3, 40, SHARED, 112, 8, 1), (22400, 1152, 2, 33, SHARED, 96, 3, 1),
           (24592, 1152, 1, 64, SHARED, 112, 2, 1), (32784, 1152, 2, 48, SHARED, 80, 3, 1)]


@pytest.mark.parametrize("N,K,l2,M,kernel,cols,slices,groups_k", SPLITS)
@pytest.mark.parametrize("bps", [1, 0])
def test_few_rows_callers_slices(dev, N, K, l2, M, kernel, cols, slices, groups_k, bps):
    entry = None if bps else "ga_mxfp8_bf16_noBpreShuffle_128x128_splitK"
    p = run(dev, M, N, K, 8, bps, l2=l2, pad_d=4, alpha=0.5, beta=2.0, seed=N + M, entry=entry)
    assert (p.kernel, p.cols, p.k_slices, p.k_workgroups) == (kernel, cols, slices, groups_k)
    if bps:
        p = run(dev, M, N, 2 * K, 4, 1, l2=l2, pad_d=4, seed=N + M)
        assert (p.kernel, p.k_slices) == (kernel, slices)


@pytest.mark.parametrize("fa,fb", [(1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M,N,K,l2,kernel", [(12, 8208, 5120, 0, FEW), (40, 8192, 12544, 0, FEW),
                                             (20, 8192, 1152, 2, SPLIT), (24, 28656, 2048, 3, SPLIT),
                                             (40, 28656, 2048, 3, SHARED), (64, 32784, 1152, 2, SHARED)])
def test_few_rows_formats(dev, M, N, K, l2, kernel, fa, fb):
    assert run(dev, M, N, K, 8, 1, fa, fb, l2=l2, pad_d=4, seed=M).kernel == kernel
