"""GPU parity of the MXFP4 path (e2m1 operands behind the f4gemm ABI).

The reference drives aiter's f4gemm_bf16_per1x32Fp4 code objects
(asm_f4gemm/README.md:1-40); these tests follow its regression sweep
(asm_f4gemm/run_tests.sh) on the MXFP4 manifest: heuristic shapes, every
manifest kernel at M=300 N=2048 K=1024, split-K, edge tiles, and the device
quantiser. Expected GEMM values come from oracle.gemm_mx_fp32acc(bits=4)
(exact 128-K step sums accumulated in fp32 in the kernel's K order) rounded
to bf16: for e2m1 operands that is the oracle's MFMA model itself (a product
of two e2m1 values has at most 4 significant bits and the exponent sums of one
group span at most 6 binades, so the MFMA's 13-bit alignment truncates
nothing), so outputs are held to the north-star rule, with the same capped
residual allowance as MXFP8 for what the model leaves out (the hardware's
second alignment of the terms of a step, which shows on long-K outputs that
cancel); quantised codes, scales and packing are compared bit for bit with
the oracle.
"""
import numpy as np
import pytest
import torch

import oracle
from gcnasm_amd import f4gemm, ops
from gcnasm_amd._lib import GaError
from helpers import assert_parity, bf16_compare

pytestmark = pytest.mark.gpu


def mx4_operands(M, N, K, seed=1, rule=0, spread=4):
    xa = oracle.gen_mx_input(M, K, seed * 7919 + 1, 1.0, spread)
    xb = oracle.gen_mx_input(N, K, seed * 7919 + 2, 1.0, spread)
    qa, sa = oracle.quant_mxfp4(xa, rule)
    qb, sb = oracle.quant_mxfp4(xb, rule)
    return qa, sa, qb, sb


def cfg4(name):
    for c in f4gemm.manifest_fp4():
        if c.knl_name == name:
            return c
    raise KeyError(name)


def run_mx4(dev, qa, sa, qb, sb, cfg, log2_k_split=0):
    M, Kp = qa.shape
    K = 2 * Kp
    N = qb.shape[0]
    sh = f4gemm.Shape(M, N, K, elem_bits=4)
    a_pad = np.zeros((sh.a_rows_pad(), Kp), dtype=np.uint8)
    a_pad[:M] = qa
    A = torch.from_numpy(a_pad).to(dev)
    bh = f4gemm.shuffle_weight_16x16(qb, N, Kp) if cfg.bpreshuffle else qb.reshape(-1)
    B = torch.from_numpy(np.ascontiguousarray(bh)).to(dev)
    SA = torch.from_numpy(f4gemm.shuffle_scale(sa, M, K // 32, sh.scale_a_rows(),
                                               sh.scale_cols())).to(dev)
    SB = torch.from_numpy(f4gemm.shuffle_scale(sb, N, K // 32, sh.scale_b_rows(),
                                               sh.scale_cols())).to(dev)
    D = torch.full((sh.d_rows_pad(), N), float("nan"), dtype=torch.bfloat16, device=dev)
    ld = f4gemm.make_launch(cfg, M, N, K, log2_k_split)
    args = f4gemm.fill_args(D, None, A, B, SA, SB, M, N, K, N, sh.scale_cols(), sh.scale_cols(),
                            1.0, 0.0, ld.log2_k_split)
    k = f4gemm.Kernel().load(None, cfg)
    print("launch %s M=%d N=%d K=%d grid=(%d,%d,%d)" % (cfg.knl_name, M, N, K, ld.gdx, ld.gdy,
                                                         ld.gdz), flush=True)
    k.launch(args, ld.gdx, ld.gdy, ld.gdz)
    torch.cuda.synchronize()
    return D[:M].view(torch.int16).cpu().numpy().view(np.uint16)


def check4(got, qa, sa, qb, sb, l2, label):
    want = oracle.to_bf16_bits(oracle.gemm_mx_fp32acc(qa, sa, qb, sb, 4, l2))
    ok, st = bf16_compare(got, want, oracle.mx4_absdot(qa, sa, qb, sb))
    assert_parity(st, label)
    return st


FP4_MANIFEST = ["ga_mxfp4_bf16_BpreShuffle_%s" % t for t in
                ("256x256", "256x128", "128x256", "128x128", "64x256", "32x256")] + \
               ["ga_mxfp4_bf16_BpreShuffle_%s_splitK" % t for t in
                ("256x256", "256x128", "128x256", "128x128", "64x256", "32x256", "32x512")] + \
               ["ga_mxfp4_bf16_noBpreShuffle_256x256", "ga_mxfp4_bf16_noBpreShuffle_256x128",
                "ga_mxfp4_bf16_noBpreShuffle_128x128_splitK"] + \
               ["ga_mxfp4_bf16_BpreShuffle_96x640", "ga_mxfp4_bf16_BpreShuffle_128x512",
                "ga_mxfp4_bf16_BpreShuffle_96x640_splitK",
                "ga_mxfp4_bf16_BpreShuffle_128x512_splitK"]

# Tile names in the reference's own (aiter) form: the ones its files name
# (asm_f4gemm/README.md:25-31 and :174, run_tests.sh:51-52) and more shapes of
# that naming; ga_kernel_find resolves each (the tile fixes the grid and the
# split contract; the library runs its own compiled tile for the shape).
AITER_TILES = ["BpreShuffle_256x256", "BpreShuffle_96x640", "BpreShuffle_128x512",
               "noBpreShuffle_256x256", "BpreShuffle_32x128", "BpreShuffle_64x384",
               "BpreShuffle_160x256", "BpreShuffle_224x256", "BpreShuffle_192x128"]


def aiter_cfg(tile):
    import re
    m = re.search(r"(\d+)x(\d+)$", tile)
    name = "f4gemm_bf16_per1x32Fp4_%s.co" % tile
    return f4gemm.Config(int(m.group(1)), int(m.group(2)), 1, int(not tile.startswith("no")),
                         name, name)


def test_manifest_fp4_rows():
    """The MXFP4 manifest carries the MXFP8 manifest's tiles in its order."""
    rows = f4gemm.manifest_fp4()
    assert [c.knl_name for c in rows] == FP4_MANIFEST
    assert [c.knl_name.replace("mxfp4", "mxfp8") for c in rows] == \
        [c.knl_name for c in f4gemm.manifest()]
    assert f4gemm.manifest_fp4_csv().splitlines()[0] == \
        "tile_M,tile_N,splitK,bpreshuffle,knl_name,co_name"


@pytest.mark.parametrize("name", FP4_MANIFEST)
def test_every_fp4_kernel(dev, name):
    M, N, K = 300, 2048, 1024
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=3)
    got = run_mx4(dev, qa, sa, qb, sb, cfg4(name))
    st = check4(got, qa, sa, qb, sb, 0, name)
    assert st["exact"] > 0.95


@pytest.mark.parametrize("tile", AITER_TILES)
def test_aiter_tile_names(dev, tile):
    """Every manifest kernel at M=300 N=2048 K=1024 (run_tests.sh:43-49),
    found by its aiter name."""
    M, N, K = 300, 2048, 1024
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=3)
    got = run_mx4(dev, qa, sa, qb, sb, aiter_cfg(tile))
    check4(got, qa, sa, qb, sb, 0, "aiter %s" % tile)


@pytest.mark.parametrize("tile", ["BpreShuffle_256x256", "BpreShuffle_128x512"])
@pytest.mark.parametrize("l2", [1, 2, 3, 4])
def test_aiter_tile_splitk(dev, tile, l2):
    """The reference's split-K sweep (run_tests.sh:51-57): M=256 N=1024 K=4096
    with log2_k_split 1..4 on its 256x256 and 128x512 tiles."""
    M, N, K = 256, 1024, 4096
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=20 + l2)
    got = run_mx4(dev, qa, sa, qb, sb, aiter_cfg(tile), l2)
    check4(got, qa, sa, qb, sb, l2, "aiter %s L=%d" % (tile, l2))


@pytest.mark.parametrize("shape", [(256, 256, 512), (1, 512, 256), (17, 784, 1280),
                                   (520, 784, 2304), (256, 4096, 256), (2048, 1024, 1024)])
def test_fp4_edge_shapes(dev, shape):
    """Partial M and N tiles, one or an odd number of 256-K steps, one row."""
    M, N, K = shape
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=M + N + K)
    for name in ("ga_mxfp4_bf16_BpreShuffle_256x256", "ga_mxfp4_bf16_noBpreShuffle_256x256",
                 "ga_mxfp4_bf16_BpreShuffle_128x128", "ga_mxfp4_bf16_noBpreShuffle_256x128"):
        got = run_mx4(dev, qa, sa, qb, sb, cfg4(name))
        check4(got, qa, sa, qb, sb, 0, "%s %s" % (shape, name))


@pytest.mark.parametrize("l2", [1, 2, 3])
@pytest.mark.parametrize("name", ["ga_mxfp4_bf16_BpreShuffle_256x256_splitK",
                                  "ga_mxfp4_bf16_BpreShuffle_128x128_splitK",
                                  "ga_mxfp4_bf16_noBpreShuffle_128x128_splitK"])
def test_fp4_splitk(dev, l2, name):
    M, N, K = 96, 1024, 4096
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=7 + l2)
    got = run_mx4(dev, qa, sa, qb, sb, cfg4(name), l2)
    check4(got, qa, sa, qb, sb, l2, "%s L=%d" % (name, l2))


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("NKL", [(784, 1280, 0), (784, 1280, 1), (4096, 2048, 0),
                                 (4096, 2048, 2), (1808, 3072, 3)])
def test_fp4_decode_path(dev, M, NKL):
    """Up to 64 rows, K slices summed in slice order: the few-row kernel for 1-16
    rows with a split, the K-split kernel for the rest of these small weights."""
    N, K, l2 = NKL
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=M * 31 + N + l2)
    name = ("ga_mxfp4_bf16_BpreShuffle_256x256_splitK" if l2 else
            "ga_mxfp4_bf16_BpreShuffle_256x256")
    got = run_mx4(dev, qa, sa, qb, sb, cfg4(name), l2)
    check4(got, qa, sa, qb, sb, l2, "decode M=%d N=%d K=%d L=%d" % (M, N, K, l2))


@pytest.mark.parametrize("M", [1, 12, 16])
@pytest.mark.parametrize("NKL", [(16384, 2048, 1), (16384, 2304, 2), (4096, 4096, 3),
                                 (784, 1280, 2), (16384, 16384, 0), (28672, 8192, 1)])
def test_fp4_decode_sequential_slices(dev, M, NKL):
    """1-16 rows, MXFP4: several K slices per wave (one fp32 chain each,
    summed in slice order), as for MXFP8; at 12 and 16 rows with wide N the
    A panel in LDS (K = 16384 fills its 128 KB)."""
    N, K, l2 = NKL
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=M * 17 + l2)
    got = run_mx4(dev, qa, sa, qb, sb, cfg4("ga_mxfp4_bf16_BpreShuffle_256x256_splitK"), l2)
    check4(got, qa, sa, qb, sb, l2, "decode sequential slices M=%d N=%d K=%d L=%d" %
           (M, N, K, l2))


def test_fp4_decode_deep(dev):
    """33-64 rows of 64 MB of weights and long K: the K-split kernel."""
    M, N, K = 40, 8192, 16384
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=77)
    got = run_mx4(dev, qa, sa, qb, sb, cfg4("ga_mxfp4_bf16_BpreShuffle_256x128_splitK"), 0)
    check4(got, qa, sa, qb, sb, 0, "decode deep M=%d N=%d K=%d" % (M, N, K))


@pytest.mark.parametrize("MNKL", [(64, 8192, 32768, 1), (64, 8192, 65536, 2),
                                  (24, 8192, 32768, 1)])
def test_fp4_decode_deep_k_split(dev, MNKL):
    """Weights from memory in a caller's 2 or 4 slices of at least 64 steps each."""
    M, N, K, l2 = MNKL
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=M + l2)
    got = run_mx4(dev, qa, sa, qb, sb, cfg4("ga_mxfp4_bf16_BpreShuffle_256x128_splitK"), l2)
    check4(got, qa, sa, qb, sb, l2, "decode deep M=%d N=%d K=%d L=%d" % (M, N, K, l2))


@pytest.mark.parametrize("name", ["ga_mxfp4_bf16_BpreShuffle_256x256",
                                  "ga_mxfp4_bf16_BpreShuffle_256x256_splitK",
                                  "ga_mxfp4_bf16_noBpreShuffle_256x256"])
def test_fp4_persistent_many_tiles(dev, name):
    """272 tiles of 256x256 on a persistent grid of one workgroup per CU:
    workgroups compute a second tile; every output checked."""
    M, N, K = 4352, 4096, 512
    cfg = cfg4(name)
    l2 = 1 if cfg.splitK else 0
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=4352)
    got = run_mx4(dev, qa, sa, qb, sb, cfg, l2)
    check4(got, qa, sa, qb, sb, l2, "persistent %s" % name)


@pytest.mark.parametrize("M", [33, 64])
def test_fp4_few_rows_wide_n(dev, M):
    """33-64 rows over wide N that is not a multiple of 256."""
    N, K = 28672 - 16, 512
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=M + 5)
    got = run_mx4(dev, qa, sa, qb, sb, cfg4("ga_mxfp4_bf16_BpreShuffle_256x128_splitK"), 0)
    check4(got, qa, sa, qb, sb, 0, "few rows wide N M=%d" % M)


def test_fp4_decode_plain_b(dev):
    M, N, K = 16, 1024, 2048
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=77)
    got = run_mx4(dev, qa, sa, qb, sb, cfg4("ga_mxfp4_bf16_noBpreShuffle_256x256"))
    check4(got, qa, sa, qb, sb, 0, "decode plain B")


@pytest.mark.parametrize("M", [24, 64])
@pytest.mark.parametrize("bps", [True, False])
@pytest.mark.parametrize("NKL", [(1040, 4096, 2), (8192, 2048, 2), (19216, 512, 0),
                                 (28672 - 16, 512, 0), (28672 - 16, 1024, 1),
                                 (19216, 2048, 2)])
def test_fp4_decode_split_across_workgroups(dev, M, bps, NKL):
    """17-64 rows in a caller's slices or one, ragged columns."""
    N, K, l2 = NKL
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=M + 9)
    name = ("ga_mxfp4_bf16_BpreShuffle_256x256_splitK" if bps else
            "ga_mxfp4_bf16_noBpreShuffle_128x128_splitK")
    got = run_mx4(dev, qa, sa, qb, sb, cfg4(name), l2)
    check4(got, qa, sa, qb, sb, l2, "decode split %s M=%d" % (name, M))


@pytest.mark.parametrize("MNKB", [(64, 32784, 1792, True), (40, 20480, 2304, False),
                                  (33, 24576, 1280, True)])
def test_fp4_decode_shared_a(dev, MNKB):
    """33-64 rows at one slice over wide N, 5 to 9 steps, at the shapes of the
    shared-A variant, which takes such N from 96 MB of weights on
    (test_gpu_mx_routes.py)."""
    M, N, K, bps = MNKB
    qa, sa, qb, sb = mx4_operands(M, N, K, seed=M + K)
    name = ("ga_mxfp4_bf16_BpreShuffle_256x256" if bps else
            "ga_mxfp4_bf16_noBpreShuffle_256x256")
    got = run_mx4(dev, qa, sa, qb, sb, cfg4(name), 0)
    check4(got, qa, sa, qb, sb, 0, "decode shared-A %s M=%d N=%d K=%d" % (name, M, N, K))


def test_fp4_k_not_multiple_of_256_is_rejected(dev):
    M, N, K = 64, 256, 384
    sh = f4gemm.Shape(M, N, K, elem_bits=4)
    A = torch.zeros((sh.a_rows_pad(), K // 2), dtype=torch.uint8, device=dev)
    B = torch.zeros((N, K // 2), dtype=torch.uint8, device=dev)
    S = torch.full((sh.scale_b_rows() * sh.scale_cols(),), 127, dtype=torch.uint8, device=dev)
    D = torch.empty((sh.d_rows_pad(), N), dtype=torch.bfloat16, device=dev)
    cfg = cfg4("ga_mxfp4_bf16_BpreShuffle_256x256")
    ld = f4gemm.make_launch(cfg, M, N, K, 0)
    args = f4gemm.fill_args(D, None, A, B, S, S, M, N, K, N, sh.scale_cols(), sh.scale_cols(),
                            1.0, 0.0, 0)
    with pytest.raises(GaError):
        f4gemm.Kernel().load(None, cfg).launch(args, ld.gdx, ld.gdy, ld.gdz)


def edge_input(rows, K, seed):
    x = oracle.gen_mx_input(rows, K, seed, 1.0, 6)
    flat = x.reshape(-1)
    mids = np.array([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], np.float32)
    flat[:64] = np.concatenate([mids, -mids, [0.0, -0.0, 6.0, -6.0, 7.5, 1e-40, -1e-40,
                                              np.inf, -np.inf, np.nan]]
                               + [np.zeros(64 - 24, np.float32)])[:64]
    x[1, :32] = 0.0                                  # zero block
    x[2, :32] = np.float32(1e-42)                    # subnormal block
    x[3, 5] = 6.0 * 2.0 ** 9                         # exact block maximum
    return x


@pytest.mark.parametrize("rule", [0, 1, 2])
@pytest.mark.parametrize("in_dtype", [torch.float32, torch.bfloat16])
def test_quant_mxfp4_bit_exact(dev, rule, in_dtype):
    rows, K = 96, 1024
    x = edge_input(rows, K, 40 + rule)
    xt = torch.from_numpy(x).to(dev).to(in_dtype)
    xr = xt.float().cpu().numpy()                    # the values the kernel sees
    q, s = ops.quant_mxfp4(xt, scale_rule=rule)
    wq, ws = oracle.quant_mxfp4(xr, rule)
    np.testing.assert_array_equal(s.cpu().numpy(), ws)
    np.testing.assert_array_equal(q.cpu().numpy(), wq)


def test_e2m1_encoder_every_bf16_value(dev):
    """Every 1x32 block holds 6.0 and 31 test values, so its scale exponent is 0
    (rule 0: floor(log2(amax/6))) and each code is e2m1(x) itself: every bf16
    bit pattern of magnitude <= 6 (and every NaN) goes through the device
    encoder and is compared with the oracle's."""
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    vals = oracle.bf16_bits_to_f32(bits)
    keep = np.isnan(vals) | (np.abs(vals) <= 6.0)
    v = vals[keep]
    nblk = (v.size + 30) // 31
    v = np.concatenate([v, np.zeros(nblk * 31 - v.size, np.float32)]).reshape(nblk, 31)
    x = np.concatenate([np.full((nblk, 1), 6.0, np.float32), v], axis=1)
    rows = 64
    nb = (nblk + rows - 1) // rows
    xp = np.zeros((rows * nb, 32), np.float32)
    xp[:, 0] = 6.0
    xp[:nblk] = x
    x = np.ascontiguousarray(xp.reshape(rows, nb * 32))
    for t in (torch.from_numpy(x).to(dev),
              torch.from_numpy(oracle.to_bf16_bits(x).view(np.int16)).to(dev).view(torch.bfloat16)):
        q, s = ops.quant_mxfp4(t, scale_rule=0)
        torch.cuda.synchronize()
        wq, ws = oracle.quant_mxfp4(x, 0)
        assert (ws == 127).all()
        np.testing.assert_array_equal(s.cpu().numpy(), ws)
        np.testing.assert_array_equal(q.cpu().numpy(), wq)


def test_mxfp4_gemm_one_call(dev):
    """ops.mxfp4_gemm (device quantiser, device shuffles, heuristic over the MXFP4
    manifest) against the oracle on the codes the device produced."""
    M, N, K = 384, 1536, 2048
    xa = torch.from_numpy(oracle.gen_mx_input(M, K, 5, 1.0, 4)).to(dev)
    xb = torch.from_numpy(oracle.gen_mx_input(N, K, 6, 1.0, 4)).to(dev)
    a = ops.prepare_mx4_a(xa)
    b = ops.prepare_mx4_b(xb)
    out, idx, ld = ops.mxfp4_gemm(a, b)
    torch.cuda.synchronize()
    qa, sa = ops.quant_mxfp4(xa)
    qb, sb = ops.quant_mxfp4(xb)
    got = out[:M].view(torch.int16).cpu().numpy().view(np.uint16)
    check4(got, qa.cpu().numpy(), sa.cpu().numpy(), qb.cpu().numpy(), sb.cpu().numpy(),
           ld.log2_k_split, "one-call")
