"""The kernels that MX launches run, as the host plans them for a device of 256
compute units (CPU only)."""
import pytest

from gcnasm_amd import _lib, f4gemm


def plan(name, M, N, K, l2, num_cu=256, fmt=(0, 0)):
    """(ga_mx_plan, gdz) of a launch of the entry `name`."""
    cfg = [c for c in f4gemm.manifest() + f4gemm.manifest_fp4() if c.knl_name == name][0]
    ld = f4gemm.make_launch(cfg, M, N, K, l2)
    args = f4gemm.fill_args(None, None, None, None, None, None, M, N, K, N, K // 32, K // 32,
                            1.0, 0.0, ld.log2_k_split)
    return f4gemm.Kernel().load(None, cfg).plan(args, ld.gdz, num_cu, *fmt), ld.gdz


@pytest.mark.parametrize("name", ["ga_mxfp8_bf16_BpreShuffle_256x256_splitK",
                                  "ga_mxfp4_bf16_BpreShuffle_256x256_splitK"])
@pytest.mark.parametrize("num_cu", [256, 304, 80])
def test_every_workgroup_along_k_has_a_slice(name, num_cu):
    """17-64 rows split over workgroups along K: each runs ceil(slices /
    workgroups) consecutive slices and writes their partials into a workspace
    of `slices` slices, so the last one's first slice has to be one of them."""
    seen = set()
    for l2 in (1, 2, 3):
        for K in (512, 1280, 1536, 5120, 8192, 28672, 65536):
            for N in range(16, 20000, 176):
                for M in (17, 64):
                    p, gdz = plan(name, M, N, K, l2, num_cu)
                    assert 1 <= p.k_workgroups <= gdz
                    if p.kernel != _lib.GA_MX_RUNS_FEW_ROWS_SPLIT:
                        continue
                    assert p.k_slices == gdz
                    per = -(-gdz // p.k_workgroups)
                    assert (p.k_workgroups - 1) * per < gdz, (M, N, K, l2, gdz, p.k_workgroups)
                    assert per <= 2 or p.k_workgroups == 1  # a wave parks one chain
                    seen.add((gdz, p.k_workgroups))
    assert len(seen) >= 5, seen


# Both sides of the lines of the rule that picks a kernel, on 256 CUs: entry,
# M, N, K, log2 split -> kernel.
ENTRY, KSPLIT, TILE128, FEW, SPLIT, SHARED, SHAPE = range(7)
P8, P8R, P4 = ("ga_mxfp8_bf16_BpreShuffle_256x256", "ga_mxfp8_bf16_noBpreShuffle_256x256",
               "ga_mxfp4_bf16_BpreShuffle_256x256")
ROUTES = [
    # one slice, up to 16 rows: 32 MB of weights; few columns, many, row-major B
    (P8, 16, 8192, 4096, 0, KSPLIT), (P8, 16, 8192, 5120, 0, FEW), (P8, 1, 20480, 2048, 0, FEW),
    (P8, 16, 5120, 8192, 0, KSPLIT), (P8, 12, 4096, 10240, 0, KSPLIT), (P8R, 16, 8192, 5120, 0, KSPLIT),
    (P4, 16, 10240, 8192, 0, FEW), (P4, 16, 16384, 4096, 0, FEW), (P4, 16, 8192, 4096, 0, KSPLIT),
    (P4, 8, 49152, 2048, 0, KSPLIT), (P4, 12, 49152, 2048, 0, FEW), (P4, 4, 49152, 2048, 0, FEW),
    # ... and 17-64: 96 MB
    (P8, 64, 8192, 8192, 0, KSPLIT), (P8, 64, 28672, 8192, 0, SHARED), (P8, 32, 28672, 8192, 0, SPLIT),
    # a caller's split: even slices of weights up to 96 MB, 17-64 rows
    (P8, 40, 8192, 8192, 2, KSPLIT), (P8, 16, 8192, 8192, 2, FEW), (P8, 40, 8192, 28672, 2, SPLIT),
    # ... wide N
    (P8, 40, 20480, 4096, 1, SHARED), (P8, 32, 24576, 2048, 1, KSPLIT), (P8, 32, 24576, 2048, 2, SPLIT),
    (P8, 32, 28672, 2048, 2, KSPLIT), (P8, 32, 28672, 2048, 3, SPLIT), (P8, 32, 32768, 2048, 3, KSPLIT),
    (P8, 64, 49152, 2048, 1, KSPLIT), (P8, 64, 49152, 2048, 2, SHARED),
    # ... long rows of few columns
    (P8, 32, 2048, 28672, 1, SPLIT), (P8, 32, 256, 16384, 2, SPLIT), (P8, 32, 3072, 16384, 2, KSPLIT),
    (P8, 32, 3072, 28672, 2, SPLIT), (P8, 64, 2048, 28672, 1, KSPLIT), (P8, 64, 1024, 32768, 3, SPLIT),
    (P8, 40, 256, 16384, 2, KSPLIT), (P4, 32, 2048, 28672, 3, KSPLIT), (P8, 32, 2048, 8192, 3, KSPLIT),
    (P8, 32, 1024, 12288, 3, SPLIT), (P8, 32, 2048, 12288, 3, KSPLIT),
    # more rows: the K-split kernel up to a quarter of the CUs with a 128x128 tile,
    # the shape's four-wave tile up to half, 128x128, 128x256, the entry's own
    # (the four-wave tile for one round of 32x256 and long K only)
    (P8, 1536, 1040, 4096, 0, SHAPE), (P8, 1737, 1040, 4096, 0, KSPLIT),
    (P8, 2865, 592, 4096, 0, TILE128), (P8, 2564, 640, 7168, 0, SHAPE),
    (P8, 2815, 560, 1536, 0, KSPLIT), (P8, 1700, 1120, 512, 0, KSPLIT),
    (P8, 1100, 1040, 2048, 0, KSPLIT), (P8, 3204, 464, 1536, 0, KSPLIT),
    (P4, 4812, 288, 3072, 0, KSPLIT), (P4, 1991, 768, 3072, 0, KSPLIT),
    (P8, 1000, 512, 8192, 0, KSPLIT), (P8, 2048, 512, 8192, 0, KSPLIT), (P8, 3000, 512, 8192, 0, SHAPE),
    (P8, 8192, 256, 4096, 0, SHAPE), (P4, 4096, 512, 4096, 0, SHAPE), (P8, 1500, 1040, 8192, 0, SHAPE),
    (P8, 16384, 128, 8192, 0, TILE128), (P8R, 4096, 512, 8192, 0, TILE128),
    (P8, 1000, 2048, 8192, 0, KSPLIT), (P8, 2048, 2048, 4096, 0, TILE128),
    (P8, 1000, 8192, 8192, 0, TILE128), (P8, 2048, 8192, 8192, 0, ENTRY),
]


@pytest.mark.parametrize("name,M,N,K,l2,kernel", ROUTES)
def test_route(name, M, N, K, l2, kernel):
    p, _ = plan(name + ("_splitK" if l2 else ""), M, N, K, l2)
    assert p.kernel == kernel


@pytest.mark.parametrize("fa,fb", [(1, 0), (0, 1), (1, 1)])
def test_route_of_other_formats(fa, fb):
    """E5M2 operands have no four-wave tile: 128x128 instead."""
    assert plan(P8, 4096, 512, 8192, 0)[0].kernel == SHAPE
    p, _ = plan(P8, 4096, 512, 8192, 0, fmt=(fa, fb))
    assert (p.kernel, p.rows, p.cols) == (TILE128, 128, 128)


@pytest.mark.parametrize("M,N,K", [(300, 2048, 1024), (3000, 512, 8192), (2048, 2048, 4096),
                                   (64, 8192, 8192)])
def test_route_is_the_same_for_every_entry(M, N, K):
    """A caller's tile name is not visible in the output."""
    for prefix in ("ga_mxfp8_bf16_BpreShuffle", "ga_mxfp4_bf16_BpreShuffle"):
        names = [c.knl_name for c in f4gemm.manifest() + f4gemm.manifest_fp4()
                 if c.knl_name.startswith(prefix)]
        plans = [plan(n, M, N, K, 0)[0] for n in names]
        assert len(names) > 8
        assert len({(p.kernel, p.rows, p.cols, p.k_slices) for p in plans}) == 1
