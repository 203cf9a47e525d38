"""The kernels that MX launches run, as the host plans them for a device of 256
compute units (CPU only)."""
import pytest

from gcnasm_amd import _lib, f4gemm


def plan(name, M, N, K, l2, num_cu=256):
    """(ga_mx_plan, gdz) of a launch of the entry `name`."""
    cfg = [c for c in f4gemm.manifest() + f4gemm.manifest_fp4() if c.knl_name == name][0]
    ld = f4gemm.make_launch(cfg, M, N, K, l2)
    args = f4gemm.fill_args(None, None, None, None, None, None, M, N, K, N, K // 32, K // 32,
                            1.0, 0.0, ld.log2_k_split)
    return f4gemm.Kernel().load(None, cfg).plan(args, ld.gdz, num_cu), ld.gdz


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
