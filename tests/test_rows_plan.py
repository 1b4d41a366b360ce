"""Into how many ranges of k a product of many rows goes, and its launch shape: what the kernel library answers from the sizes (no GPU is asked)."""
import pytest

from tiny_llm_infer_amd.kernels.ops import load_library


@pytest.mark.parametrize("nk", [(2048, 2048), (4096, 4096), (2048, 8192), (5120, 5120), (7168, 5120), (5120, 17408), (1040, 904), (12288, 1536)])
def test_one_plan_for_all_rows_of_a_block(nk):
    """A recorded step is filled up to a multiple of 32 rows: its products have the same order of sums only if every number of
    rows of a block of 128 has the same plan."""
    lib = load_library()
    N, K = nk

    def plan(M):
        splits = lib.tli_gemm_rows_splits(M, N, K)
        return splits, [lib.tli_gemm_rows_shape(M, N, K, gated, splits) for gated in (0, 1)]
    for last in list(range(256, 1537, 128)) + [2048, 3072, 3200]:
        want = plan(last)
        assert all(plan(M) == want for M in range(last - 127, last)), last


# (rows, columns, k), the ranges that were the faster, gated or columns a matrix; both measured
@pytest.mark.parametrize("mnk, gated, every, want", [((256, 8192, 4096), 0, 2048, 4), ((129, 8192, 4096), 0, 2048, 4), ((129, 8192, 3072), 0, 2048, 4),
                                                     ((512, 4096, 4096), 0, 1024, 4), ((640, 8192, 2048), 0, 2048, 1), ((1024, 4096, 1024), 0, 1024, 1),
                                                     ((640, 8192, 1024), 1, 0, 1), ((512, 4096, 4096), 1, 0, 4), ((129, 8192, 4096), 1, 0, 4),
                                                     ((256, 4096, 4096), 1, 0, 4)])
def test_ranges_for_the_shape_that_runs(mnk, gated, every, want):
    """Gated products and stacked matrices do not run in the shape that a plain product of their sizes would."""
    assert load_library().tli_gemm_rows_splits_of(*mnk, gated, every) == want


def test_ranges_of_every_kind_leave_four_slices_each():
    lib = load_library()
    for M in (129, 256, 257, 1000, 3000):
        for N in (512, 1024, 4096, 12288):
            for K in (8, 128, 904, 1024, 4096, 17408):
                for gated, every in ((0, 0), (1, 0), (0, 256), (0, 512)):
                    splits = lib.tli_gemm_rows_splits_of(M, N, K, gated, every)
                    assert 1 <= splits <= 16 and (splits == 1 or splits * 4 <= (K + 127) // 128)


@pytest.mark.parametrize("mnk", [(3200, 12288, 17408), (3200, 12288, 1536), (640, 16384, 1024), (1024, 12288, 17408), (512, 8192, 24576)])
def test_sizes_that_were_not_measured_keep_the_first_plan(mnk):
    """Ranges of k only until there are three workgroups of 128 x 256 outputs for every four compute units, four slices of 128 in each."""
    lib = load_library()
    M, N, K = mnk
    groups, splits = -(-N // 256) * -(-M // 128), 1
    while groups * splits < 3 * lib.tli_device_compute_units() // 4 and splits * 8 <= -(-K // 128) and splits < 16:
        splits *= 2
    assert lib.tli_gemm_rows_splits(M, N, K) == splits
