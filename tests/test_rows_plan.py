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
