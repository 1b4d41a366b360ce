"""Which float32 decode steps are one launch from the projections: what the kernel library answers from the sizes (no GPU is asked)."""
import pytest

from tiny_llm_infer_amd.kernels.ops import load_library


# rows, heads, kv heads, head size, keys and whether one launch was the sooner done; all measured
@pytest.mark.parametrize("size, one", [((1, 16, 4, 64, 128), 1), ((5, 16, 4, 64, 64), 1), ((8, 32, 8, 128, 1024), 1), ((16, 8, 2, 256, 2048), 1), ((200, 16, 4, 64, 512), 1),
                                       ((512, 32, 8, 64, 128), 0), ((512, 32, 8, 64, 512), 1), ((512, 32, 8, 128, 128), 0), ((512, 8, 2, 192, 128), 0), ((512, 8, 2, 192, 256), 1),
                                       ((512, 8, 2, 256, 128), 0), ((512, 16, 4, 256, 512), 0), ((1024, 16, 16, 64, 128), 1), ((512, 16, 16, 64, 512), 0),
                                       ((128, 16, 16, 128, 1024), 0), ((128, 16, 16, 128, 512), 1), ((64, 8, 8, 256, 2048), 1), ((128, 8, 8, 256, 1024), 0), ((8, 16, 16, 64, 16384), 1)])
def test_one_launch_where_it_was_the_sooner_done(size, one):
    assert load_library().tli_qkv_attention_f32_one(*size) == one


@pytest.mark.parametrize("dim, most", [(64, 16), (128, 16), (192, 8), (256, 6)])
def test_edges_of_the_rule_for_short_rows(dim, most):
    lib = load_library()
    rows = most * lib.tli_device_compute_units() // 8
    assert lib.tli_qkv_attention_f32_one(rows, 8, 2, dim, 128) and not lib.tli_qkv_attention_f32_one(rows + 1, 8, 2, dim, 128)
