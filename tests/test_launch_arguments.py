"""Arguments of the kernels of a few microseconds, read from the code objects in the
runtime library: few enough for the short way through the launch call
(cheap_arguments in gemm_common.h)."""
import os

import pytest

from test_registers import LIBRARY, _code_objects, _kernels


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(LIBRARY):
        import __graft_entry__
        __graft_entry__.build()
    return [k for elf in _code_objects(open(LIBRARY, "rb").read()) for k in _kernels(elf)]


@pytest.mark.parametrize("name", ["k_gemm_i8_skinnyI", "k_gemm_i8_batched_flatI", "k_quant_flatI", "k_quant_tiledI", "k_quant_lastaxisI",
                                  "k_quant_gatherI", "k_dequant8_flatI", "k_dequant8_gatherI", "k_dql_small",
                                  "k_gemm_i8I", "k_gemm_i8_dmaI", "k_gemm_i8_bsI", "k_gemm_i8_dma_bsI", "k_sum_partsI", "k_dql_gridI", "k_dql_repair"])
def test_short_kernels_are_cheap_to_launch(kernels, name):
    forms = [k for k in kernels if name in k[".name"]]
    assert forms
    for k in forms:
        pointers = sum(a[".value_kind"] == "global_buffer" for a in k[".args"])
        assert not any(a[".value_kind"].startswith("hidden") for a in k[".args"]), k[".name"]
        assert -(-k[".kernarg_segment_size"] // 16) * 16 + 8 * pointers < 128, (k[".name"], k[".kernarg_segment_size"], pointers)

