"""The one-lane record paths at block edges (test_gpu_records.py) in the other two
modes with FP32 columns, whose staged kernels are compilations of their own."""
import pytest

from test_gpu_records import data, test_records_at_block_edges as at_block_edges  # noqa: F401 (data: a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64_pivot", "fp32_hw_trig"])
@pytest.mark.parametrize("name", ["aos", "minv", "wafr", "fext", "ref", "fused", "split"])
def test_modes_at_block_edges(rbd, data, name, precision):  # noqa: F811
    at_block_edges(rbd, data, name, precision)
