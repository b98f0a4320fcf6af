"""Split decode attention whose second phase also quantises the row, against attention and quantiser one after the other: the same bits for every number of parts that
one launch takes, and one more (two launches), rows shorter than the workgroup, and every group of query heads."""
import pytest
import torch  # noqa: F401 (before the library: its HIP runtime is the process's)

from qserve_amd._lib import lib
from test_attention_gpu import test_attention_quant_fusion_is_bit_identical_to_the_pair as _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("int4", [True, False], ids=["kv4", "kv8"])
@pytest.mark.parametrize("parts", [2, 3, 7, 8, 9])
@pytest.mark.parametrize("H, Hkv", [(1, 1), (3, 1), (10, 2), (32, 32), (32, 4), (40, 8)])          # (40 heads: a row of more than 4096 values is two launches)
def test_parts_and_quantiser_in_one_launch(gpu, H, Hkv, parts, int4):
    lib.qs_set_attention_variant(100 + parts)
    try:
        _same(gpu, 3, H, Hkv, 1100, parts % 2 == 0, int4)
    finally:
        lib.qs_set_attention_variant(0)
