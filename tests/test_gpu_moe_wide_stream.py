"""The GELU bank's one-kernel form, 32 rows a workgroup: hidden sizes that end inside a ring of fetches, last chunks of Ie in which some
wavefronts have no block of fc_in, one chunk and several, output blocks that do not fill a group."""
import pytest

from test_gpu_moe_grouped import test_grouped_gelu_expert_bank_reference_form as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,E,k,H,Ie,e5m2", [
    (70, 3, 3, 2048, 1088, False), (40, 2, 2, 1920, 576, True), (33, 2, 1, 640, 1408, False), (50, 2, 2, 896, 704, True), (48, 2, 1, 512, 64, False),
    (20, 9, 2, 1024, 2048, False), (33, 1, 1, 128, 1984, False),
])
def test_sizes_around_the_fetch_stream(cf, dev, rows, E, k, H, Ie, e5m2):
    check(cf, dev, rows, E, k, H, Ie, e5m2)
