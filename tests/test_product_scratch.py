"""How much scratch a product asks for, and with that which deep products go by parts of their depth."""
import pytest

from swifttransformer_amd.ops import kernels as K

DEEP = [(150, 2048, 8192), (575, 4096, 16384), (768, 768, 8192)]


@pytest.mark.parametrize("shape", DEEP)
def test_it_does_not_depend_on_where_products_go_at_the_time(shape):
    """A product first met while the rule sends it elsewhere has its scratch once the rule is the default again."""
    K._gemm_scratch.cache_clear()
    try:
        K.gemm_library_rule(min_rows=1 << 20)
        first = K._gemm_scratch(*shape, K.BF16, False)
    finally:
        K.gemm_library_rule(-2, -2, -2)
    assert first == K._lib().st_gemm_scratch(*shape, K.BF16, 0) > 0 and K._gemm_scratch(*shape, K.BF16, False) == first


@pytest.mark.parametrize("features,depth", [(2048, 8192), (768, 3072), (4096, 16384), (2048, 16384), (2560, 10240), (260, 704)])
@pytest.mark.parametrize("most", [70, 200, 577, 768, 2048])
def test_the_most_is_enough_for_any_rows(most, features, depth):
    room = K._gemm_scratch(most, features, depth, K.BF16, True)
    assert all(K._gemm_scratch(m, features, depth, K.BF16, False) <= room for m in range(1, most + 1))


@pytest.mark.parametrize("rows,features,depth,taken", [
    (150, 768, 8192, False), (192, 640, 8192, False), (96, 512, 8192, False), (512, 512, 8192, False), (512, 7168, 7168, False),
    (480, 8192, 8192, False), (512, 5120, 5120, False), (512, 4096, 5376, False), (704, 4096, 8192, False), (575, 5120, 5120, False),
    (192, 768, 12288, True), (320, 512, 12288, True), (704, 768, 8192, True), (512, 4096, 16384, True), (512, 2048, 8192, True),
    (575, 4096, 16384, True), (576, 5120, 13824, True), (640, 2048, 16384, True), (256, 2048, 8192, True), (66, 2048, 8192, True)])
def test_deep_products_go_by_parts_where_that_is_faster(rows, features, depth, taken):
    """Of 256 compute units; times of both beside the rule."""
    assert (K._lib().st_gemm_scratch(rows, features, depth, K.BF16, 0) > 0) == taken
