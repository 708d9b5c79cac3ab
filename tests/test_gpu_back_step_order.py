"""The joint backward pass of up to 256 rows where its order can go wrong: one tile of 64 labels less than it has ranges, as many, one
more (the first tile of a range is then its only one, or not whole), rows whose fetches of G do not come out even among the eight
waves, and the sizes from which it stores past the caches.  Checks and bounds are those of test_gpu_back_step.py."""
import pytest
import test_gpu_back_step as back

pytestmark = pytest.mark.gpu


# 768 dims: 40 ranges on 256 CUs; 128 dims: 256
@pytest.mark.parametrize("B,L,d", [(129, 39 * 64 - 5, 768), (193, 40 * 64, 768), (209, 40 * 64 + 1, 768), (17, 81 * 64 - 63, 768),
                                   (145, 255 * 64 + 3, 128), (225, 256 * 64 + 8, 128), (1, 513 * 64 - 1, 128),
                                   (209, 50001, 768), (161, 200003, 200)])
def test_update(dev, B, L, d):
    back.test_update_in_one_pass(dev, B, L, d, 8)


@pytest.mark.parametrize("B,L,d", [(200, 40 * 64 + 9, 768), (33, 39 * 64 + 63, 768), (177, 260007, 160)])
def test_accumulation(dev, B, L, d):
    back.test_accumulation_in_one_pass(dev, B, L, d, 4, 0.5)
