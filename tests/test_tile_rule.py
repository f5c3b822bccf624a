"""Which prompt-sized products the tiled kernel takes: at sizes where both sides were measured (us, bf16, cold weights)."""
import pytest

from swiftllm_amd.worker.kernels.linear import _tile_pays


@pytest.mark.parametrize("m,rows,k,act,ours,library", [
    (374, 88, 2304, False, 13.6, 5.9), (300, 96, 2560, False, 15.4, 9.0), (368, 1024, 2560, False, 15.4, 11.8), (561, 336, 2560, False, 15.3, 10.7),
    (497, 384, 768, False, 7.1, 5.9), (402, 1024, 2048, False, 13.2, 10.4), (446, 128, 1024, False, 7.4, 6.2), (470, 2048, 4096, False, 23.0, 19.9),
    (1367, 1024, 8192, False, 41.4, 37.6), (417, 112, 2560, True, 16.0, 12.6), (473, 384, 4096, True, 21.9, 14.6), (350, 4096, 8192, True, 58.2, 47.8),
    (424, 1024, 1024, False, 7.7, 9.7), (463, 256, 512, False, 5.5, 6.0), (1259, 1152, 2048, False, 13.6, 14.2), (668, 2048, 2560, False, 17.0, 17.5),
    (847, 1536, 1024, False, 9.1, 11.3), (423, 96, 1024, True, 7.8, 9.1), (654, 640, 2048, True, 13.4, 13.9), (375, 2048, 2560, True, 16.4, 17.6),
    (3803, 384, 4096, True, 24.3, 27.5)])
def test_the_faster_one(m, rows, k, act, ours, library):
    assert _tile_pays(m, rows, k, act) == (ours < library)


@pytest.mark.parametrize("m,rows,k,takes", [(300, 1024, 2048, True), (300, 1024, 2560, True), (300, 1024, 4096, False), (2000, 1024, 4096, True)])
def test_several_products_in_one_launch(m, rows, k, takes):
    assert _tile_pays(m, rows, k, groups=4) == takes
