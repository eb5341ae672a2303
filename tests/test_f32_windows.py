"""32-bit attention behind short windows and chunks: as many waves as there are tiles to see, small heads without padding."""
import pytest

from test_f32_kernels import test_attention_over_tiles_of_32_keys as over_tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,hd,ps,vis,span", [(6, 3, 48, 8, "window", 8), (4, 2, 16, 4, "window", 9), (4, 4, 32, 16, "window", 34),
                                                (2, 1, 16, 4, "chunk", 16), (3, 1, 96, 32, "window", 98), (4, 2, 16, 16, "window", 99),
                                                (2, 2, 32, 16, "full", 0), (2, 1, 128, 32, "chunk", 96)])
def test_waves_and_head_sizes(H, G, hd, ps, vis, span):
    over_tiles(H, G, hd, ps, vis, span)
