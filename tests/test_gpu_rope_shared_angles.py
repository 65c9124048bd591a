"""256-column tiles share the rotary angles between their two heads: both rotating, the second one a value head, both value heads."""
import pytest

from test_gpu_qkv_rope import TILES, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,M", [("256x256", 256), ("256x256", 768), ("128x256", 128), ("128x256", 384)])
@pytest.mark.parametrize("n_q,n_kv", [(4, 1), (2, 2), (2, 3)])
@pytest.mark.parametrize("norm", [True, False])
def test_heads_of_a_tile(lib, oracle, tile, M, n_q, n_kv, norm):
    _run(lib, oracle, M, 256, n_q, n_kv, TILES[tile], 1, norm=norm, pre=n_kv == 3)
