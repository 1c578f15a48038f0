"""The density workspace's size never falls as the node count grows: a caller
may size it by all nodes, terminals among them, and have fewer cells."""
import pytest

from dreamplace_amd import _native as N


@pytest.mark.parametrize("dtype", [N.DP_FLOAT32, N.DP_FLOAT64], ids=["f32", "f64"])
@pytest.mark.parametrize("arith", [0, N.DP_ARITH_BIN_RELATIVE], ids=["reference", "bin_relative"])
def test_monotone(dtype, arith):
    size = lambda n: N.query("dp_density_map_workspace_bytes", 512, 512, n, 64,
                             N.DP_SCATTER_TILED | arith, dtype)
    for edge in (1 << 12, 1 << 13, 1 << 20, 1 << 21, 1 << 22):
        sizes = [size(n) for n in range(edge - 300, edge + 300)]
        assert sizes == sorted(sizes)
