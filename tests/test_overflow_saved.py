"""The density ops can be saved and copied whole, before a call and after."""
import copy
import pickle

import pytest

from _util import design, to_dev


@pytest.mark.parametrize("copy_of", [copy.deepcopy, lambda x: pickle.loads(pickle.dumps(x))],
                         ids=["copied", "saved"])
def test_saved(copy_of):
    from dreamplace_amd.electric_overflow import ElectricOverflow
    d = design(1, scale=0.001)
    t = to_dev(d, "cpu")
    op = ElectricOverflow(
        t["node_size_x"], t["node_size_y"], t["bin_center_x"], t["bin_center_y"],
        d.target_density, d.xl, d.yl, d.xh, d.yh, d.bin_size_x, d.bin_size_y, d.num_movable_nodes,
        d.num_terminals, d.num_filler_nodes, 0, True, t["sorted_node_map"])
    filler = list(op.uniform_filler_arg())  # as a call forms it
    got = copy_of(op)
    assert len(filler) == 5 and list(got.uniform_filler_arg()) == filler
