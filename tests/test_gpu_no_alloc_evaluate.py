"""An evaluation of the objective allocates nothing, from the first on: what it
needs is made with the objective (code that captures it, or serves with memory
given out beforehand, counts on that)."""
import numpy as np
import pytest
import torch

from _util import design

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,precision", [(np.float64, "fp64"), (np.float32, "bf16x3")],
                         ids=["f64", "bf16x3"])
def test_evaluate(gpu, dtype, precision):
    from dreamplace_amd.engine import DeviceDesign, PlacementObjective
    print("case no allocation in evaluate %s" % precision, flush=True)
    d = design(1, scale=0.002, dtype=dtype)
    dd = DeviceDesign(d, gpu)
    obj = PlacementObjective(dd, d.wa_gamma, density_weight=0.2, algorithm="tiled",
                             precision=precision, schedule="pins")
    torch.cuda.synchronize()
    count = lambda: torch.cuda.memory_stats(gpu)["allocation.all.allocated"]
    before = count()
    for _ in range(3):
        obj.evaluate(dd.pos)
    assert count() == before
