"""Engine forces over subsets of the potentials, bit for bit the sum of the
separate executions: only slots of bonded terms, only sums in sorted order, and
atoms whose slot lists are empty, shorter and longer than a group of lanes."""

import numpy as np
import pytest

from timemachine_amd import _lib
from timemachine_amd import testsystems as ts
from timemachine_amd.lib import LangevinIntegrator, custom_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds", [("Harmonic",), ("NonbondedAllPairs", "Nonbonded"), ("Torsion", "Nonbonded"), ("",)])
def test_engine_forces_of_potential_subsets(gpu, kinds):
    sys = ts.ligand_in_water()
    picked = [bp for bp in sys.bound_potentials() if any(k in type(bp).__name__ for k in kinds)]
    assert picked
    intg = LangevinIntegrator(300.0, 0.0015, 1.0, sys.masses, 7).impl()
    bps = [bp.bound_impl(np.float32) for bp in picked]
    ctx = custom_ops.Context(sys.x, np.zeros_like(sys.x), sys.box, intg, bps)
    ctx.step(0.3)
    raw = np.zeros(sys.N * 3, dtype=np.uint64)
    _lib.call("tm_context_get_du_dx_t_minus_1", ctx.handle, _lib.pu64(raw))
    total = np.zeros(sys.N * 3, dtype=np.uint64)
    for bp in picked:
        total += bp.unbound_impl(np.float32).execute_fixed_raw(sys.x, bp.params, sys.box, 0.3)[0]
    np.testing.assert_array_equal(raw, total)
