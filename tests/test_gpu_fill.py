"""Ghost cells on the GPU against the oracle over corner combinations of the
boundary codes, on domains down to one cell thick (a ghost cell is then several
periods or reflections away from the cell it is filled from), and steps on such
domains."""
import numpy as np
import pytest

from helpers import rel_err, run_gpu, run_oracle
from mesoflow_amd import abi, cases, runtime

pytestmark = pytest.mark.gpu

PER, FOE, EXT, WALL = abi.BC_PERIODIC, abi.BC_FOEXTRAP, abi.BC_EXT_DIR, abi.BC_WALL
# (lo, hi) codes of x, y, z
MIXES = [((PER, PER), (PER, PER), (PER, PER)),
         ((WALL, WALL), (WALL, WALL), (WALL, WALL)),
         ((EXT, FOE), (PER, PER), (WALL, WALL)),
         ((WALL, EXT), (EXT, WALL), (FOE, PER)),
         ((EXT, EXT), (WALL, FOE), (EXT, WALL))]


def _case(n, mix, geometry="none"):
    c = cases.porous_reactor(n_cell=n, nspec=5, nreact=2, geometry=geometry, rmin=1.0, rmax=2.0, order_hyp=5, seed=3)
    for d, (lo, hi) in enumerate(mix):
        if PER in (lo, hi):
            lo = hi = PER
        c.params.lo_bc[d], c.params.hi_bc[d] = lo, hi
        c.geom.is_periodic[d] = int(lo == PER)
    return c


@pytest.mark.parametrize("n", [(1, 1, 1), (1, 2, 3), (2, 3, 1), (3, 1, 2), (3, 3, 3), (5, 4, 7), (70, 2, 3)])
@pytest.mark.parametrize("mix", range(len(MIXES)))
def test_ghost_cells(n, mix):
    from oracle.pyoracle import OracleLevel
    c = _case(n, MIXES[mix])
    s = cases.perturbed_state(c, seed=5)
    O = OracleLevel(c)
    O.set_state(s)
    want = O.fill_ghosts(0.0)
    ctx = runtime.Context(c)
    L = runtime.Level(ctx)
    L.set_state(s)
    L.fill_ghosts(0.0)
    got = L.padded_state()
    L.close()
    ctx.close()
    err = rel_err(want, got)
    print("fill n=%s mix=%d max %.2e" % (n, mix, err.max()), flush=True)
    # copies and sign changes, at the ext_dir cells externalbc: a few products and
    # quotients, each within 1 ulp (the parity bar of the library is 1e-11)
    assert np.all(err <= 1e-14)


@pytest.mark.parametrize("n,mix,boxes", [((24, 1, 1), 2, None), ((16, 2, 1), 0, None), ((2, 12, 3), 1, None),
                                         ((12, 2, 2), 2, [((0, 0, 0), (5, 1, 1)), ((6, 0, 0), (11, 1, 0)),
                                                          ((6, 0, 1), (11, 1, 1))])])
def test_steps_on_thin_domains(n, mix, boxes):
    c = _case(n, MIXES[mix])
    c.boxes = boxes or []
    s = cases.perturbed_state(c, seed=6)
    want, winfo = run_oracle(c, 3, state=s)
    got, ginfo = run_gpu(c, 3, state=s)
    err = rel_err(want, got)
    print("steps n=%s mix=%d max %.2e" % (n, mix, err.max()), flush=True)
    assert np.all(err <= 1e-11)
    assert ginfo[2] == winfo[2] and abs(ginfo[0] - winfo[0]) <= 1e-11 * abs(winfo[0])
