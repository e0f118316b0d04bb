"""The two forms of the level's cut-cell pass (eight lanes a cell on short lists,
one on lists of at least 600000 cells) on both sides of the line between them,
against the oracle: nearly every cell of a block is cut, with random volume
fractions, and the list ends inside a block."""
import numpy as np
import pytest

from helpers import rel_err, run_gpu, run_oracle
from mesoflow_amd import abi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncut", [1, 33, 599999, 600000, 600131])
def test_level_cut_cells(ncut):
    n = (96, 96, 80) if ncut > 1000 else (12, 10, 8)
    c = cases.porous_reactor(n_cell=n, nspec=5, nreact=2, geometry="none", order_hyp=5, seed=3)
    s = cases.perturbed_state(c, seed=ncut % 97)
    r = np.random.default_rng(ncut)
    vf = np.ones(s.shape[1:])
    vf.flat[r.permutation(vf.size)[:ncut]] = r.uniform(0.05, 0.95, ncut)
    s[abi.VFRAC] = vf
    want, _ = run_oracle(c, 1, state=s)
    got, _ = run_gpu(c, 1, state=s)
    err = rel_err(want, got)
    print("%d cut cells: max %.2e" % (ncut, err.max()), flush=True)
    assert np.all(err <= 1e-11)
