"""The chemistry of the post-step kernels over the forms its rate constants are
held in (a column of LDS for 5 species, registers for 10) with no, one and the
largest number of reactions, on boxes that end inside a block, against the
oracle: the per-box call, and steps of a level."""
import numpy as np
import pytest

from helpers import rel_err, run_gpu, run_oracle
from mesoflow_amd import abi, cases, runtime

pytestmark = pytest.mark.gpu


def _case(nspec, nreact):
    c = cases.porous_reactor(n_cell=(18, 14, 12), nspec=nspec, nreact=nreact, geometry="none", order_hyp=5, seed=13)
    for r in range(nreact):
        c.plugin.log_A[r] = np.log(3.0e10) + 0.3 * r
        c.plugin.Ea[r] = 90.0e3 + 2.0e3 * r
    s = cases.perturbed_state(c, seed=3)
    r = np.random.default_rng(nspec + nreact)
    ctot = s[abi.FLO_NVARS:abi.FLO_NVARS + nspec - 1].sum(axis=0)
    for q in range(1, nspec):      # every reactant present
        s[abi.FLO_NVARS + q] += 0.01 * ctot * r.uniform(0.5, 1.5, ctot.shape)
    return c, s


@pytest.mark.parametrize("nspec,nreact", [(5, 0), (5, 1), (5, 8), (10, 1), (10, 8)])
def test_box_post_chemistry(nspec, nreact):
    import torch
    from oracle.pyoracle import box_post
    c, s = _case(nspec, nreact)
    lo, hi = (2, 1, 3), (12, 9, 9)      # 11*9*7 cells: the last block is partly idle
    fab = np.ascontiguousarray(s[:, lo[2]:hi[2] + 1, lo[1]:hi[1] + 1, lo[0]:hi[0] + 1])
    want = fab.copy()
    flags = abi.MF_POST_CHEMISTRY | abi.MF_POST_PRIMITIVES
    assert box_post(c, (lo, hi), (want, lo), 2.0e-7, flags) == abi.MF_OK
    ctx = runtime.Context(c)
    t = torch.from_numpy(fab.copy()).to("cuda:0")
    torch.cuda.synchronize()
    runtime.check(runtime.lib().mf_box_post(ctx.h, abi.make_box(lo, hi),
                                            abi.make_array4(t.data_ptr(), lo, [h + 1 for h in hi], ctx.nv), 2.0e-7, flags),
                  "mf_box_post")
    ctx.sync()
    err = rel_err(want, t.cpu().numpy())
    ctx.close()
    print("ns %d reactions %d: max %.2e" % (nspec, nreact, err.max()), flush=True)
    assert np.all(err <= 1e-11)
    if nreact:
        assert np.any(want[abi.FLO_NVARS:] != fab[abi.FLO_NVARS:])


@pytest.mark.parametrize("nspec,nreact", [(5, 8), (10, 8)])
def test_level_chemistry(nspec, nreact):
    c, s = _case(nspec, nreact)
    want, _ = run_oracle(c, 2, state=s)
    got, _ = run_gpu(c, 2, state=s, tile=[(64, 4, 1), (32, 8, 1), (32, 1, 8), (16, 4, 2)])
    err = rel_err(want, got)
    print("ns %d reactions %d level: max %.2e" % (nspec, nreact, err.max()), flush=True)
    assert np.all(err <= 1e-11)
