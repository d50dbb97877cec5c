"""The CI sum's table of determinants (slater_combine) on the device.

Its size follows the plan: from two groups (one walker a wavefront) to 64
groups of eight configurations (two electrons, eight orbitals), the largest any
plan can have; in a batch every wavefront has room for its launch's largest.
"""
import numpy as np
import pytest
import torch

from qmctorch_amd.scf import Molecule
from qmctorch_amd.serving import BatchRunner, SystemContext, WalkerSet, catalog, sweep_each
from tests import helpers

pytestmark = pytest.mark.gpu


def _h2():
    return Molecule("H 0 0 -0.7; H 0 0 0.7", basis="cc-pvdz", unit="bohr", name="h2_dz")


def _pair(mol, configs, precision="fp64"):
    wf, orc = helpers.make_pair(mol, configs=configs, w_ee=1.0, w_en=1.0, precision=precision)
    ci = torch.as_tensor(0.3 * np.random.default_rng(wf.nci).standard_normal(wf.nci))
    ci[0] = 1.0
    with torch.no_grad():
        wf.fc.weight.copy_(ci.view(1, -1))
        orc.fc_weight.copy_(ci.view(1, -1))
    return wf, orc


@pytest.mark.parametrize("configs,nconf", [("cas(2,2)", 2), ("cas(2,6)", 6), ("cas(2,8)", 8)])
def test_largest_tables(configs, nconf):
    """67 walkers of two electrons: two full wavefronts of 64 groups and a third of three walkers."""
    print("case combine H2", configs, flush=True)
    mol = _h2()
    wf, orc = _pair(mol, configs)
    assert wf.device_plan().tables.nconf_up == nconf
    pos = helpers.positions(mol, 67, seed=3)
    psi, psi_o = wf(pos.cuda()).detach().cpu().view(-1), orc(pos).detach().view(-1)
    assert float(((psi - psi_o).abs() / psi_o.abs()).max()) < 1e-10
    e, e_o = wf.local_energy(pos.cuda()).cpu().view(-1), orc.local_energy(pos).detach().view(-1)
    assert float(((e - e_o).abs() / e_o.abs().clamp(min=1.0)).max()) < 1e-9


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tables_of_unequal_size_in_one_launch(precision):
    """Plans of six columns, two to six configurations and 12 to 64 groups, share a
    launch: each walker gets what its own launch gives it."""
    print("case combine batch", precision, flush=True)
    ctx = [SystemContext(_pair(mol, configs, precision)[0]) for mol, configs in
           ((_h2(), "cas(2,6)"), (catalog.molecule("h2o"), "cas(2,2)"), (catalog.molecule("lih"), "cas(2,5)"))]
    assert {c.plan.bucket for c in ctx} == {6}
    make = lambda: [WalkerSet(c, helpers.positions(c.wf.mol, n, seed=n).cuda(), n) for c, n in zip(ctx, (65, 31, 100))]
    mixed, alone = make(), make()
    runner = BatchRunner(8)
    runner.sweep([(w, 7) for w in mixed])
    sweep_each([(w, 7) for w in alone])
    e = [torch.empty(w.nw, dtype=torch.float64, device="cuda") for w in mixed]
    runner.local_energy(list(zip(mixed, e)))
    for w, v, en in zip(mixed, alone, e):
        assert torch.equal(w.pos, v.pos) and torch.equal(w.logabs, v.logabs) and int(w.naccept.sum()) > 0
        assert torch.equal(en, w.ctx.wf.local_energy_parts(w.pos, "fp64")["eloc"])
