"""Small-matrix (minors) kernels on the device at every size and spin split.

Chains of n hydrogen atoms with one unpaired electron: the up block is
(n + 1) / 2 columns and the down block one fewer, so each size from 2 to 7
runs with a group completed by unit rows, and 8 is the first size of the
eliminations.  psi, the local energy and the gradient against the float64
oracle; log|psi| far from every nucleus, where products of orbital values
leave the double range, against the sum of the single-electron decays; blocks
near a node, which are eliminated; the same sizes in mixed precision.
"""
import numpy as np
import pytest
import torch

from qmctorch_amd.scf import Molecule
from tests import helpers, systems

pytestmark = pytest.mark.gpu


def _chain(n):
    atoms = "; ".join("H %.3f %.3f %.3f" % (0.3 * (k % 2), 0.2 * (k % 3), 1.6 * k) for k in range(n))
    return Molecule(atoms, basis="cc-pvdz", unit="bohr", spin=n % 2, mo_coeffs="random", name="h%d" % n)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 7, 9, 11, 13, 14, 15])
def test_every_block_size(n):
    print("case minors H%d" % n, flush=True)
    mol = _chain(n)
    wf, orc = helpers.make_pair(mol, w_ee=None if n == 1 else 1.0, w_en=1.0)
    pos = helpers.positions(mol, 67, seed=n, sigma=1.0)
    x = pos.cuda()
    psi, psi_o = wf(x).detach().cpu().view(-1), orc(pos).detach().view(-1)
    # rounding of the orbitals (1e-15) times the condition of the blocks
    assert float(((psi - psi_o).abs() / psi_o.abs()).max()) < 1e-9
    e, e_o = wf.local_energy(x).cpu().view(-1), orc.local_energy(pos).detach().view(-1)
    assert float(((e - e_o).abs() / e_o.abs().clamp(min=1.0)).max()) < 1e-8
    p = pos.clone().requires_grad_()
    g_o = torch.autograd.grad(orc(p).sum(), p)[0]
    g = wf.gradients_jacobi(x).cpu()
    assert float((g - g_o).abs().max() / g_o.abs().max()) < 1e-9


@pytest.mark.parametrize("n", [5, 9, 13])
def test_rows_far_from_the_nuclei(n):
    """Every electron is moved out so far that its orbitals are below 1e-80: the
    block's products underflow, its logarithm does not."""
    print("case minors far H%d" % n, flush=True)
    mol = _chain(n)
    wf, orc = helpers.make_pair(mol, w_ee=1.0, w_en=1.0)
    rng = np.random.default_rng(n)
    d = rng.standard_normal((33, n, 3))
    d *= 40.0 / np.linalg.norm(d, axis=2, keepdims=True)
    pos = torch.as_tensor((d + np.asarray(mol.atom_coords)[None]).reshape(33, 3 * n))
    la, sg = wf.log_psi(pos.cuda())
    mo = orc.mo(orc.ao(pos)).detach()
    scale = mo.abs().amax(-1, keepdim=True)
    rows = (mo / scale)[..., :wf.highest_occ_mo]
    su, lu = torch.linalg.slogdet(rows[:, :mol.nup, :mol.nup])
    sd, ld = torch.linalg.slogdet(rows[:, mol.nup:, :mol.ndown])
    ref = lu + ld + scale.log().sum((1, 2)) + orc.jastrow(pos).detach().view(-1).log()
    print("  log|psi| from %.0f to %.0f, largest difference %.1e" % (ref.min(), ref.max(),
                                                                   (la.cpu() - ref).abs().max()), flush=True)
    assert float(ref.max()) < -745.0  # below the smallest double
    # exponentials of arguments near -200 are good to 200 eps = 5e-14 of their
    # value, which the blocks' condition (only the most diffuse orbitals are
    # left out there) carries into the n rows' determinant
    cond = torch.linalg.cond(rows[:, :mol.nup, :mol.nup]) + torch.linalg.cond(rows[:, mol.nup:, :mol.ndown])
    bound = 5e-14 * n * cond
    ok = bound < 1e-3  # the others' determinants have no correct digits in double
    assert int(ok.sum()) >= 20
    assert ((la.cpu() - ref).abs() <= bound)[ok].all() and torch.equal(sg.cpu()[ok], (su * sd)[ok])


@pytest.mark.parametrize("n", [6, 8, 16])
def test_ci_terms_far_from_the_nuclei(n):
    """The configurations' determinants, all below the double range and of
    different powers of two (at n = 16 eliminated, with one exponent each), meet in
    the CI sum without leaving it."""
    print("case minors CI far H%d" % n, flush=True)
    mol = _chain(n)
    wf, orc = helpers.make_pair(mol, configs="cas(2,2)", w_ee=1.0, w_en=1.0)
    ci = torch.linspace(1.0, 0.1, wf.nci, dtype=torch.float64)
    with torch.no_grad():
        wf.fc.weight.copy_(ci.view(1, -1))
    rng = np.random.default_rng(n)
    d = rng.standard_normal((33, n, 3))
    d *= 40.0 / np.linalg.norm(d, axis=2, keepdims=True)
    pos = torch.as_tensor((d + np.asarray(mol.atom_coords)[None]).reshape(33, 3 * n))
    la, sg = wf.log_psi(pos.cuda())
    mo = orc.mo(orc.ao(pos)).detach()
    scale = mo.abs().amax(-1, keepdim=True)
    rows = mo / scale
    lg, s, cond = [], [], 0.0
    for cu, cd in zip(*wf.configs):
        up, dn = rows[:, :mol.nup][..., cu.long()], rows[:, mol.nup:][..., cd.long()]
        (su, lu), (sd, ld) = torch.linalg.slogdet(up), torch.linalg.slogdet(dn)
        lg.append(lu + ld)
        s.append(su * sd)
        cond = cond + torch.linalg.cond(up) + torch.linalg.cond(dn)
    lg, s = torch.stack(lg, 1), torch.stack(s, 1)
    top = lg.amax(1, keepdim=True)
    terms = ci * s * (lg - top).exp()
    tot = terms.sum(1)
    ref = tot.abs().log() + top.view(-1) + scale.log().sum((1, 2)) + orc.jastrow(pos).detach().view(-1).log()
    assert float(ref.max()) < -745.0
    # as above, carried through each determinant and a sum that may cancel
    bound = 5e-14 * n * cond * terms.abs().sum(1) / tot.abs()
    ok = bound < 1e-3
    print("  log|psi| from %.0f to %.0f, %d walkers compared, largest difference %.1e"
          % (ref.min(), ref.max(), int(ok.sum()), (la.cpu() - ref).abs()[ok].max()), flush=True)
    assert int(ok.sum()) >= 5
    assert ((la.cpu() - ref).abs() <= bound)[ok].all() and torch.equal(sg.cpu()[ok], tot.sign()[ok])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_psi_of_seven_columns_on_both_sides_of_the_wave_rule(precision):
    """1024 wavefronts of N2 expand minors, 1025 eliminate: the same rows, so the
    determinants differ by roundings times the condition of the blocks."""
    print("case minors N2 wave rule", precision, flush=True)
    mol = systems.n2()
    wf, orc = helpers.make_pair(mol, w_ee=0.9, w_en=1.0)
    pos = helpers.positions(mol, 4100, seed=2)
    few, many = wf.log_psi(pos[:4096].cuda(), precision), wf.log_psi(pos.cuda(), precision)
    mo = orc.mo(orc.ao(pos[:4096])).detach()
    rows = mo / mo.abs().amax(-1, keepdim=True)
    cond = torch.linalg.cond(rows[:, :7, :7]) + torch.linalg.cond(rows[:, 7:, :7])
    # 7^2 roundings of 1.1e-16 in either way
    assert ((few[0] - many[0][:4096]).abs().cpu() <= 2 * 49 * 1.1e-16 * cond).all()
    ok = cond < 1e12
    assert torch.equal(few[1].cpu()[ok], many[1][:4096].cpu()[ok]) and int(ok.sum()) > 4000
    if precision == "fp64":
        psi, psi_o = wf(pos.cuda()).detach().cpu().view(-1)[-300:], orc(pos[-300:]).detach().view(-1)
        assert float(((psi - psi_o).abs() / psi_o.abs()).max()) < 1e-9

def _beside_the_chain(mol, nw, rho, seed):
    """Electrons of both spins alternating along the chain, each rho from its atom
    and the chain's axis: far from every nucleus, their rows well apart."""
    rng = np.random.default_rng(seed)
    atom = np.empty(mol.nelec, dtype=int)
    atom[:mol.nup], atom[mol.nup:] = np.arange(0, mol.nelec, 2), np.arange(1, mol.nelec, 2)
    phi = rng.uniform(0, 2 * np.pi, (nw, mol.nelec))
    d = np.stack([rho * np.cos(phi), rho * np.sin(phi), rng.uniform(-0.3, 0.3, phi.shape)], -1)
    return torch.as_tensor((np.asarray(mol.atom_coords)[atom] + d).reshape(nw, -1))


def test_mixed_ci_terms_whose_product_leaves_the_double_range():
    """FP32 rows near 1e-30: each determinant of six is a double, no product of an
    up and a down one is."""
    print("case minors CI far H12 mixed", flush=True)
    mol = _chain(12)
    wf, orc = helpers.make_pair(mol, configs="cas(2,2)", w_ee=1.0, w_en=1.0)
    ci = torch.linspace(1.0, 0.1, wf.nci, dtype=torch.float64)
    with torch.no_grad():
        wf.fc.weight.copy_(ci.view(1, -1))
    pos = _beside_the_chain(mol, 33, 23.5, 1)
    la, sg = (v.cpu() for v in wf.log_psi(pos.cuda(), "mixed"))
    ref, ref_sg = (v.cpu() for v in wf.log_psi(pos.cuda(), "fp64"))
    rows = orc.mo(orc.ao(pos)).detach()
    rows = rows / rows.abs().amax(-1, keepdim=True)
    cond, terms = 0.0, []
    for c, cu, cd in zip(ci, *wf.configs):
        up, dn = rows[:, :mol.nup][..., cu.long()], rows[:, mol.nup:][..., cd.long()]
        cond = cond + torch.linalg.cond(up) + torch.linalg.cond(dn)
        terms.append(c * torch.linalg.det(up) * torch.linalg.det(dn))
    terms = torch.stack(terms, 1)
    # an exponential of an FP32 argument near -67, itself good to 4 roundings, is
    # good to 2e-5; carried through the determinants and the sum
    bound = 2e-5 * mol.nelec * cond * terms.abs().sum(1) / terms.sum(1).abs()
    ok = bound < 0.3
    print("  log|psi| from %.0f to %.0f, %d walkers compared, largest difference %.1e"
          % (ref.min(), ref.max(), int(ok.sum()), (la - ref).abs()[ok].max()), flush=True)
    slater = ref - orc.jastrow(pos).detach().view(-1).log()
    assert float(slater.max()) < -745.0 and int(ok.sum()) >= 15  # below the smallest double
    assert ((la - ref).abs() <= bound)[ok].all() and torch.equal(sg[ok], ref_sg[ok])

@pytest.mark.parametrize("n", [2, 5, 9, 13])
def test_mixed_drift_beside_an_electron_beyond_the_fp32_range(n):
    """An up electron so far out that its FP32 orbitals are zero: psi is zero, its
    block has no part in the drift (the up electrons keep the Jastrow factor's),
    the down electrons' is what it is."""
    print("case minors zero row H%d" % n, flush=True)
    mol = _chain(n)
    wf, orc = helpers.make_pair(mol, w_ee=1.0, w_en=1.0)
    pos = helpers.positions(mol, 67, seed=n).view(67, n, 3)
    pos[:, 0, 0] += 60.0
    pos = pos.reshape(67, -1)
    drift, la, _ = (v.cpu() for v in wf.drift(pos.cuda(), "mixed"))
    assert bool((la == -float("inf")).all())
    x = pos.clone().requires_grad_()
    mo = orc.mo(orc.ao(x))
    dn = mo[:, mol.nup:, :mol.ndown]
    log = torch.linalg.slogdet(dn)[1].sum() if mol.ndown else 0.0
    ref = torch.autograd.grad(log + orc.jastrow(x).log().sum(), x)[0].view(67, n, 3)
    # FP32 rows are good to about 10 roundings of 6e-8 of their terms' sum without
    # signs, their gradients to 2 sqrt(13) = 7 times that (the tightest exponent);
    # the inverse carries both into the drift
    ao = orc.ao(pos).detach()
    terms = ao.abs() @ orc.mo(torch.eye(ao.shape[-1]).to(ao)[None])[0].detach().abs()
    inv = torch.linalg.matrix_norm(torch.linalg.inv(dn.detach()), 2)
    bound = 4.2e-6 * (1.0 + inv * terms[..., :mol.ndown].amax((1, 2)))[:, None] * (1.0 + ref.norm(dim=-1))
    assert ((drift - ref).norm(dim=-1) <= bound).all()
    assert float((bound < 1e-2).double().mean()) > 0.5  # and mean something


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_drift_of_an_expansion_with_a_zero_determinant(precision):
    """A virtual orbital that is zero everywhere: the configurations that hold it
    have no determinant and no part in the drift."""
    print("case minors zero configuration", precision, flush=True)
    mol = _chain(6)
    wf, _ = helpers.make_pair(mol, configs="cas(2,2)", w_ee=1.0, w_en=1.0)
    one, _ = helpers.make_pair(mol, w_ee=1.0, w_en=1.0)
    with torch.no_grad():
        wf.mo.mo_modifier[:, mol.nup] = 0.0
    x = helpers.positions(mol, 67, seed=4).cuda()
    got, want = wf.drift(x, precision), one.drift(x, precision)
    # two instances of the kernel: rows one rounding apart (1e-16, 6e-8), times the
    # blocks' condition, below 1e4 for 67 walkers around their atoms
    tol = 1e-10 if precision == "fp64" else 1e-3
    assert float(((got[0] - want[0]).norm(dim=-1) / (1.0 + want[0].norm(dim=-1))).max()) < tol
    assert torch.equal(got[2], want[2])


def _fp32_amplification(orc, mol, pos):
    """Largest sum of a row's terms without signs times the norm of the blocks'
    inverses, per walker: what an FP32 rounding of the rows becomes in the
    inverse's products with them."""
    ao = orc.ao(pos).detach()
    terms = ao.abs() @ orc.mo(torch.eye(ao.shape[-1]).to(ao)[None])[0].detach().abs()
    mo = orc.mo(ao).detach()
    out = torch.ones(len(pos), dtype=torch.float64)
    for rows, n in ((slice(0, mol.nup), mol.nup), (slice(mol.nup, None), mol.ndown)):
        if n:
            inv = torch.linalg.matrix_norm(torch.linalg.inv(mo[:, rows, :n]), 2)
            out = out + inv * terms[:, rows, :n].amax((1, 2))
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 7, 9, 11, 13, 14, 15])
def test_every_block_size_in_mixed_precision(n):
    """The FP32 instances (unscaled rows, no fallback) against the FP64 ones."""
    print("case minors mixed H%d" % n, flush=True)
    mol = _chain(n)
    wf, orc = helpers.make_pair(mol, w_ee=None if n == 1 else 1.0, w_en=1.0)
    pos = helpers.positions(mol, 67, seed=n, sigma=1.0)
    d32, l32, s32 = (v.cpu() for v in wf.drift(pos.cuda(), "mixed"))
    d64, l64, s64 = (v.cpu() for v in wf.drift(pos.cuda(), "fp64"))
    lpsi, spsi = (v.cpu() for v in wf.log_psi(pos.cuda(), "mixed"))
    amp = _fp32_amplification(orc, mol, pos)
    # about 10 roundings of 6e-8 a row entry, n rows; gradients 2 sqrt(13) = 7 times
    ok = 6e-7 * n * amp < 0.1
    assert int(ok.sum()) >= 50
    for l, s in ((l32, s32), (lpsi, spsi)):
        assert ((l - l64).abs() <= 6e-7 * n * amp)[ok].all() and torch.equal(s[ok], s64[ok])
    err = (d32 - d64).norm(dim=-1).amax(1) / (1.0 + d64.norm(dim=-1).amax(1))
    assert (err <= 4.2e-6 * n * amp)[ok].all()


def _close_pair(mol, nw, seed):
    """Ordinary positions; in every second walker two up electrons 1e-6 to 1e-2 bohr apart."""
    pos = helpers.positions(mol, nw, seed=seed).view(nw, mol.nelec, 3)
    rng = np.random.default_rng(seed)
    step = rng.standard_normal((nw, 3))
    step *= (10.0 ** rng.uniform(-6, -2, nw) / np.linalg.norm(step, axis=1))[:, None]
    pos[1::2, 1] = pos[1::2, 0] + torch.as_tensor(step[1::2])
    return pos.reshape(nw, -1)


@pytest.mark.parametrize("n,configs", [(6, "ground_state"), (7, "ground_state"), (13, "ground_state"),
                                       (6, "cas(2,2)"), (10, "cas(2,2)"), (12, "cas(2,2)")])
def test_weak_blocks_beside_strong_ones(n, configs):
    """Blocks near a node are eliminated, the others of the wavefront expanded: psi,
    the drift, the local energy and both adjoints, for one and for several
    configurations up to seven columns."""
    print("case minors weak H%d" % n, configs, flush=True)
    mol = _chain(n)
    wf, orc = helpers.make_pair(mol, configs=configs, w_ee=1.0, w_en=1.0)
    ci = torch.linspace(1.0, 0.1, wf.nci, dtype=torch.float64)
    with torch.no_grad():
        wf.fc.weight.copy_(ci.view(1, -1))
        orc.fc_weight.copy_(ci.view(1, -1))
    orc.bas_exp.requires_grad_(False)
    orc.atom_coords.requires_grad_(False)
    wf.ao.bas_exp.requires_grad_(False)
    pos = _close_pair(mol, 67, seed=n)
    x = pos.cuda()
    ao, dao, d2ao = orc.ao(pos, "all")
    mo = orc.mo(ao).detach()
    kin = orc.kinetic_operator(pos, ao, dao, d2ao, orc.mo(ao)).detach()
    kin = kin.reshape(mo.shape)
    rows = mo / 2.0 ** torch.frexp(mo.abs().amax(-1, keepdim=True))[1]
    psi_o = orc(pos).detach().view(-1)
    cond, amp = torch.ones(67, dtype=torch.float64), torch.ones(67, dtype=torch.float64)
    det0, terms = None, []
    for c, cu, cd in zip(ci, *wf.configs):
        part, tr = c * torch.ones(67, dtype=torch.float64), 0.0
        for sl, cf in ((slice(0, mol.nup), cu.long()), (slice(mol.nup, None), cd.long())):
            A = mo[:, sl][..., cf]
            cond = torch.maximum(cond, torch.linalg.cond(rows[:, sl][..., cf]))
            tr = tr + (torch.linalg.inv(A).transpose(1, 2) * kin[:, sl][..., cf]).abs().sum((1, 2))
            part = part * torch.linalg.det(A)
        det0 = torch.linalg.det(rows[:, :mol.nup][..., cu.long()]) if det0 is None else det0
        terms.append((part, tr))
    total = sum(p for p, _ in terms).abs()
    cancel = sum(p.abs() for p, _ in terms) / total  # of the CI sum
    amp = amp + sum(p.abs() * t for p, t in terms) / total
    weak = det0.abs() < 1e-6
    assert int(weak.sum()) >= 5 and int((~weak).sum()) >= 30
    eps = 1.1e-16 * n * n * cond * cancel  # relative error of an inverse or a determinant, either way
    ok = 1e3 * eps < 0.1
    assert int((ok & weak).sum()) >= 5
    la, sg = (v.cpu() for v in wf.log_psi(x, "fp64"))
    assert ((la - psi_o.abs().log()).abs() <= 10 * eps)[ok].all() and torch.equal(sg[ok], psi_o.sign()[ok])
    dr = wf.drift(x, "fp64")[0].cpu()
    ref = (orc.gradients_jacobi(pos.clone().requires_grad_()).detach() / psi_o[:, None]).view(67, n, 3)
    assert ((dr - ref).norm(dim=-1).amax(1) <= 100 * eps * (1.0 + ref.norm(dim=-1).amax(1)))[ok].all()
    e, e_o = wf.local_energy(x).cpu().view(-1), orc.local_energy(pos).detach().view(-1)
    assert ((e - e_o).abs() <= 100 * eps * (amp + e_o.abs()))[ok].all()
    # adjoints walker by walker, the best conditioned of either kind; the local
    # energy's is a difference of products of two inverses with the rows, each
    # rounded in its terms
    Y = torch.stack([torch.linalg.matrix_norm(torch.linalg.inv(mo[:, sl][..., cf[0].long()]), 2)
                     for sl, cf in ((slice(0, mol.nup), wf.configs[0]), (slice(mol.nup, None), wf.configs[1]))]).amax(0)
    size = orc.mo_scf.abs().max() * ao.detach().norm(dim=(1, 2)) * Y * Y * kin.norm(dim=(1, 2))
    order = torch.argsort(eps)
    close = [0, 0]
    for k in [int(i) for i in order if weak[i]][:4] + [int(i) for i in order if not weak[i]][:2]:
        one = pos[k:k + 1]
        for f, f_o, extra in ((lambda v: wf(v).abs().log(), lambda v: orc(v).abs().log(), 0.0),
                              (wf.local_energy_autodiff, orc.local_energy, float(size[k]))):
            wf.zero_grad()
            f(one.cuda()).sum().backward()
            g_o = torch.autograd.grad(f_o(one).sum(), [orc.mo_modifier, orc.fc_weight])
            bound = 100 * float(eps[k]) * float(g_o[0].norm()) + 10 * n * n * 1.1e-16 * extra
            err = float((wf.mo.mo_modifier.grad.cpu() - g_o[0]).norm())
            assert err <= bound
            close[extra != 0.0] += int(bool(weak[k]) and bound < 0.1 * float(g_o[0].norm()))
            if wf.nci > 1:
                err = float((wf.fc.weight.grad.cpu() - g_o[1]).norm())
                assert err <= 100 * float(eps[k]) * (float(g_o[1].norm()) + float(amp[k]))
    # weak walkers whose gradients the bounds pin to a tenth
    assert close[0] == 4 and close[1] >= 1


@pytest.mark.parametrize("n,configs", [(11, "ground_state"), (13, "ground_state"), (10, "cas(2,2)"),
                                       (12, "cas(2,2)")])
def test_hmc_of_six_and_seven_columns_replays_the_oracle(n, configs):
    from oracle import vmc_oracle as O
    from qmctorch_amd.sampler import Hamiltonian
    from tests.test_gpu_hmc import _host_noise

    print("case minors hmc H%d" % n, configs, flush=True)
    mol = _chain(n)
    wf, orc = helpers.make_pair(mol, configs=configs, w_ee=1.0, w_en=1.0)
    nw, nstep, L, eps, seed = 7, 2, 3, 0.05, 0x1234_5678
    q = helpers.positions(mol, nw, seed=n)
    s = Hamiltonian(nwalkers=nw, nstep=nstep, step_size=eps, L=L, ntherm=0, ndecor=1, nelec=n,
                    init=mol.domain("normal"), cuda=True, seed=seed)
    kept = s(wf.pdf, pos=q.cuda().clone(), with_tqdm=False).detach().cpu().view(nstep, nw, -1)
    for step in range(nstep):
        p, u = _host_noise(seed, nw, n, step)
        q, acc = O.hmc_step(orc.pdf, q, p, eps, L, u)
        # as test_hmc_fp64_replays_oracle_step
        torch.testing.assert_close(kept[step], q, rtol=0, atol=1e-8)


def test_slater_functions_of_several_r_powers():
    """Contractions over Slater primitives of different r powers: one record per
    primitive, the entry's parts delivered one after the other."""
    print("case several r powers", flush=True)
    mol = systems.hydrogen_atom("sto", 1.0)
    b = mol.basis
    # an s of r^0, r^1 and r^2, and p functions x, y, z of r^0 and r^1
    b.nao = b.nmo = 4
    b.nshells, b.nao_per_atom = np.array([9]), np.array([4])
    b.index_ctr = np.array([0, 0, 0, 1, 1, 2, 2, 3, 3])
    b.nctr_per_ao = np.array([3, 2, 2, 2])
    b.bas_exp = np.array([1.6, 0.9, 0.7] + 3 * [1.1, 0.6])
    b.bas_coeffs = np.array([0.5, 0.4, 0.2] + 3 * [0.6, 0.5])
    b.bas_kr = np.array([0, 1, 2] + 3 * [0, 1])
    b.bas_kx = np.array([0, 0, 0, 1, 1, 0, 0, 0, 0])
    b.bas_ky = np.array([0, 0, 0, 0, 0, 1, 1, 0, 0])
    b.bas_kz = np.array([0, 0, 0, 0, 0, 0, 0, 1, 1])
    b.bas_n = list(b.bas_kr)
    b.mos = np.linalg.qr(np.random.default_rng(0).standard_normal((4, 4)))[0]
    mol.nelec, mol.nup, mol.ndown, mol.spin = 3, 2, 1, 1
    mol.atomic_number, mol.atomic_nelec = [3], [3]
    wf, orc = helpers.make_pair(mol, w_ee=0.7, w_en=1.0)
    pos = helpers.positions(mol, 67, seed=5)
    x = pos.cuda()
    psi, psi_o = wf(x).detach().cpu().view(-1), orc(pos).detach().view(-1)
    assert float(((psi - psi_o).abs() / psi_o.abs()).max()) < 1e-10
    e, e_o = wf.local_energy(x).cpu().view(-1), orc.local_energy(pos).detach().view(-1)
    assert float(((e - e_o).abs() / e_o.abs().clamp(min=1.0)).max()) < 1e-9
    g_o = torch.autograd.grad(orc(pos).abs().log().sum(), [orc.mo_modifier, orc.bas_exp])
    wf.zero_grad()
    wf(x).abs().log().sum().backward()
    for a, o in zip((wf.mo.mo_modifier.grad, wf.ao.bas_exp.grad), g_o):
        torch.testing.assert_close(a.cpu(), o, rtol=1e-9, atol=1e-9)
    wf.zero_grad()
    wf.ao.bas_exp.requires_grad_(False)
    orc.bas_exp.requires_grad_(False)
    wf.local_energy_autodiff(x).sum().backward()
    g_o = torch.autograd.grad(orc.local_energy(pos).sum(), [orc.mo_modifier])[0]
    torch.testing.assert_close(wf.mo.mo_modifier.grad.cpu(), g_o, rtol=1e-8, atol=1e-8)
