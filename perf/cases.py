"""What this framework's speed is judged by: the work that its users have it do.

Every case goes through public entry points (`molgw_amd.gw.Engine`, `molgw_amd.serving.Server`), from device-resident
RI tensors where such a program holds them, with host arrays for what the callers hold on the host (orbitals,
energies). Sizes are the shapes of the repository's own molecules (alkanes CnH2n+2, water clusters (H2O)m in
cc-pVDZ / cc-pVTZ with their RI bases). RI tensors and orbitals are drawn from the synthetic recipe of
`molgw_amd.workloads` at molecular magnitudes (scale 0.3); the integral cases take real geometries and basis files.

Paths (the "path" of a case):

* jk         Hartree and exchange matrices through the resident RI tensor: one iteration of the device RI-HF.
* integrals  (mu nu|P) on the GPU and B = (mu nu|Q) V^-1/2, left resident and handed back packed: the start of
             every molecule that the front end makes.
* grid       new orbitals, then W on the imaginary axis and Sigma(i omega): the calls that the Fortran drop-in makes.
* pade       a whole G0W0 solve from RI tensor and orbitals to quasiparticle energies (imaginary axis + Pade), as a
             serving slot runs it.
* oneshot    a whole G0W0 solve with the analytic Casida W: the reference's default GW.
* contour    a whole G0W0 solve by contour deformation.
* poles      the pole self-energy of every state on a resident W: one-shot GW's real grid, or the one point of an
             eigenvalue self-consistent step (GnW0).
* qs         the QSGW self-energy matrix on a resident W: one step of the QSGW loop.
* serving    a batch of molecules through the continuous-batching server.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from molgw_amd.frontend import Molecule, alkane, water_cluster
from molgw_amd.frontend.basis import BasisSet
from molgw_amd.gw import Engine, selfenergy_set_state_range
from molgw_amd.serving import Request, Server
from molgw_amd.workloads import BASIS_DIR, DeviceSystem, alkane_shape, upper_pairs, water_cluster_shape

DEVICE = 'cuda' if torch.cuda.is_available() else 'cpu'
NOMEGA_CHI, NOMEGA_CALC = 32, 16      # the serving stream's imaginary grid and Pade points
STEP_CALC = 0.03
NIMAG, NREAL = 16, 6                  # the contour benchmark's W grids
NSIGMA, STEP, ETA = 51, 0.01, 0.001   # the reference's real grid
WINDOW = 8                            # HOMO-7 .. LUMO+8


# ------------------------------------------------------------------ cases
def _case(path, mol, n, basis='cc-pVDZ', **more):
    return dict({'path': path, 'mol': mol, 'n': n, 'basis': basis}, **more)


def listed():
    def named(name, case):
        return dict(case, name=name)
    return [
        # an SCF iteration of a small molecule: launches and latency
        named('jk_water2', _case('jk', 'water', 2)),
        # an SCF iteration of the stream's largest molecule
        named('jk_water32', _case('jk', 'water', 32)),
        # the RI tensor of a mid-size molecule from its basis sets
        named('integrals_alkane8', _case('integrals', 'alkane', 8)),
        # the FP64 drop-in's imaginary-axis calls on a mid-size molecule
        named('grid_alkane16_fp64', _case('grid', 'alkane', 16, precision='fp64')),
        # the smallest request of the stream: launches and latency
        named('pade_water1_fp16x3', _case('pade', 'water', 1, precision='fp16x3')),
        # an ordinary request of the stream
        named('pade_alkane12_fp16x3', _case('pade', 'alkane', 12, precision='fp16x3')),
        # the largest request of the stream
        named('pade_water32_fp16x3', _case('pade', 'water', 32, precision='fp16x3')),
        # the reference's default GW on a small molecule
        named('oneshot_water2_fp64', _case('oneshot', 'water', 2)),
        # contour deformation at the benchmark's (H2O)8 shape
        named('contour_water8_fp64', _case('contour', 'water', 8)),
        # Sigma of every state on the one-shot grid, triple-zeta propane
        named('poles_alkane3_tz', _case('poles', 'alkane', 3, 'cc-pVTZ', nomega=NSIGMA)),
        # one QSGW step
        named('qs_water4', _case('qs', 'water', 4)),
        # a batch of small molecules through the server
        named('serving_alkanes', {'path': 'serving', 'count': 16, 'nmin': 1, 'nmax': 8, 'stream': 0}),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(['jk', 'jk', 'integrals', 'grid', 'grid', 'pade', 'pade', 'pade', 'oneshot', 'contour', 'poles',
                       'poles', 'qs', 'serving'])
    mol = rng.choice(['alkane', 'water'])
    if path == 'jk':
        return _case(path, mol, _between(rng, 1, 24 if mol == 'alkane' else 32))
    if path == 'integrals':
        if rng.random() < 0.3:
            return _case(path, 'alkane', _between(rng, 1, 4), 'cc-pVTZ')
        return _case(path, mol, _between(rng, 1, 10))
    if path == 'grid':
        return _case(path, mol, _between(rng, 1, 16), precision='fp64')
    if path == 'pade':
        return _case(path, mol, _between(rng, 1, 24 if mol == 'alkane' else 32), precision='fp16x3')
    if path == 'oneshot':
        return _case(path, mol, _between(rng, 1, 4))
    if path == 'contour':
        return _case(path, mol, _between(rng, 2, 8))
    if path == 'poles':
        return _case(path, mol, _between(rng, 1, 4), rng.choice(['cc-pVDZ', 'cc-pVTZ']) if mol == 'alkane' else 'cc-pVDZ',
                     nomega=rng.choice([1, NSIGMA]))
    if path == 'qs':
        return _case(path, mol, _between(rng, 1, 5))
    return {'path': 'serving', 'count': rng.randint(6, 16), 'nmin': 1, 'nmax': rng.randint(4, 8),
            'stream': rng.randint(1, 999)}


def _shape(case):
    """(nbf, naux, nocc) of the case's molecule."""
    return (alkane_shape if case['mol'] == 'alkane' else water_cluster_shape)(case['n'], case['basis'])


def _stream_shapes(case):
    sizes = np.random.default_rng(case['stream']).integers(case['nmin'], case['nmax'] + 1, case['count'])
    return [alkane_shape(int(n)) for n in sizes]


# ------------------------------------------------------------------ inputs
class _Inputs:
    """A synthetic molecule: packed RI tensor on the device (torch (naux, npair) = column-major (npair, naux),
    diagonal pairs x 1/2), pair list, orbitals, energies and occupations on the host."""

    def __init__(self, nbf, naux, nocc, seed):
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed(seed * 7919 + nbf)
        def randn(*shape):
            return torch.randn(*shape, generator=gen, device=DEVICE, dtype=torch.float64)
        self.nbf, self.naux, self.nocc = nbf, naux, nocc
        self.ib = upper_pairs(nbf)
        self.npair = self.ib.shape[1]
        sv = (1.0 + torch.arange(naux, device=DEVICE, dtype=torch.float64)) ** -1.5
        lmat = (randn(naux, naux) * sv[None, :]) @ randn(naux, naux) * (0.3 / naux)
        self.packed = torch.empty(naux, self.npair, device=DEVICE, dtype=torch.float64)
        for p0 in range(0, self.npair, 65536):
            p1 = min(self.npair, p0 + 65536)
            self.packed[:, p0:p1] = lmat @ randn(naux, p1 - p0)
        self.packed[:, torch.from_numpy(self.ib[0] == self.ib[1]).to(DEVICE)] *= 0.5
        q, r = torch.linalg.qr(randn(nbf, nbf))
        self.c = np.asfortranarray((q * torch.sign(torch.diagonal(r))[None, :]).cpu().numpy())
        host = np.random.default_rng(seed)
        self.energy = np.concatenate([np.sort(host.uniform(-1.2, -0.3, nocc)),
                                      np.sort(host.uniform(0.05, 3.0, nbf - nocc))])
        self.occupation = np.concatenate([np.full(nocc, 2.0), np.zeros(nbf - nocc)])

    def system(self):
        return DeviceSystem('synthetic', self.nbf, self.naux, self.nocc, self.packed, self.ib, self.c, self.energy,
                            self.occupation)

    def window(self):
        rng = selfenergy_set_state_range(self.occupation)
        rng.nsemin = max(rng.nsemin, rng.nhomo_G - WINDOW + 1)
        rng.nsemax = min(rng.nsemax, rng.nhomo_G + WINDOW)
        return rng

    def load(self, eng):
        eng.set_eri_3center_device(self.packed.data_ptr(), self.npair, self.naux, self.ib, self.nbf)
        eng.set_mo(self.c, self.energy, self.occupation)

    def omega_calc(self):
        return (0.5 * (self.energy[self.nocc - 1] + self.energy[self.nocc]) + 1j * STEP_CALC * np.arange(NOMEGA_CALC))


def _molecule(case, seed):
    mol = alkane(case['n']) if case['mol'] == 'alkane' else water_cluster(case['n'], seed=seed)
    shift = np.random.default_rng(seed).normal(0.0, 0.05, np.shape(mol.coords))   # a vibrating geometry (bohr)
    return Molecule(list(mol.atoms), np.asarray(mol.coords) + shift)


class _ServerState:
    def __init__(self, case, seed):
        self.server = Server()
        self.systems = [_Inputs(*shape, seed * 101 + k).system() for k, shape in enumerate(_stream_shapes(case))]

    def __del__(self):
        self.server.close()


def prepare(case, seed):
    path = case['path']
    if path == 'serving':
        state = _ServerState(case, seed)
        torch.cuda.synchronize()
        return case, state
    eng = Engine(0)
    if path == 'integrals':
        mol = _molecule(case, seed)
        bs = BasisSet(mol.atoms, mol.coords, case['basis'], BASIS_DIR)
        aux = BasisSet(mol.atoms, mol.coords, case['basis'] + '-RI', BASIS_DIR)
        kept, _, _ = eng.inverse_sqrt_eri_2center(eng.eri_2center_ao(aux), copy=False)
        ib = upper_pairs(bs.nbf)
        out = torch.empty(kept, ib.shape[1], device=DEVICE, dtype=torch.float64)
        return case, (eng, bs, aux, ib, out)
    inp = _Inputs(*_shape(case), seed)
    torch.cuda.synchronize()              # the engine reads the RI tensor on a stream of its own
    if path in ('jk', 'grid', 'poles', 'qs'):
        inp.load(eng)
        inp.packed = None                 # the engine holds its own copy
    if path in ('poles', 'qs'):
        eng.polarizability(selfenergy_set_state_range(inp.occupation))
    return case, (eng, inp)


# ------------------------------------------------------------------ one pass
def run(state):
    case, st = state
    path = case['path']
    if path == 'serving':
        res = st.server.run([Request(k, s) for k, s in enumerate(st.systems)], realtime=False)
        return [(r.energy_qp, r.zz, r.en_rpa, r.en_gw) for r in res]
    if path == 'integrals':
        eng, bs, aux, ib, out = st
        eng.eri_3center_ao(bs, aux, ib, copy=False)
        eng.build_eri_3center_resident(ib, bs.nbf, out_ptr=out.data_ptr())
        return out
    eng, inp = st
    if path == 'jk':
        return eng.hartree_exchange_ri(inp.c[:, :inp.nocc])
    if path == 'grid':
        rng = inp.window()
        eng.set_mo(inp.c, inp.energy, inp.occupation)
        om, wt = _imaginary_grid(NOMEGA_CHI)
        erpa, egw, _ = eng.polarizability_grid(rng, om, wt, precision=case['precision'])
        return erpa, egw, eng.gw_selfenergy_imag(rng, inp.omega_calc())
    if path == 'poles':
        rng = selfenergy_set_state_range(inp.occupation)
        return eng.gw_selfenergy(rng, _real_grid(case['nomega']), inp.energy)
    if path == 'qs':
        return eng.gw_selfenergy_qs(selfenergy_set_state_range(inp.occupation))[0]
    inp.load(eng)
    if path == 'pade':
        out = eng.g0w0(inp.window(), technique='imaginary_pade', precision=case['precision'],
                       nomega_chi_imag=NOMEGA_CHI, nomega_sigma_calc=NOMEGA_CALC, return_sigma=False)
        return out.energy_qp, out.zz, out.energy_qp_lin, out.en_rpa, out.en_gw
    if path == 'oneshot':
        out = eng.g0w0()
        return out.energy_qp, out.zz, out.energy_qp_lin, out.sigma, out.en_rpa, out.en_gw
    out = eng.g0w0(inp.window(), technique='contour', nomega_chi_imag=NIMAG, nomega_chi_real=NREAL)
    return out.energy_qp, out.zz, out.energy_qp_lin, out.sigma


# ------------------------------------------------------------------ what a pass cannot do without
def _solve_work(nbf, naux, nocc, nse):
    """Imaginary-axis G0W0 from orbitals: transforms, chi0, factor and inverse, W.B."""
    npole, ng = nocc * (nbf - nocc), nbf
    flops = (2.0 * naux * nbf * nbf * nocc + 2.0 * naux * nbf * npole + 2.0 * naux * nbf * ng * nse +
             NOMEGA_CHI * (naux * (naux + 1.0) * (npole + ng * nse) + 2.0 / 3.0 * naux ** 3))
    return flops, 8.0 * (naux * nbf * (nbf + 1) / 2 + nbf * nbf)


def work(case):
    path = case['path']
    if path == 'serving':
        parts = [_solve_work(*s, min(2 * WINDOW, s[2] + WINDOW)) for s in _stream_shapes(case)]
        return {'flops': sum(f for f, _ in parts), 'bytes': sum(b for _, b in parts)}
    nbf, naux, nocc = _shape(case)
    npair, npole, nv = nbf * (nbf + 1) // 2, nocc * (nbf - nocc), nbf - nocc
    nse = min(nocc, WINDOW) + min(nv, WINDOW)
    if path == 'jk':
        return {'bytes': 8.0 * (naux * npair + nbf * nocc + 2 * nbf * nbf),
                'flops': 2.0 * naux * nbf * nbf * nocc + naux * nocc * nbf * (nbf + 1.0) + 4.0 * naux * npair}
    if path == 'integrals':
        # the integrals themselves depend on contractions and classes: only the product with V^-1/2 is counted
        return {'bytes': 8.0 * npair * naux, 'flops': 2.0 * npair * naux * naux}
    if path in ('grid', 'pade'):
        flops, nbytes = _solve_work(nbf, naux, nocc, nse)
        return {'flops': flops, 'bytes': nbytes}
    if path == 'oneshot':
        poles = 2.0 * npole * nbf * nbf * naux + 8.0 * NSIGMA * npole * nbf * nbf
        return {'bytes': 8.0 * (naux * npair + nbf * nbf),
                'flops': 2.0 * naux * nbf * nbf * nbf + naux * (npole + 1.0) * npole + 10.0 / 3.0 * npole ** 3 +
                2.0 * naux * npole * npole + poles}
    if path == 'contour':
        nf = NIMAG + NREAL
        return {'bytes': 8.0 * (naux * npair + nbf * nbf),
                'flops': 2.0 * naux * nbf * nbf * (nocc + nse) + 2.0 * naux * nbf * npole +
                nf * (naux * (naux + 1.0) * npole + 10.0 / 3.0 * naux ** 3 + 2.0 * naux * naux * nbf * nse)}
    if path == 'poles':
        return {'bytes': 8.0 * (naux * npair + naux * npole),
                'flops': 2.0 * naux * nbf ** 3 + 2.0 * npole * nbf * nbf * naux + 8.0 * case['nomega'] * npole * nbf * nbf}
    return {'bytes': 8.0 * (naux * npair + naux * npole + nbf * nbf),
            'flops': 2.0 * naux * nbf ** 3 + 2.0 * npole * nbf * nbf * naux + 2.0 * npole * nbf ** 3}


# ------------------------------------------------------------------ the same results in plain 64 bits
def _imaginary_grid(n):
    x, w = np.polynomial.legendre.leggauss(n)
    x, w = 0.5 * (x + 1.0), 0.5 * w
    return 2.0 * x / (1.0 - x), 2.0 * w / (1.0 - x) ** 2


def _real_grid(nomega):
    return STEP * np.arange(-(nomega // 2), nomega // 2 + 1)


def _dense(inp):
    k, l = (torch.from_numpy((inp.ib[d] - 1).astype(np.int64)).to(DEVICE) for d in (0, 1))
    b = torch.zeros(inp.naux, inp.nbf, inp.nbf, device=DEVICE, dtype=torch.float64)
    b[:, k, l] += inp.packed
    b[:, l, k] += inp.packed
    return b                              # the halved diagonal pairs were added twice


def _mo(inp, b, lo, hi):
    """(P|p m) for all p and m in [lo, hi) of the dense b(P, k, l), as (naux, nbf, hi - lo)."""
    c = torch.from_numpy(np.ascontiguousarray(inp.c)).to(DEVICE)
    h = (b.reshape(-1, inp.nbf) @ c[:, lo:hi].contiguous()).reshape(inp.naux, inp.nbf, hi - lo)
    return torch.cat([torch.matmul(c.T.contiguous(), h[p:p + 64]) for p in range(0, inp.naux, 64)])


def _transitions(inp, b):
    """X(P, t) with t = (i outer, a inner), and the transition energies."""
    x = _mo(inp, b, 0, inp.nocc)[:, inp.nocc:, :].transpose(1, 2).reshape(inp.naux, -1).contiguous()
    e = torch.from_numpy(inp.energy).to(DEVICE)
    return x, (e[None, inp.nocc:] - e[:inp.nocc, None]).reshape(-1)


def _exact_grid(inp, b, rng):
    """(E_RPA, E_GW, Sigma(i omega)[ncalc, nse]) on the imaginary axis."""
    x, de = _transitions(inp, b)
    lo, hi = rng.nsemin - 1, rng.nsemax
    bm = _mo(inp, b, lo, hi).reshape(inp.naux, -1)            # columns (p, m)
    om, wt = _imaginary_grid(NOMEGA_CHI)
    one = torch.eye(inp.naux, device=DEVICE, dtype=torch.float64)
    n2 = (x * x).sum(0)
    erpa = egw = 0.0
    wc = inp.omega_calc()
    sigma = np.zeros((len(wc), hi - lo), dtype=np.complex128)
    ep = inp.energy[:, None]
    for w, q in zip(om, wt):
        s = 4.0 * de / (w * w + de * de)
        m = one + (x * s[None, :]) @ x.T
        h0 = float((s * n2).sum())
        chol = torch.linalg.cholesky(m)
        inv = torch.cholesky_inverse(chol)
        erpa += (2.0 * float(torch.log(torch.diagonal(chol)).sum()) - h0) * q / (2.0 * math.pi)
        egw += (inp.naux - float(torch.diagonal(inv).sum()) - h0) * q / (2.0 * math.pi)
        v = (((inv - one) @ bm) * bm).sum(0).reshape(inp.nbf, hi - lo).cpu().numpy()
        for k, z in enumerate(wc):
            g = 1.0 / (z - ep + 1j * w) + 1.0 / (z - ep - 1j * w)
            sigma[k] -= q / (2.0 * math.pi) * (g * v).sum(0)
    return erpa, egw, sigma


def _exact_casida(inp, b):
    """Poles and residues w_s(P, s) of W, and E_RPA."""
    x, de = _transitions(inp, b)
    sq = torch.sqrt(de)
    m = 4.0 * (x * sq[None, :]).T @ (x * sq[None, :])
    m.diagonal().add_(de * de)
    lam, z = torch.linalg.eigh(m)
    om = torch.sqrt(lam)
    ws = math.sqrt(2.0) * ((x * sq[None, :]) @ z) / torch.sqrt(om)[None, :]
    erpa = 0.5 * float(om.sum()) - 0.5 * float(de.sum()) - float((x * x).sum())
    return om, ws, erpa


def _exact_poles(inp, b, omega):
    """(Sigma[nomega, nstate], E_GW) on energy0 + omega, and E_RPA."""
    om, ws, erpa = _exact_casida(inp, b)
    e = torch.from_numpy(inp.energy).to(DEVICE)
    grid = torch.from_numpy(omega).to(DEVICE)
    mo = _mo(inp, b, 0, inp.nbf)
    sigma = torch.zeros(len(omega), inp.nbf, device=DEVICE, dtype=torch.complex128)
    egw = 0.0
    for p in range(inp.nbf):
        w2 = (ws.T @ mo[:, p, :].contiguous()) ** 2                       # (s, i)
        for k in range(len(omega)):
            d = (e[p] + grid[k] - e)[None, :]
            lo = d[:, :inp.nocc] + om[:, None]
            hi = d[:, inp.nocc:] - om[:, None]
            sigma[k, p] = ((w2[:, :inp.nocc] * (lo + 1j * ETA) / (lo * lo + ETA * ETA)).sum() +
                           (w2[:, inp.nocc:] * (hi - 1j * ETA) / (hi * hi + ETA * ETA)).sum())
        if p < inp.nocc:
            egw += 2.0 * float((w2[:, inp.nocc:] / ((e[p] - e[inp.nocc:])[None, :] - om[:, None])).sum())
    return sigma.cpu().numpy(), egw, erpa


def _exact_qs(inp, b):
    om, ws, _ = _exact_casida(inp, b)
    e = torch.from_numpy(inp.energy).to(DEVICE)
    mo = _mo(inp, b, 0, inp.nbf)
    sig = torch.zeros(inp.nbf, inp.nbf, device=DEVICE, dtype=torch.float64)
    for i in range(inp.nbf):
        w = ws.T @ mo[:, :, i].contiguous()                               # (s, p)
        d = (e - e[i])[None, :] + (om[:, None] if i < inp.nocc else -om[:, None])
        sig += w.T @ (w * (d / (d * d + ETA * ETA)))
    return (0.5 * (sig + sig.T)).cpu().numpy()


def _exact_contour(inp, b, rng):
    """Sigma[nomega, nse] by contour deformation with the low-rank W (|lambda / (1 - lambda)| > 1e-3)."""
    x, de = _transitions(inp, b)
    lo, hi = rng.nsemin - 1, rng.nsemax
    bm = _mo(inp, b, lo, hi).reshape(inp.naux, -1)
    e, e0, omega = inp.energy, inp.energy[lo:hi], _real_grid(NSIGMA)
    z = e0[None, :] + omega[:, None]                                      # (k, m)
    d_occ = e[None, None, :inp.nocc] - z[:, :, None]
    d_emp = z[:, :, None] - e[None, None, inp.nocc:]
    de_max = max([0.0] + [float(d[d >= -ETA].max()) for d in (d_occ, d_emp) if (d >= -ETA).any()])
    om, wt = _imaginary_grid(NIMAG)
    om_re = np.arange(NREAL) / (NREAL - 1) * de_max
    v = []
    for w2 in list(-om ** 2) + list(om_re ** 2):
        lam, u = torch.linalg.eigh(-(x * (4.0 * de / (de * de - w2))[None, :]) @ x.T)
        eta = lam / (1.0 - lam)
        eta = torch.where(eta.abs() > 1.0e-3, eta, torch.zeros_like(eta))
        v.append(((u.T @ bm) ** 2 * eta[:, None]).sum(0).reshape(inp.nbf, hi - lo).cpu().numpy())
    sigma = np.zeros((len(omega), hi - lo))
    for k in range(len(omega)):
        for m in range(hi - lo):
            xx = z[k, m] - e
            far = np.abs(xx) > ETA
            for f in range(NIMAG):
                sigma[k, m] -= wt[f] / (2.0 * math.pi) * np.sum((2.0 * xx / (xx * xx + om[f] ** 2) * v[f][:, m])[far])
            for p in range(inp.nbf):
                d = -xx[p] if p < inp.nocc else xx[p]
                if d < -ETA:
                    continue
                j = int(np.argmin(np.abs(om_re - abs(d))))
                r = v[NIMAG + j][p, m] * (0.5 if abs(d) < ETA else 1.0)
                sigma[k, m] += -r if p < inp.nocc else r
    return sigma.astype(np.complex128), omega


def _pade(wc, sc, omega):
    """Thiele's continued fraction through (wc, sc) and the conjugate points, at omega +- i eta."""
    z = np.concatenate([wc[:0:-1].conj(), wc])
    out = np.zeros((len(omega), sc.shape[1]), dtype=np.complex128)
    for m in range(sc.shape[1]):
        g = np.concatenate([sc[:0:-1, m].conj(), sc[:, m]])
        a = [g[0]]
        for p in range(1, len(z)):
            g[p:] = (g[p - 1] - g[p:]) / ((z[p:] - z[p - 1]) * g[p:])
            a.append(g[p])
        zo = omega + 1j * ETA * np.where(omega - wc[0].real >= 0.0, -1.0, 1.0)
        a0, a1, b0, b1 = 0.0, a[0], 1.0, 1.0
        for p in range(1, len(z)):
            f = (zo - z[p - 1]) * a[p]
            a0, a1 = a1, a1 + f * a0
            b0, b1 = b1, b1 + f * b0
        out[:, m] = a1 / b1
    return out


def _quasiparticles(sigma, omega, se_e0, e0, first, nstate, energy):
    """Graphical and linearised quasiparticle energies of the states first .. first + nse."""
    qp, zz, lin = energy.copy(), np.ones(nstate), energy.copy()
    n0 = len(omega) // 2
    for m in range(sigma.shape[1]):
        s = sigma[:, m].real
        x = omega + se_e0[m]
        g = s + e0[m] - x
        best = None
        for k in range(1, len(x)):
            if g[k - 1] * g[k] < 0.0:
                slope = (g[k] - g[k - 1]) / (x[k] - x[k - 1])
                z = -1.0 / slope
                if z >= 1.0e-5 and (best is None or z > best[0]):
                    best = (z, x[k - 1] - g[k - 1] / slope)
        p = first + m
        zz[p], qp[p] = best if best else (1.0, e0[m] + s[n0])
        z = min(max(1.0 / (1.0 - (s[n0 + 1] - s[n0 - 1]) / (omega[n0 + 1] - omega[n0 - 1])), 0.0), 1.0)
        lin[p] = se_e0[m] + z * (e0[m] - se_e0[m] + s[n0])
    return qp, zz, lin


def _exact_pade(inp):
    rng = inp.window()
    erpa, egw, sc = _exact_grid(inp, _dense(inp), rng)
    wc = inp.omega_calc()
    omega = wc[0].real + _real_grid(NSIGMA)
    sigma = _pade(wc, sc, omega)
    lo, hi = rng.nsemin - 1, rng.nsemax
    return _quasiparticles(sigma, omega, np.zeros(hi - lo), inp.energy[lo:hi], lo, inp.nbf, inp.energy), erpa, egw


def exact(case, seed):
    path = case['path']
    if path == 'integrals':
        return None                       # Gaussian integrals have no short plain form
    if path == 'serving':
        out = []
        for k, shape in enumerate(_stream_shapes(case)):
            (qp, zz, _), erpa, egw = _exact_pade(_Inputs(*shape, seed * 101 + k))
            out.append((qp, zz, erpa, egw))
        return out
    inp = _Inputs(*_shape(case), seed)
    if path == 'pade':
        (qp, zz, lin), erpa, egw = _exact_pade(inp)
        return qp, zz, lin, erpa, egw
    b = _dense(inp)
    if path == 'jk':
        x = torch.from_numpy(np.ascontiguousarray(inp.c[:, :inp.nocc])).to(DEVICE)
        h = (b.reshape(-1, inp.nbf) @ x).reshape(inp.naux, inp.nbf, inp.nocc)
        gamma = 2.0 * (h * x[None]).sum((1, 2))
        k = torch.zeros(inp.nbf, inp.nbf, device=DEVICE, dtype=torch.float64)
        for p in range(inp.naux):
            k -= h[p] @ h[p].T
        return (gamma @ b.reshape(inp.naux, -1)).reshape(inp.nbf, inp.nbf).cpu().numpy(), k.cpu().numpy()
    if path == 'grid':
        return _exact_grid(inp, b, inp.window())
    if path == 'qs':
        return _exact_qs(inp, b)
    if path == 'poles':
        sigma, egw, _ = _exact_poles(inp, b, _real_grid(case['nomega']))
        return sigma, egw
    if path == 'oneshot':
        omega = _real_grid(NSIGMA)
        sigma, egw, erpa = _exact_poles(inp, b, omega)
        return (*_quasiparticles(sigma, omega, inp.energy, inp.energy, 0, inp.nbf, inp.energy), sigma, erpa, egw)
    rng = inp.window()
    sigma, omega = _exact_contour(inp, b, rng)
    lo, hi = rng.nsemin - 1, rng.nsemax
    e0 = inp.energy[lo:hi]
    return (*_quasiparticles(sigma, omega, e0, e0, lo, inp.nbf, inp.energy), sigma)
