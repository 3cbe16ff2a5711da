'''Performance cases of the UPPE and paraxial steppers: what users of the framework have it do.

A case is one call pattern of the public API on one of the repository's own workloads (searay_amd.configs), with
sizes between its test grids and its benchmark grids:

* 'step'     -- a stepper handle: load a field, advance it over a number of subcycles, read the field back
                (``RunSetup.make_stepper``, ``set_field`` / ``advance`` / ``finish``), as the benchmark, the
                optimisation loops and direct users of the C ABI do. The handle, its basis and its medium are kept.
* 'plane'    -- ``uppe_kernel.propagator``, the reference's per-plane call, with every diagnostic it returns.
* 'batch'    -- ``batch.Batch``: a parameter scan, many radial instances stepped together.
* 'gradient' -- ``adjoint.SpectralPhaseProblem.value_and_grad``: a loss and its gradient.

Outputs of FP32 and BF16x3 handles hold single-precision numbers in complex128 arrays; ``run`` hands them on as
complex64, the type they have.

``exact`` repeats the propagation in 64 bits with torch alone. The tables that a handle is loaded with (wavenumbers,
densities, the radial basis, rate coefficients, the initial field) are inputs of both and come from the workload
builders.
'''
import numpy as np
import torch

from searay_amd import adjoint, batch, configs, paraxial_kernel, uppe_kernel

SINGLE = ('fp32', 'bf16x3')


# ---------------------------------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # a design study's quick look: the smallest radial grid, a few steps; launches and latency are all it costs
        dict(name='radial_kerr_65x16_fp64', kind='step', workload='kerr', precision='fp64', nw=65, nr=16, nk=16,
             n2=1, subcycles=10),
        # the headline benchmark: Kerr propagation in air over 1 m, 100 fixed steps, in its fast precision
        dict(name='radial_kerr_513x128_bf16x3', kind='step', workload='kerr', precision='bf16x3', nw=513, nr=128,
             nk=128, n2=1, subcycles=100),
        # the same physics in the default precision, with fewer radial modes than cells (a ragged contraction)
        dict(name='radial_kerr_513x128_fp64', kind='step', workload='kerr', precision='fp64', nw=513, nr=128,
             nk=100, n2=1, subcycles=50),
        # ionisation and plasma on the large radial grid, adaptive steps
        dict(name='radial_o2_2049x256_bf16x3', kind='step', workload='o2', precision='bf16x3', nw=2049, nr=256,
             nk=256, n2=1, subcycles=100),
        # the series rate model in FP32, on a wide beam: many radial cells, an odd number of modes
        dict(name='radial_series_1025x512_fp32', kind='step', workload='series', precision='fp32', nw=1025, nr=512,
             nk=391, n2=1, subcycles=40),
        # N2 with its rotational states, a non-axisymmetric beam of four azimuthal points
        dict(name='radial_raman_513x64x4_fp32', kind='step', workload='raman', precision='fp32', nw=513, nr=64,
             nk=64, n2=4, subcycles=40),
        # the drop-in call of the reference's plugin, one diagnostic plane with all its outputs, default precision
        dict(name='plane_o2_1025x128_fp64', kind='plane', workload='o2', precision='fp64', nw=1025, nr=128, nk=128,
             n2=1, subcycles=50),
        # three-dimensional filamentation: bound by memory, many strips
        dict(name='cartesian_513x128x128_fp32', kind='step', workload='filament', precision='fp32', nw=513, nr=128,
             nk=128, n2=128, subcycles=100),
        # a small three-dimensional run in the default precision, an oblong window
        dict(name='cartesian_129x64x32_fp64', kind='step', workload='filament', precision='fp64', nw=129, nr=64,
             nk=64, n2=32, subcycles=30),
        # the paraxial envelope model: the focused air filament of the reference's examples
        dict(name='envelope_256x256_bf16x3', kind='step', workload='envelope', precision='bf16x3', nw=256, nr=256,
             nk=128, n2=1, subcycles=100),
        # a scan over energies and gases: 16 instances of four radial sizes in one batch
        dict(name='batch_16x513_bf16x3', kind='batch', workload='scan', precision='bf16x3', nw=513, nr=256, nk=256,
             n2=1, members=16, subcycles=40),
        # pulse shaping: the loss and its gradient with respect to the input phase
        dict(name='gradient_513x128_fp32', kind='gradient', workload='kerr', precision='fp32', nw=513, nr=128,
             nk=128, n2=1, subcycles=50, every=10),
    ]


def draw(rng):
    def pow2(lo, hi):
        return 2 ** rng.randint(lo, hi)

    pick = rng.random()
    if pick < 0.55:
        # radial handles and planes: every workload and precision, 33 to 2049 frequencies, 8 to 512 cells
        workload = rng.choice(['kerr', 'kerr', 'o2', 'o2', 'series', 'raman'])
        precision = rng.choice(['fp64', 'fp32', 'bf16x3'])
        kind = 'plane' if rng.random() < 0.2 else 'step'
        nw = pow2(5, 11 if workload in ('o2', 'series') else 9) + 1
        if workload in ('o2', 'series'):
            nw = max(nw, 129)  # the pulse has to fit the time window, which shortens with the grid
        else:
            nw = max(nw, 65)
        nr = pow2(3, 9)
        while nw * nr > 1 << 20:
            nr //= 2
        n2 = rng.choice([2, 4]) if nr <= 64 and kind == 'step' and rng.random() < 0.15 else 1
        nk = nr if rng.random() < 0.6 else rng.randint(max(4, nr // 2), nr)
        return dict(kind=kind, workload=workload, precision='fp64' if kind == 'plane' else precision, nw=nw, nr=nr,
                    nk=nk, n2=n2, subcycles=rng.randint(5, 90))
    if pick < 0.7:
        precision = rng.choice(['fp64', 'fp32', 'fp32'])
        nw = pow2(6, 9) + 1
        nr, n2 = pow2(4, 8), pow2(4, 8)
        while nw * nr * n2 > (1 << 22 if precision == 'fp64' else 1 << 23):
            if nr >= n2:
                nr //= 2
            else:
                n2 //= 2
        return dict(kind='step', workload='filament', precision=precision, nw=nw, nr=nr, nk=nr, n2=n2,
                    subcycles=rng.randint(3, 40))
    if pick < 0.8:
        nr = pow2(5, 8)
        return dict(kind='step', workload='envelope', precision=rng.choice(['fp64', 'fp32', 'bf16x3']),
                    nw=pow2(6, 8), nr=nr, nk=rng.randint(nr // 3, nr), n2=1, subcycles=rng.randint(5, 100))
    if pick < 0.9:
        return dict(kind='batch', workload='scan', precision=rng.choice(['fp64', 'fp32', 'bf16x3']), nw=513, nr=256,
                    nk=256, n2=1, members=rng.randint(2, 16), subcycles=rng.randint(9, 40))
    nr = pow2(4, 7)
    return dict(kind='gradient', workload=rng.choice(['kerr', 'kerr', 'o2']),
                precision=rng.choice(['fp64', 'fp32']), nw=pow2(7, 9) + 1, nr=nr, nk=nr, n2=1,
                subcycles=rng.randint(10, 50), every=rng.choice([5, 10]))


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------
def _volume(case, seed):
    '''The input dictionary of the case's workload on its grid, as an input file would build it.'''
    w, nw, nr = case['workload'], case['nw'], case['nr']
    kind = case['kind']
    if w in ('kerr', 'raman'):
        build = configs.radial_kerr_air if w == 'kerr' else configs.radial_raman_air
        vol = build(scale=512 // (nw - 1), steps=100, seed=seed)
        vol['wave grid'] = (nw, nr, case['n2'], 2)
        vol['radial modes'] = case['nk']
    elif w in ('o2', 'series'):
        # subcycles of 0.5 mm, each one adaptive step or a few, at the critical power (well above it the collapse
        # makes the step sequence depend on the last bit); the gradient takes fixed steps of 40 um. Whole planes and
        # gradients cover their own subcycles only
        count = case['subcycles'] if kind in ('plane', 'gradient') else 400
        scale = 2048 // (nw - 1)
        vol = configs.radial_o2_ionization(scale=scale, steps=count, seed=seed, power=1.0,
                                           rate='explicit' if w == 'o2' else 'series',
                                           length='%g mm' % ((0.04 if kind == 'gradient' else 0.5) * count), nr=nr)
        vol['wave grid'] = (nw, nr, case['n2'], 2)
        vol['radial modes'] = case['nk']
        # small grids shorten the time window rather than cut the pulse's band off
        vol['frequency band'] = (0.0, max(2.0, 8.0 / scale))
        vol['nonlinear band'] = (0.0, min(4.0, vol['frequency band'][1]))
        if kind == 'gradient':
            vol['minimum step'] = vol['size'][2] / count
    elif w == 'filament':
        vol = configs.cartesian_filamentation(scale=512 // (nw - 1), steps=200, seed=seed)
        vol['wave grid'] = (nw, nr, case['n2'], 2)
    else:
        vol = configs.paraxial_air_filament(steps=400, seed=seed)
        vol['wave grid'] = (nw, nr, 1, 20)
        vol['radial modes'] = case['nk']
    if kind in ('plane', 'gradient') and w in ('kerr', 'raman'):
        x, y, length = vol['size']
        vol['size'] = (x, y, length * case['subcycles'] / 100)
        vol['subcycles'] = case['subcycles']
        vol['minimum step'] = vol['size'][2] / vol['subcycles']
    if case['n2'] > 1 and w != 'filament':
        plain = vol['incoming wave']
        vol['incoming wave'] = lambda w_, r, phi: plain(w_, r, phi) * (
            1.0 + 0.3 * np.cos(phi) + 0.2 * np.sin(2 * phi))[None, None, :]
    return vol


def _setup(case, seed):
    module = paraxial_kernel if case['workload'] == 'envelope' else uppe_kernel
    return module.RunSetup(_volume(case, seed))


def _scan(case):
    return configs.batched_radial(n=case['members'], scale=1024 // (case['nw'] - 1), steps=200)[0]


def _scan_fields(setups, seed):
    '''The members' initial fields, each with a spectral phase of its own.'''
    rng = np.random.default_rng([seed, 11])
    return [rs.A0 * np.exp(0.2j * np.pi * (rng.random(rs.w.shape) - 0.5))[:, None, None] for rs in setups]


def _phases(case, seed):
    '''Input spectral phase coefficients and the target spectrum of a gradient case.'''
    rng = np.random.default_rng([seed, 7])
    return 0.3 * rng.standard_normal(16), rng.uniform(-1.0, 1.0, case['nw'])


def _sigma(case):
    return configs.kerr_pulse_sigma() if case['workload'] == 'kerr' else configs.ionizing_pulse_sigma()


def _target(rs, xi):
    return 0.5 * np.abs(rs.A0[:, 0, 0]) ** 2 * (1 + 0.1 * xi)


def prepare(case, seed):
    state = dict(case=case, single=case['precision'] in SINGLE)
    if case['kind'] == 'batch':
        b = batch.Batch(_scan(case), precision=case['precision'])
        state.update(batch=b, fields=_scan_fields(b.setups, seed),
                     lengths=[rs.plane(0)[2] * case['subcycles'] for rs in b.setups])
        return state
    rs = _setup(case, seed)
    state['rs'] = rs
    if case['kind'] == 'gradient':
        c, xi = _phases(case, seed)
        state.update(c=c, problem=adjoint.SpectralPhaseProblem(
            _volume(case, seed), _sigma(case), precision=case['precision'], checkpoint_every=case['every'],
            n_phase=16, target=_target(rs, xi)))
        return state
    factory = uppe_kernel.hip_stepper_factory(case['precision'])
    if case['kind'] == 'plane':
        rs.mat.stepper_factory = factory
        return state
    state.update(field=rs.stepper_field(), stepper=rs.make_stepper(factory))
    return state


def run(state):
    case = state['case']

    def typed(a):
        return a.astype(np.complex64) if state['single'] else a

    if case['kind'] == 'batch':
        b = state['batch']
        b.set_fields(state['fields'])
        b.advance(max_steps=case['subcycles'])
        return [typed(m.finish(z, want_diagnostics=False)[0]) for m, z in zip(b.members, state['lengths'])]
    if case['kind'] == 'gradient':
        loss, grad = state['problem'].value_and_grad(state['c'])
        return (np.float32(loss), grad.astype(np.float32)) if state['single'] else (loss, grad)
    rs = state['rs']
    zi, zf, length = rs.plane(0)
    if case['kind'] == 'plane':
        return uppe_kernel.propagator(None, rs.field_tool, rs.window_speed, rs.A0, rs.mat, rs.ionizer, rs.rotator,
                                      rs.NL_band, rs.subcycles, zi, zf, rs.dzmin)
    st = state['stepper']
    st.set_field(state['field'])
    st.advance(zi, length, 0, case['subcycles'], rs.dzmin)
    return typed(st.finish(length * case['subcycles'], want_diagnostics=False)[0])


def work(case):
    '''Bytes and operations of one pass. Per grid point of one right-hand side: the field and the current each written
    once and read once between the transverse and the time transforms, the state read, the slope written, the
    propagation tables read; the transforms' and the contractions' operations. One step per subcycle.'''
    nw, c = case['nw'], (8 if case['precision'] in SINGLE else 16)
    if case['kind'] == 'batch':
        cells = [rs['wave grid'][1] for rs in _scan(case)]
        grids = [(n, n, 1) for n in cells]
    else:
        grids = [(case['nr'], case['nk'], case['n2'])]
    nt = nw if case['workload'] == 'envelope' else 2 * (nw - 1)
    fft = 4 if case['workload'] == 'envelope' else 1.5
    total = dict(bytes=0.0, flops=0.0)
    for nr, nk, n2 in grids:
        points = nw * nr * n2
        flops = fft * 5 * nt * np.log2(nt) * nr * n2
        if case['workload'] == 'filament':
            flops += 2 * 5 * points * np.log2(nr * n2)
        else:
            flops += 2 * 4.0 * nw * nk * nr * n2
        rounds = 4 * case['subcycles'] * (3 if case['kind'] == 'gradient' else 1)
        total['bytes'] += points * (rounds * (7 * c + 8) + 2 * c)
        total['flops'] += rounds * flops
    return total


# ---------------------------------------------------------------------------------------------------------------
# the same propagation in 64 bits
# ---------------------------------------------------------------------------------------------------------------
class _Exact:
    '''Interaction-picture RK4 in complex128 on torch arrays of shape (frequency, x1, x2).'''

    def __init__(self, rs, envelope):
        self.dev = torch.device('cuda' if torch.cuda.is_available() else 'cpu')
        zi, _, length = rs.plane(0)
        rs.mat.UpdateMaterial(zi + 0.5 * length)
        mat = rs.mat
        self.envelope = envelope
        self.w = self.t(mat.w if envelope else rs.w)[:, None, None]
        kz = self.t(mat.kz)
        self.ki = kz.imag.contiguous()
        if envelope:
            self.rate_z, self.kzc, self.div = kz.real.contiguous(), None, self.t(np.real(mat.k0))
            self.nt = mat.w.shape[0]
            self.dt = paraxial_kernel.source_dt(mat.w)
            nl, cond = np.ones(self.nt), np.ones(self.nt)
            ion = rs.ionizer
        else:
            self.rate_z, self.kzc, self.div = kz.real + self.t(mat.kg)[:, None, None], kz, kz.real
            self.nt = 2 * (rs.w.shape[0] - 1)
            self.dt, nl, cond, ion = rs.dt, rs.nl_filter, rs.cond_filter, rs.ionizer
        self.band = self.t((nl != 0) * 1.0)[:, None, None]
        if not envelope:
            self.band[:4] = 1.0  # the update covers the conditioner's bins (the current is zero there)
        self.nl, self.cond = self.t(nl)[:, None, None], self.t(cond)[:, None, None]
        self.ng = self.t(np.broadcast_to(mat.ngas, mat.kz.shape[1:]).copy())[None]
        self.chi3 = float(mat.redchi3)
        self.ion = None if ion is None else ion.kernel_params()
        self.rot = rs.rotator
        self.dzmin, self.length = float(rs.dzmin), float(length)
        tool = rs.field_tool.GetTransverseTool()
        self.H = None
        if hasattr(tool, 'H'):
            h = np.asarray(tool.H, dtype=np.float64).reshape(tool.Nk, rs.N[1], rs.N[2])
            lam = np.asarray(tool.Lambda, dtype=np.float64).reshape(-1)
            # row k, column j of the forward operator of azimuthal mode m: H[k, j, m] L_j / L_k, and back
            self.H = self.t(h.transpose(2, 0, 1) * lam[None, None, :] / lam[None, :tool.Nk, None])
            self.Hinv = self.t(h.transpose(2, 1, 0) * lam[None, None, :tool.Nk] / lam[None, :, None])

    def t(self, a):
        return torch.as_tensor(np.ascontiguousarray(a), device=self.dev)

    def _modes(self, op, a):
        out = []
        for m in range(a.shape[2]):
            x = a[:, :, m].transpose(0, 1).contiguous()
            out.append(torch.complex(op[m] @ x.real, op[m] @ x.imag).transpose(0, 1))
        return torch.stack(out, dim=2)

    def to_k(self, a):
        if self.H is None:
            return torch.fft.fft2(a, dim=(1, 2))
        if a.shape[2] > 1:
            a = torch.fft.fft(a, dim=2)
        k = self._modes(self.H, a)
        pad = a.shape[1] - k.shape[1]
        if pad:
            k = torch.cat([k, torch.zeros((a.shape[0], pad, a.shape[2]), dtype=k.dtype, device=k.device)], dim=1)
        return k

    def to_r(self, k):
        if self.H is None:
            return torch.fft.ifft2(k, dim=(1, 2))
        a = self._modes(self.Hinv, k[:, :self.H.shape[1]])
        return torch.fft.ifft(a, dim=2) if a.shape[2] > 1 else a

    def propagate(self, q, z):
        return torch.polar(torch.exp(-self.ki * z), self.rate_z * z) * q

    def ionise(self, ea):
        if self.ion is None:
            return torch.zeros_like(ea)
        p = self.ion
        em = p['e_conv'] * ea + p['e_cutoff']
        if p['kind'] == 1:
            r = p['rate_conv'] * p['c_pre'] * em ** p['c_pow'] * torch.exp(p['c_exp'] / em)
        else:
            lg, acc = torch.log(em), 0.0
            for k in range(5, -1, -1):
                acc = acc * lg + p['c'][k]
            r = p['rate_conv'] * torch.exp(acc)
        r = torch.cat([r[:-1], torch.zeros_like(r[:1])], dim=0)
        total = torch.flip(torch.cumsum(torch.flip(r, (0,)), 0), (0,))
        ne = self.ng * -torch.expm1(-self.dt * (total - 0.5 * r))
        if self.envelope:
            return ne
        n, N = torch.arange(self.nt, device=self.dev, dtype=torch.float64), self.nt

        def ramp(x):
            x = x / 64.0
            return 10 * x ** 3 - 15 * x ** 4 + 6 * x ** 5

        win = torch.ones_like(n)
        win = torch.where((n < 4) | (n > N - 5), torch.zeros_like(n), win)
        win = torch.where((n >= 4) & (n < 68), win * ramp(n - 4), win)
        win = torch.where((n <= N - 5) & (n > N - 69), win * ramp(N - 5 - n), win)
        return ne * win[:, None, None]

    def rotate(self, drive):
        if self.rot is None:
            return 0.0
        N = drive.shape[0]
        m = torch.arange(N, device=self.dev, dtype=torch.float64)[:, None, None]
        f = torch.flip(drive, (0,)) * (0.5 * self.rot.dalpha / self.rot.hbar)
        total = torch.zeros_like(drive)
        for j in range(2, len(self.rot.Tj)):
            W = complex(self.rot.Wj[j]) * self.dt
            c = float(self.rot.Tj[j]) * (2.0 * j * (j - 1) / (15.0 * (2 * j - 1))) * 2.0 * self.rot.dalpha

            def power(k):
                return torch.polar(torch.exp(-0.5 * W.imag * k), 0.5 * W.real * k)

            term = f * power(2 * m + 1)
            rho = -1j * self.dt * (torch.cumsum(term, 0) - term)
            total = total + c * torch.imag(rho * torch.conj(power(2 * m)) * W)
        return torch.flip(torch.cumsum(total * self.ng, 0), (0,))

    def source(self, e_w):
        '''The current of the field (the envelope: of A), with chi and the electron density.'''
        if self.envelope:
            e, a = torch.fft.ifft(1j * self.w * e_w, dim=0), torch.fft.ifft(e_w, dim=0)
            e2 = e.real ** 2 + e.imag ** 2
            ne = self.ionise(torch.sqrt(e2))
            chi = 0.75 * self.ng * self.chi3 * e2 + self.rotate(0.5 * e2)
            cur = ne * (0.25 * (a.real ** 2 + a.imag ** 2) - 1.0) * a
            return -1j * self.w * torch.fft.fft(chi * e, dim=0) + torch.fft.fft(cur, dim=0), chi, ne
        e = torch.fft.irfft(e_w, n=self.nt, dim=0)
        ne = self.ionise(torch.abs(e))
        chi = self.ng * self.chi3 * e * e + self.rotate(e * e)
        j = -1j * self.w * torch.fft.rfft(chi * e, dim=0)
        if self.ion is not None:
            j = j + torch.fft.rfft(ne * e, dim=0) / (0.1 - 1j * self.w)
        return self.nl * j, chi, ne

    def slope(self, q, z):
        a = self.propagate(q, z)
        if not self.envelope:
            a = 1j * self.kzc * a
        j = self.to_k(self.source(self.to_r(a))[0])
        s = 0.5j * torch.polar(torch.exp(self.ki * z), -self.rate_z * z) * j / self.div
        return s * self.band

    def step_size(self, q, k1, z):
        if self.dzmin >= self.length:
            return self.length - z
        amin = 0.01 * float(torch.max(torch.abs(q)))
        r = k1 * torch.conj(q) / (q.real ** 2 + q.imag ** 2 + amin ** 2)
        rate = 0.5 * 0.4 / self.length + torch.abs(r.imag) - torch.clamp(r.real, max=0.0)
        rate = torch.where(self.band > 0, rate, torch.zeros_like(rate))
        dz = max(0.4 / float(torch.max(rate)), self.dzmin)
        return self.length - z if z + dz > self.length else dz

    def advance(self, q, subcycles):
        L, steps = self.length, 0
        for sub in range(subcycles):
            z, z0 = 0.0, sub * L
            while True:
                k1 = self.slope(q, z0 + z)
                dz = self.step_size(q, k1, z)
                k2 = self.slope(self.cond * (q + 0.5 * dz * k1), z0 + z + 0.5 * dz)
                k3 = self.slope(self.cond * (q + 0.5 * dz * k2), z0 + z + 0.5 * dz)
                k4 = self.slope(self.cond * (q + dz * k3), z0 + z + dz)
                q = q + dz / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
                q = self.band * self.cond * q + (1 - self.band) * q
                z += dz
                steps += 1
                if not (z < L and (z - L) ** 2 > (L / 1e6) ** 2):
                    break
        return q, steps

    def field(self, q, z):
        return self.to_r(self.propagate(q, z))


def _host(x):
    return x.detach().cpu().numpy()


def exact(case, seed):
    if case['kind'] == 'batch':
        out = []
        setups = [uppe_kernel.RunSetup(vol) for vol in _scan(case)]
        for rs, a0 in zip(setups, _scan_fields(setups, seed)):
            m = _Exact(rs, False)
            q, _ = m.advance(m.to_k(m.t(a0)), case['subcycles'])
            out.append(_host(m.field(q, case['subcycles'] * m.length)))
        return out
    rs = _setup(case, seed)
    m = _Exact(rs, case['workload'] == 'envelope')
    if case['kind'] == 'gradient':
        c, xi = _phases(case, seed)
        basis = m.t(adjoint.legendre_basis(rs.w, 1.0, _sigma(case), 16))
        coef = m.t(c).requires_grad_(True)
        a0 = m.t(rs.A0) * torch.exp(1j * (coef @ basis))[:, None, None]
        q, _ = m.advance(m.to_k(a0), case['subcycles'])
        a = m.field(q, case['subcycles'] * m.length)[:, 0, 0]
        loss = torch.sum((a.real ** 2 + a.imag ** 2 - m.t(_target(rs, xi))) ** 2)
        loss.backward()
        return float(loss), _host(coef.grad)
    with torch.no_grad():
        q, steps = m.advance(m.to_k(m.t(rs.stepper_field())), case['subcycles'])
        a = m.field(q, case['subcycles'] * m.length)
        if case['kind'] == 'step':
            return _host(a)
        # the diagnostics take kz at the index of the radial cell
        j, chi, ne = m.source(1j * m.kzc * a)
        return (_host(a), _host(j), _host(torch.fft.rfft(chi + 0.0 * ne, dim=0)), _host(torch.fft.rfft(ne, dim=0)),
                4 * steps)
