"""Timed cases of the per-wavelength FEM + scattering-matrix path.

What a user's program does with this package falls into a few kinds of call,
and each case is one of them through the public entry points:

  films      plane-wave modes of a homogeneous film for a list of lights
             (batch.calc_films_many); the smallest call, all latency;
  cascade    the star-product cascade of given layer matrices for a batch of
             points (Context.star_cascade), as in a sweep over layer
             thickness or wavelength with the modes in hand;
  grating    a 1D grating between two half spaces: mode solve of a list of
             lights, film modes, cascade (calc_modes_many, calc_films_many,
             calc_scat_many);
  slab       the same for a 2D-periodic layer on a triangular FEM mesh;
  bands      the propagation constants of a 2D-periodic layer alone, in the
             mixed-precision form (its beta are FP64 Rayleigh quotients);
  stack      three 2D-periodic layers with two films between them, the layers
             solved by calc_modes_stack on several worker contexts, as
             bench.py's step does at full size.

Mesh sizes, mode counts and numbers of lights run from the reference cases'
(about 500 triangles, 40 modes, one light) to the benchmark's (8,000
triangles, 200 modes, several lights per call).  Everything is complex128
except the complex64 factor of the mixed form.
"""
import atexit
import os
import shutil
import tempfile

import numpy as np

PERIOD = 600.0
_meshes = {}
_dir = None


def listed():
    return [
        # film modes of a 64-point sweep, as bench.py asks for each film
        dict(name='films_64', kind='films', lights=64, order=4),
        # one structured layer at one wavelength: the call after each single solve
        dict(name='cascade_1', kind='cascade', points=1, order=2, modes=40, layers=3),
        # the benchmark's stack for a 64-point batch
        dict(name='cascade_64', kind='cascade', points=64, order=4, modes=200, layers=7),
        # a two-inclusion grating at one light, and a short spectrum of it
        dict(name='grating_1', kind='grating', lights=1, order=5, modes=60, elements=200),
        dict(name='grating_16', kind='grating', lights=16, order=5, modes=60, elements=200),
        # the reference's nanowire cell size, one light: interactive use
        dict(name='slab_500_1', kind='slab', tri=500, lights=1, order=2, modes=40),
        # the same cell over a short spectrum
        dict(name='slab_500_8', kind='slab', tri=500, lights=8, order=2, modes=40),
        # a converged ordinary cell, two lights
        dict(name='slab_1500_2', kind='slab', tri=1500, lights=2, order=2, modes=80),
        # propagation constants in the mixed-precision form
        dict(name='bands_1500_4', kind='bands', tri=1500, lights=4, order=2, modes=80),
        # three layers solved concurrently by worker contexts
        dict(name='stack_1000_4', kind='stack', tri=1000, lights=4, order=2, modes=61),
        # the benchmark's layer, one light: largest single solve
        dict(name='slab_8000_1', kind='slab', tri=8000, lights=1, order=4, modes=200),
        # the benchmark's layer, a batch of lights
        dict(name='slab_8000_4', kind='slab', tri=8000, lights=4, order=4, modes=200),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(('films', 'cascade', 'cascade', 'grating', 'slab', 'slab', 'slab', 'bands', 'stack'))
    if kind == 'films':
        return dict(kind=kind, lights=_log(rng, 4, 256), order=rng.randint(1, 5))
    if kind == 'cascade':
        order = rng.randint(1, 4)
        return dict(kind=kind, points=_log(rng, 1, 64), order=order, modes=2 * _n_orders(order) + rng.randint(7, 100),
                    layers=rng.choice((3, 5, 7)))
    if kind == 'grating':
        return dict(kind=kind, lights=_log(rng, 1, 16), order=rng.randint(3, 6), modes=rng.randint(30, 61),
                    elements=rng.randint(160, 240))
    tri = _log(rng, 300, 3000 if kind == 'stack' else 8000)
    order = rng.randint(1, 2) if tri < 1000 else rng.randint(1, 3)
    modes = 2 * _n_orders(order) + rng.randint(11, 40 if tri < 1000 else 80)
    most = max(1, min(8, int(0.4 * 8000 * 200 * 4 / (tri * modes * (3 if kind == 'stack' else 1)))))
    return dict(kind=kind, tri=tri, lights=_log(rng, 1, most), order=order, modes=modes)


def _orders(order):
    """Plane waves (px, py) of the circular truncation on a square lattice,
    the test evaluated in nm (it decides the orders on the circle)."""
    p = np.arange(-order, order + 1)
    px, py = np.repeat(p, p.size), np.tile(p, p.size)
    keep = (px / PERIOD) ** 2 + (py / PERIOD) ** 2 <= (order / PERIOD) ** 2
    return px[keep], py[keep]


def _n_orders(order):
    return int(_orders(order)[0].size)


# ------------------------------------------------------------------- inputs


def _mesh(tri, k=0):
    """A cell with a elliptical inclusion, written once per process."""
    global _dir
    from emustack_amd import EMUstack, mesher
    if (tri, k) not in _meshes:
        if _dir is None:
            _dir = tempfile.mkdtemp(prefix='emu_cells_')
            atexit.register(shutil.rmtree, _dir, ignore_errors=True)
        path = os.path.join(_dir, 'cell_%d_%d.mail' % (tri, k))
        mesher.write_mail(path, mesher.ellipse_cell_ntri(PERIOD, PERIOD, 150.0 - 20.0 * k, 115.0 - 10.0 * k, tri, seed=k + 1))
        _meshes[tri, k] = path
    path = _meshes[tri, k]
    EMUstack.mesh(path)  # loaded and analysed once, as any program that solves on it more than once has it
    return path


def _lights(rng, case, phi=True):
    from emustack_amd import objects
    n = case['lights']
    start = rng.uniform(450.0, 600.0)
    wls = start + np.arange(n) * rng.uniform(4.0, 20.0)
    theta, ph = rng.uniform(5.0, 40.0), rng.uniform(5.0, 85.0) if phi else 0.0
    return [objects.Light(float(w), max_order_PWs=case['order'], theta=theta, phi=ph) for w in wls]


def _layer(rng, tri, k=0):
    from emustack_amd import materials, objects
    n = complex(rng.uniform(1.8, 3.8), rng.uniform(0.005, 0.05))
    return objects.NanoStruct('2D_array', PERIOD, 300, height_nm=float(rng.uniform(80, 250)), background=materials.Air,
                              inclusion_a=materials.Material(n), loss=True, make_mesh_now=False,
                              mesh_file=_mesh(tri, k))


def _half_spaces(period, world_1d=False):
    from emustack_amd import materials, objects
    sub = objects.ThinFilm(period, height_nm='semi_inf', material=materials.Material(1.5 + 0j), loss=False,
                           world_1d=world_1d)
    sup = objects.ThinFilm(period, height_nm='semi_inf', material=materials.Air, loss=False, world_1d=world_1d)
    return sub, sup


def _film(rng):
    from emustack_amd import materials, objects
    return objects.ThinFilm(PERIOD, height_nm=50.0, material=materials.Material(complex(rng.uniform(1.3, 2.5), 0.01)))


def _cascade_arrays(case, seed):
    """Layer matrices of a batch of stacks, with the structure real ones have:
    J^dagger a left inverse of J up to coupling, impedances near 1, and
    propagation constants that are real for the leading modes and decay for
    the rest."""
    rng = np.random.default_rng(seed)
    nb, L, m, npw = case['points'], case['layers'], case['modes'], _n_orders(case['order'])
    d = 2 * npw
    kinds = [i % 2 for i in range(L)]

    def cplx(*shape):
        return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)

    def props(n):
        k = np.sort(rng.uniform(1.0, 14.0, (nb, n)), axis=1)[:, ::-1] + 0.02j
        lead = max(2, n // 5)
        k[:, lead:] = 0.05 + 1j * np.sort(rng.uniform(0.5, 40.0, (nb, n - lead)), axis=1)
        return k
    kz, Z, J, Jd = [], [], [], []
    for kind in kinds:
        kz.append(props(m if kind else d))
        Z.append(None if kind else 1.0 + 0.2 * cplx(nb, d))
        if kind:
            q = np.linalg.qr(cplx(nb, m, d))[0]
            J.append(np.conj(q.transpose(0, 2, 1)) + 0.05 * cplx(nb, d, m) / np.sqrt(m))
            Jd.append(q + 0.05 * cplx(nb, m, d) / np.sqrt(m))
        else:
            J.append(None)
            Jd.append(None)
    heights = rng.uniform(0.05, 0.4, (nb, L))
    heights[:, 0] = heights[:, -1] = 0.0
    Zair = 1.0 + 0.1 * cplx(nb, d)
    d_minus = np.zeros((nb, d), complex)
    d_minus[:, 0] = 1.0
    nprop = np.tile(np.array([3, 3, 4], np.int64), (nb, 1))
    return kinds, kz, Z, J, Jd, heights, Zair, d_minus, nprop


def prepare(case, seed):
    from emustack_amd import EMUstack, materials, objects
    rng = np.random.default_rng(seed)
    kind = case['kind']
    if kind == 'films':
        return dict(kind=kind, film=_film(rng), lights=_lights(rng, case))
    if kind == 'cascade':
        return dict(kind=kind, args=_cascade_arrays(case, seed), ctx=EMUstack.context())
    if kind == 'grating':
        g = objects.NanoStruct('1D_array', 400.0, 80.0, diameter2=120.0, height_nm=150.0,
                               background=materials.Material(1.45 + 0j),
                               inclusion_a=materials.Material(complex(rng.uniform(1.9, 2.4), 0.01)),
                               inclusion_b=materials.Material(complex(rng.uniform(2.8, 3.6), 0.01)), loss=True,
                               lc_bkg=1.0 / case['elements'])
        EMUstack.mesh_1d(g.x_arr, g.table_nod, g.type_el)
        sub, sup = _half_spaces(400.0, world_1d=True)
        return dict(kind=kind, layer=g, lights=_lights(rng, case, phi=False), sub=sub, sup=sup, modes=case['modes'])
    if kind == 'stack':
        from emustack_amd.batch import preload_meshes
        layers = [_layer(rng, case['tri'], k) for k in range(3)]
        preload_meshes(layers, groups=2, workers=3)
        sub, sup = _half_spaces(PERIOD)
        return dict(kind=kind, layers=layers, lights=_lights(rng, case), film=_film(rng), sub=sub, sup=sup,
                    modes=case['modes'])
    sub, sup = _half_spaces(PERIOD)
    return dict(kind=kind, layer=_layer(rng, case['tri']), lights=_lights(rng, case), sub=sub, sup=sup,
                modes=case['modes'])


# --------------------------------------------------------------------- runs


def _scattering(stacks):
    """The cascade of the stacks and what a user reads from them."""
    from emustack_amd.batch import calc_scat_many
    calc_scat_many(stacks, pol='TE', want_nets=True)
    return dict(R=np.array([np.asarray(s.R_net) for s in stacks]), T=np.array([np.asarray(s.T_net) for s in stacks]),
                a=np.array([s.a_list for s in stacks]), r=np.array([s.r_list for s in stacks]),
                t=np.array([s.t_list for s in stacks]))


def run(state):
    from emustack_amd import Stack
    from emustack_amd.batch import calc_films_many, calc_modes_many, calc_modes_stack
    kind = state['kind']
    if kind == 'films':
        films = calc_films_many(state['film'], state['lights'])
        return dict(k_z=np.array([f.k_z for f in films]), Z=np.array([f.Z() for f in films]))
    if kind == 'cascade':
        a, r, t, R, T = state['ctx'].star_cascade(*state['args'], want_nets=True)
        return dict(a=a, r=r, t=t, R=R, T=T)
    lights = state['lights']
    if kind == 'bands':
        sims = calc_modes_many(state['layer'], lights, num_BMs=state['modes'], precision='mixed')
        return dict(k_z=np.array([s.k_z for s in sims]))
    subs, sups = calc_films_many(state['sub'], lights), calc_films_many(state['sup'], lights)
    if kind == 'stack':
        sims = calc_modes_stack(state['layers'], lights, num_BMs=state['modes'], groups=2, workers=3)
        films = calc_films_many(state['film'], lights)
        out = _scattering([Stack((subs[i], sims[0][i], films[i], sims[1][i], films[i], sims[2][i], sups[i]))
                           for i in range(len(lights))])
        return dict(out, k_z=np.array([[m.k_z for m in s] for s in sims]))
    sims = calc_modes_many(state['layer'], lights, num_BMs=state['modes'])
    out = _scattering([Stack(layers) for layers in zip(subs, sims, sups)])
    if kind == 'slab':
        # (a grating's deepest evanescent k_z carry the rounding of the solve
        # well above 1e-9; they do not reach the scattering matrices)
        out['k_z'] = np.array([s.k_z for s in sims])
    return out


# --------------------------------------------------------------------- work


def work(case):
    """Bytes and flops that the path cannot do without.  Mode solves: the
    assembled pencil written once, the factor (entries ~ 1.15 n^1.5 at n
    unknowns, fitted on the meshes of this range) written once and read once
    per block of eight operator applications, one Krylov basis of 2.5 modes
    + 3 columns read twice per block; factorisation flops ~ 36 factor
    entries^1.22, eight per entry and application, Gram-Schmidt 16 n m^2."""
    kind = case['kind']
    if kind == 'films':
        n = case['lights'] * _n_orders(case['order'])
        return dict(bytes=16.0 * n * 5, flops=100.0 * n)
    if kind == 'cascade':
        return _cascade_work(case['points'], 2 * _n_orders(case['order']), case['modes'], case['layers'] // 2)
    if kind == 'grating':
        n, entries = 8.0 * case['elements'], 60.0 * 8.0 * case['elements']
        npw, nnz, layers = 2 * case['order'] + 1, 121.0 * case['elements'], 1
    else:
        n = 12.0 * case['tri']
        entries, nnz = 1.15 * n ** 1.5, 411.0 * case['tri']
        npw, layers = _n_orders(case['order']), 3 if kind == 'stack' else 1
    m, inst = 2.5 * case['modes'] + 3, 2.0 * case['lights'] * layers
    blocks = m / 8.0
    wide = 0.5 if kind == 'bands' else 1.0  # the mixed form reads a complex64 factor
    nbytes = inst * (32.0 * nnz + 16.0 * entries * (1.0 + blocks * wide) + 16.0 * nnz * blocks + 16.0 * n * m * blocks)
    flops = inst * (36.0 * entries ** 1.22 + 8.0 * (entries + nnz) * m + 16.0 * n * m * m)
    if kind != 'bands':
        c = _cascade_work(case['lights'], 2 * npw, case['modes'], layers)
        nbytes, flops = nbytes + c['bytes'], flops + c['flops']
    return dict(bytes=nbytes, flops=flops)


def _cascade_work(points, d, m, structured):
    """Per structured layer: the inverse of I + B A, two solves and the
    products between them; inputs J, J^dagger read, R_net and T_net written."""
    flops = 8.0 * structured * (2.0 * m ** 3 + 5.0 * m * m * d + 4.0 * m * d * d + d ** 3)
    return dict(bytes=16.0 * points * (structured * (2.0 * d * m + m) + 2.0 * d * d + 6.0 * d), flops=points * flops)


# -------------------------------------------------------------------- exact


def exact(case, seed):
    if case['kind'] == 'films':
        return _exact_films(case, seed)
    if case['kind'] == 'cascade':
        return _exact_cascade(case, seed)
    return None


def _exact_films(case, seed):
    """k_z = sqrt(k^2 - alpha^2 - beta^2) and Z = (1/n) k/k_z, (1/n) k_z/k in
    the order of the free-space k_z (propagating first, by decreasing k_z,
    then by increasing decay)."""
    state = prepare(case, seed)
    n = complex(state['film'].material.n(500.0))
    px, py = _orders(case['order'])
    kzs, Zs = [], []
    for light in state['lights']:
        kx, ky = light.k_pll * PERIOD
        alpha, beta = kx + 2 * np.pi * px, ky + 2 * np.pi * py
        k0 = 2 * np.pi * PERIOD / light.wl_nm
        air = np.sqrt((k0 ** 2 - alpha ** 2 - beta ** 2).astype(complex))
        order = np.argsort(-air.real + air.imag)
        kz = np.sqrt((n * k0) ** 2 - alpha ** 2 - beta ** 2)[order]
        ratio = n * k0 / kz
        kzs.append(np.concatenate((kz, kz)))
        Zs.append(np.concatenate((ratio / n, 1.0 / (n * ratio))))
    return dict(k_z=np.array(kzs), Z=np.array(Zs))


def _exact_cascade(case, seed):
    kinds, kz, Z, J, Jd, heights, Zair, d_minus, nprop = _cascade_arrays(case, seed)
    out = [_exact_point([kinds, [k[b] for k in kz], [z if z is None else z[b] for z in Z],
                         [j if j is None else j[b] for j in J], [j if j is None else j[b] for j in Jd]],
                        heights[b], Zair[b], d_minus[b], nprop[b]) for b in range(case['points'])]
    return dict(zip(('a', 'r', 't', 'R', 'T'), (np.array(v) for v in zip(*out))))


def _exact_point(layers, heights, Zair, d_minus, nprop):
    """One stack: interface matrices of every layer against air, the net
    matrices grown upwards through infinitesimal air gaps, then the fluxes of
    the amplitudes in each gap."""
    kinds, kz, Z, J, Jd = layers
    d = Zair.size
    eye = np.eye(d)
    faces = []
    for kind, z, j, jd in zip(kinds, Z, J, Jd):
        if not kind:
            r = np.diag((z - Zair) / (z + Zair))
            t = np.diag(2.0 * np.sqrt(z) * np.sqrt(Zair) / (z + Zair))
            faces.append((r, t, -r, t))
            continue
        w = np.sqrt(1.0 / Zair)
        A, B = w[:, None] * j, jd * w[None, :]
        inv = np.linalg.inv(np.eye(A.shape[1]) + B @ A)
        T12 = 2.0 * inv @ B
        faces.append((A @ T12 - eye, T12, 2.0 * inv - np.eye(A.shape[1]), 2.0 * A @ inv))
    t_net, r_net = faces[0][1], faces[0][0]
    r_nets, gaps, bodies, props = [r_net], [], [], []

    def gap(i, t_net, r_net):
        R12, T12, R21, T21 = faces[i]
        g = np.linalg.solve(eye - R12 @ r_net, T21)
        gaps.append(g)
        return t_net @ g, R21 + T12 @ r_net @ g
    for i in range(1, len(kinds) - 1):
        t_net, r_net = gap(i, t_net, r_net)
        r_nets.append(r_net)
        R12, T12, R21, T21 = faces[i]
        p = np.exp(1j * kz[i] * heights[i])
        prp = p[:, None] * r_net * p[None, :]
        b = np.linalg.solve(np.eye(p.size) - R21 @ prp, T12)
        t_net, r_net = t_net @ (p[:, None] * b), R12 + T21 @ prp @ b
        bodies.append(b)
        props.append(p)
        r_nets.append(r_net)
    t_net, r_net = gap(len(kinds) - 1, t_net, r_net)
    npw, (n_air, n_in, n_out) = d // 2, nprop

    def power(v, n):
        return np.linalg.norm(v[:n]) ** 2 + np.linalg.norm(v[npw:npw + n]) ** 2

    def flux(f, g):
        s = 0.0
        for pol, sign in ((0, -1j), (npw, 1j)):
            a, c = f[pol:pol + npw], g[pol:pol + npw]
            s += np.sum(np.abs(a[:n_air]) ** 2 - np.abs(c[:n_air]) ** 2)
            s += np.sum(np.conj(a[n_air:]) * sign * c[n_air:] - np.conj(c[n_air:]) * sign * a[n_air:])
        return s
    up = power(r_net @ d_minus, n_in)
    down = [power(d_minus, n_in)]
    f = gaps[-1] @ d_minus
    for j in range(len(bodies)):
        down.append(flux(f, r_nets[-2 * j - 1] @ f))
        f = gaps[-j - 2] @ (props[-j - 1] * (bodies[-j - 1] @ f))
    down.append(power(faces[0][1] @ f, n_out))
    inner = range(1, len(down) - 1)
    a = [abs(abs(down[i]) - abs(down[i + 1])) for i in inner] + [abs(down[0] - down[-1] - up)]
    t = [abs(down[i + 1]) / abs(down[i - 1]) for i in inner] + [abs(down[-1] / down[0])]
    return np.array(a), abs(up / down[0]), np.array(t), r_net, t_net
