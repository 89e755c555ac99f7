"""Lines and particles at the edges of the compiled code's common path
(xt_fast.h): element parameters on both sides of the rules that choose a
form, coordinates on both sides of every guard."""
import numpy as np

import xtrack_amd as xt

P0C = 7e12


def edge_particles(n, seed):
    """Beam-like particles with every guard's edge values mixed in: zeros of
    both signs, slopes around 2^-960, momenta around the entry bounds 2^-7 and
    2^-4 of the polar chains, |x| around 1, delta around +-1/4, and momenta
    that leave pz = 1 - 2^-53 (a significand of all ones)."""
    rng = np.random.default_rng(seed)
    z = {k: rng.normal(0, s, n) for k, s in (('x', 1e-3), ('px', 1e-4), ('y', 1e-3),
                                             ('py', 1e-4), ('zeta', 0.05), ('delta', 1e-3))}

    def put(name, values, k):
        at = rng.choice(n, k, replace=False)
        z[name][at] = rng.choice(np.asarray(values, dtype=float), k)
        return at

    k = n // 12
    for f in ('x', 'px', 'y', 'py', 'zeta', 'delta'):
        put(f, [0.0, -0.0], k)
    for f in ('px', 'py'):
        put(f, [s * 2.0 ** e for e in (-958, -960, -962, -1030, -1074) for s in (1, -1)], k)
        put(f, [s * v for b in (2.0 ** -7, 2.0 ** -4, 0.25) for s in (1, -1)
                for v in (b, np.nextafter(b, 0), np.nextafter(b, 1))], k)
        at = put(f, [2.0 ** -26.5, 1.05e-8, 1.2e-8], k)
        z['delta'][at[::2]] = 0.0
        z['py' if f == 'px' else 'px'][at[::2]] = 0.0
    put('x', [1.0, -1.0, np.nextafter(1, 0), np.nextafter(1, 2), 0.99, 3.0, np.inf, np.nan], k)
    put('y', [1.0, -1.0, 0.5, 1e200, np.nan], k)
    put('delta', [0.25, -0.25, np.nextafter(0.25, 1), np.nextafter(-0.25, -1), 0.4, -0.6,
                  -2.0 ** -53, 2.0 ** -52], k)
    return xt.Particles(p0c=P0C, **z)


def _line(els):
    line = xt.Line(elements=els)
    line.particle_ref = xt.Particles(p0c=P0C)
    return line


def bend_line(angle, length, **kw):
    """Two bends: the angle and the number of kicks decide between the
    small-angle form of the polar drift, its general form, a loop over equal
    steps and the general code."""
    return _line([xt.Bend(length=length, angle=angle, **kw), xt.Drift(length=0.3),
                  xt.Bend(length=length, angle=angle, knl=[0, 0, 0.02], **kw)])


def quad_line(k1, length):
    return _line([xt.Quadrupole(length=length, k1=k1), xt.Drift(length=0.4),
                  xt.Quadrupole(length=length, k1=-k1, knl=[0, 0, 0.03])])


def kick_line(knl, ksl):
    """Thin multipoles with every pattern of zero coefficients, and exact
    drifts."""
    return _line([xt.Multipole(knl=knl, ksl=ksl), xt.Drift(length=0.5, model='exact'),
                  xt.Multipole(knl=knl, ksl=ksl), xt.Drift(length=0.5),
                  xt.Sextupole(length=0.3, k2=0.4, k2s=0.1)])


def gap_line(sign=1.0, other=0.9):
    """Apertures along drifts: checks that others imply, a different
    aperture inside the run, and a drift of the other sign."""
    def rect(f=1.0):
        return xt.LimitRect(min_x=-2e-3 * f, max_x=2e-3 * f, min_y=-1e-3, max_y=1.5e-3)

    els = []
    for k in range(8):
        els += [rect()]
        for j in range(6):
            els += [xt.Drift(length=sign * (0.7 if (k, j) != (3, 2) else -1.4)),
                    rect(other if (k + j) % 5 == 0 else 1.0)]
        els += [xt.Multipole(knl=[0, 0.05 * (-1) ** k])]
    return _line(els)


def bend_steps(angle, length, kicks):
    return bend_line(angle, length, num_multipole_kicks=kicks)


def bend_model(angle, length, model):
    return bend_line(angle, length, model=model)


CASES = ([('bend', bend_line, (a, L)) for a, L in
          ((0.0057, 14.3), (0.0114, 6.0), (0.05, 3.0), (1e-7, 1.0))]
         + [('bend', bend_steps, v) for v in ((0.02, 2.0, 1), (0.13, 2.0, 1), (0.2, 2.0, 1),
                                              (0.9, 2.0, 1), (0.01, 20.0, 40))]
         + [('bend', bend_model, (0.006, 10.0, m)) for m in
            ('rot-kick-rot-low-order', 'rot-kick-rot-high-order', 'drift-kick-drift-exact')]
         + [('quad', quad_line, v) for v in ((0.0085, 3.1), (0.4, 1.0), (2.0, 1.0), (1e-7, 0.5),
                                             (1e-12, 1.0))]
         + [('kick', kick_line, v) for v in (([0, 0.1], [0, 0]), ([0, 0], [0, 0.1]),
                                             ([0.001, 0, 2.0], [0, 0, 0]),
                                             ([0, 0, 0, 5.0], [0.001, 0, 0, 1.0]))]
         + [('gap', gap_line, v) for v in ((1.0,), (-1.0,), (1.0, 1.0))])
IDS = [f'{n}-{"-".join(str(v) for v in a)}' for n, _, a in CASES]
