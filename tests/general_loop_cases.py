"""Lines on both sides of the rule that chooses between the loop over units
and the element loop over general code: elements without unit code alone, in
runs of thin elements, and among magnets that have it."""
import xtrack_amd as xt


def _quad(k, **kw):
    return xt.Quadrupole(length=0.5, k1=0.05 * (-1) ** k, **kw)


def _thin(k):
    return [xt.Drift(length=0.4), xt.Multipole(knl=[0, 0.02 * (-1) ** k, 0.4], ksl=[0, 0.001]),
            xt.LimitRect(min_x=-4e-3, max_x=5e-3, min_y=-4e-3, max_y=4e-3), xt.Marker(),
            xt.LimitEllipse(a=6e-3, b=5e-3)]


def _cavity(**kw):
    return xt.Cavity(voltage=1e5, frequency=400e6, lag=170.0, **kw)


# name: (elements of cell k, number of cells, loop over units)
CELLS = {
    'off_quads': (lambda k: [xt.Quadrupole(length=0.3, k1=0.0)] + _thin(k), 12, False),
    'off_and_on_quads': (lambda k: [xt.Quadrupole(length=0.3, k1=0.0), _quad(k)] + _thin(k), 8,
                         True),
    'cavities': (lambda k: [_cavity()] + _thin(k), 12, False),
    'cavities_and_quads': (lambda k: [_cavity(), _quad(k)] + _thin(k), 8, True),
    'rf_multipoles': (lambda k: [xt.RFMultipole(voltage=1e3, frequency=400e6, lag=10.0,
                                                knl=[1e-6, 1e-5], pn=[10.0, 20.0])] + _thin(k),
                      10, False),
    'rotated_bends': (lambda k: [xt.Bend(length=1.0, angle=0.01, rot_s_rad=1e-3)] + _thin(k), 6,
                      False),
    'matrix_bends': (lambda k: [xt.Bend(length=1.0, angle=0.01, k1=0.01,
                                        model='mat-kick-mat')] + _thin(k), 6, False),
    'tilted_kicks': (lambda k: [xt.Multipole(knl=[0, 0.01], rot_x_rad=1e-4)] + 5 * _thin(k), 4,
                     True),
    'shifted_along_s': (lambda k: [xt.Multipole(knl=[0, 0.01], shift_s=2e-4)] + _thin(k), 12,
                        True),
    'strong_bends': (lambda k: [xt.Bend(length=1.0, angle=0.5)] + _thin(k), 2, False),
}


def cell_line(name):
    cell, n, _ = CELLS[name]
    line = xt.Line(elements=[el for k in range(n) for el in cell(k)])
    line.particle_ref = xt.Particles(p0c=7e12)
    return line
