"""The compiled code's common path on the GPU against the oracle, bit for
bit, at the edges of its forms and guards (fast_path_cases)."""
import pytest

from fast_path_cases import CASES, IDS, edge_particles
from helpers import compare_exact, random_particles
from oracle_backend import OracleBackend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('name,make,args', CASES, ids=IDS)
def test_edges_of_forms_and_guards(name, make, args):
    lg, lc = make(*args), make(*args)
    lg.build_tracker(device='cuda:0', compile=True)
    lc.build_tracker(backend=OracleBackend())
    for p in (edge_particles(1500, seed=5), random_particles(100_003, seed=6, scale=6e-4,
                                                             p0c=7e12)):
        pg, pc = p.copy(_context='cuda:0'), p.copy()
        lg.track(pg, num_turns=2)
        lc.track(pc, num_turns=2)
        assert not compare_exact(pg, pc)


@pytest.mark.parametrize('name,make,args', CASES, ids=IDS)
def test_compiled_backtracking(name, make, args):
    lg, lc = make(*args), make(*args)
    lg.build_tracker(device='cuda:0', compile=True)
    lc.build_tracker(backend=OracleBackend())
    for p in (edge_particles(1500, seed=7), random_particles(20_003, seed=8, scale=6e-4,
                                                             p0c=7e12)):
        pg, pc = p.copy(_context='cuda:0'), p.copy()
        lg.track(pg, num_turns=2, backtrack=True)
        lc.track(pc, num_turns=2, backtrack=True)
        assert not compare_exact(pg, pc)
