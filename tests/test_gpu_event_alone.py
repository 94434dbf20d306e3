"""Events one by one (csrc/nsm.hip, event_alone), where rounds would keep few:
domains of a few voxels in every bucket of species and reactions, neighbour rows
longer than a wavefront, types, the textbook selection, one crowded voxel among
many empty ones, ensembles, batches, and a replay stream that ends."""
import numpy as np
import pytest

from oracle import oracle_py
from spatialpy_amd import _abi
from spatialpy_amd.core import model as M
from spatialpy_amd.core.domain import Domain
from spatialpy_amd.core.errors import SimulationError
from spatialpy_amd.engine import Engine, mt19937_64_stream
from spatialpy_amd.ensemble import Ensemble
from spatialpy_amd.lowering import K_FIRST, K_ZERO
from spatialpy_amd.solver import Solver
from test_gpu_event_rounds import lattice_model

pytestmark = pytest.mark.gpu


def follows_the_oracle(sa, n_words=400_000, least=300):
    words, expo = mt19937_64_stream(5, n_words)
    cap = 100_000
    eng = Engine(sa, trace_capacity=cap)
    res = eng.run(words=words, expo=expo)
    ev, nev = eng.trace(cap)
    o = oracle_py.Oracle(sa)
    o.set_trace(cap)
    ref = o.run(seed=5)
    oev, onev = o.trace(cap)
    assert nev == onev and nev > least
    assert np.array_equal(ev, oev)
    assert np.array_equal(res["xx"], ref["xx"])
    st, ost = eng.stats(), o.stats()
    assert (st.reactions, st.diffusions, st.rng_words_used) == (ost.reactions, ost.diffusions, ost.rng_words_used)


@pytest.mark.parametrize("nx,ny,S,R,per_voxel", [
    (1, 2, 1, 1, 60.0), (2, 2, 2, 2, 30.0), (4, 5, 2, 2, 10.0), (2, 2, 3, 4, 20.0),
    (4, 8, 4, 3, 4.0), (2, 3, 5, 6, 10.0), (8, 8, 8, 8, 2.0), (10, 10, 7, 8, 1.0), (1, 3, 9, 12, 10.0),
    (3, 3, 16, 16, 5.0), (16, 16, 16, 16, 0.2), (12, 12, 9, 9, 1.0)])
def test_few_voxels(nx, ny, S, R, per_voxel):
    follows_the_oracle(lattice_model(nx, ny, S, R, per_voxel, seed=nx + ny))


def test_without_reactions():
    """As with one that never fires, which the oracle follows."""
    sa = lattice_model(2, 2, 2, 0, 30.0, seed=4)
    words, expo = mt19937_64_stream(5, 400_000)
    got = Engine(sa).run(words=words, expo=expo, fields=("xx",))["xx"]
    sa.reactions = [(K_FIRST, 0, 0, 0.0, 0, {0: 1}, {})]
    sa.build_sparse()
    sa = sa.normalized()
    follows_the_oracle(sa)
    assert np.array_equal(got, Engine(sa).run(words=words, expo=expo, fields=("xx",))["xx"])


def test_rows_longer_than_a_wavefront():
    sa = lattice_model(10, 10, 5, 5, 1.0, seed=4, D=1e4)
    sa.h = 20.0
    follows_the_oracle(sa.normalized())


def _custom(side, S):
    """S species in a ring, each turned into the next by a function of both, one
    of them with a data function, one for one half of the domain only."""
    class Slope(M.DataFunction):
        def map(self, point):
            return 1.0 + point[0]

    m = M.Model("ring")
    d = Domain.create_2D_domain(xlim=(0, 1), ylim=(0, 1), numx=side, numy=side, type_id=1, fixed=True)
    d.type_id[d.vertices[:, 0] > 0.5] = "type_2"
    m.add_domain(d)
    m.add_data_function(Slope(name="slope"))
    m.add_species([M.Species(f"X{k}", 0.4 / side ** 2 * (1 + k % 3)) for k in range(S)])
    m.add_parameter(M.Parameter("k1", expression=0.5))
    for k in range(S):
        a, b = f"X{k}", f"X{(k + 1) % S}"
        text = {0: f"k1*{a}/(1+{b}/4)", 1: f"k1*{a}*slope", 2: f"{a}/2 + k1*{a}"}[k % 3]
        m.add_reaction(M.Reaction(f"r{k}", reactants={a: 1}, products={b: 1}, propensity_function=text,
                                  restrict_to=[2] if k == 1 else None))
        m.add_initial_condition(M.ScatterInitialCondition(a, 30, seed=k))
    m.timespan(M.TimeSpan.linspace(t=2, num_points=3, timestep_size=0.25))
    return Solver(m).lower()


@pytest.mark.parametrize("side,S", [(1, 3), (2, 5), (2, 8), (7, 8), (2, 9), (3, 16), (9, 16)])
def test_custom_propensities(side, S):
    follows_the_oracle(_custom(side, S), least=50)


def test_types_and_textbook_selection():
    sa = lattice_model(4, 4, 3, 3, 12.0, seed=6)
    sa.type = 1 + (np.arange(sa.n) % 2).astype(np.int32)
    sa.n_types = 2
    sa.diffusion_matrix = np.repeat(sa.diffusion_matrix, 2, axis=1) * np.array([1.0, 0.6])
    sa.reactions = [(*r[:4], 1 << 1 if k == 1 else 0, *r[5:]) for k, r in enumerate(sa.reactions)]
    sa.flags |= _abi.FLAG_TEXTBOOK_SELECTION
    sa.build_sparse()
    follows_the_oracle(sa.normalized())


@pytest.mark.parametrize("S,R", [(1, 1), (2, 2), (6, 5)])
def test_one_crowded_voxel(S, R):
    """More voxels than the front and the near list hold fill up from it."""
    sa = lattice_model(40, 40, S, R, 0.0, seed=3, D=0.5, nt=3)
    sa.reactions = [r for r in sa.reactions if r[0] != K_ZERO]      # (none that fires in an empty voxel)
    sa.u0[820] = 2500 // S
    sa.build_sparse()
    follows_the_oracle(sa.normalized())


def test_ensembles_and_batches_of_small_models():
    sa = lattice_model(3, 4, 3, 3, 8.0, seed=2)
    seeds = np.arange(300, dtype=np.uint64) + 11
    many = Engine(sa).run_batch(seeds, fields=())["xx"]
    few = Engine(sa).run_batch(seeds[:5], fields=())["xx"]
    totals, counts = Ensemble([sa] * 3).run(seeds[:3], counts=True)
    for b in range(3):
        one = Engine(sa).run(seed=int(seeds[b]), fields=("xx",))["xx"]
        assert np.array_equal(one, many[b]) and np.array_equal(one, few[b]) and np.array_equal(one, counts[b])
        assert np.array_equal(totals[b], one.sum(axis=1))


def test_a_replay_stream_that_ends():
    sa = lattice_model(2, 2, 2, 2, 20.0, seed=2)
    eng = Engine(sa)
    words, expo = mt19937_64_stream(9, 100_000)
    eng.run(words=words, expo=expo, fields=("xx",))
    used = int(eng.stats().rng_words_used)
    for short in (1, 2, 3, 4, 5, 64, used // 2):
        with pytest.raises(SimulationError) as err:
            eng.run(words=words[:used - short], expo=expo[:used - short], fields=("xx",))
        assert err.value.code == 9
    full = eng.run(words=words[:used], expo=expo[:used], fields=("xx",))["xx"]
    assert np.array_equal(full, eng.run(words=words, expo=expo, fields=("xx",))["xx"])
