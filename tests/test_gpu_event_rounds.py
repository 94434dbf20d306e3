"""The event loop's rounds (csrc/nsm.hip) where they can go wrong: domains
around the 64 voxels of a node and of the front, every bucket of species and
reactions, trajectories with one wavefront and with several, exactly equal
firing times, and a replay stream that ends inside a round."""
import numpy as np
import pytest

from spatialpy_amd import workloads
from spatialpy_amd.core.errors import SimulationError
from spatialpy_amd.engine import Engine, mt19937_64_stream
from spatialpy_amd.lowering import K_2X, K_AB, K_FIRST, K_ZERO
from oracle import oracle_py

pytestmark = pytest.mark.gpu


def lattice_model(nx, ny, S, R, per_voxel, seed, nt=4, D=4.0):
    """A static nx x ny lattice with S species of different mobility (one of
    them immobile) and R reactions cycling through the mass-action kinds."""
    x = np.array([(float(i), float(j), 0.0) for i in range(nx) for j in range(ny)])
    n = len(x)
    rng = np.random.default_rng(seed)
    rx = []
    for r in range(R):
        a, b, c = r % S, (r + 1) % S, (r + 2) % S
        kind = (K_FIRST, K_AB, K_2X, K_ZERO)[r % 4]
        if kind == K_FIRST:
            rx.append((kind, a, 0, 0.03, 0, {a: 1}, {b: 1} if b != a else {}))
        elif kind == K_AB and b != a:
            rx.append((kind, a, b, 0.02, 0, {a: 1, b: 1}, {c: 1} if c not in (a, b) else {}))
        elif kind == K_ZERO:
            rx.append((kind, a, 0, 0.05, 0, {}, {a: 1}))
        else:
            rx.append((K_2X, a, 0, 0.01, 0, {a: 2}, {b: 1} if b != a else {a: 1}))
    Ds = D * (1.0 + np.arange(S)) / S
    if S > 1:
        Ds[S - 1] = 0.0
    sa = workloads.SystemArrays(
        x=x, type=np.ones(n, np.int32), mass=np.ones(n), rho=np.ones(n), nu=np.ones(n), fixed=np.ones(n, np.int32),
        n_types=1, dimension=2, h=2.2, dt=1.0, nt=nt, output_steps=np.arange(nt + 1, dtype=np.uint32), static_domain=1,
        bbox=workloads.bounding_box(x), u0=rng.poisson(per_voxel, (n, S)).astype(np.uint32),
        diffusion_matrix=Ds.reshape(S, 1), reactions=rx)
    sa.build_sparse()
    return sa.normalized()


@pytest.mark.parametrize("nx,ny,S,R,per_voxel", [
    (2, 1, 1, 1, 3.0), (3, 3, 1, 2, 2.0), (7, 9, 2, 2, 1.0), (8, 8, 3, 4, 1.0), (5, 13, 4, 3, 0.5),
    (13, 10, 5, 6, 0.5), (16, 16, 8, 8, 0.3), (11, 12, 9, 12, 0.3), (12, 12, 16, 16, 0.2), (30, 40, 2, 1, 0.2)])
def test_rounds_follow_the_oracle_event_by_event(nx, ny, S, R, per_voxel):
    sa = lattice_model(nx, ny, S, R, per_voxel, seed=nx)
    words, expo = mt19937_64_stream(5, 600_000)
    cap = 200_000
    eng = Engine(sa, trace_capacity=cap)
    res = eng.run(words=words, expo=expo)
    ev, nev = eng.trace(cap)
    o = oracle_py.Oracle(sa)
    o.set_trace(cap)
    ref = o.run(seed=5)
    oev, onev = o.trace(cap)
    assert nev == onev and nev > 0
    assert np.array_equal(ev, oev)
    assert np.array_equal(res["xx"], ref["xx"])


def test_trajectories_with_one_and_with_several_wavefronts_are_the_same():
    """Up to 256 trajectories get several wavefronts each, more get one."""
    sa = lattice_model(40, 50, 2, 2, 0.4, seed=3, nt=2)
    seeds = np.arange(300)
    many = Engine(sa).run_batch(seeds, fields=())["xx"]
    eng = Engine(sa)
    for b in (0, 137, 299):
        assert np.array_equal(eng.run(seed=int(seeds[b]), fields=("xx",))["xx"], many[b])


@pytest.mark.parametrize("n_side", [5, 30])
def test_equal_firing_times_go_by_voxel_at_any_node_width(monkeypatch, n_side):
    """A stream of equal words gives every interior voxel the same firing
    time, more of them than the near list holds at 30 x 30: the run ends, keeps
    its molecules and does not depend on how the queue is cut into nodes."""
    sa = lattice_model(n_side, n_side, 1, 0, 0.0, seed=1, nt=2)
    sa.u0[:] = 1
    words = np.full(60_000, 1 << 63, np.uint64)
    expo = np.full(words.size, float(np.log(2.0)))
    runs = []
    for width in (1, 4):
        monkeypatch.setenv("SSASDPD_EVENT_TREE_PL", str(width))
        runs.append(Engine(sa).run(words=words, expo=expo, fields=("xx",))["xx"])
    assert np.array_equal(runs[0], runs[1])
    assert (runs[0].sum(axis=(1, 2)) == sa.n).all()


def test_a_replay_stream_that_ends_is_reported_wherever_it_ends():
    sa = lattice_model(8, 8, 2, 2, 1.0, seed=2)
    eng = Engine(sa)
    words, expo = mt19937_64_stream(9, 100_000)
    eng.run(words=words, expo=expo, fields=("xx",))
    used = int(eng.stats().rng_words_used)
    for short in (1, 2, 3, 4, 63, 64, 65, used // 2):
        with pytest.raises(SimulationError) as err:
            eng.run(words=words[:used - short], expo=expo[:used - short], fields=("xx",))
        assert err.value.code == 9
    full = eng.run(words=words[:used], expo=expo[:used], fields=("xx",))["xx"]
    assert np.array_equal(full, eng.run(words=words, expo=expo, fields=("xx",))["xx"])
