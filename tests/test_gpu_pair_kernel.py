"""The forces-only pair kernel against the energy kernel and the oracle at
sizes where its tiles, windows and table reads have edges."""
import numpy as np
import pytest

from gmxapi_amd import nbx, systems as S
from tests.helpers import oracle_for, rms

pytestmark = pytest.mark.gpu


def _system(name):
    if name == "water70":  # fewer clusters than wavefronts, one-tile i-entries
        return S.water_box(70, 2.05, seed=3, rc=0.9, rlist=1.0)
    if name == "water1001":
        return S.water_box(1001, None, seed=4)
    return S.hetero_chains(2410, 2.9, ntypes=7, seed=5)  # rc 1.2: windows overflow


@pytest.mark.parametrize("options", [dict(), dict(ewald_correction="analytical"), dict(coulomb="reaction-field"),
                                     dict(vdw_modifier="force-switch", rvdw_switch=0.7)],
                         ids=["table", "analytical", "rf", "force-switch"])
@pytest.mark.parametrize("name", ["water70", "water1001", "chains2410"])
def test_forces_only_kernel_matches_energy_kernel(name, options):
    # the two kernels round the same pair terms in another order and, with
    # the table, read it at positions that differ by the rounding of
    # r * scale + 1 (6e-5 of an entry, 1.3e-6 of the correction's force):
    # a few 1e-7 of the RMS force, here bounded by 4e-6
    print(f"[forces only] {name} {options}", flush=True)
    s = _system(name)
    ctx = nbx.context_for(s, **options)
    f = ctx.compute(s.x)
    fe = ctx.compute(s.x, energy=True)
    assert rms(f - fe) <= 4e-6 * rms(fe)
    if not options:
        r64 = oracle_for(s, "f64").compute(s.x)
        assert rms(f - r64["f"]) <= 5e-4 * rms(r64["f"])


@pytest.mark.parametrize("options", [dict(), dict(ewald_correction="analytical"), dict(coulomb="reaction-field"),
                                     dict(vdw_modifier="force-switch", rvdw_switch=0.7),
                                     dict(vdw_modifier="potential-switch", rvdw_switch=0.7), dict(vdw_type="pme"),
                                     dict(vdw_cutoff=0.8)],
                         ids=["table", "analytical", "rf", "force-switch", "potential-switch", "lj-pme", "twin"])
@pytest.mark.parametrize("far", [1e6, 1e19, 3e38])
def test_atom_far_outside_leaves_the_others_finite(far, options):
    # an atom that has left the box by any float distance is beyond every
    # cut-off: the atoms listed with it keep the forces they have without it
    print(f"[far atom] {far} {options}", flush=True)
    s = S.water_box(500, None, seed=6)
    ctx = nbx.context_for(s, **options)
    x = s.x.astype(np.float32)
    x[7] = (1e5, 1e5, 1e5)
    near = ctx.compute(x)
    x[7] = (far, far, -far)
    others = np.arange(s.natoms) != 7
    for energy in (False, True):
        f = ctx.compute(x, energy=energy)
        assert np.isfinite(f[others]).all()
        assert rms(f[others] - near[others]) <= 4e-6 * rms(near[others])


@pytest.mark.parametrize("molecules", [280, 1000, 3000, 9001])
def test_group_size_rule_keeps_forces(molecules):
    # the group size chosen for the system's size (1, 2, 4, ... as the
    # clusters outgrow the wavefronts) against a forced one: the same pair
    # terms, summed in another order (float sums of a few hundred terms)
    s = S.water_box(molecules, None, seed=molecules)
    ctx = nbx.context_for(s)
    print(f"[group size] {molecules} molecules: {ctx.work_groups()['group_size']}", flush=True)
    f = ctx.compute(s.x, energy=True)
    e = ctx.energies()
    for forced in (1, 8):
        other = nbx.context_for(s, kernel_group_size=forced)
        g = other.compute(s.x, energy=True)
        assert rms(f - g) <= 4e-6 * rms(g)
        np.testing.assert_allclose(e, other.energies(), rtol=1e-6)


def test_results_follow_the_last_step():
    # energies, virial and shift forces are those of the last step, whichever
    # is read first and however many steps ran since the last read
    s = S.water_box(1001, None, seed=4)
    moved = (s.x + 0.01 * np.random.default_rng(1).normal(size=s.x.shape)).astype(np.float32)

    def results(ctx, order):
        read = dict(e=lambda: np.array(ctx.energies()), v=ctx.virial, f=ctx.shift_forces)
        got = {k: read[k]() for k in order}
        return [got[k] for k in "evf"]

    flags = dict(energy=True, virial=True, shift_forces=True, reproducible=True)
    want = []
    for x in (s.x, moved):
        ctx = nbx.context_for(s)
        ctx.compute(x, **flags)
        want.append(results(ctx, "evf"))
    ctx = nbx.context_for(s)
    for which, order in ((0, "vef"), (1, "fve"), (0, "efv")):
        ctx.compute((s.x, moved)[1 - which], **flags)
        ctx.compute((s.x, moved)[which], **flags)
        for a, b in zip(results(ctx, order), want[which]):
            np.testing.assert_array_equal(a, b)
    ctx.compute(s.x)
    with pytest.raises(nbx.NbxStateError):
        ctx.energies()


@pytest.mark.parametrize("natoms,ntypes,correction,bar", [
    (1500, 31, "table", 2e-3),       # the most types: the smallest windows, which overflow
    (1500, 24, "analytical", 1e-4),  # one copy of the C6/C12 accumulators
    (1010, 1, "analytical", 1e-4),   # fewer tiles than wavefronts
])
def test_adjoint_at_the_limits_of_its_lds(natoms, ntypes, correction, bar):
    # the adjoint's bars (test_gpu_adjoint.py) where its LDS is shared out
    # differently: FP32 pair terms against the FP64 reference gradient
    from oracle import adjoint as A

    print(f"[adjoint] {natoms} atoms, {ntypes} types, {correction}", flush=True)
    s = S.hetero_chains(natoms, max(2.51, (natoms / 100.0) ** (1 / 3)), ntypes=ntypes, seed=ntypes)
    g = np.random.default_rng(2).normal(size=s.x.shape)
    ref = A.forces_and_gradient(s, g, s.c6_matrix(), s.c12_matrix(), pairs=A.pair_table(s.x, s.box, s.rcoulomb))
    gx, gq, g6, g12 = nbx.context_for(s, ewald_correction=correction).compute_adjoint(s.x, g)
    assert rms(gx - ref["grad_x"]) <= bar * rms(ref["grad_x"])
    assert rms((gq - ref["grad_q"])[:, None]) <= bar * rms(ref["grad_q"][:, None])
    for got, want in ((g6, ref["grad_c6"]), (g12, ref["grad_c12"])):
        got, want = A.symmetrized(got), A.symmetrized(want)
        assert np.abs(got - want).max() <= bar * np.abs(want).max()


@pytest.mark.parametrize("switch_streams", [False, True])
def test_parameters_follow_queued_steps(switch_streams):
    # new LJ parameters are uploaded behind the stream's queued steps, which
    # keep the ones they were queued with; a step on another stream sees the
    # last ones set, also where their upload is still behind the old stream's
    # work when the context moves
    import torch

    s = S.water_box(1001, None, seed=4)
    m6, m12 = nbx.nblib_c6c12_matrices(s.c6, s.c12)
    scales = [1.0, 1.5, 0.5, 1.25, 0.75, 1.1]
    want = []
    for k in scales:
        ctx = nbx.context_for(s)
        ctx.set_nonbonded_parameters(k * m6, k * m12)
        want.append(ctx.compute(s.x))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    x = torch.from_numpy(s.x.astype(np.float32)).cuda()
    out = [torch.empty_like(x) for _ in scales]
    busy = torch.ones(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    ctx = nbx.context_for(s)
    ctx.set_stream(streams[0].cuda_stream)
    for n, k in enumerate(scales):
        if switch_streams:
            ctx.synchronize()  # the steps share the context's buffers
            with torch.cuda.stream(streams[n % 2]):
                for _ in range(20):
                    busy = busy @ busy * 0.0 + 1.0
        ctx.set_nonbonded_parameters(k * m6, k * m12)
        if switch_streams:
            ctx.set_stream(streams[(n + 1) % 2].cuda_stream)
        ctx.compute_device(x.data_ptr(), out[n].data_ptr())
    torch.cuda.synchronize()
    for got, w in zip(out, want):
        assert rms(got.cpu().numpy() - w) <= 4e-6 * rms(w)


def _capture_step(ctx, x, f, flags):
    """A graph of one step on a stream of its own (eager first: the launch
    attributes and buffers are then there); returns the graph and the stream."""
    import torch

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    ctx.set_stream(stream.cuda_stream)
    ctx.compute_device(x.data_ptr(), f.data_ptr(), flags)
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.compute_device(x.data_ptr(), f.data_ptr(), flags)
    return graph, stream


def test_getters_wait_for_a_replayed_step():
    # a step captured by the caller: energies, virial and shift forces are
    # those of the last replay, also where it is still queued behind other work
    import torch

    s = S.water_box(1001, None, seed=4)
    rng = np.random.default_rng(7)
    moved = [(s.x + 0.01 * rng.normal(size=s.x.shape)).astype(np.float32) for _ in range(4)]
    ctx = nbx.context_for(s)
    want = []
    for xm in moved:
        f = ctx.compute(xm, energy=True, virial=True, shift_forces=True, reproducible=True)
        want.append((f, np.array(ctx.energies()), ctx.virial(), ctx.shift_forces()))
    flags = (nbx.COMPUTE_FORCES | nbx.COMPUTE_ENERGY | nbx.COMPUTE_SHIFT_FORCES | nbx.COMPUTE_VIRIAL
             | nbx.COMPUTE_REPRODUCIBLE)
    x = torch.from_numpy(s.x.astype(np.float32)).cuda()
    xs = [torch.from_numpy(xm).cuda() for xm in moved]
    f = torch.zeros_like(x)
    busy = torch.ones(4096, 4096, device="cuda")
    graph, stream = _capture_step(ctx, x, f, flags)
    for n, (wf, we, wv, ws) in enumerate(want):
        print(f"[replay] {n}", flush=True)
        with torch.cuda.stream(stream):
            for _ in range(20):
                busy = busy @ busy * 0.0 + 1.0
            x.copy_(xs[n])
            graph.replay()
            np.testing.assert_array_equal(np.array(ctx.energies()), we)
            np.testing.assert_array_equal(ctx.virial(), wv)
            np.testing.assert_array_equal(ctx.shift_forces(), ws)
            np.testing.assert_array_equal(f.cpu().numpy(), wf)


@pytest.mark.parametrize("energy", [False, True])
def test_replayed_step_takes_the_parameters_set_last(energy):
    # a captured step reads the LJ parameters from the context's tables: set
    # after the capture they hold for the replays, also for a type that had no
    # LJ then (water's hydrogens) or has none any more
    import torch

    s = S.water_box(1001, None, seed=4)
    m6, m12 = nbx.nblib_c6c12_matrices(s.c6, s.c12)
    every = nbx.nblib_c6c12_matrices(np.maximum(s.c6, 1e-4), np.maximum(s.c12, 1e-8))
    sets = [(m6, m12), every, (0.5 * m6, 0.5 * m12), (0.0 * m6, 0.0 * m12), (m6, m12)]
    want = []
    for c6, c12 in sets:
        ctx = nbx.context_for(s)
        ctx.set_nonbonded_parameters(c6, c12)
        want.append((ctx.compute(s.x, energy=True), np.array(ctx.energies())))
    assert rms(want[1][0] - want[0][0]) > 1e-2 * rms(want[0][0])  # the hydrogens' LJ shows
    ctx = nbx.context_for(s)
    x = torch.from_numpy(s.x.astype(np.float32)).cuda()
    f = torch.zeros_like(x)
    graph, stream = _capture_step(ctx, x, f, nbx.COMPUTE_FORCES | (nbx.COMPUTE_ENERGY if energy else 0))
    for n, ((c6, c12), (wf, we)) in enumerate(zip(sets, want)):
        print(f"[replay] parameters {n}", flush=True)
        ctx.set_nonbonded_parameters(c6, c12)
        with torch.cuda.stream(stream):
            graph.replay()
            got = f.cpu().numpy()
        # the forces-only kernel's sums differ by rounding (above)
        assert rms(got - wf) <= 4e-6 * rms(wf)
        if energy:
            np.testing.assert_allclose(ctx.energies(), we, rtol=1e-12)


def test_stream_switch_inside_a_capture_after_new_parameters():
    # the context moves to the captured stream inside the capture, with
    # parameters set on its last stream (their upload is waited for, not captured)
    import torch

    s = S.water_box(1001, None, seed=4)
    m6, m12 = nbx.nblib_c6c12_matrices(s.c6, s.c12)
    ctx = nbx.context_for(s)
    want = []
    for k in (1.5, 0.5):
        ctx.set_nonbonded_parameters(k * m6, k * m12)
        want.append(ctx.compute(s.x))
    x = torch.from_numpy(s.x.astype(np.float32)).cuda()
    f = torch.zeros_like(x)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    ctx.set_stream(streams[0].cuda_stream)
    ctx.set_nonbonded_parameters(1.5 * m6, 1.5 * m12)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[1]):
        ctx.set_stream(streams[1].cuda_stream)
        ctx.compute_device(x.data_ptr(), f.data_ptr())
    for n, k in enumerate((1.5, 0.5, 1.5)):
        ctx.set_nonbonded_parameters(k * m6, k * m12)
        with torch.cuda.stream(streams[1]):
            graph.replay()
            got = f.cpu().numpy()
        assert rms(got - want[n % 2]) <= 4e-6 * rms(want[n % 2])


def test_parameters_are_in_place_for_a_replay_on_another_stream():
    # with a step in a graph, set_nonbonded_parameters returns when the tables
    # hold the new parameters: the graph may be replayed on any stream next,
    # without the context's own stream having been waited for
    import torch

    s = S.water_box(1001, None, seed=4)
    m6, m12 = nbx.nblib_c6c12_matrices(s.c6, s.c12)
    scales = [1.5, 0.5, 1.25, 1.0]
    ctx = nbx.context_for(s)
    want = []
    for k in scales:
        ctx.set_nonbonded_parameters(k * m6, k * m12)
        want.append(ctx.compute(s.x))
    x = torch.from_numpy(s.x.astype(np.float32)).cuda()
    f = torch.zeros_like(x)
    graph, stream = _capture_step(ctx, x, f, nbx.COMPUTE_FORCES)
    own = torch.cuda.Stream()
    torch.cuda.synchronize()
    ctx.set_stream(own.cuda_stream)
    for k, w in zip(scales, want):
        ctx.set_nonbonded_parameters(k * m6, k * m12)
        with torch.cuda.stream(stream):
            graph.replay()
            got = f.cpu().numpy()
        assert rms(got - w) <= 4e-6 * rms(w)


def test_many_contexts_keep_their_own_results():
    # contexts share pinned memory for their results (64 blocks a slab): more
    # of them than a slab holds, destroyed and created in between, on two threads
    from concurrent.futures import ThreadPoolExecutor

    s = S.water_box(70, 2.05, seed=3, rc=0.9, rlist=1.0)
    m6, m12 = nbx.nblib_c6c12_matrices(s.c6, s.c12)

    def open_context(k):
        ctx = nbx.context_for(s)
        ctx.set_nonbonded_parameters((1.0 + k) * m6, (1.0 + k) * m12)
        ctx.compute(s.x, energy=True)
        return k, ctx

    one = nbx.context_for(s)
    one.compute(s.x, energy=True)
    lj, coulomb = one.energies()

    def check(contexts):
        for k, ctx in contexts:
            # LJ is linear in the parameters (float pair terms)
            np.testing.assert_allclose(ctx.energies(), ((1.0 + k) * lj, coulomb), rtol=1e-5)

    with ThreadPoolExecutor(2) as pool:
        contexts = list(pool.map(open_context, range(140)))
        check(contexts)
        for _, ctx in contexts[::2]:
            ctx.close()
        contexts = contexts[1::2] + list(pool.map(open_context, range(140, 170)))
        check(contexts)
    for _, ctx in contexts:
        ctx.close()
    one.compute(s.x, energy=True)
    np.testing.assert_allclose(one.energies(), (lj, coulomb), rtol=1e-12)
