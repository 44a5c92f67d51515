"""Parity of the gfx950 Slater-Jastrow path (through the C ABI) with the CPU
oracle's Sherman-Morrison runner on the same Philox streams, in FP64 and in
mixed precision; independence of the result from lanes-per-walker;
heterogeneous systems in one launch; zero-variance anchors (1s and 2p); the
FP64 log-determinants carried through the updates and their drift; the
singular-pivot guard on planted singular configurations."""
import numpy as np
import pytest

import mole_amd as M
from mole_amd import systems as S
from oracle import sj_ffi as SJ

pytestmark = pytest.mark.gpu

E_TOL = 1e-10


def bits(a):
    return np.asarray(a, dtype=np.float64).view(np.uint64)


def run_device(systems, W, steps, B, *, precision=M.PREC_FP64, lu=16, lanes=None, seed=0, side=0.6,
               hamiltonian=M.H_ELECTRONIC, proposal=M.PROPOSAL_BOX):
    dev = [M.slater_jastrow(s, W, hamiltonian=hamiltonian) for s in systems]
    with M.Context(dev, seed=seed, step=side, block_size=B, flags=M.FLAG_TRACE, record_sweeps=steps,
                   precision=precision, lu_period=lu, proposal=proposal) as ctx:
        if lanes is not None:
            for k in range(len(systems)):
                ctx.set_walker_lanes(lanes, sys=k)
        ctx.init_walkers()
        ctx.run(steps)
        total = (steps // B) * B
        out = []
        for k in range(len(systems)):
            masks, el = ctx.trace(total, total - B, sys=k)
            out.append(dict(masks=masks, el=el, cfg=ctx.get_configs(sys=k), stats=ctx.stats(sys=k),
                            sr=ctx.sr_sums(sys=k), lanes=ctx.walker_lanes(sys=k)))
    return out


def run_oracle(system, W, steps, B, *, precision=SJ.PREC_FP64, lu=16, seed=0, side=0.6, sys=0,
               hamiltonian=0, proposal=SJ.BOX):
    wv = SJ.SjWave(system, hamiltonian=hamiltonian)
    return SJ.run(wv, seed=seed, walkers=W, steps=steps, block_size=B, box_side=side,
                  precision=precision, lu_period=lu, sys=sys, n_threads=8, proposal=proposal, tau=side)


@pytest.mark.parametrize("Z", [3, 6, 10])
def test_fp64_parity_with_oracle(Z):
    W, steps, B = 70, 30, 10
    system = S.atom(Z)
    d = run_device([system], W, steps, B)[0]
    o = run_oracle(system, W, steps, B)
    assert np.array_equal(d["masks"], o["accept_mask"]), "accept/reject decisions differ"
    assert np.array_equal(bits(d["cfg"]), bits(o["cfg"]))
    rel = np.abs(d["el"] - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
    assert np.max(rel) <= E_TOL
    st = d["stats"]
    assert st["n_accepted"] == o["n_accepted"] and st["n_moves"] == o["n_moves"]
    assert abs(st["sum_e"] - o["sum_e"]) <= 1e-10 * o["n_samples"] * max(1.0, abs(o["sum_e"] / o["n_samples"]))
    assert st["max_condition"] > 1.0


@pytest.mark.parametrize("Z", [3, 6])
def test_mixed_precision_parity_with_oracle(Z):
    W, steps, B = 64, 30, 10
    system = S.atom(Z)
    d = run_device([system], W, steps, B, precision=M.PREC_MIXED, lu=64)[0]
    o = run_oracle(system, W, steps, B, precision=SJ.PREC_MIXED, lu=64)
    assert np.array_equal(d["masks"], o["accept_mask"])
    assert np.array_equal(bits(d["cfg"]), bits(o["cfg"]))
    rel = np.abs(d["el"] - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
    assert np.max(rel) <= E_TOL


@pytest.mark.parametrize("Z,lanes,steps", [(3, 2, 30), (4, 2, 12), (5, 2, 10), (6, 4, 10), (7, 4, 8), (8, 4, 8),
                                           (9, 4, 8), (10, 4, 10)])
def test_mixed_precision_parity_at_workload_width(Z, lanes, steps):
    # the atoms workload's width (65,536 walkers, LU refresh every 64 moves)
    # with the lanes per walker its autotuning picks: every accept decision,
    # the configurations and the FP32 inverses' consequences bit for bit
    W, B = 65536, 2
    print(f"workload width Z={Z} W={W} lanes={lanes} sweeps={steps}", flush=True)
    system = S.atom(Z)
    d = run_device([system], W, steps, B, precision=M.PREC_MIXED, lu=64, lanes=lanes, seed=1)[0]
    o = run_oracle(system, W, steps, B, precision=SJ.PREC_MIXED, lu=64, seed=1)
    assert d["lanes"] == lanes
    assert np.array_equal(d["masks"], o["accept_mask"]), "accept/reject decisions differ"
    assert np.array_equal(bits(d["cfg"]), bits(o["cfg"]))
    rel = np.abs(d["el"] - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
    assert np.max(rel) <= 1e-9
    assert d["stats"]["n_accepted"] == o["n_accepted"]


def tile_footprint(system, lanes):
    """LDS bytes of one full tile of the system at the given lanes per walker
    (a one-tile context's launch shape)."""
    with M.Context([M.slater_jastrow(system, 64 // lanes)], seed=0, step=0.6, block_size=2,
                   precision=M.PREC_MIXED, lu_period=64) as c:
        c.set_walker_lanes(lanes)
        return c.launch_info()[1]


def test_heterogeneous_batch_at_workload_shape():
    # the heterogeneous workload's launches: 256 systems of 2..40 electrons,
    # 2^20 walkers split in proportion to N, the lanes its autotuning picked,
    # mixed precision.  The tiles are grouped into LDS footprint classes (one up
    # to an eighth of a CU's 160 KiB, 4 KiB steps above it), one launch per class
    # with blockIdx.x restarting at 0 in each, longest tiles first within a class.
    # The system with the fewest electrons, the one with the largest tile
    # footprint and the largest system of a third class against their own oracle
    # runs (systems are independent streams)
    from mole_amd import autotune
    from mole_amd import workloads as WL
    lanes = {n: 4 if n <= 4 else 8 if n <= 16 else 16 if n <= 27 else 32 for n in range(2, 41)}
    sys_list = WL.hetero_systems(256, 3)
    Ns = np.array([s.n_electrons for s in sys_list])
    W = np.maximum(1, np.floor(Ns / Ns.sum() * (1 << 20))).astype(int)
    W[np.argmax(Ns)] += (1 << 20) - W.sum()
    lds = np.array([tile_footprint(s, lanes[int(n)]) for s, n in zip(sys_list, Ns)])
    cls = (np.maximum(lds, 163840 // 8) + 4095) // 4096
    assert np.unique(cls).size >= 3
    first, largest = int(np.argmin(Ns)), int(np.argmax(lds))
    others = [k for k in np.argsort(Ns, kind="stable") if cls[k] not in (cls[first], cls[largest])]
    picks = [first, largest, int(others[-1])]
    assert np.unique(cls[picks]).size == 3
    steps, B = 4, 2
    print(f"heterogeneous batch: {len(sys_list)} systems, {int(W.sum())} walkers, checking {picks}", flush=True)
    dev = [M.slater_jastrow(s, int(w)) for s, w in zip(sys_list, W)]
    with M.Context(dev, seed=3, step=0.6, block_size=B, flags=M.FLAG_TRACE, record_sweeps=steps,
                   precision=M.PREC_MIXED, lu_period=64) as ctx:
        autotune.apply(ctx, sys_list, lanes)
        ctx.init_walkers()
        ctx.run(steps)
        got = {k: (ctx.trace(steps, steps - B, sys=k), ctx.get_configs(sys=k)) for k in picks}
    for k in picks:
        (masks, el), cfg = got[k]
        o = SJ.run(SJ.SjWave(sys_list[k]), seed=3, walkers=int(W[k]), steps=steps, block_size=B, box_side=0.6,
                   precision=SJ.PREC_MIXED, lu_period=64, sys=k, n_threads=8)
        assert np.array_equal(masks, o["accept_mask"]), f"system {k}: accept/reject decisions differ"
        assert np.array_equal(bits(cfg), bits(o["cfg"])), f"system {k}"
        rel = np.abs(el - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
        assert np.max(rel) <= 1e-9, f"system {k}"


def test_results_independent_of_lanes_per_walker():
    system = S.atom(7)
    ref = None
    for L in (2, 4, 8, 16, 32, 64):
        d = run_device([system], 40, 20, 5, lanes=L)[0]
        assert d["lanes"] == L
        if ref is None:
            ref = d
            continue
        assert np.array_equal(d["masks"], ref["masks"]), L
        assert np.array_equal(bits(d["cfg"]), bits(ref["cfg"])), L
        assert np.array_equal(bits(d["el"]), bits(ref["el"])), L
        for k in ("sum_o", "sum_oe", "sum_oo"):
            assert np.array_equal(d["sr"][k], ref["sr"][k]), (L, k)


def test_heterogeneous_systems_in_one_launch():
    systems = [S.helium_product(1.7, 0.5), S.atom(4), S.hydrogen_chain(4), S.random_molecule(9, seed=2),
               S.atom(10)]
    W, steps, B = 33, 20, 5
    dev = run_device(systems, W, steps, B)
    for k, system in enumerate(systems):
        o = run_oracle(system, W, steps, B, sys=k)
        assert np.array_equal(dev[k]["masks"], o["accept_mask"]), k
        assert np.array_equal(bits(dev[k]["cfg"]), bits(o["cfg"])), k
        rel = np.abs(dev[k]["el"] - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
        assert np.max(rel) <= E_TOL, k


@pytest.mark.parametrize("wide", [0, 2])
def test_small_footprints_share_a_launch(wide):
    # tiles up to an eighth of a CU's LDS (20 KiB) are one class whatever their
    # footprints, larger ones classes of their own: every system at the fewest
    # lanes below the line, then the last two at the most lanes above it
    systems = [S.helium_product(1.7, 0.5), S.hydrogen_chain(6), S.atom(10), S.random_molecule(14, seed=3),
               S.hydrogen_chain(24)]
    lanes = []
    for k, s in enumerate(systems):
        above = k >= len(systems) - wide
        L = 64
        while L > 2 and tile_footprint(s, L) > 20480:
            L //= 2
        while L > 2 and tile_footprint(s, L // 2) <= 20480:
            L //= 2
        lanes.append(L // 2 if above and L > 2 else L)
    print(f"small footprints: lanes {lanes}", flush=True)
    W, steps, B = 33, 6, 2
    dev = [M.slater_jastrow(s, W) for s in systems]
    with M.Context(dev, seed=5, step=0.6, block_size=B, flags=M.FLAG_TRACE, record_sweeps=steps,
                   precision=M.PREC_MIXED, lu_period=64) as ctx:
        for k, L in enumerate(lanes):
            ctx.set_walker_lanes(L, sys=k)
        ctx.init_walkers()
        ctx.run(steps)
        got = [(ctx.trace(steps, steps - B, sys=k), ctx.get_configs(sys=k)) for k in range(len(systems))]
    for k, system in enumerate(systems):
        (masks, el), cfg = got[k]
        o = run_oracle(system, W, steps, B, sys=k, precision=SJ.PREC_MIXED, lu=64, seed=5)
        assert np.array_equal(masks, o["accept_mask"]), k
        assert np.array_equal(bits(cfg), bits(o["cfg"])), k
        rel = np.abs(el - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
        assert np.max(rel) <= E_TOL, k


def test_zero_variance_anchors():
    d = run_device([S.hydrogenic(1)], 128, 20, 5)[0]
    assert np.max(np.abs(d["el"] + 0.5)) <= 1e-12
    # the 2p eigenfunctions x_q exp(-Z r/2): E_L = -Z^2/8 for every sample
    for axis in range(3):
        d = run_device([S.hydrogenic_2p(2, axis)], 128, 20, 5)[0]
        assert np.max(np.abs(d["el"] + 0.5)) <= 1e-11
    d = run_device([S.helium_product(2.0, 0.0)], 128, 20, 5, hamiltonian=M.H_IONIC)[0]
    assert np.max(np.abs(d["el"] + 4.0)) <= 1e-12


def test_helium_product_anchor_through_determinants():
    zeta = 1.5
    sysd = M.slater_jastrow(S.helium_product(zeta, 0.0), 4096)
    with M.Context([sysd], seed=9, step=1.0, block_size=50, lu_period=32) as ctx:
        ctx.init_walkers()
        ctx.run(1000)
        st = ctx.stats()
    mean = st["sum_e"] / st["n_samples"]
    nb = st["n_blocks"]
    err = np.sqrt((st["sum_block_mean2"] / nb - (st["sum_block_mean"] / nb) ** 2) / (nb - 1))
    assert abs(mean - (zeta**2 - 27 * zeta / 8)) < 4 * err


def test_graph_replays_match_eager_sweeps():
    # a captured [sweep, advance] launch replayed several times, with eager
    # work and synchronisations between replays, equals the eager sequence
    systems = [S.atom(4), S.random_molecule(6, seed=4)]

    def make():
        dev = [M.slater_jastrow(s, 50) for s in systems]
        ctx = M.Context(dev, seed=5, step=0.6, block_size=4, precision=M.PREC_MIXED, lu_period=16)
        ctx.init_walkers()
        return ctx

    snaps = []
    for use_graph in (False, True):
        ctx = make()
        g = ctx.capture(5, sample=True) if use_graph else None
        out = []
        for r in range(4):
            if use_graph:
                g.launch(1)
            else:
                ctx.sweep(5, sample=True)
            ctx.synchronize()
            ctx.sweep(2)  # eager work between replays
            out.append((ctx.get_configs(0), ctx.get_configs(1), ctx.stats(0), ctx.sr_sums(1), ctx.get_stream()))
        if g is not None:
            g.launch(2)
            out.append((ctx.get_configs(0), ctx.get_configs(1), ctx.stats(0), ctx.sr_sums(1), ctx.get_stream()))
            g.close()
        else:
            ctx.sweep(5, sample=True)
            ctx.sweep(5, sample=True)
            out.append((ctx.get_configs(0), ctx.get_configs(1), ctx.stats(0), ctx.sr_sums(1), ctx.get_stream()))
        ctx.close()
        snaps.append(out)
    for a, b in zip(*snaps):
        assert np.array_equal(bits(a[0]), bits(b[0]))
        assert np.array_equal(bits(a[1]), bits(b[1]))
        assert a[2] == b[2]
        for k in ("sum_o", "sum_oe", "sum_oo"):
            assert np.array_equal(a[3][k], b[3][k])
        assert a[4] == b[4]


def test_graph_goes_stale_when_lanes_change():
    dev = [M.slater_jastrow(S.atom(3), 32)]
    with M.Context(dev, seed=1, step=0.6, block_size=4, lu_period=16) as ctx:
        ctx.init_walkers()
        g = ctx.capture(2)
        g.launch(1)
        ctx.set_walker_lanes(2)
        with pytest.raises(M.MoleError) as ei:
            g.launch(1)
        assert ei.value.status == M.ERR_INVALID_ARGUMENT
        g.close()


# ------------------------------------------------ drift-diffusion proposal

@pytest.mark.parametrize("Z,precision", [(3, M.PREC_FP64), (7, M.PREC_FP64), (4, M.PREC_MIXED)])
def test_diffusion_parity_with_oracle(Z, precision):
    # MetropolisDiffuse (metrop.rs:150-197, single-row Green's functions):
    # same Box-Muller normals, drift and accept decisions as the oracle
    W, steps, B, tau = 48, 24, 8, 0.05
    system = S.atom(Z)
    d = run_device([system], W, steps, B, precision=precision, lu=16, side=tau,
                   proposal=M.PROPOSAL_DIFFUSE)[0]
    o = run_oracle(system, W, steps, B, precision=precision, lu=16, side=tau, proposal=SJ.DIFFUSE)
    assert np.array_equal(d["masks"], o["accept_mask"]), "accept/reject decisions differ"
    assert np.array_equal(bits(d["cfg"]), bits(o["cfg"]))
    rel = np.abs(d["el"] - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
    assert np.max(rel) <= E_TOL


def test_diffusion_heterogeneous_and_lane_independent():
    systems = [S.helium_product(1.7, 0.5), S.random_molecule(6, seed=8)]
    ref = None
    for L in (2, 8, 32):
        dev = run_device(systems, 24, 12, 4, lanes=L, side=0.1, proposal=M.PROPOSAL_DIFFUSE)
        if ref is None:
            ref = dev
            for k, system in enumerate(systems):
                o = run_oracle(system, 24, 12, 4, side=0.1, sys=k, proposal=SJ.DIFFUSE)
                assert np.array_equal(dev[k]["masks"], o["accept_mask"]), k
                assert np.array_equal(bits(dev[k]["cfg"]), bits(o["cfg"])), k
        else:
            for k in range(len(systems)):
                assert np.array_equal(bits(dev[k]["cfg"]), bits(ref[k]["cfg"])), (L, k)
                assert np.array_equal(bits(dev[k]["el"]), bits(ref[k]["el"])), (L, k)


def test_diffusion_helium_product_anchor():
    zeta = 1.5
    sysd = M.slater_jastrow(S.helium_product(zeta, 0.0), 4096)
    with M.Context([sysd], seed=3, step=0.3, block_size=50, lu_period=32,
                   proposal=M.PROPOSAL_DIFFUSE) as ctx:
        ctx.init_walkers()
        ctx.run(1000)
        st = ctx.stats()
    mean = st["sum_e"] / st["n_samples"]
    nb = st["n_blocks"]
    err = np.sqrt((st["sum_block_mean2"] / nb - (st["sum_block_mean"] / nb) ** 2) / (nb - 1))
    assert abs(mean - (zeta**2 - 27 * zeta / 8)) < 4 * err


# ------------------------------------------------ log-determinants, singular blocks

@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED])
def test_logdet_carried_through_updates_matches_oracle(precision):
    # det A_s carried through every accepted move as mantissa x 2^exponent:
    # the drift against each re-inversion (the FP32 chain's error in mixed
    # precision) bit for bit as the oracle's, the final log-determinants as
    # the oracle carries them, and (FP64) as the LU of the final configuration
    W, steps, B = 64, 60, 20
    system = S.atom(9)
    dev = [M.slater_jastrow(system, W)]
    with M.Context(dev, seed=2, step=0.6, block_size=B, precision=precision, lu_period=64) as ctx:
        ctx.init_walkers()
        ctx.run(steps)
        st = ctx.stats()
        ld, sg = ctx.logdet()
        cfg = ctx.get_configs()
    wv = SJ.SjWave(system)
    o = SJ.run(wv, seed=2, walkers=W, steps=steps, block_size=B, box_side=0.6, precision=precision, lu_period=64,
               n_threads=8, record=False)
    assert np.array_equal(bits(cfg), bits(o["cfg"]))
    assert st["max_logdet_drift"] == o["max_ld_drift"]
    assert st["n_singular"] == 0 == o["n_singular"]
    want = np.array([[SJ.logdet_value(o["ld"][w, 2 * q], o["ld"][w, 2 * q + 1]) for q in (0, 1)] for w in range(W)])
    assert np.max(np.abs(ld - want)) <= 1e-12 * np.max(np.abs(want))
    assert np.array_equal(sg, np.sign(o["ld"][:, [0, 2]]))
    if precision == M.PREC_FP64:
        assert 0.0 < st["max_logdet_drift"] < 1e-10
        for w in range(W):
            for q in (0, 1):
                lu, s_lu = SJ.logdet(wv, cfg[w], q)
                assert abs(ld[w, q] - lu) < 1e-10 and sg[w, q] == s_lu
    else:
        assert st["max_logdet_drift"] > 1e-8


def test_planted_singular_configuration_is_counted():
    # walkers 0..7 start with spin-up electrons 0 and 1 at the same point
    # (identical rows, det A_up = 0): the re-inversion counts the block and
    # skips its division instead of writing Inf/NaN into the walker; the
    # guarded path then follows the oracle's bit for bit, and the other
    # walkers' determinants stay finite
    W, steps, B = 16, 20, 10
    system = S.atom(6)
    cfg = np.random.default_rng(7).normal(scale=1.2, size=(W, 3 * system.n_electrons))
    cfg[:8, 3:6] = cfg[:8, 0:3]
    dev = [M.slater_jastrow(system, W)]
    with M.Context(dev, seed=4, step=0.6, block_size=B, flags=M.FLAG_TRACE, record_sweeps=steps, lu_period=8) as ctx:
        ctx.set_configs(cfg)
        ld0, sg0 = ctx.logdet()
        n0 = ctx.stats()["n_singular"]
        ctx.run(steps)
        masks, _ = ctx.trace(steps, 0)
        st = ctx.stats()
        out = ctx.get_configs()
    assert n0 == 8
    assert np.all(ld0[:8, 0] == -np.inf) and np.all(sg0[:8, 0] == 0.0)
    assert np.all(np.isfinite(ld0[8:])) and np.all(np.isfinite(ld0[:, 1]))
    o = SJ.run(SJ.SjWave(system), seed=4, walkers=W, steps=steps, block_size=B, box_side=0.6, lu_period=8,
               cfg=cfg, n_threads=8)
    assert np.array_equal(masks, o["accept_mask"])
    assert np.array_equal(bits(out), bits(o["cfg"]))
    assert st["n_singular"] == o["n_singular"] >= 8
    assert np.all(np.isfinite(out))


# ------------------------------------------------ reference anchors

H2ION_E = -0.43720930232581723   # quadrature of <E> of the product function (R = 2.5)
H2ION_STD = 0.5052200457935744


def test_h2_ion_product_reference_anchor():
    # tests/hydrogen_molecular_ion_lcao.rs:100-142 on the device: H2+ at
    # R = 2.5 with psi = exp(-r_A) exp(-r_B) (a constant orbital times the e-n
    # Pade factor, a = 1, d = 0), MetropolisBox(1.0), Runner::run(.., 100);
    # the reference asserts |E + 0.565| < std of the samples.  The device's
    # short run also follows the oracle bit for bit, and its long run's mean
    # sits on the quadrature value within the blocking error.
    system = S.h2_ion_product()
    d = run_device([system], 64, 40, 10, side=1.0, seed=4)[0]
    o = run_oracle(system, 64, 40, 10, side=1.0, seed=4)
    assert np.array_equal(d["masks"], o["accept_mask"])
    assert np.array_equal(bits(d["cfg"]), bits(o["cfg"]))
    with M.Context([M.slater_jastrow(system, 8192)], seed=0, step=1.0, block_size=100, lu_period=64) as ctx:
        ctx.init_walkers()
        ctx.run(3000)
        st = ctx.stats()
    n = st["n_samples"]
    mean = st["sum_e"] / n
    std = np.sqrt(st["sum_e2"] / n - mean * mean)
    nb = st["n_blocks"]
    err = np.sqrt((st["sum_block_mean2"] / nb - (st["sum_block_mean"] / nb) ** 2) / (nb - 1))
    assert abs(mean - (-0.565)) < std
    assert abs(mean - H2ION_E) < 4 * err, (mean, err)
    assert abs(std - H2ION_STD) < 0.02 * H2ION_STD


@pytest.mark.parametrize("workgroups", [0, 3])
def test_persistent_schedule_matches_class_launches(workgroups):
    # every tile of the context in one persistent launch (the tiles drawn from
    # a device ticket, longest first; 3 workgroups: each takes many tiles)
    # against one launch per footprint class: the same walkers, bit for bit,
    # eagerly and replayed from a captured graph (the ticket's reset is part
    # of the capture)
    systems = [S.atom(4), S.random_molecule(9, seed=2), S.hydrogen_chain(6), S.atom(10)]
    W, B = 70, 5

    def run(schedule):
        dev = [M.slater_jastrow(s, W) for s in systems]
        with M.Context(dev, seed=6, step=0.6, block_size=B, flags=M.FLAG_TRACE, record_sweeps=30,
                       precision=M.PREC_MIXED, lu_period=16) as ctx:
            for k, L in enumerate((4, 8, 16, 8)):
                ctx.set_walker_lanes(L, sys=k)
            ctx.set_tile_schedule(schedule, workgroups)
            if schedule == M.SCHEDULE_PERSISTENT:
                wg, _ = ctx.launch_info()
                assert wg == (workgroups or wg) and wg >= 1
            ctx.init_walkers()
            ctx.run(10)
            g = ctx.capture(5, sample=True)
            for _ in range(3):
                g.launch(1)
                ctx.synchronize()
                ctx.sweep(1)
            g.close()
            return [(ctx.get_configs(k), ctx.trace(28, 24, sys=k), ctx.stats(k)) for k in range(len(systems))]

    a = run(M.SCHEDULE_CLASSES)
    b = run(M.SCHEDULE_PERSISTENT)
    for k in range(len(systems)):
        assert np.array_equal(bits(a[k][0]), bits(b[k][0])), k
        assert np.array_equal(a[k][1][0], b[k][1][0]), k
        assert np.array_equal(bits(a[k][1][1]), bits(b[k][1][1])), k
        assert a[k][2] == b[k][2], k


@pytest.mark.parametrize("make,precision,proposal", [
    (lambda: S.atom(3), M.PREC_FP64, M.PROPOSAL_BOX),
    (lambda: S.atom(8), M.PREC_MIXED, M.PROPOSAL_BOX),
    (lambda: S.h2_lcao(), M.PREC_FP64, M.PROPOSAL_DIFFUSE),
])
def test_exponent_scale_parameter_parity_with_oracle(make, precision, proposal):
    # six parameters: the basis exponents are s zeta_m on both sides (same
    # products), so the trajectories match bit for bit, and the per-walker
    # sums of the six log-derivatives match the oracle's samples
    system = make()
    s0 = 1.15
    W, steps, B = 48, 24, 4
    side = 0.6 if proposal == M.PROPOSAL_BOX else 0.05
    p6 = list(system.jastrow) + [s0]
    dev = [M.slater_jastrow(system, W, params=p6)]
    with M.Context(dev, seed=2, step=side, block_size=B, flags=M.FLAG_TRACE, record_sweeps=steps,
                   precision=precision, lu_period=16, proposal=proposal) as ctx:
        ctx.init_walkers()
        ctx.run(steps)
        total = (steps // B) * B
        masks, el = ctx.trace(total, total - B)
        cfg = ctx.get_configs()
        sr = ctx.sr_sums()
        assert np.array_equal(ctx.get_params(), p6)
    wv = SJ.SjWave(system, params=p6)
    o = SJ.run(wv, seed=2, walkers=W, steps=steps, block_size=B, box_side=side, tau=side,
               precision=SJ.PREC_FP64 if precision == M.PREC_FP64 else SJ.PREC_MIXED, lu_period=16,
               n_threads=8, proposal=SJ.BOX if proposal == M.PROPOSAL_BOX else SJ.DIFFUSE)
    assert np.array_equal(masks, o["accept_mask"])
    assert np.array_equal(bits(cfg), bits(o["cfg"]))
    rel = np.abs(el - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
    assert np.max(rel) <= E_TOL
    dl = o["dlog"].reshape(-1, 6)
    assert sr["sum_o"].shape == (6,) and abs(sr["sum_o"][5]) > 0.0
    assert np.allclose(sr["sum_o"], dl.sum(axis=0), rtol=1e-9, atol=1e-9)
    assert np.allclose(sr["sum_oo"], dl.T @ dl, rtol=1e-9, atol=1e-9)
    assert np.allclose(sr["sum_oe"], dl.T @ o["e_local"].ravel(), rtol=1e-9, atol=1e-7)


def test_sho_steepest_descent_reaches_the_ground_state():
    # tests/sho_optimize.rs:117-141 on the device: a 3D Gaussian trial
    # function exp(-s r^2) (a = 1: s = 1) under T + r^2/2 with the drift-
    # diffusion proposal, steepest descent on the exponent from the energy
    # gradient 2(<E O> - <E><O>); the ground state s = 1/2 has E = 3/2 with
    # zero variance.  (The reference's step 1e-3 applies to its Q1-scaled
    # gradient; with the log-derivative a step of 0.2 converges in ~10
    # iterations.)  The last energy lies within its blocking error of 1.5.
    system = S.harmonic_oscillator(1.0, a=1.0)
    h = M.harmonic_hamiltonian(1.0)
    p = np.array(list(system.jastrow) + [1.0])
    dev = [M.slater_jastrow(system, 1024, params=p)]
    energies = []
    with M.Context(dev, seed=0, step=0.1, block_size=10, proposal=M.PROPOSAL_DIFFUSE) as ctx:
        ctx.set_hamiltonian(h)
        ctx.init_walkers()
        ctx.sweep(50)
        for it in range(20):
            ctx.reset_stats()
            ctx.run(100, 10)
            st = ctx.stats()
            mean = st["sum_e"] / st["n_samples"]
            nb = st["n_blocks"]
            err = np.sqrt(max(st["sum_block_mean2"] / nb - (st["sum_block_mean"] / nb) ** 2, 0.0) / (nb - 1))
            energies.append((mean, err, p[5]))
            dp, g = M.parameter_update(ctx.sr_sums_raw(), M.OPT_SD, 0.2)
            assert np.all(dp[:5] == 0.0)  # no Jastrow term: only the exponent moves
            p = p + dp
            ctx.set_params(p)
    e0, err0, s_first = energies[0]
    e, err, s_last = energies[-1]
    assert e0 > 1.8 and s_first == 1.0  # E(s) = 3/2 (s + 1/(4 s)) = 1.875 at s = 1
    assert abs(s_last - 0.5) < 1e-6
    assert abs(e - 1.5) <= max(err, 1e-12), (e, err)


@pytest.mark.parametrize("make,params,optimizer,step,precision", [
    (lambda: S.helium_product(1.6, 0.4), [0.4, 0.0, 0.3, 0.0, 1.0, 1.05], M.OPT_SD, 0.05, M.PREC_FP64),
    (lambda: S.atom(3), None, M.OPT_SD, 0.01, M.PREC_MIXED),
    (lambda: S.atom(3), list(S.atom(3).jastrow) + [1.0], M.OPT_SR, 0.02, M.PREC_MIXED),
    (lambda: S.harmonic_oscillator(1.0, a=1.0), [0.0, 0.0, 0.0, 0.0, 0.0, 1.0], M.OPT_SD, 0.2, M.PREC_FP64),
])
def test_device_optimisation_loop_equals_host_loop(make, params, optimizer, step, precision):
    # mole_optimize on a Slater-Jastrow system (the step kernel rewrites the
    # device system table and, with the exponent scale, the exponents)
    # against the same iterations through the host (sums read back, the
    # update on the host, mole_set_params): the same parameters, sums and
    # walkers bit for bit
    system = make()
    p0 = np.array(system.jastrow if params is None else params, dtype=float)
    W, steps, B, iters = 256, 40, 10, 4
    h = M.harmonic_hamiltonian(1.0) if system.charges.sum() == 0 else None

    def context():
        c = M.Context([M.slater_jastrow(system, W, params=p0)], seed=9, step=0.5, block_size=B,
                      precision=precision, lu_period=16)
        if h is not None:
            c.set_hamiltonian(h)
        c.init_walkers()
        return c

    with context() as ctx:
        p = p0.copy()
        host_log = []
        for _ in range(iters):
            ctx.reset_stats()
            ctx.run(steps, B)
            st = ctx.stats()
            host_log.append((st["sum_e"], st["sum_block_mean"], st["n_accepted"]))
            dp, _ = M.parameter_update(ctx.sr_sums_raw(), optimizer, step, M.SR_TEXTBOOK, 1e-3)
            p = p + dp
            ctx.set_params(p)
        cfg_host = ctx.get_configs()
    with context() as ctx:
        p_dev, log = ctx.optimize(iters, steps, B, optimizer, step, M.SR_TEXTBOOK, 1e-3)
        assert np.array_equal(ctx.get_params(), p_dev)
        cfg_dev = ctx.get_configs()
    assert np.array_equal(bits(p_dev), bits(p))
    for it in range(iters):
        assert log[it, 0] == host_log[it][0] and log[it, 2] == host_log[it][1], it
        assert log[it, 4] == host_log[it][2] and log[it, 5] == 0.0
    assert np.array_equal(bits(cfg_dev), bits(cfg_host))
    assert not np.array_equal(p_dev, p0)


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED])
def test_compat_samples_match_oracle(precision):
    # MOLE_FLAG_SAMPLES on a Slater-Jastrow system: per-sample "Energy",
    # "Wavefunction value" (psi psi)/psi from the carried determinants and
    # "Parameter gradient" O psi_s, against the oracle's parity runner
    system = S.random_molecule(6, seed=5)
    W, steps, B = 70, 30, 10
    ns = (steps // B - 1) * B
    with M.Context([M.slater_jastrow(system, W)], seed=3, step=0.6, block_size=B, flags=M.FLAG_SAMPLES,
                   record_sweeps=steps, precision=precision, lu_period=16) as ctx:
        ctx.init_walkers()
        ctx.run(steps)
        e, p, g = ctx.samples(ns)
    o = run_oracle(system, W, steps, B, precision=SJ.PREC_FP64 if precision == M.PREC_FP64 else SJ.PREC_MIXED,
                   seed=3)
    rel = np.abs(e - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))
    assert np.max(rel) <= E_TOL
    assert np.all(np.isfinite(p)) and np.all(p != 0.0)
    assert np.array_equal(np.sign(p), np.sign(o["psi"]))
    assert np.max(np.abs(p - o["psi"]) / np.abs(o["psi"])) <= 1e-9
    want = o["dlog"][:, :, :5] * o["psi"][:, :, None]
    assert g.shape == (W, ns, 5)
    scale = np.abs(o["psi"])[:, :, None] * np.maximum(1.0, np.abs(o["dlog"][:, :, :5]))
    assert np.max(np.abs(g - want) / scale) <= 1e-9


def _configs_near_nuclei(system, n, seed):
    rng = np.random.default_rng(seed)
    N = system.n_electrons
    at = rng.integers(0, system.nuclei.shape[0], (n, N))
    return system.nuclei[at] + rng.normal(0.0, 0.8, (n, N, 3))


@pytest.mark.parametrize("make", [lambda: S.atom(4), lambda: S.atom(10), lambda: S.random_molecule(6, seed=5)])
@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED])
def test_eval_matches_oracle(make, precision):
    # mole_eval on a Slater-Jastrow system (FP64 whatever the context's
    # precision): psi against the oracle's LU determinants and full Jastrow
    # sum, grad psi = psi drift, lap psi = psi kin with kin from E_L and the
    # potential, E_L and d psi/dp against the oracle's fresh-inverse local
    # energy; the context's own walkers are left as they were
    system = make()
    n, N = 37, system.n_electrons
    x = _configs_near_nuclei(system, n, 4)
    with M.Context([M.slater_jastrow(system, 8)], seed=1, step=0.6, block_size=2, precision=precision,
                   lu_period=16) as ctx:
        ctx.init_walkers()
        ctx.run(4)
        before = ctx.get_configs()
        out = ctx.eval(x)
        assert np.array_equal(bits(ctx.get_configs()), bits(before))
    wv = SJ.SjWave(system)
    R, Z = system.nuclei, system.charges.astype(float)
    v_nn = sum(Z[I] * Z[J] / np.linalg.norm(R[I] - R[J]) for I in range(len(Z)) for J in range(I + 1, len(Z)))
    for j in range(n):
        xj = x[j].ravel()
        v = SJ.value(wv, xj)
        e, dl = SJ.local_energy(wv, xj)
        assert abs(out["value"][j] - v) <= 1e-10 * abs(v), j
        assert abs(out["e_local"][j] - e) <= 1e-9 * max(1.0, abs(e)), j
        assert np.all(np.abs(out["pgrad"][j] - v * dl[:5]) <= 1e-9 * abs(v) * np.maximum(1.0, np.abs(dl[:5]))), j
        g = np.concatenate([SJ.drift(wv, xj, i) for i in range(N)])
        assert np.all(np.abs(out["grad"][j] - v * g) <= 1e-9 * abs(v) * np.maximum(1.0, np.abs(g))), j
        pos = x[j]
        V = -sum(Z[I] / np.linalg.norm(pos[i] - R[I]) for i in range(N) for I in range(len(Z)))
        V += sum(1.0 / np.linalg.norm(pos[i] - pos[k]) for i in range(N) for k in range(i + 1, N))
        kin = -2.0 * (e - V - v_nn)
        assert abs(out["lap"][j] / v - kin) <= 1e-8 * max(1.0, abs(kin)), j


def test_eval_lanes_follow_the_configurations():
    # mole_eval takes the lanes that a context of as many walkers as it is given
    # configurations would (FP64, box proposal), not those of its own context's
    # walkers, unless the caller set them; the values do not depend on them
    import ctypes as C
    sj = S.atom(10)
    cfg = np.random.default_rng(3).normal(size=(9000, 30))

    def eval_lanes(c, n):
        L = C.c_uint32()
        M.check(M.lib().mole_debug_eval_lanes(c.h, 0, n, C.byref(L)))
        return L.value

    def context(W, precision=M.PREC_FP64, proposal=M.PROPOSAL_BOX):
        return M.Context([M.slater_jastrow(sj, W)], seed=1, step=0.1, block_size=2, precision=precision,
                         proposal=proposal)

    want = {}
    for n in (1, 4096, 9000, 65536):
        with context(n) as c:
            want[n] = c.walker_lanes()
    assert want[1] != want[65536]
    res = []
    for W, precision, proposal in ((64, M.PREC_FP64, M.PROPOSAL_BOX), (65536, M.PREC_MIXED, M.PROPOSAL_BOX),
                                   (65536, M.PREC_MIXED, M.PROPOSAL_DIFFUSE)):
        with context(W, precision, proposal) as c:
            assert {n: eval_lanes(c, n) for n in want} == want
            res.append(c.eval(cfg))
            c.set_walker_lanes(32)
            assert eval_lanes(c, 65536) == 32
            res.append(c.eval(cfg))
            c.set_walker_lanes(0)
            assert eval_lanes(c, 65536) == want[65536]
    for r in res[1:]:
        for k in r:
            assert np.array_equal(bits(r[k]), bits(res[0][k])), k


@pytest.mark.parametrize("Z_or_n,W", [(2, 64), (3, 40000), (5, 9000), (10, 3000), (10, 20000), (17, 500), (36, 70)])
def test_default_lanes_leave_the_results_unchanged(Z_or_n, W):
    # the library's choice of lanes (by electrons and walkers; every width of
    # the rule is met here) against 16 lanes per walker
    sj = S.atom(Z_or_n) if Z_or_n <= 10 else S.hydrogen_chain(Z_or_n, seed=3)
    res = []
    for lanes in (0, 16):
        with M.Context([M.slater_jastrow(sj, W)], seed=9, step=0.6, block_size=2, precision=M.PREC_MIXED,
                       lu_period=16) as ctx:
            ctx.set_walker_lanes(lanes)
            ctx.init_walkers()
            ctx.sweep(2)
            ctx.sweep(2, sample=True)
            res.append((ctx.get_configs(), ctx.stats(), ctx.sr_sums(), ctx.logdet()))
    (c0, s0, r0, l0), (c1, s1, r1, l1) = res
    assert np.array_equal(bits(c0), bits(c1)) and s0 == s1
    assert all(np.array_equal(r0[k], r1[k]) for k in r0)
    assert np.array_equal(bits(l0[0]), bits(l1[0])) and np.array_equal(l0[1], l1[1])


@pytest.mark.parametrize("N,W,precision,proposal", [
    (5, 65536, M.PREC_FP64, M.PROPOSAL_BOX), (6, 65536, M.PREC_MIXED, M.PROPOSAL_DIFFUSE),
    (8, 65536, M.PREC_FP64, M.PROPOSAL_DIFFUSE), (10, 65536, M.PREC_MIXED, M.PROPOSAL_BOX),
    (16, 16384, M.PREC_FP64, M.PROPOSAL_BOX), (16, 65536, M.PREC_FP64, M.PROPOSAL_DIFFUSE),
    (36, 4096, M.PREC_MIXED, M.PROPOSAL_BOX), (3, 1, M.PREC_FP64, M.PROPOSAL_BOX)])
def test_default_lanes_take_the_shorter_rounds(N, W, precision, proposal):
    # a CU holds eight workgroups, or as many as its LDS (160 KiB) has room for;
    # a launch is a number of rounds of that many on every CU, shorter the more
    # lanes a walker has: the default is never half the lanes that need no more
    # rounds (up to the width of a move)
    cus = M.device_info()[1]

    def rounds(c):
        workgroups, lds = c.launch_info()
        return -(-workgroups // (cus * min(8, 163840 // lds)))

    with M.Context([M.slater_jastrow(S.hydrogen_chain(N, seed=3), W)], seed=1, step=0.1, block_size=2,
                   precision=precision, lu_period=16, proposal=proposal) as c:
        L = c.walker_lanes()
        default = rounds(c)
        if L < max(N, 4):
            c.set_walker_lanes(2 * L)
            assert rounds(c) > default, (L, default)


@pytest.mark.parametrize("N,W", [(1, 5461), (1, 5462), (1, 21845), (1, 21846), (2, 21846), (3, 14563), (11, 3973),
                                 (40, 200), (40, 2185)])
def test_configurations_round_trip_through_staged_transfers(N, W):
    # both sides of the staging rules (128 KiB: counted; 512 KiB: always), chunks
    # of 1 MiB with a partial last one, partial 64 x 32 tiles, more than one
    # column tile
    sj = S.hydrogenic() if N == 1 else S.hydrogen_chain(N, seed=1)
    cfg = np.random.default_rng(N).normal(size=(W, 3 * N))
    with M.Context([M.slater_jastrow(sj, W)], seed=1, step=0.5, block_size=2) as ctx:
        ctx.set_configs(cfg)
        assert np.array_equal(bits(ctx.get_configs()), bits(cfg))


@pytest.mark.parametrize("N,W", [(1, 5462), (3, 7281), (11, 1986)])
def test_transfers_before_and_after_the_staging_buffer(N, W):
    # between 128 and 512 KiB a context stages from its ninth transfer on: every
    # round trip is exact on both sides of it
    sj = S.hydrogenic() if N == 1 else S.hydrogen_chain(N, seed=1)
    rng = np.random.default_rng(N)
    with M.Context([M.slater_jastrow(sj, W)], seed=1, step=0.5, block_size=2) as ctx:
        for k in range(7):
            cfg = rng.normal(size=(W, 3 * N))
            ctx.set_configs(cfg)
            assert np.array_equal(bits(ctx.get_configs()), bits(cfg)), k


def test_one_read_does_not_pay_for_the_staging_buffer():
    # contexts of 127 and 129 KiB of walkers that are read once and closed, on
    # the two sides of the staging line: making and freeing a pinned buffer for
    # the one read would take half as long again
    import time
    best = {}
    for _ in range(20):
        for W in (2709, 2753):
            c = M.Context([M.helium(W)], seed=1, step=0.5, block_size=10)
            c.init_walkers()
            c.synchronize()
            t = time.perf_counter()
            c.get_configs()
            c.close()
            best[W] = min(best.get(W, 1.0), time.perf_counter() - t)
    print(f"one read and close: {best}", flush=True)
    assert best[2753] <= 1.25 * best[2709], best


@pytest.mark.parametrize("proposal", [M.PROPOSAL_BOX, M.PROPOSAL_DIFFUSE])
@pytest.mark.parametrize("n,per", [(4, 2), (3, 3), (5, 2), (8, 2), (9, 2)])
def test_shared_basis_tables_at_their_edges(n, per, proposal):
    # basis tables in LDS up to 8 functions (8: yes; 9, 10, 16, 18: no) and
    # coefficients up to 512 bytes (128, 144, 240, 512: yes; 720: no)
    system = S.hydrogen_chain(n, basis_per_nucleus=per, seed=2)
    W, steps, B = 37, 6, 2
    side = 0.6 if proposal == M.PROPOSAL_BOX else 0.05
    d = run_device([system], W, steps, B, lu=7, seed=4, side=side, proposal=proposal)[0]
    o = run_oracle(system, W, steps, B, lu=7, seed=4, side=side, proposal=proposal)
    assert np.array_equal(d["masks"], o["accept_mask"])
    assert np.array_equal(bits(d["cfg"]), bits(o["cfg"]))
    assert np.max(np.abs(d["el"] - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))) <= E_TOL


@pytest.mark.parametrize("N", [10, 11, 20, 21, 22, 40])
def test_spin_blocks_at_the_chunk_edges(N):
    # spin blocks of 5, 6, 10, 11 and 20: the halves and chunks of the local
    # energy's orbital registers and the rows of the re-inversion (every 5 moves)
    system = S.hydrogen_chain(N, seed=6)
    W, steps, B = 9, 4, 2
    d = run_device([system], W, steps, B, lu=5, seed=2)[0]
    o = run_oracle(system, W, steps, B, lu=5, seed=2)
    assert np.array_equal(d["masks"], o["accept_mask"])
    assert np.array_equal(bits(d["cfg"]), bits(o["cfg"]))
    assert np.max(np.abs(d["el"] - o["e_local"]) / np.maximum(1.0, np.abs(o["e_local"]))) <= E_TOL


@pytest.mark.parametrize("side", [1e-60, 1e-130, 1e-200])
def test_local_energy_outside_the_fast_roots(side):
    # an electron that stays within 1e-60 (inside the fast roots' range), 1e-130
    # (a square below it) or 1e-200 (a square that underflows: r = 0, E_L
    # infinite or NaN) of its nucleus: the electron is evaluated in full
    system = S.atom(4)
    W, steps, B = 20, 4, 2
    cfg = np.random.default_rng(2).normal(size=(W, 12))
    cfg[:, :3] = 0.0
    with M.Context([M.slater_jastrow(system, W)], seed=3, step=side, block_size=B, flags=M.FLAG_TRACE,
                   record_sweeps=steps, lu_period=64) as ctx:
        ctx.set_configs(cfg)
        ctx.set_stream(0, 12)
        ctx.run(steps)
        masks, el = ctx.trace(steps, steps - B)
        got = ctx.get_configs()
    o = SJ.run(SJ.SjWave(system), seed=3, walkers=W, steps=steps, block_size=B, box_side=side, lu_period=64, cfg=cfg,
               pos0=12)
    assert np.array_equal(masks, o["accept_mask"]) and np.array_equal(bits(got), bits(o["cfg"]))
    want = o["e_local"].reshape(el.shape)
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(el), fin) and np.array_equal(np.isnan(el), np.isnan(want))
    assert np.all(np.abs(el[fin] - want[fin]) <= E_TOL * np.maximum(1.0, np.abs(want[fin])))


@pytest.mark.parametrize("precision", [M.PREC_MIXED, M.PREC_FP64])
def test_absent_walkers_cost_a_wave_nothing(precision):
    # one workgroup with one of its 4 walkers present against the same with all
    # of them: fewer walkers never make a wave's sampled sweeps longer.  With a
    # basis of 64 functions on 16 lanes the local energy (a lane per electron) is
    # most of a sweep, and evaluating it a second time for the empty slots makes
    # it a fifth longer.
    system = S.hydrogen_chain(2, basis_per_nucleus=32, seed=2)
    ctxs = []
    for W in (1, 4):
        c = M.Context([M.slater_jastrow(system, W)], seed=1, step=0.6, block_size=10, precision=precision, lu_period=64)
        c.set_walker_lanes(16)
        c.init_walkers()
        ctxs.append(c)
    best = [np.inf, np.inf]
    for _ in range(12):
        for k, c in enumerate(ctxs):
            c.sweep(20, sample=True)
            c.synchronize()
            best[k] = min(best[k], c.last_timing()[0])
    for c in ctxs:
        c.close()
    print(f"absent walkers: {best}", flush=True)
    assert best[0] <= 1.08 * best[1], best
