"""The HIP path against the CPU oracle on seeded synthetic events (runs on an MI355X)."""
import numpy as np
import pytest

import oracle
from allen_amd import synth, velo
from tests import parity

pytestmark = pytest.mark.gpu

# Small, seeded datasets that the oracle finishes in seconds.
DATASETS = {
    "single_pv": dict(n_events=30, pileup=0, mean_tracks=120.0, seed=11),
    "pileup": dict(n_events=120, pileup=1, nu=7.6, seed=12),
    "shuffled_backward": dict(n_events=30, pileup=0, mean_tracks=150.0, backward_fraction=0.3, shuffle_sp=1,
                              seed=13),
    "v2_banks": dict(n_events=20, pileup=0, mean_tracks=100.0, bank_version=2, seed=14),
    "empty_events": dict(n_events=6, pileup=0, mean_tracks=0.0, noise_fraction=0.0, seed=15),
    "stress": dict(n_events=12, pileup=1, nu=15.0, noise_fraction=0.05, dead_asic_fraction=0.01, seed=16),
    # The same kind of events in the MEP layout (MEPTools.h:59-200), super pixels and retina clusters.
    "mep_pileup": dict(n_events=40, pileup=1, nu=7.6, seed=18),
    "mep_v2_banks": dict(n_events=20, pileup=0, mean_tracks=100.0, bank_version=2, seed=19),
    "mep_retina_v3": dict(n_events=30, pileup=1, nu=7.6, retina=1, bank_version=3, seed=20),
}


@pytest.fixture(scope="module")
def constants(geometry, beamline):
    c = velo.VeloConstants(geometry, beamline)
    yield c
    c.close()


def run_both(name, geometry, beamline, constants, fused, tuning=None, oracle_props=None, events=None):
    ev = events if events is not None else synth.generate(**DATASETS[name])
    if name.startswith("mep_"):
        ev = synth.to_mep(ev)
    print(f"[parity] dataset={name} events={ev.n_events} raw_bytes={ev.raw.size} fused={fused} tuning={tuning}",
          flush=True)
    ref = oracle.run(ev, geometry, beamline, **(oracle_props or {}))
    dev = velo.DeviceEvents(ev)
    seq = velo.VeloSequence(constants, ev.n_events, max(ev.raw.size, 4096))
    seq.set_tuning("fused_clustering", int(fused))
    for k, v in (tuning or {}).items():
        seq.set_tuning(k, v)
    seq.run(dev)
    status = seq.status()
    gpu = parity.gpu_buffers(seq, ref)
    seq.close()
    return ref, gpu, status


@pytest.mark.parametrize("fused", [True, False], ids=["fused", "per_algorithm"])
@pytest.mark.parametrize("name", list(DATASETS))
def test_sequence_matches_oracle(name, fused, geometry, beamline, constants):
    ref, gpu, status = run_both(name, geometry, beamline, constants, fused)
    assert int(ref["status"][0]) == 0, "the oracle flags a capacity overflow; pick a smaller dataset"
    assert status & velo.STATUS_OVERFLOW_MASK == 0
    errs = parity.compare(gpu, ref, fused)
    assert not errs, "\n".join(errs[:20])
    if name != "empty_events":
        assert ref["offsets_all_velo_tracks"][-1] > 0


@pytest.mark.parametrize("fused", [True, False], ids=["fused", "per_algorithm"])
def test_real_sp_banks_match_oracle(fused, geometry, beamline, constants):
    """The reference's bundled MDF file's real super-pixel banks (10 minimum-bias events, bank
    version 2, 208 banks per event): pixel maps of real data, with clusters at the edges of the
    masked window and larger than it, through the whole HIP path against the oracle."""
    import os
    from tests import textbook
    ev = textbook.load_mdf_fixture(os.path.join(os.path.dirname(__file__), "golden", "mdf_minbias_vp.npz"))
    assert ev.bank_version == 2 and ev.n_events == 10
    ref, gpu, status = run_both("mdf_minbias_vp", geometry, beamline, constants, fused, events=ev)
    assert int(ref["status"][0]) == 0
    assert status & velo.STATUS_OVERFLOW_MASK == 0
    errs = parity.compare(gpu, ref, fused)
    assert not errs, "\n".join(errs[:20])
    # The same real banks in the MEP layout.
    ref, gpu, status = run_both("mep_mdf_minbias_vp", geometry, beamline, constants, fused, events=ev)
    assert int(ref["status"][0]) == 0
    assert status & velo.STATUS_OVERFLOW_MASK == 0
    errs = parity.compare(gpu, ref, fused)
    assert not errs, "\n".join(errs[:20])
    assert ref["module_cluster_num"].sum() > 15000 and ref["offsets_all_velo_tracks"][-1] > 1000


def test_batched_persistent_graph_replays(geometry, beamline, constants):
    """The batched workload's event mix (one vertex with Poisson(120) tracks, 5 % of the events at
    nu = 20 pile-up) through the persistent work-stealing search, the whole sequence captured as
    one HIP graph and replayed three times with eager runs of other events in between: every
    replay equals the oracle bit for bit."""
    import torch
    cfg = dict(n_events=400, pileup=0, mean_tracks=120.0, high_occupancy_fraction=0.05, high_nu=20.0, seed=23)
    ev = synth.generate(**cfg)
    other = synth.generate(**dict(cfg, n_events=100, seed=24))
    print(f"[batched-graph] events={ev.n_events} raw_bytes={ev.raw.size}", flush=True)
    ref = oracle.run(ev, geometry, beamline)
    assert int(ref["status"][0]) == 0
    dev, dev_other = velo.DeviceEvents(ev), velo.DeviceEvents(other)
    seq = velo.VeloSequence(constants, ev.n_events, max(ev.raw.size, other.raw.size))
    seq.set_tuning("search_persistent", 1)
    stream = torch.cuda.Stream()
    seq.capture(dev, stream)
    stream.synchronize()
    for replay in range(3):
        seq.run(dev_other)
        torch.cuda.synchronize()
        seq.replay(stream)
        stream.synchronize()
        assert seq.status() & velo.STATUS_OVERFLOW_MASK == 0
        errs = parity.compare(parity.gpu_buffers(seq, ref), ref, True)
        assert not errs, f"replay {replay}:\n" + "\n".join(errs[:20])
    seq.close()


def test_batched_mix_graph_replays(geometry, beamline, constants):
    """The batched workload's event mix (one vertex with Poisson(120) tracks, 5 % of the events at
    nu = 20 pile-up; events of up to ~5000 hits take the mixed LDS layout) through the whole
    sequence captured as one HIP graph, as bench.py --graph runs it (one workgroup per event), and
    replayed three times with eager runs of other events in between: every replay equals the
    oracle bit for bit."""
    import torch
    cfg = dict(n_events=400, pileup=0, mean_tracks=120.0, high_occupancy_fraction=0.05, high_nu=20.0, seed=23)
    ev = synth.generate(**cfg)
    other = synth.generate(**dict(cfg, n_events=100, seed=24))
    print(f"[batched-graph] events={ev.n_events} raw_bytes={ev.raw.size}", flush=True)
    ref = oracle.run(ev, geometry, beamline)
    assert int(ref["status"][0]) == 0
    dev, dev_other = velo.DeviceEvents(ev), velo.DeviceEvents(other)
    seq = velo.VeloSequence(constants, ev.n_events, max(ev.raw.size, other.raw.size))
    seq.run(dev)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    seq.capture(dev, stream)
    stream.synchronize()
    for replay in range(3):
        seq.run(dev_other)
        torch.cuda.synchronize()
        seq.replay(stream)
        stream.synchronize()
        assert seq.status() & velo.STATUS_OVERFLOW_MASK == 0
        errs = parity.compare(parity.gpu_buffers(seq, ref), ref, True)
        assert not errs, f"replay {replay}:\n" + "\n".join(errs[:20])
    seq.close()


TUNINGS = {
    "block64": {"search_block": 64},
    "block1024": {"search_block": 1024, "search_lds_hits": 2048},
    "many_lds_hits": {"search_block": 256, "search_lds_hits": 4096},  # the ring's window gives way to them
    "mixed_lds": {"search_block": 256, "search_lds_hits": 600},   # phi + used in LDS, xyz global
    "global_hits": {"search_block": 128, "search_lds_hits": 64},  # everything in global memory
    "event_order": {"search_largest_first": 0},                   # events in their own order
    "persistent": {"search_persistent": 1},                       # resident grid, work stealing
    "persistent_block64": {"search_persistent": 1, "search_block": 64, "search_largest_first": 0},
    "clustering_resident": {"clustering_resident_grid": 1},       # clustering waves loop over items
    "split": {"search_split": 32},                                # largest 1/32 of the events on a second stream
    # the smallest LDS window of the ring and list of unused hits: forwarding reads the ring back
    # from HBM and seeding walks the pendulum in module pairs of more than 64 hits
    "small_window_list": {"search_ring_window": 64, "search_list_cap": 64},
    # half the events in the side stream's launch, small workgroups and LDS there (mixed layout)
    "split_half": {"search_split": 2, "search_big_block": 128, "search_big_lds_hits": 600},
    # consolidation and fit read every event's hits from memory (events beyond 1920 hits always do)
    "consolidate_search": {"consolidate_lds_map": 0},
}


@pytest.mark.parametrize("tuning", list(TUNINGS))
def test_sequence_tuning_variants(tuning, geometry, beamline, constants):
    """Launch geometries and LDS layouts do not change a single bit of the result."""
    ref, gpu, status = run_both("pileup", geometry, beamline, constants, True, TUNINGS[tuning])
    assert status & velo.STATUS_OVERFLOW_MASK == 0
    errs = parity.compare(gpu, ref, True)
    assert not errs, "\n".join(errs[:20])


def test_kalman_fp64_covariance_fallback(geometry, beamline, constants):
    """With the FP64 covariance fallback on, the GPU states and covariances equal the oracle's
    fallback bit for bit (same FP64 operations, no contraction on either side)."""
    ref, gpu, status = run_both("pileup", geometry, beamline, constants, True, {"kalman_fp64_fallback": 1},
                                {"kalman_fp64_fallback": 1})
    assert status & velo.STATUS_OVERFLOW_MASK == 0
    errs = parity.compare(gpu, ref, True)
    assert not errs, "\n".join(errs[:20])


def _normalised_cov_error(c32, c64):
    """|c32 - c64| per stored term; diagonal terms relative, off-diagonal ones over sqrt(c_ii c_jj)."""
    pairs = [(0, 0), (0, 2), (2, 2), (3, 3), (3, 5), (5, 5)]
    e = np.empty_like(c64)
    for k, (i, j) in enumerate(pairs):
        e[:, k] = np.abs(c32[:, k] - c64[:, k]) / np.sqrt(np.abs(c64[:, i] * c64[:, j]))
    return e


def test_stress_kalman_against_fp64(geometry, beamline, constants):
    """High-occupancy events (nu = 15, 5 % noise pixels, 1 % dead ASICs). The GPU fit equals the
    oracle's bit for bit without and with the FP64 covariance fallback. Against the FP64
    restatement of the fit, the FP32 covariance of the plain fit is off by percents on
    ill-conditioned steps (three-hit tracks included); with the fallback every track's covariance
    is within FP32 storage precision, and the states within 2e-4 mm and 1e-6 in slope."""
    cfg = dict(n_events=40, pileup=1, nu=15.0, noise_fraction=0.05, dead_asic_fraction=0.01, seed=17)
    ev = synth.generate(**cfg)
    print(f"[stress-kalman] events={ev.n_events} raw_bytes={ev.raw.size}", flush=True)
    dev = velo.DeviceEvents(ev)
    out = {}
    for fb in (0, 1):
        ref = oracle.run(ev, geometry, beamline, kalman_fp64_fallback=fb)
        seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
        seq.set_tuning("kalman_fp64_fallback", fb)
        seq.run(dev)
        assert seq.status() & velo.STATUS_OVERFLOW_MASK == 0
        gpu = parity.gpu_buffers(seq, ref)
        seq.close()
        errs = parity.compare(gpu, ref, True)
        assert not errs, "\n".join(errs[:20])
        out[fb] = ref
    ref = out[1]
    n = int(ref["offsets_all_velo_tracks"][-1])
    hits = np.diff(ref["offsets_velo_track_hit_number"][:n + 1].astype(np.int64))
    three = hits == 3
    assert n > 5000 and three.sum() > 50
    for name in ["velo_kalman_beamline_states", "velo_kalman_endvelo_states"]:
        f64 = ref[name + "_f64"][:14 * n]
        c64 = f64[6 * n:].reshape(-1, 8)[:, :6]
        s64 = f64[:6 * n].reshape(-1, 6)[:, :5]
        e = {fb: _normalised_cov_error(out[fb][name][6 * n:14 * n].reshape(-1, 8)[:, :6].astype(np.float64), c64)
             for fb in (0, 1)}
        d = np.abs(out[1][name][:6 * n].reshape(-1, 6)[:, :5].astype(np.float64) - s64)
        print(f"[stress-kalman] {name}: {n} tracks ({three.sum()} three-hit); covariance error vs FP64 "
              f"plain q99 {np.quantile(e[0], 0.99):.3g} max {e[0].max():.3g} (three-hit max {e[0][three].max():.3g}); "
              f"fallback max {e[1].max():.3g} (three-hit {e[1][three].max():.3g}); state error with fallback: "
              f"x,y {d[:, :2].max():.3g} mm, slopes {d[:, 3:].max():.3g}", flush=True)
        assert e[1].max() < 1e-5
        assert e[0][three].max() > 1e-3 > e[1][three].max()
        assert d[:, 3:].max() < 1e-6 and d[:, :2].max() < 2e-4


def test_captured_sequence_replays(geometry, beamline, constants):
    """The whole sequence captured as one HIP graph: three replays, with an eager run on other
    events in between (which overwrites the buffers), each reproduce the eager result and the
    oracle bit for bit."""
    import torch
    ev = synth.generate(**DATASETS["pileup"])
    other = synth.generate(**dict(DATASETS["pileup"], n_events=40, seed=99))
    print(f"[graph] events={ev.n_events} other={other.n_events}", flush=True)
    ref = oracle.run(ev, geometry, beamline)
    dev, dev_other = velo.DeviceEvents(ev), velo.DeviceEvents(other)
    seq = velo.VeloSequence(constants, ev.n_events, max(ev.raw.size, other.raw.size))
    seq.run(dev)
    torch.cuda.synchronize()
    eager = parity.gpu_buffers(seq, ref)
    stream = torch.cuda.Stream()
    seq.capture(dev, stream)
    stream.synchronize()
    for replay in range(3):
        seq.run(dev_other)
        torch.cuda.synchronize()
        seq.replay(stream)
        stream.synchronize()
        got = parity.gpu_buffers(seq, ref)
        # Same rules as the oracle comparison: filled slots only (gap contents are unspecified and
        # keep what the run on the other events left there).
        errs = parity.compare(got, eager, True)
        assert not errs, f"replay {replay} against the eager run:\n" + "\n".join(errs[:20])
        errs = parity.compare(got, ref, True)
        assert not errs, f"replay {replay} against the oracle:\n" + "\n".join(errs[:20])
    assert seq.status() & velo.STATUS_OVERFLOW_MASK == 0
    seq.close()


def test_times_of_the_stages_that_share_a_launch(geometry, beamline, constants):
    """The time of the three-hit filter is that of the search's launch, and the fit's that of the
    consolidation's, which hold them."""
    ev = synth.generate(n_events=400, pileup=1, nu=12.0, seed=25)
    dev = velo.DeviceEvents(ev)
    seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
    seq.run(dev)
    ms = {}
    for stage in velo.STAGES:
        if stage == "pv":
            continue
        seq.time_stage(stage)
        for _ in range(5):
            seq.run(dev)
        total, runs = seq.stage_ms()
        assert runs == 5
        ms[stage] = total
    seq.time_stage(None)
    seq.close()
    for part, whole in (("three_hit_filter", "search"), ("kalman", "consolidate")):
        assert 0.5 * ms[whole] < ms[part] < 2.0 * ms[whole]
    assert all(0.0 < v < 1.2 * ms["all"] for v in ms.values())


def test_autotune_keeps_outputs(geometry, beamline, constants):
    """A reduced autotuner sweep: every candidate reproduces the default outputs (the tuner raises
    otherwise), what they are compared with is the library's default, and the chosen knobs are applied
    to the sequence."""
    from allen_amd import autotune
    ev = synth.generate(**DATASETS["pileup"])
    dev = velo.DeviceEvents(ev)
    seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
    first = []
    set_tuning = seq.set_tuning
    seq.set_tuning = lambda k, v: (first.append((k, v)), set_tuning(k, v))
    none = autotune.tune(seq, dev, reps=3, blocks=())
    assert none.trials == [] and none.knobs == autotune.default_knobs()
    assert all((k, 0) in first for k in ("search_block", "search_lds_hits", "search_ring_window", "search_list_cap"))
    assert not any(k == "search_block" and v for k, v in first)  # the time compared with is the library's own
    res = autotune.tune(seq, dev, reps=1, blocks=(64, 256), lds_hits=(512, 1760))
    assert len(res.trials) == 16 and res.search_ms <= res.default_search_ms
    assert res.knobs["search_block"] in (0, 64, 256)
    seq.run(dev)
    ref = oracle.run(ev, geometry, beamline)
    errs = parity.compare(parity.gpu_buffers(seq, ref), ref, True)
    assert not errs, "\n".join(errs[:20])
    seq.close()


def test_throughput_autotune_on_two_streams(geometry, beamline, constants):
    """The throughput tuner over two sequences on two streams: every candidate keeps the outputs,
    the winner is applied to both, and both then reproduce the oracle."""
    import torch
    from allen_amd import autotune
    ev = synth.generate(**DATASETS["pileup"])
    print(f"[autotune-throughput] events={ev.n_events}", flush=True)
    dev = velo.DeviceEvents(ev)
    seqs = [velo.VeloSequence(constants, ev.n_events, ev.raw.size) for _ in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]

    def measure():
        torch.cuda.synchronize()
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        main = torch.cuda.current_stream()
        start.record(main)
        for st in streams:
            st.wait_event(start)
        for i in range(4):
            seqs[i % 2].run(dev, stream=streams[i % 2])
        for st in streams:
            main.wait_stream(st)
        end.record(main)
        torch.cuda.synchronize()
        return start.elapsed_time(end) / 4

    cands = ({"search_block": 128, "search_lds_hits": 512}, {"search_block": 192, "search_lds_hits": 800})
    res = autotune.tune_throughput(seqs, measure, ev.n_events, candidates=cands)
    assert len(res.trials) == 2 and res.search_ms <= res.default_search_ms
    ref = oracle.run(ev, geometry, beamline)
    for sq, st in zip(seqs, streams):
        sq.run(dev, stream=st)
        torch.cuda.synchronize()
        errs = parity.compare(parity.gpu_buffers(sq, ref), ref, True)
        assert not errs, "\n".join(errs[:20])
        sq.close()


def test_dense_module_pairs_take_the_tiled_paths(geometry, beamline, constants):
    """Events dense enough that module pairs exceed the per-wave LDS slices of clustering."""
    DATASETS["dense"] = dict(n_events=4, pileup=1, nu=60.0, noise_fraction=0.3, seed=17)
    ref, gpu, status = run_both("dense", geometry, beamline, constants, True)
    est = ref["offsets_estimated_input_size"]
    assert np.diff(est).max() > 320  # some module pair is above the cluster slice
    if int(ref["status"][0]) == 0:
        errs = parity.compare(gpu, ref, True)
        assert not errs, "\n".join(errs[:20])
    else:  # capacity overflow in the search: compare the clustering stages only
        errs = [e for e in parity.compare(gpu, ref, True) if e.split(":")[0].startswith(("sorted", "module_cluster",
                                                                                          "estimated", "offsets_est"))]
        assert not errs, "\n".join(errs[:20])


@pytest.mark.parametrize("fused", [True, False], ids=["fused", "per_algorithm"])
@pytest.mark.parametrize("version", [2, 4])
@pytest.mark.parametrize("nu,lowest", [(16.0, 193), (30.0, 440), (45.0, 513)])
def test_module_pairs_at_the_limits_of_the_clustering_slices(nu, lowest, version, fused, geometry, beamline, constants):
    """Module pairs on both sides of each limit of the per-wave slices (192 clusters placed there, 256
    non-isolated words, 512 clusters ranked there) and, per algorithm, banks of more than 64 words:
    integers and bytes equal the oracle's."""
    ev = synth.generate(n_events=3, pileup=1, nu=nu, shuffle_sp=1, bank_version=version, seed=41)
    ref, gpu, status = run_both(f"slices_nu{nu}_v{version}", geometry, beamline, constants, fused, events=ev)
    assert int(ref["status"][0]) == 0 and status & velo.STATUS_OVERFLOW_MASK == 0
    assert np.diff(ref["offsets_estimated_input_size"].astype(np.int64)).max() >= lowest
    errs = parity.compare(gpu, ref, fused)
    assert not errs, "\n".join(errs[:20])


@pytest.mark.parametrize("n_events,bytes_per_event", [(513, 0), (1025, 0), (4097, 0), (6145, 0), (513, 15000),
                                                      (513, 32000), (1025, 32000)])
def test_search_launch_shapes_by_number_of_events(n_events, bytes_per_event, geometry, beamline, constants):
    """The smallest numbers of events that take the other shapes of the search's launch than the first, and
    the shapes of crowded slices (the raw bytes are what the host knows of the events' size, and a
    slice may state more than it fills). With the shape's own hits in LDS, and with 256, where the
    events take every layout: equal to the oracle."""
    ev = synth.generate(n_events=n_events, pileup=0, mean_tracks=12.0, high_occupancy_fraction=0.02, high_nu=14.0, seed=43)
    ref = oracle.run(ev, geometry, beamline)
    assert int(ref["status"][0]) == 0
    hits = np.diff(ref["offsets_estimated_input_size"].astype(np.int64)[::26])
    assert hits.min() < 256 and hits.max() > 2048 and np.any((hits > 256) & (hits < 16 * 256 // 3))
    stated = max(ev.raw.size, bytes_per_event * n_events)
    seq = velo.VeloSequence(constants, n_events, stated)
    dev = velo.DeviceEvents(ev)
    for lds_hits in (0, 256):
        seq.set_tuning("search_lds_hits", lds_hits)
        seq.run(dev, raw_input_bytes=stated)
        assert seq.status() & velo.STATUS_OVERFLOW_MASK == 0
        errs = parity.compare(parity.gpu_buffers(seq, ref), ref, True)
        assert not errs, f"search_lds_hits {lds_hits}:\n" + "\n".join(errs[:20])
    seq.close()


@pytest.mark.parametrize("n_events,bytes_per_event", [(513, 0), (2049, 0), (2049, 15000)])
def test_masked_clustering_workgroups_by_number_of_events(n_events, bytes_per_event, geometry, beamline, constants):
    """The smallest numbers of events that take the masked clustering's smaller workgroups, and the larger
    of these for crowded slices (by the slice's stated bytes), algorithm by algorithm: the clusters of
    every module pair are the oracle's."""
    ev = synth.generate(n_events=n_events, pileup=0, mean_tracks=3.0, high_occupancy_fraction=0.005, high_nu=30.0, seed=50)
    ref = oracle.run(ev, geometry, beamline, compute_f64=0)
    stated = max(ev.raw.size, bytes_per_event * n_events)
    seq = velo.VeloSequence(constants, n_events, stated)
    seq.set_tuning("fused_clustering", 0)
    seq.run(velo.DeviceEvents(ev), raw_input_bytes=stated)
    assert seq.status() & velo.STATUS_OVERFLOW_MASK == int(ref["status"][0]) == 0
    errs = parity.compare(parity.gpu_buffers(seq, ref), ref, False)
    seq.close()
    assert not errs, "\n".join(errs[:20])


@pytest.mark.parametrize("lds_hits,list_cap", [(256, 64), (64, 64), (16, 64), (64, 512), (0, 0)])
def test_unused_hit_lists_in_the_lds_of_the_hits(lds_hits, list_cap, geometry, beamline, constants):
    """Events that are searched in memory keep the lists of unused hits where the hits would be, four
    entries of both lists a hit and at most 1024, if that is more than list_cap; module pairs beyond
    take the walk. Module pairs on both sides of 256 and of 512 hits and beyond: equal to the oracle."""
    ev = synth.generate(n_events=3, pileup=1, nu=70.0, seed=49)
    ref = oracle.run(ev, geometry, beamline)
    pairs = np.diff(ref["offsets_estimated_input_size"].astype(np.int64))
    assert int(ref["status"][0]) == 0 and pairs.max() > 512 and np.any((pairs > 64) & (pairs < 256))
    seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
    seq.set_tuning("search_lds_hits", lds_hits)
    seq.set_tuning("search_list_cap", list_cap)
    seq.run(velo.DeviceEvents(ev))
    errs = parity.compare(parity.gpu_buffers(seq, ref), ref, True)
    seq.close()
    assert not errs, "\n".join(errs[:20])


@pytest.mark.parametrize("phi_tolerance", [-0.01, 0.0, 0.2, 0.79, 2.0])
def test_search_windows_of_other_tolerances(phi_tolerance, geometry, beamline, constants):
    """Windows that are empty, that end a module pair's phis on both sides, and that are wider than what
    the phi buckets serve (8192 units, 0.786 rad): the same tracks as the oracle's."""
    ev = synth.generate(n_events=6, pileup=1, nu=7.6, seed=44)
    ref = oracle.run(ev, geometry, beamline, phi_tolerance=phi_tolerance)
    seq = velo.VeloSequence(constants, ev.n_events, max(ev.raw.size, 4096))
    seq.run(velo.DeviceEvents(ev), phi_tolerance=phi_tolerance)
    errs = parity.compare(parity.gpu_buffers(seq, ref), ref, True)
    seq.close()
    assert not errs, "\n".join(errs[:20])


@pytest.mark.parametrize("seed,phi_tolerance", [(13, 0.25), (42, 0.5), (47, 0.7), (117, 0.25)])
def test_search_walk_goes_on_through_opposite_hits(seed, phi_tolerance, geometry, beamline, constants):
    """Sparse noisy events and a scatter limit that any hit meets: the 16-bit |difference| takes a hit
    exactly opposite for one within the tolerance, so the walk goes on through it where it is the
    next one after the hits of the window. It decides a seed or an extension in each of these
    slices (rarely: one event in some ten thousand). The oracle's tracks, in every layout of the hits."""
    ev = synth.generate(n_events=1000, pileup=0, mean_tracks=3.0, noise_fraction=4.0, seed=seed)
    ref = oracle.run(ev, geometry, beamline, phi_tolerance=phi_tolerance, max_scatter=1e6)
    assert int(ref["status"][0]) == 0
    hits = np.diff(ref["offsets_estimated_input_size"].astype(np.int64)[::26])
    assert 64 < np.median(hits) < 16 * 64 // 3
    seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
    dev = velo.DeviceEvents(ev)
    for lds_hits in (0, 64, 1):  # in LDS; mostly phi and flags in LDS; from memory
        seq.set_tuning("search_lds_hits", lds_hits)
        seq.run(dev, phi_tolerance=phi_tolerance, max_scatter=1e6)
        errs = parity.compare(parity.gpu_buffers(seq, ref), ref, True)
        assert not errs, f"search_lds_hits {lds_hits}:\n" + "\n".join(errs[:20])
    seq.close()


@pytest.mark.parametrize("tuning", [{}, {"search_lds_hits": 1}, {"search_ring_window": 64}], ids=["lds", "memory", "ring"])
@pytest.mark.parametrize("max_skipped_modules", [0, 7, 8, 25])
def test_search_limits_of_skipped_modules(max_skipped_modules, tuning, geometry, beamline, constants, monkeypatch):
    """The skipped modules of an entry have three bits. Up to 7 the limit is exact, beyond it there is
    none: the rules with a field that holds any number (entries that skip 8 modules are common: tracks
    that end downstream)."""
    from tests import textbook, textbook_search as ts
    monkeypatch.setattr(ts, "SKIP_MASK", 0xFF << ts.SKIP_SHIFT)
    monkeypatch.setattr(ts, "SEED_BIT", 1 << 40)
    ev = synth.generate(n_events=5, pileup=0, mean_tracks=60.0, seed=48)
    ref = oracle.run(ev, geometry, beamline, compute_f64=0)
    zs = textbook.parse_geometry(geometry)["module_zs"]
    offsets, counts = ref["offsets_estimated_input_size"], ref["module_cluster_num"]
    seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
    for k, v in tuning.items():
        seq.set_tuning(k, v)
    seq.run(velo.DeviceEvents(ev), max_skipped_modules=max_skipped_modules)
    gpu = parity.gpu_buffers(seq, ref)
    tracks = seq.fetch("tracks", parity.TRACK, ref["tracks"].size)
    seq.close()
    for e in range(ev.n_events):
        want = ts.search(ts.event_from_container(ref["sorted_velo_cluster_container"], offsets, counts, e, zs),
                         max_skipped_modules=max_skipped_modules if max_skipped_modules <= 7 else 26)
        toff = int(np.float32(offsets[26 * e]) * np.float32(0.34))
        n, (n3, ttf) = int(gpu["number_of_velo_tracks"][e]), (int(v) for v in gpu["atomics_velo"][3 * e:3 * e + 2])
        assert [t["hits"][:t["hitsNum"]].tolist() for t in tracks[toff:toff + n]] == want["tracks"]
        assert gpu["three_hit_tracks"]["hits"][toff:toff + n3].tolist() == want["three_hit"]
        assert ttf == want["ttf"]
        h0, h1 = int(offsets[26 * e]), int(offsets[26 * (e + 1)])
        np.testing.assert_array_equal(gpu["hit_used"][h0:h1], want["used"])


def test_hit_offsets_of_an_event_that_overflows_the_ring(geometry, beamline, constants):
    """Events whose tracks to follow overflow the ring raise the status bit and have no specified tracks,
    but the offsets of the track hits still are the sums of the tracks' hit numbers, and the
    other events' tracks are the oracle's."""
    ev = synth.generate(n_events=6, pileup=0, mean_tracks=120.0, high_occupancy_fraction=0.4, high_nu=300.0, seed=47)
    ref = oracle.run(ev, geometry, beamline, compute_f64=0, max_skipped_modules=2)
    hits = np.diff(ref["offsets_estimated_input_size"].astype(np.int64)[::26])
    assert int(ref["status"][0]) == 1 and hits.min() < 3000 and 30000 < hits.max() < 65536
    seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
    seq.run(velo.DeviceEvents(ev), max_skipped_modules=2)
    assert seq.status() & velo.STATUS_OVERFLOW_MASK == 1
    off = seq.fetch("offsets_all_velo_tracks", np.uint32, ev.n_events + 1).astype(np.int64)
    hit_number = seq.fetch("velo_track_hit_number", np.uint32, int(off[-1]))
    hit_off = seq.fetch("offsets_velo_track_hit_number", np.uint32, int(off[-1]) + 1).astype(np.int64)
    ids = seq.fetch("velo_track_hits", np.uint32, int(hit_off[-1]))
    seq.close()
    np.testing.assert_array_equal(np.diff(hit_off), hit_number)
    assert np.all((hit_number >= 3) & (hit_number <= 26))
    ref_off, ref_hit_off = (ref[k].astype(np.int64) for k in ("offsets_all_velo_tracks", "offsets_velo_track_hit_number"))
    ref_ids = ref["velo_track_hits"][:4 * int(ref_hit_off[-1])].view("<u4")
    for e in np.nonzero(hits < 20000)[0]:
        a, b = (slice(o[e], o[e + 1] + 1) for o in (off, ref_off))
        np.testing.assert_array_equal(np.diff(hit_off[a]), np.diff(ref_hit_off[b]))
        np.testing.assert_array_equal(ids[hit_off[a][0]:hit_off[a][-1]], ref_ids[ref_hit_off[b][0]:ref_hit_off[b][-1]])


def test_prefix_sum_iota(constants):
    """The reference's own prefix-sum test shape (TestPrefixSum.cu:9-33): iota 1..1000."""
    import torch
    x = torch.arange(1, 1001, dtype=torch.int32, device="cuda")
    out = torch.empty(1001, dtype=torch.int32, device="cuda")
    total = velo.prefix_sum(x, 1000, out, want_total=True)
    expect = np.concatenate([[0], np.cumsum(np.arange(1, 1001))])
    assert total == expect[-1]
    np.testing.assert_array_equal(out.cpu().numpy(), expect)


@pytest.mark.parametrize("n", [0, 1, 4095, 4096, 4097, 26 * 1000, 32768, 32769, 26 * 20000 + 3])
def test_prefix_sum_sizes(n, constants):
    import torch
    rng = np.random.default_rng(n)
    host = rng.integers(0, 1 << 20, size=n, dtype=np.int64).astype(np.uint32)
    x = torch.from_numpy(host.view(np.int32)).cuda()
    out = torch.full((n + 1,), -1, dtype=torch.int32, device="cuda")
    total = velo.prefix_sum(x, n, out, want_total=True)
    expect = np.zeros(n + 1, np.uint32)
    oracle.lib().vo_prefix_sum(host.ctypes.data, n, expect.ctypes.data)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), expect)
    assert total == int(expect[-1])


def test_constants_tables_match_oracle(constants):
    mine = constants.sp_tables()
    ref = oracle.sp_tables()
    for a, b in zip(mine, ref):
        np.testing.assert_array_equal(a, b)
