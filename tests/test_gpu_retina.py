"""Retina-cluster decoding on the GPU against the CPU oracle (runs on an MI355X)."""
import ctypes

import numpy as np
import pytest

import oracle
from allen_amd import synth, velo
from tests import parity, textbook

pytestmark = pytest.mark.gpu

DATASETS = {
    "v4_pileup": dict(n_events=60, pileup=1, nu=7.6, seed=51, retina=1, bank_version=4),
    "v3_single_pv": dict(n_events=30, pileup=0, mean_tracks=120.0, seed=52, retina=1, bank_version=3),
    "v4_shuffled_backward": dict(n_events=30, pileup=0, mean_tracks=150.0, backward_fraction=0.3, shuffle_sp=1,
                                 seed=53, retina=1, bank_version=4),
    "v4_stress": dict(n_events=12, pileup=1, nu=15.0, noise_fraction=0.05, dead_asic_fraction=0.01, seed=54,
                      retina=1, bank_version=4),
    "v4_empty": dict(n_events=6, pileup=0, mean_tracks=0.0, noise_fraction=0.0, seed=55, retina=1, bank_version=4),
}


@pytest.fixture(scope="module")
def constants(geometry, beamline):
    c = velo.VeloConstants(geometry, beamline)
    yield c
    c.close()


def _events(name):
    if name == "mdf_real_v3":
        import os
        ev = textbook.load_mdf_fixture(os.path.join(os.path.dirname(__file__), "golden", "mdf_minbias_retina.npz"))
        ev.retina = True
        return ev
    return synth.generate(**DATASETS[name])


@pytest.mark.parametrize("name", list(DATASETS) + ["mdf_real_v3"])
def test_retina_sequence_matches_oracle(name, geometry, beamline, constants):
    """The whole path from retina banks: decoding (sizes, offsets, keys, permutations, sorted
    container) and everything after it equal the oracle's bit for bit."""
    ev = _events(name)
    print(f"[retina] dataset={name} events={ev.n_events} version={ev.bank_version} raw_bytes={ev.raw.size}", flush=True)
    ref = oracle.run(ev, geometry, beamline)
    seq = velo.VeloSequence(constants, ev.n_events, max(ev.raw.size, 4096))
    seq.run(velo.DeviceEvents(ev))
    assert seq.status() & velo.STATUS_OVERFLOW_MASK == 0
    gpu = parity.gpu_buffers(seq, ref)
    seq.close()
    errs = parity.compare(gpu, ref, True)
    assert not errs, "\n".join(errs[:20])
    if name != "v4_empty":
        assert ref["offsets_all_velo_tracks"][-1] > 0


@pytest.mark.parametrize("version", [3, 4])
@pytest.mark.parametrize("nu", [60.0, 150.0])
def test_module_pairs_beyond_the_keys_kept_in_lds(nu, version, geometry, beamline, constants):
    """Module pairs of more than 512 words, which are ranked tile by tile, with words that are repeated
    within a tile and in another and with zero words: keys, ranks, counts and the cluster that
    every written slot holds equal the oracle's."""
    ev = synth.generate(n_events=3, pileup=1, nu=nu, seed=57, retina=1, bank_version=version)
    raw, s16 = ev.raw.copy(), ev.sizes.view("<u2")
    for e in range(ev.n_events):
        base = int(ev.offsets[e])
        nb = int(raw[base:base + 4].view("<u4")[0])
        boff = raw[base + 4:base + 8 + 4 * nb].view("<u4").astype(np.int64)
        for b in range(0, nb, 5):
            at = base + 8 + 4 * nb + int(boff[b]) + (8 if version == 3 else 4)
            words = raw[at:base + 8 + 4 * nb + int(boff[b + 1])].view("<u4") if b + 1 < nb else raw[:0].view("<u4")
            if words.size > 8:
                words[1], words[-2], words[-1] = words[0], words[2], 0
    ev = synth.dataclasses.replace(ev, raw=raw)
    ref = oracle.run(ev, geometry, beamline, compute_f64=0)
    est = ref["offsets_estimated_input_size"].astype(np.int64)
    assert np.diff(est).max() > (1024 if nu > 100 else 512) and np.diff(est).min() < 512
    seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
    seq.run(velo.DeviceEvents(ev))
    got = {k: seq.fetch(k, ref[k].dtype, ref[k].size) for k in
           ("offsets_estimated_input_size", "module_cluster_num", "hit_sorting_key", "hit_permutations")}
    container = seq.fetch("sorted_velo_cluster_container", np.uint8, 18 * int(est[-1]))
    seq.close()
    for k, v in got.items():
        np.testing.assert_array_equal(v, ref[k], err_msg=k)
    written = np.unique(ref["hit_permutations"])
    assert written.size < est[-1]  # equal keys share a slot
    for a, b in zip(parity.cluster_views(container, int(est[-1])),
                    parity.cluster_views(ref["sorted_velo_cluster_container"], int(est[-1]))):
        np.testing.assert_array_equal(a[written].view(np.uint8), b[written].view(np.uint8))


def test_retina_drop_in_entry_points(geometry, beamline, constants):
    """calculate_number_of_retinaclusters_each_sensor_pair and decode_retinaclusters called
    one by one through the C ABI, with an event list, equal the oracle."""
    import torch
    ev = _events("v4_pileup")
    print(f"[retina-abi] events={ev.n_events}", flush=True)
    ref = oracle.run(ev, geometry, beamline)
    dev = velo.DeviceEvents(ev)
    n = ev.n_events
    slots = velo.lib().velo_retina_sensor_slots(ev.bank_version)
    cuda = lambda k, dt=torch.int32: torch.zeros(k, dtype=dt, device="cuda")
    event_list = torch.arange(n, dtype=torch.int32, device="cuda")
    sizes, bank_index = cuda(n * slots), cuda(slots)
    p = velo.RetinaSizesParams()
    p.host_number_of_events, p.host_raw_bank_version = n, ev.bank_version
    p.dev_event_list, p.event_list_size = event_list.data_ptr(), n
    p.dev_velo_retina_raw_input, p.dev_velo_retina_raw_input_offsets = dev.raw.data_ptr(), dev.offsets.data_ptr()
    p.dev_velo_retina_raw_input_sizes, p.dev_velo_retina_raw_input_types = dev.sizes.data_ptr(), dev.types.data_ptr()
    p.dev_retina_bank_index, p.dev_each_sensor_pair_size = bank_index.data_ptr(), sizes.data_ptr()
    velo.check(velo.lib().velo_calculate_number_of_retinaclusters_each_sensor_pair(ctypes.byref(p), None), "sizes")
    offsets = cuda(n * slots + 1)
    total = velo.prefix_sum(sizes, n * slots, offsets, want_total=True)
    assert total == int(ref["offsets_each_sensor_pair_size"][-1])
    n_events_dev = torch.tensor([n], dtype=torch.int32, device="cuda")
    mcn, mp_off = cuda(26 * n), cuda(26 * n + 1)
    container, perm, keys = cuda(18 * total, torch.uint8), cuda(total), cuda(total, torch.int64)
    d = velo.RetinaDecodeParams()
    d.host_total_number_of_velo_clusters, d.host_raw_bank_version, d.host_number_of_events = total, ev.bank_version, n
    d.dev_velo_retina_raw_input, d.dev_velo_retina_raw_input_offsets = dev.raw.data_ptr(), dev.offsets.data_ptr()
    d.dev_velo_retina_raw_input_sizes, d.dev_velo_retina_raw_input_types = dev.sizes.data_ptr(), dev.types.data_ptr()
    d.dev_offsets_each_sensor_pair_size, d.dev_retina_bank_index = offsets.data_ptr(), bank_index.data_ptr()
    d.dev_event_list, d.event_list_size, d.dev_number_of_events = event_list.data_ptr(), n, n_events_dev.data_ptr()
    d.dev_module_cluster_num, d.dev_offsets_module_pair_cluster = mcn.data_ptr(), mp_off.data_ptr()
    d.dev_velo_cluster_container, d.dev_hit_permutations = container.data_ptr(), perm.data_ptr()
    d.dev_hit_sorting_key, d.constants = keys.data_ptr(), constants.handle
    velo.check(velo.lib().velo_decode_retinaclusters(ctypes.byref(d), None), "decode")
    torch.cuda.synchronize()
    host = lambda t, dt: t.cpu().numpy().view(dt)
    np.testing.assert_array_equal(host(sizes, np.uint32), ref["each_sensor_pair_size"])
    np.testing.assert_array_equal(host(bank_index, np.uint32), ref["retina_bank_index"])
    np.testing.assert_array_equal(host(mcn, np.uint32), ref["module_cluster_num"])
    np.testing.assert_array_equal(host(mp_off, np.uint32), ref["offsets_estimated_input_size"])
    np.testing.assert_array_equal(host(keys, np.int64), ref["hit_sorting_key"])
    np.testing.assert_array_equal(host(perm, np.uint32), ref["hit_permutations"])
    slots_f = parity.filled_slots(ref["offsets_estimated_input_size"], ref["module_cluster_num"])
    g = parity.cluster_views(host(container, np.uint8), total)
    r = parity.cluster_views(ref["sorted_velo_cluster_container"], total)
    for a, b in zip(g, r):
        np.testing.assert_array_equal(a[slots_f].view(np.uint8), b[slots_f].view(np.uint8))


def test_module_pair_out_of_order_is_searched_alike_in_every_layout(geometry, beamline):
    """Retina words of one pixel with different fractions share a sorting key, and the slot left over
    holds whatever was there: the module pair's phis are out of order. Every layout of the hits
    (LDS, mixed, global) and workgroup size gives the same tracks."""
    from allen_amd import synth, velo
    ev = synth.generate(n_events=2180, pileup=0, mean_tracks=120.0, retina=1, seed=101 * 64 + 1, keep_truth=False)
    constants = velo.VeloConstants(geometry, beamline)
    seq = velo.VeloSequence(constants, ev.n_events, ev.raw.size)
    dev = velo.DeviceEvents(ev)
    got = {}
    for name, knobs in {"default": {}, "one_wave": {"search_block": 64}, "mixed": {"search_block": 256, "search_lds_hits": 400},
                        "global": {"search_block": 128, "search_lds_hits": 64}}.items():
        for k in ("search_block", "search_lds_hits"):
            seq.set_tuning(k, knobs.get(k, 0))
        seq.run(dev)
        assert seq.status() & velo.STATUS_OVERFLOW_MASK == 0
        n = int(seq.fetch("offsets_all_velo_tracks", np.uint32, ev.n_events + 1)[-1])
        hits = int(seq.fetch("offsets_velo_track_hit_number", np.uint32, n + 1)[-1])
        got[name] = (seq.fetch("offsets_all_velo_tracks", np.uint32, ev.n_events + 1),
                     seq.fetch("velo_track_hits", np.uint8, 16 * hits))
    est = seq.fetch("offsets_estimated_input_size", np.uint32, 26 * ev.n_events + 1).astype(np.int64)
    key = seq.fetch("hit_sorting_key", np.int64, int(est[-1]))
    mp = np.repeat(np.arange(est.size - 1), np.diff(est))
    order = np.lexsort((key, mp))
    same = (np.diff(mp[order]) == 0) & (np.diff(key[order]) == 0) & (key[order][1:] != 0x7FFFFFFFFFFFFFFF)
    assert same.any(), "no two words of a module pair share a key: the events no longer hold the case"
    for name, (offsets, track_hits) in got.items():
        np.testing.assert_array_equal(offsets, got["default"][0], err_msg=name)
        np.testing.assert_array_equal(track_hits, got["default"][1], err_msg=name)
    seq.close()
    constants.close()
