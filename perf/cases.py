"""The work that a program built on this framework has it do, as cases that can be timed and compared.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program holds
before the call, run() is one pass through the public entry points, work() what the pass cannot do
without and exact() its outputs in 64 bits where plain arithmetic gives them.

Kinds of case:
  sequence  one slice of events through VeloSequence.run on one stream (super pixels or retina clusters)
  graph     the same run captured once and replayed
  streams   several slices, one VeloSequence each, dealt to a few streams (how throughput is measured)
  chain     the nine algorithms one by one (algorithms.velo_sp_sequence), as a host scheduler binds them
  train     one Adam step of the seed scorer on a batch of labelled seeds
  score     the scorer's logits of a set of seeds
Events come from the package's seeded generator with its real geometry.
"""
import numpy as np
import torch

from allen_amd import algorithms, scorer, synth, velo

# Tracks of an event from one primary vertex, and the tracks that a pile-up collision adds.
SINGLE_PV_TRACKS = 120.0
TRACKS_PER_COLLISION = 16.0
HITS_PER_TRACK = 9.0


def listed():
    return [
        # A handful of events, as a monitor or an event display asks for: launches and the latency
        # of one event's dependent steps.
        dict(name="monitor_8", kind="sequence", n_events=8, nu=7.6),
        # The small reference workload as a captured graph, for a program that replays fixed slices.
        dict(name="single_pv_200_graph", kind="graph", n_events=200, nu=0.0),
        # The benchmark's slice: 1000 pile-up events, eager, on one stream.
        dict(name="pileup_1000", kind="sequence", n_events=1000, nu=7.6),
        # The same occupancy as retina clusters, the production decoding.
        dict(name="retina_1000", kind="sequence", n_events=1000, nu=7.6, retina=True),
        # With the primary-vertex finder behind the fit, for a program that wants vertices.
        dict(name="vertices_1000", kind="sequence", n_events=1000, nu=7.6, vertices=True),
        # With the shipped seed scorer pruning ghosts, an odd slice of the one-vertex events it was trained for.
        dict(name="pruned_777", kind="sequence", n_events=777, nu=0.0, pruned=True),
        # Crowded, noisy events with dead ASICs and the FP64 covariance fallback.
        dict(name="stress_2000", kind="sequence", n_events=2000, nu=15.0, noise=0.05, dead=0.01, fp64=True),
        # The batched workload: one-vertex events with 5 % of high occupancy, the throughput regime.
        dict(name="batched_20000", kind="sequence", n_events=20000, nu=0.0, crowded=0.05),
        # Six slices in flight on three streams with the knobs that the throughput autotuner settles on.
        dict(name="slices_6x1000", kind="streams", n_events=1000, nu=7.6, slices=6, streams=3,
             search_block=128, search_lds_hits=800, search_ring_window=256, search_list_cap=256),
        # Algorithm by algorithm, sizes through the host, as the algorithms sit in a scheduler's sequence.
        dict(name="chain_500", kind="chain", n_events=500, nu=7.6),
        # The scorer's training step at the trainer's batch size.
        dict(name="train_65536", kind="train", rows=65536),
        # The scorer over the seeds of a few thousand events; the row count is nothing round.
        dict(name="score_240459", kind="score", rows=240459),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(float(lo) * (float(hi) / float(lo)) ** rng.random()))


def draw(rng):
    kind = rng.choice(["sequence"] * 6 + ["graph", "streams", "chain", "chain", "train", "score"])
    if kind in ("train", "score"):
        return dict(kind=kind, rows=_log_uniform(rng, 1000, 200000 if kind == "train" else 1000000))
    nu = rng.choice([0.0, 0.0, round(rng.uniform(2.0, 16.0), 2)])
    case = dict(kind=kind, nu=nu)
    if nu and rng.random() < 0.3:
        case.update(noise=0.05, dead=0.01)
    if kind == "streams":
        case.update(n_events=_log_uniform(rng, 50, 1000), slices=rng.randint(2, 6), streams=rng.randint(2, 3))
        return case
    if kind == "chain":
        case.update(n_events=_log_uniform(rng, 1, 1000), bank_version=rng.choice([2, 4]), mep=rng.random() < 0.3)
        return case
    case.update(n_events=_log_uniform(rng, 1, 3000))
    option = rng.choice(["", "", "retina", "vertices", "pruned", "fp64", "v2", "shuffled"])
    if option == "v2":
        case.update(bank_version=2)
    elif option == "shuffled":
        case.update(shuffled=True)
    elif option:
        case[option] = True
    return case


def _events(case, seed, slice_=0):
    kw = dict(n_events=case["n_events"], seed=(int(seed) * 64 + slice_ + 1) & 0x7FFFFFFF, keep_truth=False)
    if case["nu"]:
        kw.update(pileup=1, nu=case["nu"])
    else:
        kw.update(pileup=0, mean_tracks=SINGLE_PV_TRACKS)
    if case.get("crowded"):
        kw.update(high_occupancy_fraction=case["crowded"], high_nu=20.0)
    if case.get("noise"):
        kw.update(noise_fraction=case["noise"])
    if case.get("dead"):
        kw.update(dead_asic_fraction=case["dead"])
    if case.get("retina"):
        kw.update(retina=1)
    if case.get("shuffled"):
        kw.update(shuffle_sp=1)
    kw.update(bank_version=case.get("bank_version", 4))
    events = synth.generate(**kw)
    return synth.to_mep(events) if case.get("mep") else events


def _constants():
    return velo.VeloConstants(synth.read_geometry(), synth.read_beamline())


def _room(case):
    """(tracks, hits, raw bytes) that no slice of this case exceeds, which a program sizes its buffers by:
    the mean of the case's events, six standard deviations of their sum and a few more."""
    n, nu = case["n_events"], case["nu"]
    mean, var = (TRACKS_PER_COLLISION * nu, 450.0 * nu) if nu else (SINGLE_PV_TRACKS, 150.0)
    if case.get("crowded"):
        high = TRACKS_PER_COLLISION * 20.0
        var = (1 - case["crowded"]) * var + case["crowded"] * (450.0 * 20.0 + (high - mean) ** 2)
        mean += case["crowded"] * (high - mean)
    tracks = int(1.02 * mean * n + 6 * (var * n) ** 0.5) + 64
    header = 1000 if case.get("bank_version", 4) == 4 else 3000
    return tracks, 10 * tracks, 64 * tracks + header * n


class _Buffer:
    """The leading `count` items of a sequence's named device buffer, for torch.as_tensor."""

    def __init__(self, seq, name, typestr, count):
        ptr, capacity = seq.buffer_ptr(name)
        if count * int(typestr[-1]) > capacity:
            raise velo.VeloError(f"{name}: {count} elements exceed the capacity")
        self.seq = seq  # the buffer lives as long as its sequence
        self.__cuda_array_interface__ = dict(shape=(count,), typestr=typestr, data=(ptr, False), version=2)


def _sequence(case, constants, events):
    """A sequence with room for the case's slices, its knobs, and tensors over the outputs of its runs.

    How many tracks a run finds is known on the device only, so the tensors cover the whole room and
    start as zeros, which the part that no track reaches stays."""
    tracks, hits, raw_bytes = _room(case)
    n = events.n_events
    seq = velo.VeloSequence(constants, n, max(raw_bytes, events.raw.size))
    for knob in ("search_block", "search_lds_hits", "search_ring_window", "search_list_cap"):
        if case.get(knob):
            seq.set_tuning(knob, case[knob])
    if case.get("fp64"):
        seq.set_tuning("kalman_fp64_fallback", 1)
    if case.get("vertices"):
        seq.set_tuning("pv_finder", 1)
    if case.get("pruned"):
        params, threshold = scorer.trained()
        seq.set_scorer(params, threshold)
    layout = [("offsets_all_velo_tracks", "<i4", n + 1), ("offsets_velo_track_hit_number", "<i4", tracks + 1),
              ("velo_track_hits", "<i4", 18 * hits // 4), ("is_backward", "|u1", tracks),
              ("velo_kalman_beamline_states", "<f4", 14 * tracks), ("velo_kalman_endvelo_states", "<f4", 14 * tracks)]
    if case.get("vertices"):
        layout.append(("number_of_multi_final_vertices", "<i4", n))
        layout.append(("multi_final_vertices", "<f4", 12 * 32 * n))
    out = {name: torch.as_tensor(_Buffer(seq, name, t, count), device="cuda") for name, t, count in layout}
    for t in out.values():
        t.zero_()
    return seq, out


def _results(case):
    """Arrays of its own that a program copies each slice's results into, with room for the case's slices."""
    tracks, hits, _ = _room(case)
    z = lambda dtype, *shape: torch.zeros(shape, dtype=dtype, device="cuda")  # noqa: E731
    out = dict(offsets_all_velo_tracks=z(torch.int32, case["n_events"] + 1),
               offsets_velo_track_hit_number=z(torch.int32, tracks + 1),
               velo_track_hits=z(torch.uint8, 16 * hits), is_backward=z(torch.uint8, tracks))
    for name in ("velo_kalman_beamline_states", "velo_kalman_endvelo_states"):
        # x, y, z, tx, ty (qop is never written), then the covariance (chi2 and ndof are not).
        out[name] = z(torch.float32, tracks, 5)
        out[name + "_covariance"] = z(torch.float32, tracks, 6)
    return out


def _seeds(rows, seed):
    """Features and labels of seeds, spread as the search's are: residuals and phi steps around zero
    with tails, slopes, a small scatter, the module pair; nearly all seeds open a true track."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 17)
    x = torch.randn(rows, 10, generator=g, device="cuda")
    x[:, 0:4] *= 0.4
    x[:, 8] = x[:, 8].square() * 0.2
    x[:, 9] = torch.randint(2, 26, (rows,), generator=g, device="cuda") / 32.0
    true = torch.rand(rows, generator=g, device="cuda") > 0.005 + 0.2 * (x[:, 8] > 0.8)
    return x.contiguous(), true.to(torch.uint8)


TRAIN_LR = 3e-3
TRAIN_STEPS_BEFORE = 200  # the step timed lies inside a training run: Adam's moments are filled


def _adam_state(seed):
    rng = np.random.default_rng(int(seed) + 29)
    m = rng.normal(0.0, 1e-3, scorer.N_PARAMS).astype(np.float32)
    v = (rng.uniform(0.5, 2.0, scorer.N_PARAMS) * 1e-5).astype(np.float32)
    return scorer.init_params(int(seed) % 9973), m, v


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "score"):
        features, labels = _seeds(case["rows"], seed)
        params, m, v = _adam_state(seed)
        net = scorer.MLP(params=params)
        net.m.copy_(torch.from_numpy(m))
        net.v.copy_(torch.from_numpy(v))
        net.step_count = TRAIN_STEPS_BEFORE
        return dict(case=case, net=net, features=features, labels=labels)
    constants = _constants()
    if kind == "chain":
        return dict(case=case, constants=constants, events=velo.DeviceEvents(_events(case, seed)),
                    results=_results(case))
    slices = []
    for i in range(case.get("slices", 1)):
        events = _events(case, seed, i)
        seq, out = _sequence(case, constants, events)
        slices.append((seq, velo.DeviceEvents(events), out))
    state = dict(case=case, constants=constants, slices=slices)
    if kind == "streams":
        state["streams"] = _streams(case["streams"])
    if kind == "graph":
        # The stream that was captured on is the one that replays; what the inputs and outputs were
        # filled by is done before.
        state["stream"], = _streams(1)
        torch.cuda.synchronize()
        seq, events, _ = slices[0]
        seq.capture(events, state["stream"])
    return state


_kept_streams = []


def _streams(count):
    """A program makes its streams once and keeps them."""
    while len(_kept_streams) < count:
        _kept_streams.append(torch.cuda.Stream())
    return _kept_streams[:count]


def _chain(state):
    events, out = state["events"], state["results"]
    args = algorithms.velo_sp_sequence(state["constants"], events, events.n_events)
    n = args.host["number_of_reconstructed_velo_tracks"]
    hits = args.host["accumulated_number_of_hits_in_velo_tracks"]
    for name, count in (("offsets_all_velo_tracks", events.n_events + 1), ("offsets_velo_track_hit_number", n + 1),
                        ("velo_track_hits", 16 * hits), ("is_backward", n)):  # id, x, y, z; phi is never written
        out[name][:count].copy_(args[name][:count])
    for name in ("velo_kalman_beamline_states", "velo_kalman_endvelo_states"):
        words = args[name][:14 * n]
        out[name][:n].copy_(words[:6 * n].view(n, 6)[:, :5])
        out[name + "_covariance"][:n].copy_(words[6 * n:].view(n, 8)[:, :6])
    return out


def run(state):
    kind = state["case"]["kind"]
    if kind == "train":
        net = state["net"]
        loss, _ = net.train_step(state["features"], state["labels"], TRAIN_LR)
        return dict(loss=loss, params=net.params, m=net.m, v=net.v)
    if kind == "score":
        return dict(logits=state["net"].score(state["features"]))
    if kind == "chain":
        return _chain(state)
    if kind == "graph":
        seq, _, out = state["slices"][0]
        seq.replay(state["stream"])
        return out
    if kind == "sequence":
        seq, events, out = state["slices"][0]
        seq.run(events)
        return out
    # Slices dealt to the streams in turn; what follows on the current stream sees all of them.
    main = torch.cuda.current_stream()
    streams = state["streams"]
    for s in streams:
        s.wait_stream(main)
    for i, (seq, events, _) in enumerate(state["slices"]):
        seq.run(events, stream=streams[i % len(streams)])
    for s in streams:
        main.wait_stream(s)
    return [out for _, _, out in state["slices"]]


def work(case):
    kind = case["kind"]
    if kind in ("train", "score"):
        rows, macs = case["rows"], 320 + 1024 + 32
        if kind == "score":
            return dict(bytes=rows * (40 + 4) + 4 * scorer.N_PARAMS, flops=2 * macs * rows)
        return dict(bytes=rows * (40 + 1) + 6 * 4 * scorer.N_PARAMS, flops=6 * macs * rows)
    tracks = TRACKS_PER_COLLISION * case["nu"] if case["nu"] else SINGLE_PV_TRACKS
    if case.get("crowded"):
        tracks = (1 - case["crowded"]) * tracks + case["crowded"] * TRACKS_PER_COLLISION * 20.0
    # Raw banks (a word of four bytes for each of about thirteen super pixels or ten clusters of a
    # track, and the headers of 104 banks), read; hits, states and flags of the tracks, written.
    raw = 4 * tracks * (10 if case.get("retina") else 13) + 104 * (4 + 4 + 2 + 1)
    bytes_ = raw + tracks * (16 * HITS_PER_TRACK + 2 * 44 + 1 + 4)
    # The fit: one update of two projections for each hit, and each hit's place found in the module pair before.
    flops = tracks * HITS_PER_TRACK * 150
    events = case["n_events"] * case.get("slices", 1)
    return dict(bytes=bytes_ * events, flops=flops * events)


def _mlp(p, x):
    """Logits in the type of its arguments, and what the backward pass needs."""
    w1, b1, w2, b2, w3, b3 = (p[o:o + int(np.prod(shape, dtype=np.int64))].reshape(shape)
                              for o, shape in scorer.LAYOUT.values())
    a1 = torch.relu(x @ w1 + b1)
    return torch.relu(a1 @ w2 + b2) @ w3 + b3


def exact(case, seed):
    """The scorer's arithmetic in 64 bits. The tracks of an event are decisions of the 32-bit path
    (which hits pass a cut), which no plain 64-bit statement gives alike."""
    if case["kind"] not in ("train", "score"):
        return None
    x, labels = _seeds(case["rows"], seed)
    params, m, v = (torch.from_numpy(a).double().cuda() for a in _adam_state(seed))
    x = x.double()
    if case["kind"] == "score":
        return dict(logits=_mlp(params, x))
    params.requires_grad_(True)
    loss = torch.nn.functional.binary_cross_entropy_with_logits(_mlp(params, x), labels.double())
    loss.backward()
    g, step = params.grad, TRAIN_STEPS_BEFORE + 1
    m = 0.9 * m + 0.1 * g
    v = 0.999 * v + 0.001 * g * g
    update = (m / (1 - 0.9 ** step)) / (torch.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
    return dict(loss=loss.item(), params=params.detach() - TRAIN_LR * update, m=m, v=v)
