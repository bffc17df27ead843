"""GPU tests of the streaming tracker server.

Bars: a request's integrated output [W][F][B] is bit-identical whether it
runs alone or mixed with other requests, and to the multi-beam tracker
(same kernel arithmetic) over the same span of voltages; against the FP64
oracle it holds the split-FP16 bar (floored relative error <= 1e-5).
A loss-masked stream equals, bit for bit, the unmasked stream with its lost
frames zeroed (include/beamformer/formats.hpp:22-32), and spectra written
in place through acquire/commit equal the same spectra ingested by copy.
The ring is kept small so that windows wrap around it.
"""
import numpy as np
import pytest

import oracle as O
from beamform_project_amd import _capi, api, serve as SV, tracker as TR
from helpers import F, incoherent_floor, rel_err_floored

pytestmark = pytest.mark.gpu
K = api.Kernel
A = 64
POS = O.regular_array(8, 8, 0.3)
FR = np.linspace(400e6, 800e6, F).astype(np.float32)


def trajectories(B, seed):
    rng = np.random.default_rng(seed)
    t = np.zeros((B, 4), np.float32)
    t[:, 0] = rng.uniform(-0.4, 0.4, B)
    t[:, 1] = rng.uniform(-0.4, 0.4, B)
    t[:, 2:] = rng.uniform(-2e-5, 2e-5, (B, 2))
    return t


def voltages(T, seed):
    return O.make_uniform_int4(T * F * A, seed).reshape(T, F, A)


def config(**kw):
    base = dict(n_freq=F, n_ant=A, ring_spectra=1024, max_window=320, max_step_spectra=4096,
                hbm_budget_bytes=64 << 20, max_requests=16, positions=POS, frequencies=FR,
                enable_graph=True)
    base.update(kw)
    return SV.ServerConfig(**base)


# (B, S, n_spectra, start, submit_at, trajectory seed): start -1 = the head
# at admission.
MIX = [
    (5, 10, 1234, 0, 0, 10),
    (64, 320, 960, 100, 0, 11),
    (17, 16, 1000, 700, 300, 12),
    (1, 320, 700, -1, 1200, 13),
    (33, 10, 333, 1500, 1500, 14),
]


def produce(srv, x, mask, producer):
    """Writes x (and mask) into the ring in place: acquire, copy each span,
    commit on the producer's stream."""
    spans = srv.acquire(x.shape[0])
    i = 0
    for sp in spans:
        n = sp["n_spectra"]
        assert sp["first_spectrum"] == srv.stats()["head"] + i
        part = np.ascontiguousarray(x[i:i + n])
        _capi.call("bf_memcpy_htod", sp["voltages"], part.ctypes.data, part.nbytes)
        if mask is not None:
            m = np.ascontiguousarray(mask[i:i + n])
            _capi.call("bf_memcpy_htod", sp["valid"], m.ctypes.data, m.nbytes)
        i += n
    srv.commit(x.shape[0], producer.handle)


def run(requests, x, chunk=100, mask=None, zero_copy=False, **kw):
    """Streams x (with validity bytes `mask`) through a server, submitting
    request i once `submit_at` spectra have been ingested; returns
    {i: (start, output)}."""
    srv = SV.TrackerServer(config(loss_masks=mask is not None, **kw))
    producer = api.Stream() if zero_copy else None
    ids = {}
    T = x.shape[0]
    for h in range(0, T, chunk):
        for i, (B, S, n, start, at, seed) in enumerate(requests):
            if at == h:
                ids[i] = srv.submit(SV.Request(trajectories(B, seed), S, n, start))
        m = None if mask is None else mask[h:h + chunk]
        if zero_copy:
            produce(srv, x[h:h + chunk], m, producer)
        else:
            srv.ingest(x[h:h + chunk], m)
        srv.step()
    srv.synchronize()
    out = {}
    for i, rid in ids.items():
        st = srv.status(rid)
        B = requests[i][0]
        assert st["state"] == SV.COMPLETE, (i, st)
        out[i] = (st["start"], srv.read(rid, 0, st["windows_total"], B))
        srv.release(rid)
    stats = srv.stats()
    srv.close()
    return out, stats


@pytest.fixture(scope="module")
def stream():
    return voltages(2400, 99)


@pytest.fixture(scope="module")
def mixed(stream):
    return run(MIX, stream)


def test_alone_equals_mixed(stream, mixed):
    out, _ = mixed
    for i, req in enumerate(MIX):
        start = out[i][0]
        alone, _ = run([(req[0], req[1], req[2], start, req[4], req[5])], stream)
        assert alone[0][0] == start
        assert np.array_equal(alone[0][1], out[i][1]), f"request {i}"


def test_alone_equals_mixed_on_the_full_size_ring(stream, mixed):
    """The same request mix on a 2^20-spectrum ring (22.5 GB at A=64,
    F=336) with a 1 GiB output budget: each request alone equals the mix,
    and both equal the small-ring results (the ring size changes only where
    a spectrum lives)."""
    big = dict(ring_spectra=1 << 20, hbm_budget_bytes=1 << 30, max_step_spectra=8192)
    out_big, _ = run(MIX, stream, **big)
    out, _ = mixed
    for i, req in enumerate(MIX[:3]):
        assert out_big[i][0] == out[i][0]
        assert np.array_equal(out_big[i][1], out[i][1]), i
        alone, _ = run([(req[0], req[1], req[2], out_big[i][0], req[4], req[5])], stream, **big)
        assert np.array_equal(alone[0][1], out_big[i][1]), i


def test_matches_multibeam_tracker_and_fp64(stream, mixed):
    out, stats = mixed
    for i, (B, S, n, _, _, seed) in enumerate(MIX):
        t0, got = out[i]
        x = np.ascontiguousarray(stream[t0:t0 + n])
        assert x.shape[0] == n
        traj = trajectories(B, seed)
        dx = api.DeviceArray.from_numpy(x)
        dpos, dfr, dtraj = (api.DeviceArray.from_numpy(a) for a in (POS, FR, traj))
        W = (n + S - 1) // S
        dout = api.DeviceArray.empty((W, F, B), np.float32)
        TR.multibeam_tracker_launch(None, dx, dout, n, F, A, B, S, dpos, dfr,
                                    trajectories=dtraj, kernel=K.SPLIT_F16)
        api.device_synchronize()
        assert np.array_equal(dout.to_numpy(), got), f"request {i} vs multibeam tracker"
        if B * n <= 64 * 1000:
            dirs = np.zeros((W, B, 3), np.float32)
            for w in range(W):
                for b in range(B):
                    dirs[w, b] = O.tracker_direction(*traj[b], w * S)
            _, ref64 = O.multibeam_tracker(x, n, F, A, B, S, POS, FR, dirs, want_f64=True)
            err = rel_err_floored(got, ref64, incoherent_floor(x, A, S))
            assert err <= 1e-5, f"request {i}: {err:.3e}"
    assert stats["windows_processed"] == sum((r[2] + r[1] - 1) // r[1] for r in MIX)
    assert stats["windows_timed"] > 0 and stats["latency_p99_ms"] > 0


def test_graph_and_eager_steps_agree(stream, mixed):
    out, _ = mixed
    eager, _ = run(MIX, stream, enable_graph=False)
    for i in out:
        assert np.array_equal(eager[i][1], out[i][1]), f"request {i}"


def test_f16_kernel_holds_its_bar(stream):
    B, S, n = 12, 320, 640
    out, _ = run([(B, S, n, 0, 0, 10)], stream, kernel=K.F16)
    x = np.ascontiguousarray(stream[:n])
    traj = trajectories(B, 10)
    W = n // S
    dirs = np.array([[O.tracker_direction(*traj[b], w * S) for b in range(B)] for w in range(W)],
                    np.float32)
    _, ref64 = O.multibeam_tracker(x, n, F, A, B, S, POS, FR, dirs, want_f64=True)
    assert rel_err_floored(out[0][1], ref64, incoherent_floor(x, A, S)) <= 2e-3


def test_admission_waits_for_hbm_budget(stream):
    B, S, n = 8, 10, 400
    per_request = (n // S) * F * B * 4
    srv = SV.TrackerServer(config(hbm_budget_bytes=2 * per_request + 256))
    ids = [srv.submit(SV.Request(trajectories(B, 40 + i), S, n)) for i in range(3)]
    srv.step()
    st = [srv.status(r) for r in ids]
    assert [s["state"] for s in st] == [SV.ACTIVE, SV.ACTIVE, SV.PENDING]
    h = 0
    while srv.status(ids[0])["state"] != SV.COMPLETE:
        srv.ingest(stream[h:h + 100])
        h += 100
        srv.step()
        srv.synchronize()
    first = srv.read(ids[0], 0, n // S, B)
    srv.release(ids[0])
    srv.ingest(stream[h:h + 100])
    h += 100
    srv.step()
    s2 = srv.status(ids[2])
    # admitted once request 0's outputs were released; it starts at the head
    assert s2["state"] == SV.ACTIVE and s2["start"] == h
    while srv.status(ids[2])["state"] != SV.COMPLETE:
        srv.ingest(stream[h:h + 100])
        h += 100
        srv.step()
        srv.synchronize()
    late = srv.read(ids[2], 0, n // S, B)
    stats = srv.stats()
    assert stats["requests_admitted"] == 3 and stats["arena_peak_bytes"] <= 2 * per_request + 256
    assert stats["mean_admission_wait_spectra"] > 0
    srv.close()
    # the same two requests on a server with room for both
    srv2 = SV.TrackerServer(config())
    r0 = srv2.submit(SV.Request(trajectories(B, 40), S, n, 0))
    r2 = srv2.submit(SV.Request(trajectories(B, 42), S, n, s2["start"]))
    for g in range(0, h, 100):
        srv2.ingest(stream[g:g + 100])
        srv2.step()
    srv2.synchronize()
    assert np.array_equal(srv2.read(r0, 0, n // S, B), first)
    assert np.array_equal(srv2.read(r2, 0, n // S, B), late)
    srv2.close()


def test_admission_waits_for_the_beam_budget(stream):
    """With max_active_beams, a request waits (FIFO) until the active
    requests' beams plus its own fit; it is admitted at completion of an
    earlier one (no release needed, the budget is compute, not memory), and
    its output equals a run on a server without the cap."""
    S, n = 10, 300
    srv = SV.TrackerServer(config(max_active_beams=40))
    with pytest.raises(_capi.InvalidArgument, match="max_active_beams"):
        srv.submit(SV.Request(trajectories(41, 1), S, n))
    ids = [srv.submit(SV.Request(trajectories(B, 50 + i), S, n))
           for i, B in enumerate((24, 16, 9))]
    srv.step()
    assert [srv.status(r)["state"] for r in ids] == [SV.ACTIVE, SV.ACTIVE, SV.PENDING]
    h = 0
    while srv.status(ids[2])["state"] == SV.PENDING:
        srv.ingest(stream[h:h + 100])
        h += 100
        srv.step()
        srv.synchronize()
    st2 = srv.status(ids[2])
    assert srv.status(ids[0])["state"] == SV.COMPLETE and st2["start"] > 0
    while srv.status(ids[2])["state"] != SV.COMPLETE:
        srv.ingest(stream[h:h + 100])
        h += 100
        srv.step()
        srv.synchronize()
    late = srv.read(ids[2], 0, n // S, 9)
    srv.close()
    srv2 = SV.TrackerServer(config())
    r2 = srv2.submit(SV.Request(trajectories(9, 52), S, n, st2["start"]))
    for g in range(0, h, 100):
        srv2.ingest(stream[g:g + 100])
        srv2.step()
    srv2.synchronize()
    assert np.array_equal(srv2.read(r2, 0, n // S, 9), late)
    srv2.close()


def test_output_ring_and_reads(stream):
    B, S, n = 3, 10, 500
    srv = SV.TrackerServer(config())
    full = srv.submit(SV.Request(trajectories(B, 7), S, n, 0))
    ring = srv.submit(SV.Request(trajectories(B, 7), S, n, 0, output_windows=8))
    for h in range(0, 500, 50):
        srv.ingest(stream[h:h + 50])
        srv.step()
        done = srv.status(ring)["windows_issued"]
        if done >= 4:
            a = srv.read(ring, done - 4, 4, B)
            b = srv.read(full, done - 4, 4, B)
            assert np.array_equal(a, b)
    with pytest.raises(_capi.OutOfRange):
        srv.read(ring, 0, 4, B)  # overwritten
    with pytest.raises(_capi.OutOfRange):
        srv.read(full, 0, n // S + 1, B)  # not yet produced
    srv.close()


def test_ring_overrun_and_request_validation(stream):
    srv = SV.TrackerServer(config(ring_spectra=1024))
    srv.submit(SV.Request(trajectories(2, 1), 320, 5000, 0))
    srv.ingest(stream[:600])
    with pytest.raises(_capi.LogicError, match="ring overrun"):
        srv.ingest(stream[600:1200])  # no step has processed the oldest spectra
    srv.step()
    srv.synchronize()
    srv.ingest(stream[600:1200])  # fine once the oldest spectra are processed
    with pytest.raises(_capi.InvalidArgument, match="n_beams"):
        srv.submit(SV.Request(np.zeros((65, 4), np.float32), 10, 100))
    with pytest.raises(_capi.InvalidArgument, match="window"):
        srv.submit(SV.Request(np.zeros((1, 4), np.float32), 640, 1000))
    with pytest.raises(_capi.InvalidArgument, match="sky"):
        srv.submit(SV.Request(np.array([[0.5, 0.5, 1e-3, 0.0]], np.float32), 10, 1000))
    old = srv.submit(SV.Request(trajectories(1, 2), 10, 100, start=0))
    srv.step()
    assert srv.status(old)["state"] == SV.REJECTED
    srv.close()


def test_past_start_back_fills_windows(stream):
    """A request admitted with an explicit start behind the processed head
    gets every window from its start (the first step after admission issues
    the ones already in the ring), equal to the multi-beam tracker on the
    same span.  Spectra 0..799 are ingested and stepped on a 1024-spectrum
    ring before the requests arrive; the stream then wraps the ring."""
    reqs = [(7, 10, 600, 0, 22), (24, 320, 900, 50, 23), (3, 16, 400, 650, 24)]
    srv = SV.TrackerServer(config(ring_spectra=1024))
    for h in range(0, 800, 100):
        srv.ingest(stream[h:h + 100])
        srv.step()
    ids = [srv.submit(SV.Request(trajectories(B, seed), S, n, start))
           for B, S, n, start, seed in reqs]
    srv.step()  # admits; nothing new ingested, the back-filled windows run now
    assert [srv.status(r)["windows_issued"] for r in ids] == [60, 2, 9]
    for h in range(800, 1600, 100):
        srv.ingest(stream[h:h + 100])
        srv.step()
    srv.synchronize()
    for (B, S, n, start, seed), rid in zip(reqs, ids):
        st = srv.status(rid)
        assert st["state"] == SV.COMPLETE and st["start"] == start, st
        got = srv.read(rid, 0, st["windows_total"], B)
        x = np.ascontiguousarray(stream[start:start + n])
        W = (n + S - 1) // S
        dx = api.DeviceArray.from_numpy(x)
        dpos, dfr, dtraj = (api.DeviceArray.from_numpy(a)
                            for a in (POS, FR, trajectories(B, seed)))
        dout = api.DeviceArray.empty((W, F, B), np.float32)
        TR.multibeam_tracker_launch(None, dx, dout, n, F, A, B, S, dpos, dfr,
                                    trajectories=dtraj, kernel=K.SPLIT_F16)
        api.device_synchronize()
        assert np.array_equal(dout.to_numpy(), got), (B, S, start)
        srv.release(rid)
    # head 1600 on a 1024-spectrum ring: spectrum 576 is the oldest held.
    late = [srv.submit(SV.Request(trajectories(2, 25), 10, 100, s0)) for s0 in (575, 576)]
    srv.step()
    assert [srv.status(r)["state"] for r in late] == [SV.REJECTED, SV.ACTIVE]
    assert srv.status(late[1])["windows_issued"] == 10
    srv.close()


def test_native_load_generator_reports_latency():
    cfg = SV.SimConfig(server=config(ring_spectra=1 << 16, max_requests=64,
                                     hbm_budget_bytes=1 << 30),
                       run_seconds=0.25, arrival_rate_hz=80.0, min_duration_s=0.02,
                       max_duration_s=0.1, output_windows_cap=256, pool_spectra=4096)
    rep = SV.simulate(cfg)
    st = rep["stats"]
    assert rep["requests_generated"] > 5
    assert st["requests_admitted"] >= 1 and st["windows_timed"] > 0
    assert 0 < st["latency_p50_ms"] <= st["latency_p99_ms"] <= st["latency_max_ms"]
    assert st["beam_samples"] > 0 and rep["beam_samples_per_s"] > 0
    assert rep["graph_used"] == 1


def loss_mask(T, seed):
    rng = np.random.default_rng(seed)
    mask = (rng.random((T, F)) > 0.2).astype(np.uint8)
    mask[450:530] = 0     # a run of lost spectra across every channel
    mask[:, 5] = 0        # a dead channel
    return mask


def test_masked_stream_equals_zeroed_payload(stream, mixed):
    mask = loss_mask(stream.shape[0], 3)
    zeroed = stream * mask[:, :, None]
    got, _ = run(MIX, stream, mask=mask)
    want, _ = run(MIX, zeroed)
    for i in want:
        assert got[i][0] == want[i][0]
        assert np.array_equal(got[i][1], want[i][1]), f"request {i}"
        assert np.all(got[i][1][:, 5, :] == 0)
    # a masked server fed every frame valid equals the unmasked server
    ones, _ = run(MIX, stream, mask=np.ones(mask.shape, np.uint8), enable_graph=False)
    for i in ones:
        assert np.array_equal(ones[i][1], mixed[0][i][1]), f"request {i}"


@pytest.mark.parametrize("n_ant,kernel", [(64, K.SPLIT_F16), (32, K.SPLIT_F16), (64, K.F16)])
def test_masked_window_lengths(stream, n_ant, kernel):
    """Windows around the length where masked ones take a body of their own (64)
    and around its groups of four tiles, across the ring's end."""
    x = np.ascontiguousarray(stream[..., :n_ant])
    kw = dict(n_ant=n_ant, positions=O.regular_array(n_ant // 8, 8, 0.3), kernel=kernel)
    requests = [(9, 63, 2300, 0, 0, 20), (9, 64, 2300, 0, 0, 21), (17, 79, 2300, 3, 0, 22),
                (3, 130, 2200, 41, 0, 23), (20, 255, 2301, 0, 0, 24)]
    mask = loss_mask(x.shape[0], 5)
    got, _ = run(requests, x, mask=mask, **kw)
    want, _ = run(requests, x * mask[:, :, None], **kw)
    for i in want:
        assert np.array_equal(got[i][1], want[i][1]), f"request {i}"


def test_zero_copy_producer_equals_ingest(stream, mixed):
    # chunks of 100 on a ring of 1024: spans wrap at 1000..1100 and 2000..2100
    got, _ = run(MIX, stream, zero_copy=True)
    for i in got:
        assert np.array_equal(got[i][1], mixed[0][i][1]), f"request {i}"
    mask = loss_mask(stream.shape[0], 4)
    masked, _ = run(MIX, stream, mask=mask, zero_copy=True)
    zeroed, _ = run(MIX, stream * mask[:, :, None])
    for i in zeroed:
        assert np.array_equal(masked[i][1], zeroed[i][1]), f"request {i}"


def test_producer_interface_contract(stream):
    srv = SV.TrackerServer(config(ring_spectra=1024))
    with pytest.raises(_capi.InvalidArgument, match="loss_masks"):
        srv.ingest(stream[:10], np.ones((10, F), np.uint8))
    with pytest.raises(_capi.LogicError, match="without an acquired"):
        srv.commit(10)
    spans = srv.acquire(100)
    assert len(spans) == 1 and spans[0]["valid"] == 0 and spans[0]["n_spectra"] == 100
    with pytest.raises(_capi.LogicError, match="already acquired"):
        srv.acquire(10)
    with pytest.raises(_capi.LogicError, match="committed before ingesting"):
        srv.ingest(stream[:10])
    with pytest.raises(_capi.InvalidArgument, match="more spectra"):
        srv.commit(101)
    srv.commit(60)             # a partial commit publishes the first 60
    assert srv.stats()["head"] == 60
    assert srv.acquire(600)[0]["first_spectrum"] == 60
    srv.commit(0)              # abandoned
    with pytest.raises(_capi.InvalidArgument, match="ring capacity"):
        srv.acquire(1024 - 320 + 1)
    srv.close()


def test_shard_descriptor_sets_the_channel_plan(stream):
    # shard 1 of the two-shard band (include/beamformer/config.hpp:64-72):
    # with no explicit frequencies the server uses channels 336..671
    from beamform_project_amd import formats as FM
    s1 = FM.default_shard_descriptor(1)
    reqs = [(4, 10, 400, 0, 0, 21)]
    by_shard, _ = run(reqs, stream[:500], frequencies=None, shard=s1)
    explicit, _ = run(reqs, stream[:500], frequencies=FM.shard_frequencies(s1))
    assert np.array_equal(by_shard[0][1], explicit[0][1])
    shard0, _ = run(reqs, stream[:500], frequencies=None)
    assert not np.array_equal(shard0[0][1], by_shard[0][1])
    bad = FM.ShardDescriptor.from_c(s1.c())
    bad.shard_count = 3
    with pytest.raises(_capi.InvalidArgument, match="shard_count"):
        SV.TrackerServer(config(shard=bad))
