"""The continuous-batching server: each request's result is the same alone and in
the mix (bit for bit), admission respects the HBM budget, and latencies are
reported."""
import pytest
import torch

from azeban_amd import init as I
from azeban_amd import initialize
from azeban_amd.ensemble import solve_one
from azeban_amd.serving import Request, Server

pytestmark = pytest.mark.gpu


def reqs():
    out = []
    specs = [(2, 64, 0.0), (2, 128, 0.001), (3, 64, 0.002), (2, 64, 0.003), (2, 256, 0.004), (3, 64, 0.005)]
    for i, (dim, N, arr) in enumerate(specs):
        u = initialize(I.fractional_brownian(dim, N, seed=100 + i))
        out.append(Request(i, dim, N, u, 0.004 if dim == 3 else 0.01, arr))
    torch.cuda.synchronize()
    return out


def test_results_same_alone_and_in_mix(cuda):
    print("[case] serving mix", flush=True)
    rs = reqs()
    srv = Server(chunk_steps=3, max_active=8)
    stats = srv.run(rs)
    torch.cuda.synchronize()
    assert stats["requests"] == len(rs)
    assert stats["peak_active"] >= 2  # work of several requests overlapped
    by_id = {r.rid: r for r in rs}
    for res in srv.results:
        r = by_id[res.rid]
        ref, n = solve_one(r.dim, r.N, r.u_hat, r.t_end)
        assert res.steps == n
        assert torch.equal(res.u_hat, ref), r.rid
    assert stats["latency_p99_s"] >= stats["latency_p50_s"] > 0


def test_budget_serialises_admission(cuda):
    """With a budget that fits one request at a time, requests still all complete
    (FIFO) and never overlap."""
    print("[case] serving budget", flush=True)
    rs = reqs()[:3]
    srv = Server(hbm_budget=1, chunk_steps=4)
    stats = srv.run(rs)
    assert stats["requests"] == 3
    assert stats["peak_active"] == 1


def test_host_side_requests_upload_asynchronously(cuda):
    """Requests whose state is in host memory are uploaded on their own stream from a
    pinned copy the server keeps until they finish; results equal those of the same
    requests given on the device."""
    print("[case] serving host inputs", flush=True)
    rs = reqs()
    host_rs = [Request(r.rid, r.dim, r.N, r.u_hat.cpu(), r.t_end, r.arrival) for r in rs]
    a, b = Server(chunk_steps=3, max_active=8), Server(chunk_steps=3, max_active=8)
    a.run(rs)
    b.run(host_rs)
    torch.cuda.synchronize()
    ra = {r.rid: r for r in a.results}
    for res in b.results:
        assert res.steps == ra[res.rid].steps
        assert torch.equal(res.u_hat, ra[res.rid].u_hat), res.rid


def test_slots_are_reused_by_later_requests(cuda):
    """More requests of one size than its class has slots: later requests join the
    running batch in slots that earlier ones left (a slot's stale progress from its
    previous request never ends the new one early); each result equals a solve alone."""
    print("[case] serving slot reuse", flush=True)
    rs = []
    for i in range(7):
        u = initialize(I.fractional_brownian(2, 64, seed=300 + i))
        rs.append(Request(i, 2, 64, u, 0.004 + 0.003 * (i % 3), 0.0005 * i))
    torch.cuda.synchronize()
    srv = Server(chunk_steps=2, slots={(2, 64): 2})
    stats = srv.run(rs)
    assert stats["requests"] == 7 and stats["peak_active"] == 2
    by_id = {r.rid: r for r in rs}
    for res in srv.results:
        r = by_id[res.rid]
        ref, n = solve_one(r.dim, r.N, r.u_hat, r.t_end)
        assert res.steps == n, r.rid
        assert torch.equal(res.u_hat, ref), r.rid


def test_serving_config_sizes_against_single_solves_and_oracle(cuda):
    """The serving workload's larger sizes (2D 512^2, 1024^2; 3D 128^3, 256^3, fractional
    Brownian data) through the server in one mix: bit-identical to solving each alone,
    and the 1024^2 and 128^3 requests match the FP64 oracle to 1e-11."""
    import numpy as np

    from oracle import azeban_oracle as O

    print("[case] serving config sizes", flush=True)
    specs = [(2, 512, 0.004), (2, 1024, 0.002), (3, 128, 0.004), (3, 256, 0.002), (2, 1024, 0.003)]
    rs = []
    for i, (dim, N, t_end) in enumerate(specs):
        u = initialize(I.fractional_brownian(dim, N, seed=500 + i))
        rs.append(Request(i, dim, N, u, t_end, 0.001 * i))
    torch.cuda.synchronize()
    srv = Server(chunk_steps=4)
    stats = srv.run(rs)
    assert stats["requests"] == len(rs) and stats["peak_active"] >= 2
    by_id = {r.rid: r for r in rs}
    for res in srv.results:
        r = by_id[res.rid]
        ref, n = solve_one(r.dim, r.N, r.u_hat, r.t_end)
        assert res.steps == n, r.rid
        assert torch.equal(res.u_hat, ref), r.rid
        if (r.dim, r.N) in ((2, 1024), (3, 128)) and r.rid != 4:
            osim = O.Simulation(O.IncompressibleEuler(O.Grid(r.dim, r.N), O.baseline_visc(r.N), workers=16),
                                r.u_hat.cpu().numpy(), 0.2)
            osim.simulate_until(r.t_end)
            err = O.l2_rel(res.u_hat.cpu().numpy(), osim.u)
            print(f"  {r.dim}D N={r.N} steps={n} rel L2 vs oracle {err:.2e}", flush=True)
            assert len(osim.dts) == n and err <= 1e-11, (r.rid, err)


def test_one_at_a_time_baseline_gives_the_same_results(cuda):
    """The sequential baseline solves the same requests to the same results."""
    from azeban_amd.serving import serve_one_at_a_time

    print("[case] serving one-at-a-time baseline", flush=True)
    rs = reqs()
    srv = Server(chunk_steps=3)
    srv.run(rs)
    base = serve_one_at_a_time(rs, chunk=3)
    assert base["requests"] == len(rs) and base["latency_p99_s"] >= base["latency_p50_s"] > 0
    got = {r.rid: r for r in base["results"]}
    for res in srv.results:
        assert res.steps == got[res.rid].steps
        assert torch.equal(res.u_hat, got[res.rid].u_hat), res.rid


def test_slots_are_reused_when_all_requests_wait(cuda):
    """Seven requests for two slots, all there from the start: both slots are in use together however
    fast a request is solved, and five requests join the batch in slots that others left."""
    print("[case] serving slot reuse, equal arrivals", flush=True)
    rs = []
    for i in range(7):
        u = initialize(I.fractional_brownian(2, 64, seed=300 + i))
        rs.append(Request(i, 2, 64, u, 0.004 + 0.003 * (i % 3), 0.0))
    torch.cuda.synchronize()
    srv = Server(chunk_steps=2, slots={(2, 64): 2})
    stats = srv.run(rs)
    assert stats["requests"] == 7 and stats["peak_active"] == 2
    assert sum(res.admitted > min(r.finished for r in srv.results) for res in srv.results) >= 4
    by_id = {r.rid: r for r in rs}
    for res in srv.results:
        r = by_id[res.rid]
        ref, n = solve_one(r.dim, r.N, r.u_hat, r.t_end)
        assert res.steps == n, r.rid
        assert torch.equal(res.u_hat, ref), r.rid
