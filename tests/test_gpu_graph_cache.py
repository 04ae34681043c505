"""A job that replays graphs at more bond dimensions than it keeps graphs for, and comes back to the first."""
import numpy as np
import pytest

from bqa_amd import instances
from bqa_amd.config import config_to_context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["single", "double"])
def test_more_graphs_than_are_kept(precision, monkeypatch):
    from bqa_amd.native import Job
    n, d = 40, 3
    nodes, edges = instances.regular_uniform(n, d, seed=5, field_sigma=0.3)
    ctx = config_to_context({"nodes": nodes, "edges": edges, "max_bond_dim": 8, "bp_eps": 1e-9,
                             "max_bp_iter_number": 60, "schedule": instances.anneal_schedule(1.0, 2),
                             "backend": "mi355x", "precision": precision})
    # (bond dimension, sweeps of a run): both lengths of graph at six bond dimensions, then short runs, then the first
    # again with a long graph's worth of sweeps and a remainder
    plan = [(2, 7), (2, 38), (3, 38), (4, 38), (5, 38), (6, 38), (7, 38), (8, 7), (2, 38), (2, 7), (3, 38), (2, 45)]
    got = []
    for graphs in ("1", "0"):
        monkeypatch.setenv("BQA_GRAPHS", graphs)
        monkeypatch.setenv("BQA_AUTOTUNE", "0")
        job = Job(ctx, precision)
        try:
            job.init_state()
            one = []
            for chi, iters in plan:
                rng = np.random.default_rng(chi)
                job.set_tensors(0, rng.normal(size=(n, 2) + (chi,) * d) + 1j * rng.normal(size=(n, 2) + (chi,) * d))
                m = np.repeat(np.eye(chi)[None] / chi, n * d, axis=0).astype(complex)
                for _ in range(11):   # eight eager runs, then replays
                    job.set_messages(m)
                    out = job.run_bp(iters, 0.0, 0.0)
                    assert out[0] == iters
                one.append(job.get_messages())
            stats = job.graph_stats()
            got.append(one)
        finally:
            job.close()
        print(f"[gpu] graph cache {precision} graphs={graphs}: {stats}", flush=True)
        if graphs == "1":
            assert stats[0] > 8 and stats[1] > 0 and stats[2] == 0
        else:
            assert stats == (0, 0, 0)
    for a, b in zip(*got):
        assert np.array_equal(a, b)
