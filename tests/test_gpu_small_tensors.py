"""Classes of many nodes with small tensors, whose sweeps, extended messages and readout go to the generic kernel: a
layer against the batched products', which the same shapes with few nodes take."""
import numpy as np
import pytest

from bqa_amd import instances
from bqa_amd.config import config_to_context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi", [(2, 9), (2, 11), (2, 13), (5, 2), (5, 3), (5, 4), (6, 2), (6, 3), (4, 5)])
def test_copies_of_a_small_graph(d, chi, precision):
    """1,100 and more nodes as copies of a graph of a few nodes: the same step on every copy as on the graph alone."""
    from bqa_amd.native import Job
    n = {2: 7, 4: 10, 5: 10, 6: 12}[d]
    copies = 1100 // n + 1
    nodes, edges = ({i: 0.1 * i for i in range(n)}, {(i, (i + 1) % n): 0.1 + 0.05 * i for i in range(n)}) if d == 2 \
        else instances.regular_uniform(n, d, seed=4, field_sigma=0.3)
    rng = np.random.default_rng(d)
    t = (rng.normal(size=(n, 2) + (chi,) * d) + 1j * rng.normal(size=(n, 2) + (chi,) * d)) / chi ** (d / 2)
    out = []
    for k in (1, copies):
        ctx = config_to_context({
            "nodes": {c * n + v: h for c in range(k) for v, h in nodes.items()},
            "edges": {(c * n + a, c * n + b): j for c in range(k) for (a, b), j in edges.items()}, "max_bond_dim": chi,
            "default_field": 0.0, "seed": 1, "bp_eps": 1e-9, "max_bp_iter_number": 30, "pinv_eps": 1e-6, "damping": 0.0,
            "measurement_threshold": 0.95, "schedule": instances.anneal_schedule(1.0, 4), "backend": "mi355x",
            "precision": precision})
        (_, lay), = ctx.degree_to_layout.items()
        job = Job(ctx, precision)
        try:
            job.init_state()
            job.set_tensors(0, t[np.asarray(lay.node_ids) % n])
            m = np.repeat(np.eye(chi)[None] / chi, k * n * d, axis=0).astype(complex)
            job.set_messages(m)
            rho = [job.density()[0]]
            job.run_layer(0.2, 0.1, 1e-6, 30, 1e-9, 0.0)
            rho.append(job.density()[0])
        finally:
            job.close()
        out.append([r.reshape(k, n, 2, 2) for r in rho])
    # products of chi d terms in the job's precision; the step's canonicalisers (pinv_eps = 1e-6) amplify their rounding
    u = 6e-8 if precision == "single" else 1.2e-16
    for a, b, tol in zip(*out, (u * (8 * d * chi + 64), u * 1e3 * (8 * d * chi + 64))):
        assert np.abs(a - b).max() < tol
