"""The split-column canonicalisers (csrc/kernels_canon_h.hpp) at every kind of n = 2 chi against the generic Jacobi
kernel, and a quench at chi = 3 against the NumPy oracle.

Where chi is no power of two an edge's lane group holds padding lanes; a lane exchange in two moves passes through
them, so it must not run where they are switched off.
"""
import numpy as np
import pytest

from bqa_amd import instances
from bqa_amd.config import config_to_context
from oracle import bqa_oracle as O

pytestmark = pytest.mark.gpu


# few edges: both sides of an edge at once; more than 1,024 (chi = 4 and 8: 2,048) waves: one side after the other
@pytest.mark.parametrize("chi,edges", [(c, 6) for c in (2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 13, 14, 15, 16)]
                         + [(3, 4096), (3, 4097), (4, 8193), (8, 2048), (8, 2049), (11, 1024), (11, 1025)]
                         + [(3, 8193), (5, 4097), (6, 4097), (7, 4097), (9, 2049), (12, 2049), (15, 2049)])
@pytest.mark.parametrize("decay", [0.0, 4.5])
def test_matches_generic(chi, edges, decay, monkeypatch):
    from bqa_amd.native import Job
    n = edges
    ctx = config_to_context({"nodes": {i: 0.2 for i in range(n)},
                             "edges": {(i, (i + 1) % n): 0.3 + 0.2 * i / n for i in range(n)}, "max_bond_dim": 2 * chi,
                             "default_field": 0.0, "seed": 1, "bp_eps": 1e-12, "max_bp_iter_number": 60,
                             "pinv_eps": 1e-6, "damping": 0.0, "measurement_threshold": 0.95,
                             "schedule": instances.anneal_schedule(1.0, 4), "backend": "mi355x", "precision": "double"})
    rng = np.random.default_rng(chi)
    t = rng.normal(size=(n, 2, chi, chi)) + 1j * rng.normal(size=(n, 2, chi, chi))
    # with a decay, eigenvalues of the extended messages fall through pinv_eps
    w = 10.0 ** (-decay * np.arange(chi) / chi)
    t = t * w[:, None] * w[None, :]
    m = np.repeat(np.eye(chi)[None] / chi, 2 * n, axis=0).astype(complex)
    out = []
    for mask in ("", "c"):
        monkeypatch.setenv("BQA_GENERIC_KERNELS", mask)
        job = Job(ctx, "double")
        try:
            job.init_state()
            job.set_tensors(0, t / np.sqrt((np.abs(t[0]) ** 2).sum()))
            job.set_messages(m)
            chi_new, err = job.simple_update(0.3, 1e-6)
            out.append((chi_new, err, job.get_lambdas().real))
        finally:
            job.close()
    # square roots of eigenvalues down to pinv_eps = 1e-6 amplify rounding by 1e3
    assert out[0][0] == out[1][0] and abs(out[0][1] - out[1][1]) < 1e-10
    assert np.abs(out[0][2] - out[1][2]).max() < 1e-10


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n,chi,steps", [(100, 3, 14), (60, 5, 12), (60, 6, 12)])
def test_quench_matches_oracle(n, chi, steps, precision):
    from bqa_amd.native import Job
    nodes, edges, _ = instances.regular_qubo(n, 3, seed=n, qmax=10)
    cfg = {"nodes": nodes, "edges": edges, "max_bond_dim": chi, "default_field": 0.0, "seed": 1, "bp_eps": 1e-10,
           "max_bp_iter_number": 75, "pinv_eps": 1e-6, "damping": 0.0, "measurement_threshold": 0.95,
           "schedule": {"total_time": 0.2 * steps, "starting_mixing": 0.5, "actions": [
               {"type": "real_time_evolution", "weight": 1.0, "steps_number": steps, "final_mixing": 0.5}]}}
    ctx_o = O.make_context(cfg)
    st = O.init_state(ctx_o)
    ctx = config_to_context(dict(cfg, backend="mi355x", precision=precision))
    job = Job(ctx, precision)
    try:
        job.init_state()
        for ins in ctx.instructions:
            if isinstance(ins, dict):
                O.run_layer(ctx_o, st, ins["xtime"], ins["ztime"])
                job.run_layer(ins["xtime"], ins["ztime"], ctx.pinv_eps, ctx.max_bp_iters_number, ctx.bp_eps, 0.0)
        bloch = job.density()[1]
        assert job.bond_dim == st.chi
    finally:
        job.close()
    # the tolerances of the parity tests: Bloch vectors of a whole run in double and in single precision
    assert np.abs(bloch - O.bloch_vectors(O.get_density_matrices(ctx_o, st))).max() < (1e-8 if precision == "double" else 1e-5)
