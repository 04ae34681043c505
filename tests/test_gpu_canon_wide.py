"""The chi = 17..32 canonicalisers (csrc/canon_wide.hip) against the generic Jacobi kernel."""
import numpy as np
import pytest

from bqa_amd import instances
from bqa_amd.config import config_to_context

pytestmark = pytest.mark.gpu


# every row padding (34, 40 | 42, 48 | 50, 56 | 58, 64 rows), kept columns even and odd, fewer than chi' = 2 chi
@pytest.mark.parametrize("chi,chi_max", [(17, 32), (20, 23), (21, 32), (24, 24), (25, 32), (28, 29), (29, 32), (32, 32)])
@pytest.mark.parametrize("decay", [0.0, 4.5])
def test_matches_generic(chi, chi_max, decay, monkeypatch):
    from bqa_amd.native import Job
    n = 5
    edges = {(i, (i + 1) % n): 0.3 + 0.1 * i for i in range(n)}
    ctx = config_to_context({"nodes": {i: 0.2 for i in range(n)}, "edges": edges, "max_bond_dim": chi_max,
                             "default_field": 0.0, "seed": 1, "bp_eps": 1e-12, "max_bp_iter_number": 60,
                             "pinv_eps": 1e-6, "damping": 0.0, "measurement_threshold": 0.95,
                             "schedule": instances.anneal_schedule(1.0, 4), "backend": "mi355x",
                             "precision": "double"})
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
            lam = job.get_lambdas().real
            job.set_symmetric_gauge()
            job.run_bp(60, 1e-12, 0.0)
            out.append((chi_new, err, lam, job.density()[0]))
        finally:
            job.close()
    a, b = out
    assert a[0] == b[0] and abs(a[1] - b[1]) < 1e-10
    assert np.abs(a[2] - b[2]).max() < 1e-10
    assert np.abs(a[3] - b[3]).max() < 1e-9     # densities after the gauge and BP: pinv_eps amplifies rounding


# the split-column kernels (chi <= 16) on either side of the edge counts where a job's two extended messages are
# factored by two lane groups at once: 2,048 waves of 16, 4, 2 and 1 edges
@pytest.mark.parametrize("chi,edges", [(2, 16384), (2, 16385), (4, 8192), (4, 8193), (8, 4095), (8, 4097), (11, 2048), (11, 2049)])
def test_split_sides_match_generic(chi, edges, monkeypatch):
    from bqa_amd.native import Job
    n = edges
    ctx = config_to_context({"nodes": {i: 0.2 for i in range(n)}, "edges": {(i, (i + 1) % n): 0.3 + 1e-5 * i for i in range(n)},
                             "max_bond_dim": 2 * chi, "default_field": 0.0, "seed": 1, "bp_eps": 1e-12, "max_bp_iter_number": 60,
                             "pinv_eps": 1e-6, "damping": 0.0, "measurement_threshold": 0.95,
                             "schedule": instances.anneal_schedule(1.0, 4), "backend": "mi355x", "precision": "double"})
    rng = np.random.default_rng(chi)
    t = rng.normal(size=(n, 2, chi, chi)) + 1j * rng.normal(size=(n, 2, chi, chi))
    m = np.repeat(np.eye(chi)[None] / chi, 2 * n, axis=0).astype(complex)
    out = []
    for mask in ("", "c"):
        monkeypatch.setenv("BQA_GENERIC_KERNELS", mask)
        job = Job(ctx, "double")
        try:
            job.init_state()
            job.set_tensors(0, t / np.sqrt((np.abs(t[0]) ** 2).sum()))
            job.set_messages(m)
            out.append((job.simple_update(0.3, 1e-6)[0], job.get_lambdas().real))
        finally:
            job.close()
    # square roots of eigenvalues down to pinv_eps = 1e-6 amplify rounding by 1e3
    assert out[0][0] == out[1][0]
    assert np.abs(out[0][1] - out[1][1]).max() < 1e-10
