"""Node tensors or messages that are not finite: the canonicalisers stay within their arrays, the lambdas of the edges
they reach are not finite, and the other edges' are as the generic canonicaliser gives them."""
import numpy as np
import pytest

from bqa_amd import instances
from bqa_amd.config import config_to_context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chi", [3, 8, 17, 24, 32])
@pytest.mark.parametrize("where", ["tensors", "element", "infinity", "messages"])
def test_not_finite(chi, where, monkeypatch):
    from bqa_amd.native import Job
    n = 5
    ctx = config_to_context({"nodes": {i: 0.2 for i in range(n)}, "edges": {(i, (i + 1) % n): 0.3 for i in range(n)},
                             "max_bond_dim": chi, "default_field": 0.0, "seed": 1, "bp_eps": 1e-12,
                             "max_bp_iter_number": 20, "pinv_eps": 1e-6, "damping": 0.0, "measurement_threshold": 0.95,
                             "schedule": instances.anneal_schedule(1.0, 4), "backend": "mi355x", "precision": "double"})
    rng = np.random.default_rng(chi)
    t = rng.normal(size=(n, 2, chi, chi)) + 1j * rng.normal(size=(n, 2, chi, chi))
    m = np.repeat(np.eye(chi)[None] / chi, 2 * n, axis=0).astype(complex)
    if where == "tensors":
        t[:] = np.nan
    elif where == "element":
        t[2, 1, chi // 2, 1] = np.nan
    elif where == "infinity":
        t[2, 0, 1] = np.inf
    else:
        m[:] = np.nan
    out = []
    for mask in ("", "c"):
        print(f"[gpu] not finite: chi {chi} {where} mask '{mask}'", flush=True)
        monkeypatch.setenv("BQA_GENERIC_KERNELS", mask)
        job = Job(ctx, "double")
        try:
            job.init_state()
            job.set_tensors(0, t)
            job.set_messages(m)
            out.append((job.simple_update(0.3, 1e-6)[0], job.get_lambdas().real))
        finally:
            job.close()
    (a, la), (b, lb) = out
    assert a == b
    if where in ("tensors", "messages"):
        assert a == 0   # no lambda above pinv_eps on any edge
        return
    bad = ~np.isfinite(la).all(axis=1)
    assert bad.sum() == 2 and np.array_equal(bad, ~np.isfinite(lb).all(axis=1))   # the two edges of the node
    assert np.abs(la - lb)[~bad].max() < 1e-10
