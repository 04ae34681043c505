"""Uploaded messages that are not Hermitian, or Hermitian and not positive, against the NumPy oracle: they need kernels
that apply every message to the ket and canonicalisers that factor any matrix."""
import numpy as np
import pytest

from bqa_amd import instances
from bqa_amd.config import config_to_context
from oracle import bqa_oracle as O

pytestmark = pytest.mark.gpu

U = {"single": 6e-8, "double": 1.2e-16}


def _state(d, n, chi, precision, kind):
    """Config, node tensors and messages as the job stores them; kind: "any", "indefinite" or "positive"."""
    if d == 2:
        nodes, edges = {i: 0.1 for i in range(n)}, {(i, (i + 1) % n): 0.1 + 0.01 * i for i in range(n)}
    else:
        nodes, edges = instances.regular_uniform(n, d, seed=3, field_sigma=0.3)
    cfg = {"nodes": nodes, "edges": edges, "max_bond_dim": min(32, 2 * chi), "default_field": 0.0, "seed": 1, "bp_eps": 1e-6,
           "max_bp_iter_number": 75, "pinv_eps": 1e-6, "damping": 0.0, "measurement_threshold": 0.95,
           "schedule": instances.anneal_schedule(1.0, 4)}
    rng = np.random.default_rng(100 * d + chi)
    store = np.complex64 if precision == "single" else np.complex128
    t = rng.normal(size=(n, 2) + (chi,) * d) + 1j * rng.normal(size=(n, 2) + (chi,) * d)
    t = (t / np.sqrt(t[0].size)).astype(store)
    m = rng.normal(size=(n * d, chi, chi)) + 1j * rng.normal(size=(n * d, chi, chi))
    if kind == "positive":
        m = m @ m.conj().transpose(0, 2, 1)
    if kind != "any":
        m = m + m.conj().transpose(0, 2, 1)
    # a trace of one, by the diagonal's mean: traces of random matrices may vanish
    m = m - (np.trace(m, axis1=1, axis2=2)[:, None, None] / chi - 1) * np.eye(chi) if kind != "positive" else m
    m = (m / np.trace(m, axis1=1, axis2=2)[:, None, None]).astype(store)
    return cfg, t.astype(np.complex128), m.astype(np.complex128)


def _job(cfg, t, m, precision):
    from bqa_amd.native import Job
    job = Job(config_to_context(dict(cfg, backend="mi355x", precision=precision)), precision)
    job.init_state()
    job.set_tensors(0, t)
    job.set_messages(m)
    return job


def _layout(cfg):
    (_, lay), = O.make_context(cfg).classes.items()
    return lay


def _sweep(cfg, t, m, d):
    """New messages in FP64: the Hermitian part of the Gram over its trace."""
    lay = _layout(cfg)
    new = np.empty_like(m)
    for k, msg in enumerate(O.pass_msgs(t, [m[lay.input_pos[j]] for j in range(d)])):
        new[lay.output_pos[k]] = msg
    # the kernels take the trace's real part
    tr = np.empty(len(m), dtype=complex)
    for k in range(d):
        ket = t
        for j in range(d):
            if j != k:
                ket = O.mode_product(ket, m[lay.input_pos[j]], j + 2)
        tr[lay.output_pos[k]] = np.trace(O.gram(t, ket, k + 2), axis1=1, axis2=2)
    new = new * tr[:, None, None]
    new = (new + new.conj().transpose(0, 2, 1)) / 2
    return new / tr.real[:, None, None]


# every kernel that moves messages to the bra side in some precision, and neighbours that do not
SHAPES = [(2, 4, 9), (2, 8, 9), (2, 12, 9), (3, 1, 8), (3, 2, 8), (3, 4, 30), (3, 6, 8), (3, 8, 10), (3, 10, 6), (3, 16, 4),
          (4, 3, 10), (4, 6, 8), (4, 8, 12), (5, 3, 8), (5, 5, 6)]


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("damping,sweeps", [(0.0, 1), (0.0, 3), (0.3, 3)])
@pytest.mark.parametrize("d,chi,n", SHAPES)
def test_sweeps(d, chi, n, damping, sweeps, precision):
    cfg, t, m = _state(d, n, chi, precision, "any")
    job = _job(cfg, t, m, precision)
    try:
        assert job.run_bp(sweeps, 0.0, damping)[0] == sweeps
        got = job.get_messages()
    finally:
        job.close()
    want = m
    for _ in range(sweeps):
        new = _sweep(cfg, t, want, d)
        want = damping * want + (1 - damping) * new
    # the last iterate is not damped.  Each of the d - 1 products sums chi terms and a Gram 2 chi^(d-1); random
    # messages cancel in the trace by about chi^((d-1)/2), and each sweep adds its own
    tol = 32 * U[precision] * ((d - 1) * chi + chi ** (d - 1) + 64) * sweeps * np.abs(new).max() * chi ** ((d - 1) / 2)
    assert np.abs(got - new).max() < tol


@pytest.mark.parametrize("variant", range(5))
@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi,n", [(2, 4, 9), (2, 8, 70), (3, 3, 8), (3, 4, 30), (3, 6, 8), (3, 8, 10), (3, 8, 600), (3, 16, 4),
                                     (4, 4, 10), (4, 8, 12), (4, 8, 300)])
def test_launch_variants_on_positive_messages(d, chi, n, precision, variant, monkeypatch):
    """One sweep of the kernels that Hermitian messages run, under each launch variant (variants that a shape does not
    have run as the first)."""
    monkeypatch.setenv("BQA_BP_VARIANT", str(variant))
    cfg, t, m = _state(d, n, chi, precision, "positive")
    job = _job(cfg, t, m, precision)
    try:
        job.run_bp(1, 0.0, 0.0)
        got = job.get_messages()
    finally:
        job.close()
    want = _sweep(cfg, t, m, d)
    # each of the d - 1 products sums chi terms, a Gram's chains a quarter of 2 chi^(d-1); nothing cancels in the trace
    tol = U[precision] * ((d - 1) * chi + chi ** (d - 1) / 2 + 64) * np.abs(want).max()
    assert np.abs(got - want).max() < tol


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi,n", SHAPES)
def test_readout(d, chi, n, precision):
    cfg, t, m = _state(d, n, chi, precision, "any")
    job = _job(cfg, t, m, precision)
    try:
        rho, _ = job.density()
    finally:
        job.close()
    lay = _layout(cfg)
    want = np.empty((n, 2, 2), dtype=complex)
    want[lay.node_ids] = O.density_matrices(t, [m[lay.input_pos[j]] for j in range(d)])
    tol = 32 * U[precision] * (d * chi + 64) * np.abs(want).max() ** 2 * chi ** (d / 2)
    assert np.abs(rho - want).max() < tol


@pytest.mark.parametrize("d,chi,n", SHAPES)
def test_extended_messages(d, chi, n, monkeypatch):
    """Lambdas through the extended messages and the generic canonicaliser, in FP64."""
    monkeypatch.setenv("BQA_GENERIC_KERNELS", "c")
    _simple_update(d, chi, n, "any")


def _simple_update(d, chi, n, kind):
    cfg, t, m = _state(d, n, chi, "double", kind)
    job = _job(cfg, t, m, "double")
    try:
        job.simple_update(0.2, 1e-6)
        lam = job.get_lambdas().real
    finally:
        job.close()
    ctx = O.make_context(cfg)
    st = O.init_state(ctx)
    st.tensors, st.msgs, st.chi = {d: t}, m, chi
    ext = O.extended_msgs(ctx, st, 0.2)
    want = O.canonicalizers(ext, 1e-6)[0].real
    # square roots of singular values down to pinv_eps = 1e-6 amplify rounding of the largest by 1e3
    tol = 1e-10 * max(1.0, np.abs(ext).max())
    assert np.abs(lam - want[:, :lam.shape[1]]).max() < tol


@pytest.mark.parametrize("kind", ["any", "indefinite", "positive"])
@pytest.mark.parametrize("d,chi,n", SHAPES + [(2, 17, 5), (2, 24, 5), (2, 32, 4)])
def test_simple_update(d, chi, n, kind):
    """Lambdas through the extended messages and the job's own canonicalisers, in FP64."""
    _simple_update(d, chi, n, kind)


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi,n", [(3, 4, 10), (3, 8, 10), (3, 10, 6), (4, 8, 12)])
def test_messages_after_a_sweep_are_the_jobs_own(d, chi, n, precision, monkeypatch):
    """Once a sweep has replaced them, the same kernels serve the messages as if they had been uploaded so, bit for
    bit; a run that keeps the upload goes on with it."""
    monkeypatch.setenv("BQA_AUTOTUNE", "0")   # launch variants differ in rounding
    cfg, t, m = _state(d, n, chi, precision, "any")
    out = []
    job = _job(cfg, t, m, precision)
    try:
        job.run_bp(2, 0.0, 0.0)
        own = job.get_messages()
        rho = job.density()[0]
        out.append((rho, (job.run_bp(2, 0.0, 0.0), job.get_messages())[1]))
    finally:
        job.close()
    job = _job(cfg, t, own, precision)
    try:
        rho = job.density()[0]
        out.append((rho, (job.run_bp(2, 0.0, 0.0), job.get_messages())[1]))
    finally:
        job.close()
    assert np.array_equal(own, own.conj().transpose(0, 2, 1))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    # any distance converges: the upload is kept, and the next run's sweep reads it
    job = _job(cfg, t, m, precision)
    try:
        assert job.run_bp(5, 1e9, 0.0)[1]
        assert np.array_equal(job.get_messages(), m)
        job.run_bp(2, 0.0, 0.0)
        assert np.array_equal(job.get_messages(), own)
    finally:
        job.close()

def test_batch_after_an_upload():
    """A serving batch's step from such messages gives what the job's own step gives."""
    from bqa_amd.native import Batch
    out = []
    for batched in (False, True):
        jobs = []
        try:
            for d, chi, n, kind in ((3, 4, 10, "any"), (3, 8, 10, "indefinite"), (4, 8, 12, "any"), (3, 8, 10, "positive")):
                cfg, t, m = _state(d, n, chi, "double", kind)
                cfg["max_bond_dim"] = chi
                jobs.append(_job(cfg, t, m, "double"))
            if batched:
                batch = Batch(len(jobs))
                batch.run_layer(jobs, 0.3, 0.2, 1e-6, 40, 1e-9, 0.0)
            else:
                for job in jobs:
                    job.run_layer(0.3, 0.2, 1e-6, 40, 1e-9, 0.0)
            out.append([job.density()[0] for job in jobs])
        finally:
            for job in jobs:
                job.close()
    for a, b in zip(*out):
        assert np.abs(a - b).max() < 1e-9   # pinv_eps = 1e-6 amplifies the rounding between launch variants
