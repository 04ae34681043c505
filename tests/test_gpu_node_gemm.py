"""Node contractions as batched matrix products (csrc/node_gemm.hip) against the NumPy oracle."""
import numpy as np
import pytest

from bqa_amd import instances
from bqa_amd.config import config_to_context
from oracle import bqa_oracle as O

pytestmark = pytest.mark.gpu


def _graph(d, n):
    if d == 2:
        edges = {(i, (i + 1) % n): 0.1 + 0.01 * i for i in range(n)}
        return {i: 0.1 for i in range(n)}, edges
    return instances.regular_uniform(n, d, seed=3, field_sigma=0.3)


def _state(d, n, chi, precision, hermitian=True):
    """Context, node tensors and messages: random, as the job stores them."""
    nodes, edges = _graph(d, n)
    ctx = config_to_context({"nodes": nodes, "edges": edges, "max_bond_dim": min(32, 2 * chi), "default_field": 0.0, "seed": 1,
                             "bp_eps": 1e-6, "max_bp_iter_number": 75, "pinv_eps": 1e-6, "damping": 0.0,
                             "measurement_threshold": 0.95, "schedule": instances.anneal_schedule(1.0, 4),
                             "backend": "mi355x", "precision": precision})
    rng = np.random.default_rng(100 * d + chi)
    store = np.complex64 if precision == "single" else np.complex128
    t = rng.normal(size=(n, 2) + (chi,) * d) + 1j * rng.normal(size=(n, 2) + (chi,) * d)
    t = (t / np.sqrt(t[0].size)).astype(store)
    a = rng.normal(size=(2, n * d, chi, chi))
    m = a[0] + 1j * a[1]
    if hermitian:
        m = m @ m.conj().transpose(0, 2, 1)
        m = (m + m.conj().transpose(0, 2, 1)) / 2
    m = (m / np.trace(m, axis1=1, axis2=2)[:, None, None]).astype(store)
    return ctx, t.astype(np.complex128), m.astype(np.complex128)


def _job(ctx, t, m, precision):
    from bqa_amd.native import Job
    job = Job(ctx, precision)
    job.init_state()
    job.set_tensors(0, t)
    job.set_messages(m)
    return job


def _sweep(ctx, t, m):
    """One sweep in FP64; the new messages are the Hermitian part of the Gram over its trace."""
    (d, lay), = ctx.degree_to_layout.items()
    new = np.empty_like(m)
    for k in range(d):
        ket = t
        for j in range(d):
            if j != k:
                ket = O.mode_product(ket, m[lay.input_msgs_position[j]], j + 2)
        new[lay.output_msgs_position[k]] = O.gram(t, ket, k + 2)
    new = (new + new.conj().transpose(0, 2, 1)) / 2
    return new / np.trace(new, axis1=1, axis2=2).real[:, None, None]


# tile edges of the rows (multiples of 8) and of the summed index (multiples of 4), odd chi (unpaired
# fibre loads), every degree, more nodes than one round of the workspace holds (degree 5, chi = 8)
SHAPES = [(2, 9, 7), (2, 12, 30), (2, 17, 5), (2, 31, 6), (2, 32, 9), (3, 9, 12), (3, 12, 10), (3, 13, 4), (3, 15, 6),
          (3, 17, 4), (3, 20, 6), (3, 24, 4), (3, 29, 4), (3, 32, 4), (4, 5, 14), (4, 6, 6), (4, 7, 8), (4, 9, 6),
          (5, 2, 6), (5, 4, 8), (5, 5, 6), (5, 8, 20), (6, 2, 8), (6, 3, 8), (6, 4, 8)]


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi,n", SHAPES)
def test_sweep_matches_oracle(d, chi, n, precision):
    ctx, t, m = _state(d, n, chi, precision)
    job = _job(ctx, t, m, precision)
    try:
        job.run_bp(1, 0.0, 0.0)
        got = job.get_messages()
    finally:
        job.close()
    want = _sweep(ctx, t, m)
    # each of the d - 1 products sums chi terms, a wave's Gram chain a quarter of 2 chi^(d-1); the products of the
    # degree-4..6 kernels and the random tensors' Grams do not cancel, so rounding stays below one unit a term
    u = 6e-8 if precision == "single" else 1.2e-16
    tol = u * ((d - 1) * chi + 2 * chi ** (d - 1) / 4 + 64) * np.abs(want).max()
    assert np.abs(got - want).max() < tol


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi,n", [(2, 12, 10), (3, 9, 6), (3, 12, 8), (3, 18, 4), (4, 6, 6), (5, 5, 6), (6, 2, 8)])
def test_extended_messages_match_generic(d, chi, n, precision, monkeypatch):
    """Lambdas of a simple update (through the extended messages) against the generic kernel's."""
    ctx, t, m = _state(d, n, chi, precision)
    lam = []
    for mask in ("", "e"):
        monkeypatch.setenv("BQA_GENERIC_KERNELS", mask)
        job = _job(ctx, t, m, precision)
        try:
            job.simple_update(0.2, 1e-6)
            lam.append(job.get_lambdas().real)
        finally:
            job.close()
    # FP64 arithmetic in both; the square roots of eigenvalues down to pinv_eps = 1e-6 amplify rounding by 1e3
    assert lam[0].shape == lam[1].shape
    assert np.abs(lam[0] - lam[1]).max() < 1e-10


def test_messages_that_are_not_hermitian():
    """Uploaded messages need not be Hermitian; they keep the contraction that does not assume it."""
    ctx, t, m = _state(3, 6, 10, "double", hermitian=False)
    job = _job(ctx, t, m, "double")
    try:
        job.run_bp(1, 0.0, 0.0)
        got = job.get_messages()
    finally:
        job.close()
    want = _sweep(ctx, t, m)
    assert np.abs(got - want).max() < 1e-10 * np.abs(want).max()


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi,chi_max,n", [(3, 8, 16, 10), (3, 11, 13, 4), (3, 12, 12, 20), (3, 16, 32, 4), (3, 31, 32, 4),
                                             (4, 5, 7, 6), (4, 8, 9, 6), (5, 4, 5, 8), (5, 5, 8, 6), (6, 3, 4, 8)])
def test_local_step_matches_generic(d, chi, chi_max, n, precision, monkeypatch):
    """Tensors and messages after the absorb alone and after the whole local step, from the same canonicalisers."""
    ctx, t, m = _state(d, n, chi, precision)
    ctx.max_bond_dim = chi_max
    got = []
    for mask in ("", "l"):
        monkeypatch.setenv("BQA_GENERIC_KERNELS", mask)
        one = []
        job = _job(ctx, t, m, precision)
        try:
            job.simple_update(0.2, 1e-6)
            one.append(job.get_tensors(0))
        finally:
            job.close()
        job = _job(ctx, t, m, precision)
        try:
            job.run_layer(0.3, 0.2, 1e-6, 1, 0.0, 0.0)
            one += [job.get_tensors(0), job.get_messages()]
        finally:
            job.close()
        got.append(one)
    u = 6e-8 if precision == "single" else 1.2e-16
    for k, (a, b) in enumerate(zip(*got)):
        # FP64 sums of d chi terms in both, rounded once to the storage type; the messages come from one sweep of them
        tol = u * 64 if precision == "single" else u * 64 * d * chi
        assert a.shape == b.shape
        assert np.abs(a - b).max() < (tol if k < 2 else 64 * tol) * np.abs(b).max()


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi,n", [(2, 9, 7), (2, 16, 40), (2, 32, 3), (3, 9, 12), (3, 16, 10), (3, 32, 4), (4, 5, 14),
                                     (4, 8, 30), (5, 4, 8), (5, 8, 20), (6, 3, 8)])
def test_density_matches_oracle(d, chi, n, precision):
    ctx, t, m = _state(d, n, chi, precision)
    job = _job(ctx, t, m, precision)
    try:
        rho, bloch = job.density()
    finally:
        job.close()
    (_, lay), = ctx.degree_to_layout.items()
    want = np.empty((n, 2, 2), dtype=np.complex128)
    want[lay.node_ids] = O.density_matrices(t, [m[lay.input_msgs_position[j]] for j in range(d)])
    # d products of chi terms each in the job's precision, summed in FP64 to entries of order one
    u = 6e-8 if precision == "single" else 1.2e-16
    tol = u * (8 * d * chi + 64)
    assert np.abs(rho - want).max() < tol
    assert np.abs(bloch[:, 2] - (want[:, 0, 0] - want[:, 1, 1]).real).max() < 2 * tol


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,chi,chi_max,n", [(2, 1, 2, 9), (2, 3, 4, 9), (2, 6, 8, 30), (3, 1, 2, 10), (3, 2, 3, 10), (3, 4, 7, 8),
                                             (3, 5, 8, 20), (4, 1, 2, 14), (4, 2, 4, 8), (5, 1, 2, 8)])
def test_growing_local_step_matches_generic(d, chi, chi_max, n, precision, monkeypatch):
    """The local step from a smaller bond dimension (the tensor padded in LDS), from the bond dimension-1 extended
    messages on."""
    test_local_step_matches_generic(d, chi, chi_max, n, precision, monkeypatch)


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("d,n", [(2, 5), (3, 10), (4, 300), (5, 8)])
def test_extended_messages_of_bond_dimension_one(d, n, precision, monkeypatch):
    ctx, t, m = _state(d, n, 1, precision)
    lam = []
    for mask in ("", "e"):
        monkeypatch.setenv("BQA_GENERIC_KERNELS", mask)
        job = _job(ctx, t, m, precision)
        try:
            job.simple_update(0.2, 1e-6)
            lam.append(job.get_lambdas().real)
        finally:
            job.close()
    assert np.abs(lam[0] - lam[1]).max() < 1e-13   # a handful of FP64 products of numbers of order one
