"""GPU: the BF16 MFMA GEMM, the network's forward and backward passes against
the NumPy oracle, training, and the learned start vector."""
import sys

import numpy as np
import pytest

import hamiltonian_diagonalization_amd as hd
from hamiltonian_diagonalization_amd import learned, models
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, flush=True)
    sys.stdout.flush()


def _bf16_bits(x):
    return mo.bf16(x).view(np.uint32) >> 16


@pytest.mark.parametrize("M,N,K", [(64, 64, 16), (128, 192, 64), (64, 256, 4096)])
def test_mfma_gemm(M, N, K):
    say("mfma gemm", M, N, K)
    rng = np.random.default_rng(M + N + K)
    A = mo.bf16(rng.normal(size=(M, K)).astype(np.float32))
    B = mo.bf16(rng.normal(size=(N, K)).astype(np.float32))
    C = learned.gemm_check(_bf16_bits(A).astype(np.uint16), _bf16_bits(B).astype(np.uint16))
    want = A.astype(np.float64) @ B.astype(np.float64).T
    assert np.max(np.abs(C - want)) <= 1e-5 * np.sqrt(K) * np.max(np.abs(want))


def _data(rng, n, n_bits):
    states = np.array([int(rng.integers(0, 1 << n_bits)) for _ in range(n)], dtype=np.uint64)
    params = rng.random((n, 3)).astype(np.float32)
    targets = np.stack([rng.normal(size=n), rng.choice([-1.0, 1.0], size=n),
                        rng.random(n) + 0.5], 1).astype(np.float32)
    return states, params, targets


@pytest.mark.parametrize("n_states", [1, 3])
def test_forward_and_gradients_match_oracle(n_states):
    say("mlp forward/backward vs oracle, amplitudes", n_states)
    rng = np.random.default_rng(1)
    n_bits = 34
    net = learned.AmplitudeNet(n_bits, 3, seed=5, n_states=n_states)
    w = net.get_weights()
    states, params, targets = _data(rng, 300, n_bits)  # 300 pads to 320 rows
    targets = np.concatenate([targets] + [_data(rng, 300, n_bits)[2] for _ in range(n_states - 1)], axis=1)
    out = net.forward(states, params)
    assert out.shape == (300, 2 * n_states)
    want, _, _ = mo.forward(w, states, params, n_bits, 3, bf=True)
    live = want[:, :2 * n_states]
    assert np.max(np.abs(out - live)) <= 2e-2 * max(1.0, np.max(np.abs(live)))
    assert np.all(want[:, 2 * n_states:] == 0)
    loss, g = net.gradients(states, params, targets, lam=0.5)
    lref, gref = mo.loss_and_grads(w, states, params, targets, n_bits, 3, lam=0.5, bf=True)
    assert abs(loss - lref) <= 1e-3 * abs(lref)
    rel = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    say("gradient relative error", rel)
    assert rel < 2e-2
    # per layer too (no layer may hide behind a larger one)
    for (gw, gb), (rw, rb) in zip(learned.unflatten(g), learned.unflatten(gref.astype(np.float32))):
        assert np.linalg.norm(gw - rw) <= 5e-2 * np.linalg.norm(rw) + 1e-6
        assert np.linalg.norm(gb - rb) <= 5e-2 * np.linalg.norm(rb) + 1e-6


def test_weight_roundtrip_and_padding():
    net = learned.AmplitudeNet(22, 3, seed=1)
    w = net.get_weights()
    layers = learned.unflatten(w)
    assert np.all(layers[0][0][:, 25:] == 0) and np.all(layers[3][0][2:] == 0)
    w2 = w.copy()
    w2[:10] += 0.5
    net.set_weights(w2)
    assert np.array_equal(net.get_weights(), w2)


def test_training_and_learned_start():
    """Train on plain-solver ground states of a small sphere at a few
    parameter points; the network's start vector must overlap the held-out
    ground state better than before training, and Lanczos from it must reach
    the same eigenvalues."""
    say("mlp training on N=6 2S=15 ground states")
    n, two_s = 6, 15
    basis = hd.FockBasis(hd.Sector.lz(0, two_s), n, two_s + 1)
    rng = np.random.default_rng(3)
    pts = learned.sample_params(rng, 8)
    data = learned.make_dataset(basis, two_s, pts, per_point=2048, seed=0, log=None)
    net = learned.AmplitudeNet(two_s + 1, 3, seed=0)
    held = learned.sample_params(np.random.default_rng(99), 1)[0]
    h = learned.sphere_hamiltonian(basis, two_s, held)
    ref = h.lanczos(nev=3, tol=1e-10, seed=0)
    psi = h.eigenvector(0)
    ov0 = learned.overlap(net, basis, held, psi)
    losses = learned.train(net, data, steps=600, batch=1024, lr=2e-3, log=None)
    say("loss", losses[0], "->", losses[-1])
    assert losses[-1] < 0.3 * losses[0]
    ov1 = learned.overlap(net, basis, held, psi)
    say("overlap untrained", ov0, "trained", ov1)
    assert ov1 > max(0.9, ov0)
    start = net.start_vector(basis, held)
    r = h.lanczos(nev=3, tol=1e-10, start=start)
    assert r.converged
    assert np.max(np.abs(r.evals - ref.evals)) < 1e-9
    # the same start vector as the reference's --use-initial file, read by the
    # C++ drop-in driver: same ground state, fewer products than a random start
    import json
    import os
    import subprocess
    import tempfile
    from hamiltonian_diagonalization_amd import fileio
    driver = os.path.join(os.path.dirname(hd.__file__), "lib", "hd_diagonalize")
    with tempfile.TemporaryDirectory() as d:
        f = os.path.join(d, "initial_vector.bin")
        v = net.write_initial_vector(basis, held, f)
        assert np.array_equal(fileio.read_initial_vector(f), v) and len(v) == basis.dim
        vm = models.coulomb_list(two_s, {1: float(held[0]), 3: float(held[1]), 5: float(held[2])})
        base = [driver, "--nbr-particles", str(n), "--nbr-orbitals", str(two_s + 1), "--lz", "0",
                "--pseudopotentials", ",".join("%.17g" % x for x in vm), "--nbr-eigenvalues", "1", "--tol", "1e-10"]
        out = [json.loads(subprocess.run(base + extra, capture_output=True, text=True, check=True,
                                         timeout=300).stdout.strip().splitlines()[-1])
               for extra in ([], ["--initial-vector", f])]
    say("drop-in matvecs random start", out[0]["matvecs"], "learned start", out[1]["matvecs"])
    assert abs(out[1]["eigenvalues"][0] - ref.evals[0]) < 1e-9
    assert out[1]["matvecs"] < out[0]["matvecs"]



def test_multi_amplitude_start_vector():
    """A network with 3 amplitudes trained on the 3 lowest eigenvectors of a
    small sphere: each amplitude overlaps its eigenvector well, the start
    vector (the sum of the normalised amplitudes) overlaps all three, and
    Lanczos from it reaches the random start's eigenvalues."""
    say("mlp with 3 amplitudes on N=6 2S=15")
    n, two_s = 6, 15
    basis = hd.FockBasis(hd.Sector.lz(0, two_s), n, two_s + 1)
    pts = learned.sample_params(np.random.default_rng(3), 8)
    data = learned.make_dataset(basis, two_s, pts, per_point=2048, seed=0, log=None, n_states=3)
    assert data.targets.shape[1] == 9
    net = learned.AmplitudeNet(two_s + 1, 3, seed=0, n_states=3)
    losses = learned.train(net, data, steps=800, batch=1024, lr=2e-3, log=None)
    say("loss", losses[0], "->", losses[-1])
    held = learned.sample_params(np.random.default_rng(99), 1)[0]
    h = learned.sphere_hamiltonian(basis, two_s, held)
    ref = h.lanczos(nev=3, tol=1e-10, seed=0)
    vecs = [h.eigenvector(k) for k in range(3)]
    amp = learned.amplitude_overlaps(net, basis, held, vecs)
    v = net.start_vector(basis, held).to_array(np.float64, basis.dim)
    v /= np.linalg.norm(v)
    over = [abs(v @ x) for x in vecs]
    say("amplitude overlaps", amp, "start vector overlaps", over)
    assert min(amp) > 0.5 and min(over) > 0.2
    # the forward outputs assemble the same start vector
    out = net.forward(basis.states(), np.repeat(np.asarray(held, dtype=np.float32)[None, :], basis.dim, axis=0))
    want = np.zeros(basis.dim)
    for s in range(3):
        a = np.exp((out[:, 2 * s] - out[:, 2 * s].max()).astype(np.float64)) * np.where(out[:, 2 * s + 1] >= 0, 1.0, -1.0)
        want += a / np.linalg.norm(a)
    assert np.max(np.abs(v - want / np.linalg.norm(want))) < 1e-12
    r = h.lanczos(nev=3, tol=1e-10, start=net.start_vector(basis, held))
    assert r.converged and np.max(np.abs(r.evals - ref.evals)) < 1e-9


@pytest.mark.parametrize("n_bits,n_params,n_states,n", [
    (34, 3, 5, 1), (20, 0, 16, 31), (22, 3, 1, 33), (61, 3, 8, 127), (30, 2, 3, 129), (34, 3, 5, 256 * 256 + 37)])
def test_inference_tiles_match_oracle(n_bits, n_params, n_states, n):
    """The inference kernel at the edges of its 32-state tiles, its 128- and
    256-state groups and its output widths.  A BF16 activation that falls on
    the other side of a rounding boundary moves by 2^-8 of itself; a few such
    flips among the 256 inputs of an output stay below 2^-8 of the outputs'
    scale.  A batch large enough for the 256-state groups gives its first
    states the outputs they have alone, bit for bit."""
    say("mlp inference", n_bits, n_params, n_states, n)
    rng = np.random.default_rng(n)
    net = learned.AmplitudeNet(n_bits, n_params, seed=2, n_states=n_states)
    w = net.get_weights()
    states = rng.integers(0, 1 << n_bits, size=n).astype(np.uint64)
    params = rng.random((n, n_params)).astype(np.float32)
    out = net.forward(states, params)
    want = mo.forward(w, states, params, n_bits, n_params, bf=True)[0][:, :2 * n_states]
    assert np.max(np.abs(out - want)) <= 2.0 ** -8 * max(1.0, np.max(np.abs(want)))
    k = min(n, 129)
    assert np.array_equal(out[:k], net.forward(states[:k], params[:k]))


def test_start_vector_large_sector_matches_forward():
    """Above 65,536 states the start vector runs 256-state groups; it equals the
    sum of the normalised amplitudes assembled from the forward outputs."""
    say("start vector N=8 2S=28, 81446 states")
    basis = hd.FockBasis(hd.Sector.lz(4, 28), 8, 29)
    net = learned.AmplitudeNet(29, 3, seed=4, n_states=9)
    p = np.array([0.7, 0.2, 0.1], dtype=np.float32)
    v = net.start_vector(basis, p).to_array(np.float64, basis.dim)
    out = net.forward(basis.states(), np.repeat(p[None, :], basis.dim, axis=0))
    want = np.zeros(basis.dim)
    for s in range(9):
        a = np.exp((out[:, 2 * s] - out[:, 2 * s].max()).astype(np.float64)) * np.where(out[:, 2 * s + 1] >= 0, 1.0, -1.0)
        want += a / np.linalg.norm(a)
    assert np.linalg.norm(v - want) <= 1e-13 * np.linalg.norm(want)


@pytest.mark.parametrize("n_states,n", [(1, 1), (2, 63), (16, 65), (5, 1000), (3, 1025), (5, 4097)])
def test_gradients_at_batch_edges(n_states, n):
    """Gradients at the edges of the 64-sample padding and of the batch splits
    (a block of at least 64 samples, 16 blocks at most) against the oracle,
    and a training step against Adam's first step on those gradients."""
    say("gradients", n_states, n)
    rng = np.random.default_rng(n)
    n_bits = 28
    net = learned.AmplitudeNet(n_bits, 3, seed=6, n_states=n_states)
    w = net.get_weights()
    states, params, _ = _data(rng, n, n_bits)
    targets = np.concatenate([_data(rng, n, n_bits)[2] for _ in range(n_states)], axis=1)
    loss, g = net.gradients(states, params, targets, lam=0.5)
    lref, gref = mo.loss_and_grads(w, states, params, targets, n_bits, 3, lam=0.5, bf=True)
    assert abs(loss - lref) <= 1e-3 * abs(lref)
    # BF16 deltas: 2^-9 relative rounding per factor, amplified by cancellation
    # in the batch sum (the bound of test_forward_and_gradients_match_oracle)
    assert np.linalg.norm(g - gref) <= 2e-2 * np.linalg.norm(gref)
    bufs = [hd.DeviceBuffer.from_array(a) for a in (states, params, targets)]
    l2 = net.train_step(*bufs, n, 0.5, 1e-3)
    assert l2 == loss
    # first step: both moments corrected to g and g^2
    want = w - np.float32(1e-3) * g / (np.abs(g) + np.float32(1e-8))
    assert np.max(np.abs(net.get_weights() - want)) <= 1e-3 * 1e-4


def test_inference_special_values():
    """SiLU of the inference kernel at its ends: +inf where a sum overflows, and -0, not a
    multiple of z, where the exponential does (|z| up to the largest float)."""
    say("mlp inference, overflowing activations")
    big = np.float32(3e38)
    net = learned.AmplitudeNet(20, 0, seed=0, n_states=2)
    w = np.zeros_like(net.get_weights())
    off = 0
    for rows, cols in ((256, 64), (256, 256), (256, 256), (64, 256)):
        m = w[off:off + rows * cols].reshape(rows, cols)
        if cols == 64:
            m[:, 0:2] = big
            m[:, 2] = -big
            m[:, 3] = -1000.0
        else:
            m[:] = 1.0
        off += rows * cols + rows
    assert off == len(w)
    w[-64:] = 0.25  # the outputs' biases
    net.set_weights(w)
    states = np.array([0b0011, 0b0100, 0b1000, 0b0000], dtype=np.uint64)
    out = net.forward(states, np.zeros((4, 0), dtype=np.float32))
    assert np.all(out[0] == np.inf)
    assert np.all(out[1:] == np.float32(0.25))
