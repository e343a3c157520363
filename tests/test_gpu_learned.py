"""GPU tests of the learned jump: the HIP MLP kernels against the FP64 CPU
oracle (forward, gradients, Adam), training on the plain solver's own
trajectories, the learned solve on its own (no fallback) against the plain
solve, and the verified form's fallback rule."""
import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def L():
    assert torch.cuda.is_available()
    from egg_sync import learned
    return learned


def _rand_batch(rng, B, d=3):
    F = np.concatenate([rng.random((B, d)), rng.uniform(-1, 1, (B, 2 * d)),
                        rng.normal(0, 0.5, (B, d))], 1).astype(np.float32)
    T = rng.normal(0, 0.5, (B, d)).astype(np.float32)
    return torch.from_numpy(F).cuda(), torch.from_numpy(T).cuda()


def test_forward_matches_oracle(L):
    import mlp_oracle as M
    rng = np.random.default_rng(1)
    net = L.JumpMLP(3, seed=3)
    F, _ = _rand_batch(rng, 5000)
    got = net.forward(F).cpu().numpy()
    ref, _ = M.forward(net.state(), F.cpu().numpy(), 12, 128, 3)
    assert np.abs(got - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


def test_gradients_match_oracle(L):
    import mlp_oracle as M
    rng = np.random.default_rng(2)
    net = L.JumpMLP(3, seed=4)
    F, T = _rand_batch(rng, 4096)
    g, loss = net.grad_and_loss(F, T)
    lr, gr = M.loss_and_grad(net.state(), F.cpu().numpy(), T.cpu().numpy(), 12, 128, 3)
    assert abs(loss - lr) <= 1e-5 * max(1.0, abs(lr))
    g = g.cpu().numpy()
    assert np.abs(g - gr).max() <= 2e-4 * np.abs(gr).max()
    # Adam step against the oracle's
    p0 = net.state()
    net.train_step(F, T, lr=1e-3)
    p1, _, _ = M.adam_step(p0, g.astype(np.float64), np.zeros_like(p0), np.zeros_like(p0), 1, 1e-3)
    assert np.abs(net.state() - p1).max() <= 1e-6


def test_training_on_plain_trajectories_beats_no_jump(L):
    from egg_sync import data
    torch.manual_seed(0)
    Fs, Ts = [], []
    for seed in range(8):
        X, eps = data.config1(seed=100 + seed, n=20000)
        F, T = L.trajectory_samples(X, eps)
        Fs.append(F)
        Ts.append(T)
    F, T = torch.cat(Fs[:-2]), torch.cat(Ts[:-2])
    Fv, Tv = torch.cat(Fs[-2:]), torch.cat(Ts[-2:])
    net = L.JumpMLP(3, seed=0)
    base = float((Tv ** 2).sum(1).mean())           # predicting no jump
    losses = net.fit(F, T, epochs=6, batch=4096, lr=2e-3, log=_say)
    val = float(((net.forward(Fv) - Tv) ** 2).sum(1).mean())
    _say(f"held-out squared jump error: no jump {base:.4f}, trained MLP {val:.4f}")
    assert losses[-1] < losses[0]
    assert val < 0.8 * base


def _trained_net(L):
    net = L.JumpMLP(3, seed=0)
    Fs, Ts = [], []
    for seed in range(6):
        from egg_sync import data
        X, eps = data.config1(seed=200 + seed, n=20000)
        F, T = L.trajectory_samples(X, eps)
        Fs.append(F)
        Ts.append(T)
    net.fit(torch.cat(Fs), torch.cat(Ts), epochs=4, batch=4096, lr=2e-3)
    return net


@pytest.fixture(scope="module")
def net(L):
    return _trained_net(L)


def test_learned_solve_unverified(L, net, O):
    """The learned solve on its own (verify=False, no fallback): one plain pass,
    the jump, plain passes to EGG-SynC's stop rule.  Its labels are the cell
    rule applied to its own final positions, and at this size (the regime the
    network was trained in) its partition is within 1% of the plain solve's."""
    from egg_sync import data, metrics, solver
    X, eps = data.config1(seed=300, n=20000)
    r = L.solve_learned(X, eps, net, t0=1, alpha=0.5, clip=0.5, verify=False)
    assert r["fallback"] is False and "same_partition" not in r
    assert O.same_partition(r["labels"], O.egg_labels(r["X"], eps))
    p = solver.solve(X, eps)
    dis = metrics.disagreement(r["labels"], p["labels"])
    _say(f"learned: {r['iterations']} passes {r['seconds']*1e3:.1f} ms; plain "
         f"{p['stats']['iterations']} passes; disagreement {dis}")
    assert dis["unmatched"] + dis["noise_differs"] <= 0.01 * len(X)


def test_learned_solve_verify_falls_back_only_on_disagreement(L, net):
    """verify=True returns the learned labels when the partitions agree and the
    plain ones (fallback) when they do not; a zero-length jump keeps the plain
    trajectory's partition and does not fall back."""
    from egg_sync import data, metrics, solver
    X, eps = data.config1(seed=301, n=20000)
    u = L.solve_learned(X, eps, net, t0=1, alpha=0.5, clip=0.5, verify=False)
    v = L.solve_learned(X, eps, net, t0=1, alpha=0.5, clip=0.5, verify=True)
    p = solver.solve(X, eps)
    same = metrics.same_partition(u["labels"], p["labels"])
    _say(f"jump alpha=0.5: same partition {same}, fallback {v['fallback']}")
    assert v["same_partition"] == same and v["fallback"] == (not same)
    assert np.array_equal(v["labels"], u["labels"] if same else p["labels"])
    z = L.solve_learned(X, eps, net, t0=1, alpha=0.0, verify=True)
    assert z["same_partition"] and not z["fallback"]
    assert np.array_equal(z["labels"], L.solve_learned(X, eps, net, t0=1, alpha=0.0)["labels"])


@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 129, 65_537])
def test_forward_at_tile_edges(L, n):
    """Remainders of the 32-point MFMA tiles and of a workgroup's four.  Bound: every product and
    sum of the three layers rounds once, at most 12 + 128 + 128 deep and six of them for the
    biases and the halves, so the error is within 280 * 2^-24 of the same network on absolute
    values (no ReLU: it only shrinks them)."""
    import mlp_oracle as M
    _say("forward", n)
    net = L.JumpMLP(3, seed=3)
    F, _ = _rand_batch(np.random.default_rng(n), n)
    got = net.forward(F).cpu().numpy()
    X = F.cpu().numpy().astype(np.float64)
    ref, _ = M.forward(net.state(), X, 12, 128, 3)
    q = {k: np.abs(v) for k, v in M.unpack(net.state(), 12, 128, 3).items()}
    mag = (((np.abs(X) @ q["W1"].T + q["b1"]) @ q["W2"].T + q["b2"]) @ q["W3"].T + q["b3"])
    assert (np.abs(got - ref) <= 280 * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("B", [1, 31, 33, 257, 4097, 12_289, 33_000])
def test_gradients_at_slice_edges(L, B):
    """Batches at the edges of the training step's slices: 16, 32, 48 ... samples per workgroup,
    a last workgroup of one sample, and one batch past 32,768.  Tolerances as in
    test_gradients_match_oracle."""
    import mlp_oracle as M
    _say("train step", B)
    net = L.JumpMLP(3, seed=5)
    F, T = _rand_batch(np.random.default_rng(100 + B), B)
    p0 = net.state()
    g, loss = net.train_step(F, T, lr=1e-3)
    lr, gr = M.loss_and_grad(p0, F.cpu().numpy(), T.cpu().numpy(), 12, 128, 3)
    assert abs(loss - lr) <= 1e-5 * max(1.0, abs(lr))
    g = g.cpu().numpy()
    assert np.abs(g - gr).max() <= 2e-4 * np.abs(gr).max()
    p1, _, _ = M.adam_step(p0, g.astype(np.float64), np.zeros_like(p0), np.zeros_like(p0), 1, 1e-3)
    assert np.abs(net.state() - p1).max() <= 1e-6


def test_gradients_of_a_batch_beyond_the_partial_tiles(L):
    """A layer of 70,000 x 64 outputs does not fit the 4,194,304 floats of split-K partial tiles:
    its rows are taken in parts.  Tolerances as in test_gradients_match_oracle."""
    import mlp_oracle as M
    _say("train step 8-64-64-2, 70,000 samples")
    net = L.JumpMLP(2, hidden=64, seed=6)
    F, T = _rand_batch(np.random.default_rng(7), 70_000, d=2)
    g, loss = net.grad_and_loss(F, T)
    lr, gr = M.loss_and_grad(net.state(), F.cpu().numpy(), T.cpu().numpy(), 8, 64, 2)
    assert abs(loss - lr) <= 1e-5 * max(1.0, abs(lr))
    assert np.abs(g.cpu().numpy() - gr).max() <= 2e-4 * np.abs(gr).max()


@pytest.mark.parametrize("d", [1, 2, 3, 5, 20])
def test_features_at_row_edges(L, O, d):
    """Rows of the features at the remainders of a wavefront's 64, into memory aligned to 16 bytes
    and not: positions as given, means within 1e-6 of FP64 sums over the oracle's cells (totals
    compensated to a few 2^-24 of values up to 1), displacements as their FP32 formula."""
    nat, eps = L.nat, 0.3
    rng = np.random.default_rng(200 + d)
    for n in (1, 63, 64, 65, 1000):
        X = rng.random((n, d)).astype(np.float32)
        prev = rng.random((n, d)).astype(np.float32)
        cell = np.empty(n, np.int64)
        g = O.build_grid(X, eps)
        cell[g["order"]] = g["cell_of"]
        cnt = np.bincount(cell, minlength=g["C"])[:, None]
        mean = [np.stack([np.bincount(cell, f(X[:, l].astype(np.float64)), g["C"])
                          for l in range(d)], 1) / cnt for f in (np.sin, np.cos)]
        inv = np.float32(1.0) / np.float32(eps)
        Xd, Pd = torch.from_numpy(X).cuda(), torch.from_numpy(prev).cuda()
        for shift in (0, 1):
            for p in (Pd, None):
                _say("features", n, d, shift, p is not None)
                buf = torch.full((n * 4 * d + 2,), -7.0, device="cuda")
                rc = nat.lib().egg_sync_features_device(nat.ptr(Xd), nat.ptr(p), n, d, eps,
                                                        nat.ptr(buf[shift:]), None)
                nat.check(rc, "egg_sync_features_device")
                out = buf.cpu().numpy()
                assert np.all(out[:shift] == -7.0) and np.all(out[shift + n * 4 * d:] == -7.0)
                F = out[shift:shift + n * 4 * d].reshape(n, 4, d)
                assert np.array_equal(F[:, 0], X)
                assert np.abs(F[:, 1] - mean[0][cell]).max() <= 1e-6
                assert np.abs(F[:, 2] - mean[1][cell]).max() <= 1e-6
                want = (X - prev) * inv if p is not None else np.zeros_like(X)
                assert np.array_equal(F[:, 3], want)
