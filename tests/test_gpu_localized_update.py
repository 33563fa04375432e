"""The localised EnKF update at the edges of its matrix tiles (16 members,
16 observations, 16 nodes), and with an observation that is not finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def setup(N, m, seed):
    from tests.test_gpu_enkf import ensemble
    base, ens = ensemble(N)
    rng = np.random.RandomState(seed)
    X = 1000.0 + rng.normal(scale=30.0, size=(N, ens.n_dofs))
    obs = np.sort(rng.permutation(ens.n_dofs)[:m]).astype(np.int64)
    y = 1000.0 + rng.normal(scale=5.0, size=m)
    R = np.diag(rng.uniform(1.0, 4.0, m))
    return base, ens, X, obs, y, R, rng.normal(0.0, 1.5, (N, m))


def update(ens, base, fn, cutoff, X, obs, y, R, noise):
    import torch
    from adamantine_amd.ensemble import DataAssimilator
    da = DataAssimilator(fn, cutoff)
    da.update_dof_mapping(ens, base.node_coordinates()[obs])
    dev = torch.tensor(X, device="cuda")
    da.update_ensemble(ens, dev, y, R, noise=noise)
    return dev.cpu().numpy()


@pytest.mark.parametrize("fn", ["step_function", "gaspari_cohn"])
@pytest.mark.parametrize("N,m", [(2, 1), (15, 16), (16, 17), (17, 15),
                                 (33, 31), (48, 33), (49, 20), (64, 40)])
def test_localized_update_edges(N, m, fn):
    from adamantine_amd.ensemble import LOCALIZATION
    from tests.test_gpu_enkf import oracle_analysis
    base, ens, X, obs, y, R, noise = setup(N, m, 7 * N + m)
    got = update(ens, base, fn, 0.9e-3, X, obs, y, R, noise)
    want, _ = oracle_analysis(base, X.copy(), None, obs, y, R, noise,
                              LOCALIZATION[fn], 0.9e-3)
    scale = np.abs(want - X).max()
    # the bar of test_gpu_enkf: solves of two precisions
    assert np.abs(got - want).max() <= 1e-10 * scale + 1e-12 * 1000


def test_localized_update_not_finite():
    """Nodes out of the observation's reach keep their values."""
    base, ens, X, obs, y, R, noise = setup(5, 1, 3)
    y[0] = np.inf
    got = update(ens, base, "gaspari_cohn", 0.6e-3, X, obs, y, R, noise)
    xyz = base.node_coordinates()
    far = np.linalg.norm(xyz - xyz[obs[0]], axis=1) > 0.6e-3
    assert far.any() and not far.all()
    np.testing.assert_allclose(got[:, far], X[:, far], rtol=1e-14)
    assert not np.isfinite(got[:, obs[0]]).any()


def test_localized_update_not_finite_reaches_all():
    """An observation that is not finite makes the gains of all of them so,
    also of those out of its reach."""
    base, ens, X, obs, y, R, noise = setup(5, 3, 3)
    xyz = base.node_coordinates()
    obs = np.array([0, ens.n_dofs // 2, ens.n_dofs - 1])
    assert np.linalg.norm(xyz[obs[0]] - xyz[obs[2]]) > 0.4e-3
    y[0] = np.inf
    got = update(ens, base, "gaspari_cohn", 0.4e-3, X, obs, y, R, noise)
    far = (np.linalg.norm(xyz[:, None] - xyz[obs], axis=2) > 0.4e-3).all(1)
    assert far.any()
    np.testing.assert_allclose(got[:, far], X[:, far], rtol=1e-14)
    assert not np.isfinite(got[:, obs]).any()


def direct_update(X, xyz, obs, y, R, noise, fn, cutoff):
    """x_j + rho o (A^T S) (rho o (S^T S) / (N-1) + R)^-1 d_j / (N-1)."""
    def rho(d):
        if fn == "step_function":
            return (d <= cutoff).astype(float)
        q = 2.0 * d / cutoff
        near = ((((-0.25 * q + 0.5) * q + 0.625) * q - 5.0 / 3.0) * q * q
                + 1.0)
        s = np.maximum(q, 1.0)
        far = ((((s / 12.0 - 0.5) * s + 0.625) * s + 5.0 / 3.0) * s - 5.0) \
            * s + 4.0 - 2.0 / (3.0 * s)
        return np.where(q < 1.0, near, np.where(q < 2.0, far, 0.0))
    N = len(X)
    A = X - X.mean(0)
    S, xo = A[:, obs], xyz[obs]
    dist = np.linalg.norm(xo[:, None] - xo, axis=2)
    E = np.linalg.solve(rho(dist) * (S.T @ S) / (N - 1) + R,
                        (noise + y - X[:, obs]).T)
    out = X.copy()
    for k in range(len(obs)):
        w = rho(np.linalg.norm(xyz - xo[k], axis=1)) * (S[:, k] @ A) / (N - 1)
        out += np.outer(E[k], w)
    return out


@pytest.mark.parametrize("fn", ["step_function", "gaspari_cohn"])
@pytest.mark.parametrize("N,m,cutoff", [
    (2, 1, 0.2e-3), (2, 17, 3e-3), (5, 3, 1e-3), (8, 64, 3e-3),
    (16, 2, 0.5e-3), (16, 40, 3e-3), (17, 1, 1e-3), (17, 20, 1e-3),
    (32, 1, 0.2e-3), (32, 33, 1e-3), (33, 1, 1e-3)])
def test_localized_update_large(N, m, cutoff, fn):
    """A mesh on which some sizes take the lane-per-node kernel and some the
    matrix tiles."""
    from adamantine_amd.ensemble import EnsembleDevice, Member
    from adamantine_amd.workloads import plain_large
    base = plain_large(n_cells=(61, 32, 17))
    ens = EnsembleDevice(base, [Member() for _ in range(N)])
    rng = np.random.RandomState(100 * N + m)
    X = 1000.0 + rng.normal(scale=30.0, size=(N, ens.n_dofs))
    obs = np.sort(rng.permutation(ens.n_dofs)[:m]).astype(np.int64)
    y = 1000.0 + rng.normal(scale=5.0, size=m)
    R, noise = np.diag(rng.uniform(1.0, 4.0, m)), rng.normal(0.0, 1.5, (N, m))
    got = update(ens, base, fn, cutoff, X, obs, y, R, noise)
    want = direct_update(X, base.node_coordinates(), obs, y, R, noise, fn,
                         cutoff)
    scale = np.abs(want - X).max()
    assert scale > 0.1
    assert np.abs(got - want).max() <= 1e-10 * scale + 1e-12 * 1000
