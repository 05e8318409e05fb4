"""POD products at the edges of their tiles: Gram matrices around multiples of
64 snapshots (tiles below the diagonal are mirrored), bases around 64 modes (the
narrow product), rows that end inside a stage of 32. Bars: singular values within
1e-12 of the largest (FP64 Gram eigenvalues of well-separated values), an
orthonormal basis to 1e-12, and the modes' projector to 1e-9 against numpy's SVD
(gaps of 10 %, perturbations of 1e-12)."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ns,k", [(97, 1, 1), (1000, 63, 10), (4096, 64, 40), (4097, 65, 64), (9001, 130, 65),
                                    (8192, 128, 30)])
def test_pod_matches_svd(n, ns, k):
    print(f"[gpu] POD n={n} ns={ns} k={k}", flush=True)
    rng = np.random.default_rng(n + ns)
    u = np.linalg.qr(rng.standard_normal((n, ns)))[0]
    v = np.linalg.qr(rng.standard_normal((ns, ns)))[0]
    s = 0.9 ** np.arange(ns)
    S = (u * s) @ v.T
    phi, sigma = shaw_amd.pod_basis(S, k)
    assert np.abs(sigma[:k] - s[:k]).max() <= 1e-12
    assert np.abs(phi.T @ phi - np.eye(k)).max() <= 1e-12
    # singular vectors of separated values: the overlap with the exact ones is 1 up to the square of the error
    overlap = np.abs(np.einsum("ij,ij->j", phi, u[:, :k]))
    assert np.abs(overlap - 1.0).max() <= 1e-9
