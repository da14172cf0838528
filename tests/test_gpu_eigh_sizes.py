"""The batched dense eigensolver around the sizes where its kernels change (one wave to 64 rows, rows per
lane to 128, 192 and 256, the general form above) against LAPACK."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 65, 128, 129, 169, 192, 193, 256, 257])
def test_dense_eigh_kernel_sizes(gpu, n):
    # a random matrix, one with degenerate levels, and a block-diagonal one whose columns need no
    # reflector (zero below the diagonal) among others; few pairs, and so many that the inverse
    # iteration's factors leave the LDS. Bounds: n·eps·|H| ≈ 6e-14·|H| for values and residuals
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    q, _ = np.linalg.qr(a)
    levels = np.repeat(np.arange((n + 2) // 3), 3)[:n].astype(float)
    block = (a + a.conj().T) / 2
    block[: n // 2, n // 2:] = block[n // 2:, : n // 2] = 0
    block[3, :] = block[:, 3] = 0
    hs = [(a + a.conj().T) / 2, (q * levels) @ q.conj().T, block]
    for nb in (1, 8, 40):
        print("eigh", n, nb, flush=True)
        w, v = gpu.dense_eigh(np.stack(hs), nb)
        for i, h in enumerate(hs):
            norm = np.linalg.norm(h, 2)
            assert np.abs(w[i] - np.linalg.eigvalsh(h)[:nb]).max() < 2e-13 * norm
            assert np.linalg.norm(h @ v[i] - v[i] * w[i], axis=0).max() < 1e-11 * norm
            assert np.abs(v[i].conj().T @ v[i] - np.eye(nb)).max() < 1e-10


@pytest.mark.parametrize("n", [40, 64, 65, 100, 169, 240, 257])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_dense_eigh_passes_nan_on(gpu, n, bad):
    # a NaN or an infinity in the first column reaches every eigenvalue and vector, whichever kernel runs
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    h = (a + a.conj().T) / 2
    h[5, 0] = h[0, 5] = bad
    print("eigh", n, bad, flush=True)
    w, v = gpu.dense_eigh(h[None], 6)
    assert np.isnan(w).all() and np.isnan(v).all()
