"""The Rayleigh-Ritz step spread over the chip (bases of 512 plane waves and more off the fused small grids)
through a solve: the filtered eigensolver against the dense one at block widths on both sides of 16, and with
more k-points than the spread form takes."""
import numpy as np
import pytest

from conftest import SI_UPF

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [6, 8, 9, 20])
def test_filtered_solve_above_512_plane_waves(gpu, nb):
    # Si2 at 25 Ry: 537 plane waves on 24³; blocks of nb + 8 vectors: 14, 16, 17, 28. Both solves stop at
    # 1e-9 e/Å³, so the energies agree to the convergence, far below 1e-7 eV
    from pwk import scf

    a = 10.26 * 0.529177210903 / 2
    deck = scf.CrystalDeck([[0, a, a], [a, 0, a], [a, a, 0]], [[0, 0, 0], [0.25] * 3], [0, 0], [SI_UPF])
    out = {}
    for eig in (0, 1):
        p = scf.ScfParams(ecut_ev=25 * 13.605693122994, kgrid=(2, 2, 2), n_bands=nb, conv_threshold=1e-9,
                          energy_threshold=1e-7, smearing_sigma=0.136, eigensolver=eig)
        print("rr split: bands", nb, "eigensolver", eig, flush=True)
        out[eig] = scf.run_scf(gpu, deck, p)
        assert out[eig]["converged"] and out[eig]["npw"] >= 512
    assert abs(out[0]["e_total"] - out[1]["e_total"]) < 1e-7
    assert np.abs(out[0]["eigenvalues"] - out[1]["eigenvalues"]).max() < 1e-5


@pytest.mark.parametrize("nb", [6, 17])
def test_filtered_solve_with_many_k_points(gpu, nb):
    # 512 k-points of 537 plane waves: blocks of 14 vectors (a workgroup each) and of 25 (spread), against the
    # dense eigensolver. Both solves stop at an energy change of 1e-6 eV, which bounds what they differ by
    from pwk import scf

    a = 10.26 * 0.529177210903 / 2
    deck = scf.CrystalDeck([[0, a, a], [a, 0, a], [a, a, 0]], [[0, 0, 0], [0.25] * 3], [0, 0], [SI_UPF])
    out = {}
    for eig in (0, 1):
        p = scf.ScfParams(ecut_ev=25 * 13.605693122994, kgrid=(8, 8, 8), n_bands=nb, conv_threshold=1e-7,
                          energy_threshold=1e-6, smearing_sigma=0.136, eigensolver=eig, use_symmetry=False)
        print("rr split: 512 k-points, bands", nb, "eigensolver", eig, flush=True)
        out[eig] = scf.run_scf(gpu, deck, p)
        assert out[eig]["converged"] and out[eig]["npw"] >= 512 and len(out[eig]["eigenvalues"]) == 512
    assert abs(out[0]["e_total"] - out[1]["e_total"]) < 1e-6
    assert np.abs(out[0]["eigenvalues"] - out[1]["eigenvalues"]).max() < 1e-4
