"""The z-plane passes of the sphere-pruned transforms (square grids) against numpy in 64 bits, at the
sizes where their layout changes: planes per workgroup, sums in registers or LDS, bases whose columns
are two runs of rows or every row, band counts around the planes per workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def sphere(dims, m):
    """Miller indices with |n|² ≤ m² in n1 → n2 → n3 order, and their flat grid index."""
    r = np.arange(-m, m + 1)
    n = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3)
    n = n[(n * n).sum(1) <= m * m]
    i = [n[:, d] % dims[d] for d in range(3)]
    return n.astype(np.int32), (i[0] * dims[1] + i[1]) * dims[2] + i[2]


def setup(acc, dims, m):
    miller, idx = sphere(dims, m)
    acc.prepare_buffers(dims, np.ones(int(np.prod(dims))))
    acc.set_basis(miller)
    acc.set_nk(1)
    acc.set_kinetic(0, (miller.astype(float) ** 2).sum(1))
    return miller, idx


def bands(rng, nb, npw):
    psi = rng.standard_normal((nb, npw)) + 1j * rng.standard_normal((nb, npw))
    return psi / np.linalg.norm(psi, axis=1)[:, None]


def to_grid(psi, idx, dims):
    g = np.zeros((len(psi), int(np.prod(dims))), dtype=complex)
    g[:, idx] = psi
    return np.fft.ifftn(g.reshape((len(psi),) + tuple(dims)), axes=(1, 2, 3)) * np.prod(dims)


# (grid, sphere radius). Bases within a quarter of every axis take the pruned passes, the others the
# general ones: 15 with every row carrying sticks and 16 with all but one, 25 and 27 with several planes
# per workgroup, 45 and 48 around the register limit of the FP64 sums, 64 and 72 with sums in LDS, 81 the
# longest line; radii at the quarter (25/6, 45/11, 60/14) and far below it.
PLANES = [((15, 15, 18), 7), ((16, 16, 12), 5), ((25, 25, 25), 6), ((27, 27, 27), 13), ((27, 27, 32), 6),
          ((45, 45, 16), 7), ((45, 45, 45), 11), ((48, 48, 9), 4), ((48, 48, 20), 4), ((60, 60, 10), 4),
          ((60, 60, 60), 14), ((64, 64, 15), 7), ((64, 64, 30), 7), ((72, 72, 8), 3), ((72, 72, 81), 3),
          ((81, 81, 72), 3), ((81, 81, 12), 5), ((75, 75, 15), 3), ((80, 80, 16), 3), ((80, 80, 30), 9),
          # nx != ny: pruned (held rows moved between launches), at the quarter, and the whole-grid transforms;
          # 64 and 72 points along x on both sides of the FP64 limit
          ((50, 25, 25), 6), ((25, 50, 27), 6), ((16, 81, 15), 3), ((80, 18, 20), 4), ((20, 25, 15), 7),
          ((54, 30, 20), 4), ((60, 24, 27), 5), ((64, 32, 30), 7), ((72, 36, 30), 7)]


@pytest.mark.parametrize("dims,m", PLANES)
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 4e-6)])
def test_density_planes(gpu, dims, m, prec, tol):
    # tolerance: three axes of log2(N) ≈ 6 roundings each on ψ, doubled by the square (FP32: 18 ·
    # 6e-8 · 2 = 2.1e-6 of the largest value)
    gpu.set_fused_hpsi(False)  # the plane passes also where a fused small-grid kernel exists
    try:
        miller, idx = setup(gpu, dims, m)
        rng = np.random.default_rng(31)
        for nb in (1, 2, 3, 11, 12):
            psi = bands(rng, nb, len(miller))
            fw = rng.uniform(0.1, 2.0, nb)
            fw[nb // 2] = 0.0 if nb > 2 else fw[nb // 2]  # a band without weight is left out
            rho0 = rng.uniform(0.0, 1e-3, int(np.prod(dims)))
            print("density planes", dims, m, prec, "bands", nb, flush=True)
            got = gpu.density(psi, fw, rho0, prec)
            ref = rho0 + (fw[:, None] * np.abs(to_grid(psi, idx, dims).reshape(nb, -1)) ** 2).sum(0)
            assert np.abs(got - ref).max() < tol * np.abs(ref).max()
        psi[:] = np.nan  # bands without weight are not read
        assert np.array_equal(gpu.density(psi, np.zeros(nb), rho0, prec), rho0)
    finally:
        gpu.set_fused_hpsi(True)


@pytest.mark.parametrize("dims,m", PLANES)
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-14), ("fp32", 4e-6)])
def test_hpsi_planes(gpu, dims, m, prec, tol):
    # tolerance relative to the largest |Hψ|: six line transforms of about 6 roundings each (FP32: 36 ·
    # 6e-8 = 2.2e-6, FP64 36 · 1.1e-16 = 4e-15)
    gpu.set_fused_hpsi(False)
    try:
        miller, idx = setup(gpu, dims, m)
        rng = np.random.default_rng(32)
        n = int(np.prod(dims))
        v = rng.uniform(-13.6, 13.6, dims)
        gpu.set_veff((np.fft.fftn(v) / n).reshape(-1))
        # a few bands, and enough of them for several planes per workgroup, the last one not full
        many = [245] if dims[0] <= 16 else [107] if dims[0] <= 32 else [74] if dims[0] <= 48 else []
        for nb in [1, 2, 5] + many:
            psi = bands(rng, nb, len(miller))
            print("hpsi planes", dims, m, prec, "bands", nb, flush=True)
            got = gpu.hpsi(0, psi, prec)
            w = np.fft.fftn(to_grid(psi, idx, dims) * v, axes=(1, 2, 3)).reshape(nb, -1)[:, idx] / n
            ref = w + (miller.astype(float) ** 2).sum(1) * psi
            assert np.abs(got - ref).max() < tol * np.abs(ref).max()
    finally:
        gpu.set_fused_hpsi(True)


@pytest.mark.parametrize("dims,m", [((25, 25, 25), 6), ((27, 27, 27), 9), ((27, 25, 32), 6), ((15, 15, 15), 3)])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 6e-6), ("split_bf16", 2e-5)])
@pytest.mark.parametrize("channels,counts", [((7, 7, 7), (3, 1, 18)), ((80, 80), (33, 161)), ((5, 0, 5), (2, 2, 2)),
                                             ((3, 3, 6, 6, 6), (2, 1, 2, 3, 1)), ((2,) * 17, (1,) * 17), ((4,) * 130, (1, 2) * 65)])
def test_hpsi_batch_sticks(gpu, dims, m, prec, tol, channels, counts):
    # k × band batches: one launch per pass and grouped projector products (one fused launch on the small grid)
    # for up to 128 consecutive entries with one channel count. Tolerance relative to the largest |Hψ|:
    # the transforms as above plus sums over npw (projection) and nch terms, √npw ≈ 60 roundings
    # (FP32 3.6e-6, split-bf16 2^-16 per product: 1.5e-5)
    miller, idx = setup(gpu, dims, m)
    npw, n = len(miller), int(np.prod(dims))
    rng = np.random.default_rng(33)
    v = rng.uniform(-13.6, 13.6, dims)
    gpu.set_veff((np.fft.fftn(v) / n).reshape(-1))
    gpu.set_nk(len(channels))
    kin, proj = [], []
    for ik, nch in enumerate(channels):
        kin.append((miller.astype(float) ** 2).sum(1) * (1 + 0.1 * ik))
        gpu.set_kinetic(ik, kin[-1])
        b = (rng.standard_normal((npw, nch)) + 1j * rng.standard_normal((npw, nch))) / np.sqrt(npw)
        d = rng.standard_normal((nch, npw)) + 1j * rng.standard_normal((nch, npw))
        proj.append((b, d))
        gpu.set_nonlocal(ik, b, d)
    order = list(range(len(channels)))[::-1]  # entries in another order than the k-points
    nbands = [counts[i] for i in order]
    psi = bands(rng, sum(nbands), npw)
    print("hpsi batch", dims, prec, channels, nbands, flush=True)
    for _ in range(2):
        got = gpu.hpsi_batch(order, nbands, psi, prec)
    w = np.fft.fftn(to_grid(psi, idx, dims) * v, axes=(1, 2, 3)).reshape(len(psi), -1)[:, idx] / n
    b0 = 0
    for ik, nb in zip(order, nbands):
        p = psi[b0:b0 + nb]
        w[b0:b0 + nb] += kin[ik] * p + (proj[ik][0] @ (proj[ik][1] @ p.T)).T
        b0 += nb
    assert np.abs(got - w).max() < tol * np.abs(w).max()
    # fewer entries next
    got = gpu.hpsi_batch(order[:1], nbands[:1], psi[:nbands[0]], prec)
    assert np.abs(got - w[:nbands[0]]).max() < tol * np.abs(w).max()


# batches run between the replays of one with k-points 2, 0, 1 and 5, 3, 4 bands (or 18 entries): fewer
# entries, the same size with other k-points and counts, more entries, more bands
OTHERS = [([2, 0], [5, 3]), ([1], [12]), ([0, 1, 2], [4, 5, 3]), ([1, 1, 0, 2, 0], [1, 2, 3, 1, 9])]


@pytest.mark.parametrize("dims", [(25, 25, 25), (27, 25, 32), (15, 15, 15), (20, 20, 20)])
@pytest.mark.parametrize("order,nbands", [([2, 0, 1], [5, 3, 4]), ([0, 2, 1] * 6, [1] * 18)])
def test_hpsi_batch_captured(gpu, dims, order, nbands):
    # replays of a captured batch equal the same batch run directly, whatever other batches (of either
    # precision) run between them: on the stick path and on the fused small grids
    import torch

    miller, _ = setup(gpu, dims, 6 if dims[0] > 20 else 3)
    npw, nch = len(miller), 7
    rng = np.random.default_rng(34)
    gpu.set_veff((np.fft.fftn(rng.uniform(-13.6, 13.6, dims)) / np.prod(dims)).reshape(-1))
    gpu.set_nk(3)
    for ik in range(3):
        gpu.set_kinetic(ik, (miller.astype(float) ** 2).sum(1) * (1 + 0.1 * ik))
        b = (rng.standard_normal((npw, nch)) + 1j * rng.standard_normal((npw, nch))) / np.sqrt(npw)
        gpu.set_nonlocal(ik, b, b.conj().T.copy())
    most = max([sum(nbands)] + [sum(nb) for _, nb in OTHERS])
    psi = torch.from_numpy(bands(rng, most, npw).astype(np.complex64)).cuda()
    psi64 = psi.to(torch.complex128)
    out, other, other64 = torch.empty_like(psi), torch.empty_like(psi), torch.empty_like(psi64)
    torch.cuda.synchronize()

    def batch():
        gpu.hpsi_batch_dev(order, nbands, psi.data_ptr(), out.data_ptr(), "fp32")

    def others():
        for ks, nb in OTHERS:
            gpu.hpsi_batch_dev(ks, nb, psi.data_ptr(), other.data_ptr(), "fp32")
            yield ks
            gpu.hpsi_batch_dev(ks, nb, psi64.data_ptr(), other64.data_ptr(), "fp64")
            yield ks

    list(others())  # workspaces
    out.zero_()
    torch.cuda.synchronize()
    batch()
    gpu.sync()
    want = out.cpu()
    print("captured batch", dims, flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(torch.cuda.ExternalStream(gpu.stream)):
        graph.capture_begin(capture_error_mode="thread_local")
        try:
            batch()
        finally:
            graph.capture_end()
        for ks in others():
            gpu.sync()
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out.cpu(), want), ks
        out.zero_()
        batch()
        gpu.sync()
        assert torch.equal(out.cpu(), want)


# more bands than the sticks and held rows of one launch sequence take (256 MiB), and than a launch has rows
@pytest.mark.parametrize("dims,m,nb", [((27, 25, 32), 6, 2500), ((9, 8, 8), 1, 66000)])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 4e-6)])
def test_unequal_axes_many_bands(gpu, dims, m, nb, prec, tol):
    # tolerances as for the same passes above (FP64: plus nb·eps / 10 of the sums over the bands)
    miller, idx = setup(gpu, dims, m)
    npw, n = len(miller), int(np.prod(dims))
    rng = np.random.default_rng(38)
    v = rng.uniform(-13.6, 13.6, dims)
    gpu.set_veff((np.fft.fftn(v) / n).reshape(-1))
    psi = bands(rng, nb, npw)
    fw = rng.uniform(0.1, 2.0, nb)
    fw[::7] = 0.0
    rho0 = rng.uniform(0.0, 1e-3, n)
    print("many bands", dims, nb, prec, flush=True)
    got = gpu.hpsi(0, psi, prec)
    rho = gpu.density(psi, fw, rho0, prec)
    ref, diff, top = rho0.copy(), 0.0, 0.0
    for b in range(0, nb, 500):
        g = to_grid(psi[b:b + 500], idx, dims)
        w = np.fft.fftn(g * v, axes=(1, 2, 3)).reshape(len(g), -1)[:, idx] / n
        w += (miller.astype(float) ** 2).sum(1) * psi[b:b + 500]
        diff, top = max(diff, np.abs(got[b:b + 500] - w).max()), max(top, np.abs(w).max())
        ref += (fw[b:b + 500, None] * np.abs(g.reshape(len(g), -1)) ** 2).sum(0)
    assert diff < tol * top
    assert np.abs(rho - ref).max() < (tol + nb * 2.3e-17) * np.abs(ref).max()


@pytest.mark.parametrize("dims,m", [((25, 25, 25), 6), ((27, 25, 32), 6), ((27, 27, 27), 13)])
def test_density_captured(gpu, dims, m):
    # a captured density reads the caller's weights at each replay, also where a band gains or loses its weight
    import torch

    miller, _ = setup(gpu, dims, m)
    rng = np.random.default_rng(35)
    nb, n = 7, int(np.prod(dims))
    psi = bands(rng, nb, len(miller))
    dev = torch.from_numpy(psi).cuda()
    rho = torch.zeros(n, dtype=torch.float64, device="cuda")
    fw = rng.uniform(0.1, 2.0, nb)
    torch.cuda.synchronize()
    gpu.density_dev(nb, dev.data_ptr(), fw, rho.data_ptr(), "fp64")  # workspaces
    gpu.sync()
    print("captured density", dims, m, flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(torch.cuda.ExternalStream(gpu.stream)):
        graph.capture_begin(capture_error_mode="thread_local")
        try:
            gpu.density_dev(nb, dev.data_ptr(), fw, rho.data_ptr(), "fp64")
        finally:
            graph.capture_end()
        for zero in ([], [2], [0, 6]):
            fw[:] = rng.uniform(0.1, 2.0, nb)
            fw[zero] = 0.0
            rho.zero_()
            graph.replay()
            torch.cuda.synchronize()
            want = gpu.density(psi, fw, None, "fp64")
            # sums over other groups of the bands: a rounding per band
            assert np.abs(rho.cpu().numpy() - want).max() < nb * 2.3e-16 * want.max()


@pytest.mark.parametrize("dims,m", [((25, 25, 25), 6), ((27, 25, 32), 6), ((27, 27, 27), 13)])
@pytest.mark.parametrize("first", [[2, 3, 4, 5, 6], list(range(7))])
def test_density_captured_after_unoccupied_bands(pwk_mod, gpu, dims, m, first):
    # the call before the capture has bands without weight (or nothing but such bands); the captured one uses
    # every band
    import torch

    acc = pwk_mod.GpuAccelerator(0)  # workspaces as that first call leaves them
    try:
        miller, _ = setup(acc, dims, m)
        rng = np.random.default_rng(37)
        nb, n = 7, int(np.prod(dims))
        psi = bands(rng, nb, len(miller))
        dev = torch.from_numpy(psi).cuda()
        rho = torch.zeros(n, dtype=torch.float64, device="cuda")
        fw = rng.uniform(0.1, 2.0, nb)
        weights = fw.copy()
        fw[first] = 0.0
        torch.cuda.synchronize()
        print("captured density after zero weights", dims, m, first, flush=True)
        acc.density_dev(nb, dev.data_ptr(), fw, rho.data_ptr(), "fp64")
        acc.sync()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(torch.cuda.ExternalStream(acc.stream)):
            graph.capture_begin(capture_error_mode="thread_local")
            try:
                acc.density_dev(nb, dev.data_ptr(), fw, rho.data_ptr(), "fp64")
            finally:
                graph.capture_end()
            fw[:] = weights
            want = acc.density(psi, fw, None, "fp64")
            for _ in range(3):
                rho.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert np.abs(rho.cpu().numpy() - want).max() < nb * 2.3e-16 * want.max()
    finally:
        acc.close()


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-13), ("fp32", 2e-5), ("split_bf16", 5e-5)])
def test_zgemm_column_blocks(gpu, prec, tol):
    # column counts around the tiles of 16, 32 and 48 columns (FP64: 32 at most) with and without split K, row
    # counts that make few and many tiles, reductions around the two-step turn of the main loop and around the
    # split-K chunk; the product stored, and added to what is there
    import torch

    rng = np.random.default_rng(34)
    dt = torch.complex128 if prec == "fp64" else torch.complex64
    edges = (1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 96, 97, 161)
    sizes = [(63, 143, 31), (65, 160, 33), (1, 161, 17), (256, 160, 1000), (3000, 80, 48), (512, 144, 2001), (130, 289, 255),
             (16, 16, 257)] + [(70, n, 1030) for n in edges] + [(9000, n, 40) for n in edges]
    for (m, n, k) in sizes:
        A = rng.standard_normal((m, k)) + 1j * rng.standard_normal((m, k))
        B = rng.standard_normal((k, n)) + 1j * rng.standard_normal((k, n))
        dA, dB = (torch.from_numpy(np.ascontiguousarray(x.T)).to(dt).cuda() for x in (A, B))
        dC = torch.full((n, m), float("nan"), dtype=dt).cuda()
        torch.cuda.synchronize()
        ref = A @ B
        for add in (False, True):
            gpu.zgemm_dev(m, n, k, dA.data_ptr(), m, dB.data_ptr(), k, dC.data_ptr(), m, precision=prec, accumulate=add)
            gpu.sync()
            err = np.abs(dC.cpu().numpy().T - (2 if add else 1) * ref).max() / np.abs(ref).max()
            print("zgemm", prec, (m, n, k), add, f"{err:.2e}", flush=True)
            assert err < tol, (m, n, k, add)


@pytest.mark.parametrize("dims", [(25, 25, 25), (27, 25, 32)])
def test_captured_workspaces_survive_growth(pwk_mod, gpu, dims):
    # replays of a captured H·ψ batch and density after larger direct calls, which grow every workspace that
    # the graph's kernels use
    import torch

    acc = pwk_mod.GpuAccelerator(0)  # workspaces of its own, as small as the first calls need
    try:
        miller, _ = setup(acc, dims, 6)
        npw, nch, n = len(miller), 40, int(np.prod(dims))
        rng = np.random.default_rng(36)
        acc.set_veff((np.fft.fftn(rng.uniform(-13.6, 13.6, dims)) / n).reshape(-1))
        acc.set_nk(2)
        for ik in range(2):
            acc.set_kinetic(ik, (miller.astype(float) ** 2).sum(1) * (1 + 0.1 * ik))
            b = (rng.standard_normal((npw, nch)) + 1j * rng.standard_normal((npw, nch))) / np.sqrt(npw)
            acc.set_nonlocal(ik, b, b.conj().T.copy())
        fw = rng.uniform(0.1, 2.0, 96)
        psi = torch.from_numpy(bands(rng, 96, npw)).cuda()
        out, rho = torch.zeros_like(psi), torch.zeros(n, dtype=torch.float64, device="cuda")
        other, rho2 = torch.zeros_like(psi), torch.zeros_like(rho)
        torch.cuda.synchronize()

        def calls(nb, h, r):
            acc.hpsi_batch_dev([1, 0], [nb, nb - 1], psi.data_ptr(), h.data_ptr(), "fp64")
            acc.density_dev(nb, psi.data_ptr(), fw, r.data_ptr(), "fp64")

        calls(2, out, rho)
        acc.sync()
        want = out.cpu(), rho.cpu()
        print("captured, then larger calls", dims, flush=True)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(torch.cuda.ExternalStream(acc.stream)):
            graph.capture_begin(capture_error_mode="thread_local")
            try:
                calls(2, out, rho)
            finally:
                graph.capture_end()
            for nb in (5, 17, 48):
                calls(nb, other, rho2)
                acc.sync()
                out.zero_()
                rho.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(out.cpu(), want[0]) and torch.equal(rho.cpu(), want[1]), nb
    finally:
        acc.close()
