"""The blocked Cholesky at the edges of its blocks: one matrix row either side of the four-column
groups and the eight-block superblocks, a size whose far updates come in four shares, a batch, and a
smaller matrix on the same handle (its exchange words and block mask lie elsewhere).  The reference is
numpy's float64 solve of the float32 matrix."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spd(n, rng):
    J = rng.normal(size=(n, max(4, n // 8))) / np.sqrt(max(4, n // 8))
    A = J @ J.T + np.diag(np.exp(rng.normal(size=n)) + 0.2)
    return (0.5 * (A + A.T)).astype(np.float32)


@pytest.mark.parametrize("n,batch", [(255, 2), (257, 1), (512, 1), (513, 2), (577, 1), (2881, 1)])
def test_group_and_superblock_edges(gpu_device, n, batch):
    import torch

    from sap_warp_amd.blocked_cholesky import BlockCholeskySolverBatched

    rng = np.random.default_rng(n)
    solver = BlockCholeskySolverBatched(n, batch, refine=2)
    for m in (n, n - 64 if n > 64 else n, n):
        A = np.stack([_spd(m, rng) for _ in range(batch)])
        Ad = torch.tensor(A, device="cuda:0")
        solver.factorize(Ad, m)
        for _ in range(2):  # a second right-hand side on the same factor
            b = rng.normal(size=(batch, m))
            rhs, x = torch.tensor(b, device="cuda:0"), torch.zeros((batch, m), dtype=torch.float64, device="cuda:0")
            print(f"chol n {n} of {m} batch {batch}", flush=True)
            solver.solve(rhs, x)
            assert np.all(solver.info() == 0)
            for k in range(batch):
                # condition below 1e2: two float64-residual refinements of a float32 factor leave 1e-12
                ref = np.linalg.solve(A[k].astype(np.float64), b[k])
                assert np.max(np.abs(x[k].cpu().numpy() - ref)) <= 1e-10 * np.max(np.abs(ref)), (m, k)
    solver.close()


def unrefined_error(n, matrices):
    """Geometric mean over matrices of the relative 2-norm error of a solve without refinement."""
    import torch

    from sap_warp_amd.blocked_cholesky import BlockCholeskySolverBatched

    solver = BlockCholeskySolverBatched(n, 1, refine=0)
    logs = []
    for seed in range(matrices):
        rng = np.random.default_rng(1000 * n + seed)
        A, b = _spd(n, rng), rng.normal(size=n)
        rhs = torch.tensor(b[None], device="cuda:0")
        x = torch.zeros_like(rhs)
        solver.factorize(torch.tensor(A[None], device="cuda:0"), n)
        solver.solve(rhs, x)
        assert np.all(solver.info() == 0)
        ref = np.linalg.solve(A.astype(np.float64), b)
        logs.append(np.log(np.linalg.norm(x[0].cpu().numpy() - ref) / np.linalg.norm(ref)))
    solver.close()
    return float(np.exp(np.mean(logs)))


@pytest.mark.parametrize("n", [200, 500, 1000, 1536])
def test_unrefined_error(gpu_device, n):
    """Nothing but the float32 rounding of a 64-wide right-looking elimination is left in an unrefined
    solve.  Such an elimination with float32 sums and 64-wide substitution measures 3.5e-7 to 3.9e-7 on
    these matrices; one sum over the four columns of a group, or an inverse of 512 unknowns summed in
    float32, adds to it (5.0e-7 to 5.3e-7 from order 500 on)."""
    error = unrefined_error(n, 10)
    print(f"chol n {n} unrefined error {error:.3e}", flush=True)
    assert error <= 4.1e-7


def test_solves_on_several_streams(gpu_device):
    """Two handles whose solves each fill the chip (512 workgroups, two a CU) on a stream each, and a third
    of another size beside them: every solve ends where it ends alone, bit for bit, and none times out."""
    import torch

    from sap_warp_amd.blocked_cholesky import BlockCholeskySolverBatched

    rng = np.random.default_rng(3)
    handles = []
    for n, batch in ((200, 128), (512, 64), (1100, 12)):
        A = torch.tensor(np.stack([_spd(n, rng) for _ in range(2)]), device="cuda:0").repeat(batch // 2, 1, 1)
        rhs = torch.tensor(rng.normal(size=(batch, n)), device="cuda:0")
        solver = BlockCholeskySolverBatched(n, batch, refine=2)
        solver.factorize(A, n)
        alone = torch.zeros_like(rhs)
        solver.solve(rhs, alone)
        assert np.all(solver.info() == 0)
        ref = torch.linalg.solve(A[:2].double().cpu(), rhs[:2].cpu())
        assert float((alone[:2].cpu() - ref).abs().max()) <= 1e-10 * float(ref.abs().max())
        handles.append((solver, rhs, alone, torch.zeros_like(rhs), torch.cuda.Stream()))
    torch.cuda.synchronize()
    for _ in range(20):
        for solver, rhs, _, x, stream in handles:
            with torch.cuda.stream(stream):
                solver.solve(rhs, x)
    torch.cuda.synchronize()
    for solver, _, alone, x, _ in handles:
        assert np.all(solver.info() == 0)
        assert torch.equal(x, alone)
        solver.close()
