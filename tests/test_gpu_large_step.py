"""Steps of worlds beyond the LDS layout: packed Newton matrix, contact rows listed by contact and dof.

The 256-thread kernel against the float64 oracle where its blocks and loops have their edges: a last
block of two dofs, full blocks only, the largest order (16 blocks, Newton matrix in device memory), a
Newton matrix in LDS, and more contact slots than threads.  Bars as for every step: 1e-5 in the velocities, the formed problem and the public state, which
float32 matrices of these scenes keep with two digits to spare (the solve is refined in float64)."""
import pytest

from tests import test_gpu_step as step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bodies,slots,preset,ls", [
    (11, 88, "approx32", "exact_root"),
    (16, 320, "drake", "armijo_decay"),
    (24, 96, "approx32", "exact_root"),
    (42, 168, "approx32", "exact_root"),
])
def test_block_edges(gpu_device, monkeypatch, bodies, slots, preset, ls):
    from sap_warp_amd import hetero

    monkeypatch.setattr(step, "_scene", lambda name, worlds, seed: (
        hetero.build_pile_scene(worlds, seed=seed + 5, bodies=bodies, device="cuda:0"), 2.0e-3, slots))
    step._run_and_compare(f"pile of {bodies}", preset, ls, worlds=2, steps=2, warm_steps=120, min_max_contacts=bodies)


@pytest.mark.parametrize("preset,ls", [("approx32", "exact_root"), ("drake", "armijo_decay")])
def test_articulated(gpu_device, preset, ls):
    """Contact rows over the joints of two root paths of one tree, so that the dofs' lists differ in
    length: lying humanoids (35 dofs) with so many slots that J exceeds the LDS layout."""
    step._run_and_compare("humanoid_lying", preset, ls, worlds=3, steps=2, warm_steps=50, solver_C=300, pipe_C=64,
                          min_max_contacts=25)


def test_builds_agree(gpu_device):
    """More than 512 worlds whose LDS lets three share a CU run in the build with fewer registers: the
    first worlds of such a batch end where they end in a batch of two, up to what another order of float32
    operations moves a refined solve (each build is within 1e-5 of the oracle)."""
    import numpy as np
    import torch

    from sap_warp_amd import hetero
    from sap_warp_amd.collision import SapCollisionPipeline
    from sap_warp_amd.solver_sap import SolverSAP
    from tests.helpers import world_rel_err

    ends = []
    for worlds in (2, 513):
        model = hetero.build_pile_scene(worlds, seed=8, bodies=11, device="cuda:0")
        solver = SolverSAP(model, max_rigid_contact=88, line_search_variant="exact_root", contact_preset_variant="approx32")
        pipe = SapCollisionPipeline(model, max_contacts_per_world=88)
        contacts = pipe.contacts()
        s0, s1, control = model.state(), model.state(), model.control()
        for _ in range(3):
            pipe.collide(s0, contacts)
            solver.step(s0, s1, control, contacts, 2.0e-3)
            s0, s1 = s1, s0
        torch.cuda.synchronize()
        assert int(contacts.rigid_contact_world_start[2]) > 0
        ends.append([getattr(s0, k)[:size].cpu().numpy().astype(np.float64).reshape(2, -1)
                     for k, size in (("joint_q", 2 * 77), ("joint_qd", 2 * 66))])
    for a, b in zip(*ends):
        for w in range(2):
            assert world_rel_err(b[w], a[w]) <= 2.0e-5, w


def test_block_of_device_memory(gpu_device):
    """A world of 32 free bodies with 256 contact slots takes no more device memory than its dense A, H
    and J (0.89 MB): the contact rows are listed by contact and by dof without their zeros."""
    import torch

    from sap_warp_amd import hetero
    from sap_warp_amd.solver_sap import SolverSAP

    worlds, n, slots = 128, 192, 256
    model = hetero.build_pile_scene(worlds, seed=8, bodies=32, device="cuda:0")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    solver = SolverSAP(model, max_rigid_contact=slots, line_search_variant="exact_root", contact_preset_variant="approx32")
    used = before - torch.cuda.mem_get_info()[0]
    solver.close()
    dense = 4 * (2 * n * (n + 1) + 3 * slots * (n + 1))
    # outside the block: states, warm start and statistics of a world
    assert used <= worlds * (dense + 50_000), (used / worlds, dense)
