"""One-wave step kernel: block factor and solves at the edges of their 16 x 16 blocks.

Piles of 1 to 10 free bodies (6 to 60 dofs) against the float64 oracle: a single block with its second
half empty (6), a last block of two (18), eight (24), ten (42) and twelve dofs (60), full blocks only
(48), with contact slots for the small variant alone and beside larger ones.  Bars as for every step:
1e-5 in the velocities, the formed problem and the public state.  The piles are compared while they
fall together: the errors are relative, and a body at rest has no velocity to be relative to."""
import pytest

from tests import test_gpu_step as step

pytestmark = pytest.mark.gpu


def _pile(bodies, slots):
    from sap_warp_amd import hetero

    return lambda name, worlds, seed: (
        hetero.build_pile_scene(worlds, seed=seed + 5, bodies=bodies, device="cuda:0"), 2.0e-3, slots)


@pytest.mark.parametrize("bodies,slots", [(1, 16), (3, 16), (4, 32), (7, 24), (8, 64), (10, 48)])
def test_block_edges(gpu_device, monkeypatch, bodies, slots):
    monkeypatch.setattr(step, "_scene", _pile(bodies, slots))
    step._run_and_compare(f"pile of {bodies}", "approx32", "exact_root", worlds=3, steps=2, warm_steps=45,
                          min_max_contacts=1)


@pytest.mark.parametrize("lying,slots,worlds", [(1.0, 64, 24), (0.5, 30, 24), (1.0, 64, 520), (0.5, 30, 1040)])
def test_contact_variants_agree(gpu_device, lying, slots, worlds):
    """Worlds split over the contact variants of a step (fewest contacts first, on two streams or on one)
    end where the 64-slot variant alone takes them: a variant is a choice of LDS layout, the arithmetic
    and its order are the same, so the states are equal bit for bit.  24 worlds fit on the chip at once and
    take one launch whatever the schedule; 520 with 64 slots (three launches) and 1040 with 32 (two) do not."""
    import torch

    from sap_warp_amd.collision import SapCollisionPipeline
    from sap_warp_amd.scenes import build_humanoid_scene
    from sap_warp_amd.solver_sap import SolverSAP

    model = build_humanoid_scene(worlds, seed=4, lying_fraction=lying, contact_gap=0.05, device="cuda:0")
    ends = []
    for small, fork in ((64, False), (16, True), (16, False), (32, True)):
        solver = SolverSAP(model, max_rigid_contact=slots, line_search_variant="exact_root",
                           contact_preset_variant="approx32")
        solver.set_schedule(kernel="wave", small_capacity=small, fork=fork, world_order=True)
        pipe = SapCollisionPipeline(model, max_contacts_per_world=slots)
        contacts = pipe.contacts()
        s0, s1, control = model.state(), model.state(), model.control()
        for _ in range(3):
            pipe.collide(s0, contacts)
            solver.step(s0, s1, control, contacts, 2.0e-3)
            s0, s1 = s1, s0
        torch.cuda.synchronize()
        starts = contacts.rigid_contact_world_start.cpu()
        ends.append((s0.joint_q.clone(), s0.joint_qd.clone(), s0.body_q.clone()))
    counts = (starts[1:] - starts[:-1]).tolist()
    assert max(counts) > 24 and (lying == 1.0 or min(counts) <= 16), counts
    for end in ends[1:]:
        for a, b in zip(ends[0], end):
            assert torch.equal(a, b)
