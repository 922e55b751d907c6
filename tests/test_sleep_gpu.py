"""GPU: island sleep and wake on the device world (the island pass of
world.hip: union-find islands, wakes through broadphase-connected
islands, sleep of islands whose bodies are all ready) against the
reference's own run (tests/golden/sleep_scene.npz; the oracle reproduces
it bit for bit) and, at every transition step, the whole step against the
oracle started from the device's state.

Bars: sleeping flags exact every step; states within 1e-4 relative (1e-6
absolute) of the reference's; contact events (notifications on) exact in
bodies, kinds, counts and shapes, impulse sums 1e-4; transition steps as
world_parity holds them."""
import numpy as np
import pytest

from author_cases import apply_edits
from test_author_gpu import _Ids, _world
from fyzz_amd import scenes
from oracle_bind import StepOracle
from world_parity import compare_step

from pathlib import Path

GOLDEN = Path(__file__).resolve().parent / "golden" / "sleep_scene.npz"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
def test_sleep_and_wake_match_reference(ctx, orc, torch_cuda, graph):
    g = np.load(GOLDEN)
    sc = scenes.Scene(g["half"], g["pos"], g["quat"], friction=0.5, restitution=0.0)
    steps = int(g["steps"][0])
    transitions = {49, 50, 51, 90, 91, 92, 100, 101, 110, 111}
    w = _world(ctx, sc)
    w.set_contact_notifications(True)
    so = StepOracle(orc, sc.half, threads=4)
    try:
        for s in range(steps):
            apply_edits(_Ids(w), g["edits"], s, to_id=lambda i: i + 1)
            rec = w.body_records()
            np.testing.assert_array_equal((rec["flags"] & 1).astype(np.uint8), g["sleeping"][s],
                                          err_msg=f"sleeping, step {s}")
            np.testing.assert_allclose(w.body_states(), g["state"][s], rtol=1e-4, atol=1e-6, err_msg=f"step {s}")
            if s in transitions and not graph:
                compare_step(w, so, 1 / 120, f"sleep step {s}")
            elif graph:
                w.step_graph(1 / 120)
            else:
                w.step(1 / 120)
            # events: persisting touches of sleeping islands are not reported
            ev, _ = w.contact_events()
            got = np.stack([ev["body0"], ev["body1"], ev["kind"], ev["contact_count"], ev["shape0"], ev["shape1"]],
                           1).astype(np.uint32)
            np.testing.assert_array_equal(got.reshape(-1, 6), g[f"ev_{s}"].reshape(-1, 6), err_msg=f"step {s} events")
            np.testing.assert_allclose(ev["normal_impulse"], g[f"evimp_{s}"], rtol=1e-4, atol=1e-5,
                                       err_msg=f"step {s} event impulses")
        np.testing.assert_allclose(w.body_states(), g["state"][steps], rtol=1e-4, atol=1e-6)
        assert w.stats()["flags"] == 0
    finally:
        w.close()


@pytest.mark.parametrize("n_rows", [40, 1100])
def test_island_pass_agrees_with_the_authority_on_long_rows(ctx, torch_cuda, n_rows):
    """Rows of 15 resting boxes whose bounds touch (one broadphase island
    each, one of them joined to a row of 600), slots in random order, go to
    sleep; boxes dropped at staggered heights wake some rows. In the native
    order every step compares the island pass's sleep flags with the host
    authority's and fails on a difference. 40 rows take the one-launch pass
    and 1,100 rows (17,100 boxes and more) the separate launches."""
    from fyzz_amd.world import World
    rng = np.random.default_rng(n_rows)
    length = np.full(n_rows, 15)
    length[0] = 600
    row = np.repeat(np.arange(n_rows), length)
    col = np.concatenate([np.arange(k) for k in length])
    pos = np.stack([col * 1.01, np.full(len(row), 0.5), row * 3.0], 1)
    drop = rng.choice(n_rows, n_rows // 4, replace=False)
    fall = np.stack([rng.integers(0, 15, len(drop)) * 1.01, rng.uniform(6.0, 14.0, len(drop)), drop * 3.0], 1)
    pos = np.concatenate([pos, fall]).astype(np.float32)
    pos = pos[rng.permutation(len(pos))]
    w = World(ctx, len(pos) + 1)
    try:
        fid = w.add_static_floor(0.0)
        w.set_body_material(fid, 0.5, 0.5, 0.0)
        w.add_dynamic_boxes(np.full((len(pos), 3), 0.5), pos, np.tile([0, 0, 0, 1.0], (len(pos), 1)), friction=0.5,
                            restitution=0.0)
        w.set_solver_order(True)
        asleep = []
        for s in range(230):
            w.step(1 / 120)
            if s % 10 == 9:
                asleep.append(int((w.body_records()["flags"] & 1).sum()))
        assert w.stats()["flags"] == 0
        assert max(asleep) > len(pos) // 2
        assert any(b < a for a, b in zip(asleep, asleep[1:]))  # rows woken by what fell on them
    finally:
        w.close()
