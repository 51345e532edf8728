"""Chains long enough to fill several chunks of the solo owners' interval logs (64 intervals each), whose jump
moments are formed after the chain: whole operator calls give the same bits as with the sequential walk forced,
where the chain forms every event's moments itself. Baths as long as the call make the chains long."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h", [(1500, 3.0), (6000, 1.0)])
def test_long_chains_equal_the_general_loop(gpu, n, h):
    from gamedev_amd import CollisionOperator, synth
    st = synth.clumped_3d_state(n, seed=4)
    outs = []
    for exact in (False, True):
        d = synth.to_device(st, gpu)
        op = CollisionOperator("fiducial_3d", n, st["total_mass"], seed=9)
        op.bind_soa(d["x"], d["y"], d["z"], d["size"], d["numr"])
        op.set_exact_walk(exact)
        op.set_fixed_bath(h)
        op.geometry()
        ev = []
        for step in range(3):
            print(f"[logs] n={n} exact={exact} step {step}", flush=True)
            s = op.evolve(h)
            ev.append((s["events"], s["waves"], s["max_chain_events"]))
        outs.append((ev, d["size"].cpu().numpy().tobytes(), d["numr"].cpu().numpy().tobytes(), op.rng().tobytes()))
    print("[logs]", outs[0][0], flush=True)
    assert max(e[2] for e in outs[0][0]) > 200
    assert outs[0] == outs[1]
