"""The pool of the chain's interval logs is reserved in full by a handle's first operator call, for the largest grid: a
larger run through the same handle does not free and allocate it between its launches."""
import pytest

pytestmark = pytest.mark.gpu


def test_first_call_reserves_the_whole_pool(gpu):
    from gamedev_amd import CollisionOperator, synth
    reserved = []
    for n in (300, 3000, 100000):
        st = synth.fiducial_3d_state(n, seed=3)
        d = synth.to_device(st, gpu)
        op = CollisionOperator("fiducial_3d", n, st["total_mass"], seed=1)
        op.bind_soa(d["x"], d["y"], d["z"], d["size"], d["numr"])
        op.geometry()
        op.evolve(0.01)
        reserved.append(int(op.chain_sums()[2][1]))
    print(f"[buffers] chunks reserved {reserved}", flush=True)
    assert reserved[0] > 8192 and reserved == [reserved[0]]*3
