"""Which scenes of a batch get a workgroup of their own (batch_shape.hpp): the
rule on the host over the sizes it was measured at, and on the GPU both forms
of stepping and recording with the same bits."""
import numpy as np
import pytest

from dyphur_amd import scenes
from tests import _hostmath

SLOTS, SLOTS_REC = 512, 256  # workgroups of 256 threads on 256 CUs: stepping two a CU, recording one


def _wave_max(bodies, slots):
    off = np.concatenate([[0], np.cumsum(bodies)]).astype(np.uint32)
    return _hostmath.lib().hm_batch_wave_max(off.ctypes.data, len(bodies), slots)


def _lognormal(n, median, top):
    rng = np.random.default_rng([n, median, top])
    return np.clip(np.round(median * np.exp(0.75 * rng.normal(size=n))), 8, top).astype(int) + 1


@pytest.mark.parametrize("bodies,step,record", [
    ([33] * 256, 32, 32), ([33] * 300, 32, 128), ([33] * 512, 32, 128), ([33] * 513, 128, 128), ([33] * 1024, 128, 128),
    ([64] * 256, 32, 32), ([64] * 512, 32, 128), ([64] * 600, 128, 128), ([128] * 256, 32, 32), ([128] * 600, 128, 128),
    ([65] * 256, 32, 32), ([20] * 4000, 128, 128), ([20] * 4000 + [100], 32, 32), ([300] * 50, 128, 128), ([33], 32, 32),
    (_lognormal(300, 48, 256), 32, 32), (_lognormal(600, 48, 256), 32, 32), (_lognormal(768, 48, 256), 32, 128),
    (_lognormal(1500, 48, 256), 128, 128), (_lognormal(512, 64, 512), 128, 128), (_lognormal(4096, 64, 512), 128, 128),
])
def test_workgroup_line_where_it_was_measured(bodies, step, record):
    assert _wave_max(bodies, SLOTS) == step
    assert _wave_max(bodies, SLOTS_REC) == record


@pytest.mark.gpu
@pytest.mark.parametrize("n_scenes,n_dyn", [(3, 40), (300, 32), (520, 32)])
def test_default_shape_steps_and_records_as_any_other(gpu, n_scenes, n_dyn):
    print(f"[batch shape] scenes={n_scenes} bodies={n_dyn + 1}", flush=True)
    scs = [scenes.pile_scene(n_dyn, scenes.Pcg32(k % 7)) for k in range(n_scenes)]
    out = []
    for shape in (None, (256, 32), (256, 128)):
        b, r = gpu.Batch(scs), gpu.Batch(scs)
        if shape:
            b.set_shape(*shape)
            r.set_shape(*shape)
        else:
            assert b.shape() == (256, _wave_max([n_dyn + 1] * n_scenes, SLOTS))
        b.step(6)
        d = gpu.Diff(r, 6, 3, tape_contacts_per_body=12.0)
        d.forward(6)
        adj = d.backward({"pos_y": np.ones(r.n_bodies, np.float32)})
        out.append((b.state(), r.state(), adj))
        d.close()
        b.close()
        r.close()
    for stepped, recorded, adj in out:
        for k in stepped:
            assert np.array_equal(stepped[k].view(np.uint32), out[0][0][k].view(np.uint32)), k
            assert np.array_equal(recorded[k].view(np.uint32), stepped[k].view(np.uint32)), k
        for k in adj:
            assert np.array_equal(adj[k].view(np.uint32), out[0][2][k].view(np.uint32)), k


@pytest.mark.gpu
def test_autotune_keeps_a_faster_shape_it_started_from(gpu):
    """A batch for which the default beats the six shapes keeps it, recording
    shape included; one that starts from one of the six takes the fastest of them."""
    scs = [scenes.pile_scene(62, scenes.Pcg32(k)) for k in range(64)]
    b = gpu.Batch(scs)
    assert b.shape() == (256, 32) and b.shape() not in gpu.Batch.TUNE_SHAPES[:6]
    b.step(40)
    chosen, ms = b.autotune(8)
    print(f"[autotune] kept {chosen}; the six: {[round(m, 3) for m in ms]} ms", flush=True)
    assert chosen == b.shape() == (256, 32) and len(ms) == 6 and min(ms) > 0
    b.set_shape(128, 64)
    chosen, ms = b.autotune(8)
    assert chosen == gpu.Batch.TUNE_SHAPES[int(np.argmin(ms))]
