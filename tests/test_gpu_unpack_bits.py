"""Packed and indexed primitives unpack to the same bits: the two run their loads and sums in another
order, straight from memory in small launches and through LDS in large ones."""
import numpy as np
import pytest

import vknrc_amd as v
from vknrc_amd import workloads as wl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"


@pytest.mark.parametrize("n", [777, 32768, 32769, 100003])
@pytest.mark.parametrize("seed", [1, 2])
def test_packed_and_indexed_primitives_give_the_same_bits(seed, n):
    s = wl.make_scene(seed, primitives=20000, vertices=15000, instances=30, materials=20, textures=3, texture_size=32)
    vi = np.array(s["vertex_indices"]).reshape(-1, 3)
    vi[::97, 1] = vi[::97, 0]  # degenerate triangles, whose normal angles are NaN
    ds = v.DeviceScene(torch, s["vertices"], vi.ravel(), s["texcoords"], s["texcoord_indices"], s["materials"], s["material_ids"],
                       s["transforms"], s["textures"])
    ds.pack_primitives()
    rng = np.random.default_rng(seed)
    tr = np.zeros(n, v.WIRE_TRAIN_RECORD)
    tr["packed_input"], tr["bias"] = wl.make_packed_inputs(s, n, rng), rng.uniform(0, 1, (n, 3))
    ev = np.zeros(n, v.EVAL_RECORD)
    ev["packed_input"] = tr["packed_input"]
    ev, tr = (torch.from_numpy(a.view(np.int32)).to(DEV) for a in (ev, tr))
    out = {}
    for packed in (False, True):
        ds.use_packed(packed)
        q, t = torch.full((n, 14), 7.0, device=DEV), torch.full((n, 17), 7.0, device=DEV)
        v.unpack_eval_records(ds, ev, n, q)
        v.unpack_train_records(ds, tr, n, t)
        torch.cuda.synchronize()
        out[packed] = q.cpu().numpy(), t.cpu().numpy()
    assert np.isnan(out[True][0]).any() and np.isfinite(out[True][0]).all(1).mean() > 0.9
    for a, b in zip(out[False], out[True]):
        assert np.array_equal(a, b, equal_nan=True)
    assert np.array_equal(out[True][0], out[True][1][:, :14], equal_nan=True)
