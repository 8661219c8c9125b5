"""Query fields that no encoder is written for, through the FP8 inference.

A one-blob quad of a NaN is four zeros (the clamp of five NaN knots), as it is for a value two
bins or more out of range: a record with the one gives the bits of a record with the other.  A
degenerate triangle's normal angles are NaN, so such fields do arrive."""
import numpy as np
import pytest

import vknrc_amd as v
from vknrc_amd import workloads as wl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"


@pytest.mark.parametrize("field", [3, 4, 5, 6, 7])
@pytest.mark.parametrize("enc", [v.ENCODING_TRI12, v.ENCODING_SINCOS6])
def test_nan_field_encodes_as_a_field_out_of_range(enc, field):
    q = wl.make_queries(1000, np.random.default_rng(field))
    out = []
    for value in (np.nan, -200.0 if field == 7 else 2.0):  # the roughness enters as 1 - exp(-r): -200 gives -inf
        q[::3, field] = value
        st = v.NRCState(v.NRCConfig(encoding=enc, seed=9))
        out.append(torch.full((1000, 3), 7.0, device=DEV))
        st.infer(torch.from_numpy(q).to(DEV), out[-1], path=v.PATH_FUSED_F8)
        torch.cuda.synchronize()
        st.close()
    assert torch.equal(out[0], out[1])
