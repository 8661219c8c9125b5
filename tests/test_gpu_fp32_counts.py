"""FP32 launches whose device count leaves workgroups, or all of them, without a record: the rows and the
training step are those of a call of the count's size, bit for bit."""
import numpy as np
import pytest

import vknrc_amd as v
from vknrc_amd import workloads as wl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"


@pytest.mark.parametrize("hidden,enc", [(5, v.ENCODING_TRI12), (5, v.ENCODING_SINCOS6), (4, v.ENCODING_UV_SINCOS16)])
@pytest.mark.parametrize("live", [0, 1, 16, 17, 700])
def test_fp32_counts_below_the_size(hidden, enc, live):
    n = 9000
    r = torch.from_numpy(wl.make_train_records(n, np.random.default_rng(live), wl.GaussianLights(7))).to(DEV)
    q = r[:, :14].contiguous()
    count = torch.tensor([live], dtype=torch.int32, device=DEV)
    counted, sized = (v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc, seed=3)) for _ in range(2))
    y, ref = torch.full((n, 3), 7.0, device=DEV), torch.full((n, 3), 7.0, device=DEV)
    for _ in range(2):  # the second round on trained weights
        counted.infer(q, y, count=count, path=v.PATH_PLAIN_F32)
        counted.train(r, count=count, path=v.PATH_PLAIN_F32)
        if live:
            sized.infer(q, ref, max_count=live, path=v.PATH_PLAIN_F32)
            sized.train(r, max_count=live, path=v.PATH_PLAIN_F32)
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
        a, b = counted.get_state(), sized.get_state()
        for k in ("weight", "m", "v", "ema_weight", "weights_f16", "use_weights_f16"):
            assert np.array_equal(a[k], b[k]), k
        assert a["state"]["t"] == b["state"]["t"] and a["state"]["last_count"] == b["state"]["last_count"]
    counted.close()
    sized.close()
