"""The stateless gradient's kept scratch goes back to the device on request, and calls go on after it."""
import numpy as np
import pytest

import vknrc_amd as v

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"


def test_release_scratch_frees_the_kept_blocks():
    rng = np.random.default_rng(21)
    dev = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    w = dev(rng.normal(0, np.sqrt(2 / 64), v.weight_count(5)).astype(np.float16))
    x, t = dev(rng.uniform(-1, 1, (3000, 64)).astype(np.float16)), dev(rng.uniform(0, 1, (3000, 3)).astype(np.float32))
    dw = torch.zeros((3, v.weight_count(5)), device=DEV)
    for k in range(3):
        v.mlp_gradient_f16(w, x, t, 3000, dw[k])
        if k == 2:
            break  # released with the call still in flight: the release waits for it
        torch.cuda.synchronize()
        kept = torch.cuda.mem_get_info()[0]
        v.release_scratch()
        assert torch.cuda.mem_get_info()[0] - kept >= 21_000_000
    v.release_scratch()
    v.release_scratch()  # nothing is kept: no work
    torch.cuda.synchronize()
    assert torch.equal(dw[0], dw[1]) and torch.equal(dw[0], dw[2]) and dw[0].abs().max() > 0
