"""The stateless gradient's kept scratch: back to the device on request, beside a capture that another stream
has under way, and from several host threads at once."""
import threading

import numpy as np
import pytest

import vknrc_amd as v
from vknrc_amd import workloads as wl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"


def inputs(n):
    rng = np.random.default_rng(21)
    dev = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    return (dev(rng.normal(0, np.sqrt(2 / 64), v.weight_count(5)).astype(np.float16)),
            dev(rng.uniform(-1, 1, (n, 64)).astype(np.float16)), dev(rng.uniform(0, 1, (n, 3)).astype(np.float32)))


def test_release_scratch_frees_the_kept_blocks():
    w, x, t = inputs(3000)
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


@pytest.mark.parametrize("kept", [True, False])
def test_gradient_on_one_stream_during_a_capture_on_another(kept):
    w, x, t = inputs(5000)
    q = torch.from_numpy(wl.make_queries(5000, np.random.default_rng(1))).to(DEV)
    st = v.NRCState(v.NRCConfig(seed=1))
    ref, out = torch.zeros((5000, 3), device=DEV), torch.zeros((5000, 3), device=DEV)
    st.infer(q, ref)
    dw = torch.zeros((2, v.weight_count(5)), device=DEV)
    v.mlp_gradient_f16(w, x, t, 5000, dw[0])
    torch.cuda.synchronize()
    if not kept:
        v.release_scratch()
    other, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="global"):
        v.mlp_gradient_f16(w, x, t, 5000, dw[1], stream=other)
        st.infer(q, out)
    torch.cuda.synchronize()
    assert torch.equal(dw[0], dw[1])
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
    st.close()


def test_gradient_from_several_threads():
    w, x, t = inputs(8 * 4096)
    parts = [(x[4096 * k:4096 * (k + 1)], t[4096 * k:4096 * (k + 1)]) for k in range(8)]
    one, many = torch.zeros((8, v.weight_count(5)), device=DEV), torch.zeros((8, v.weight_count(5)), device=DEV)
    for k, (xk, tk) in enumerate(parts):
        v.mlp_gradient_f16(w, xk, tk, 4096, one[k])
        torch.cuda.synchronize()
    errors = []

    def work(k):
        try:
            stream = torch.cuda.Stream()
            for _ in range(10):
                v.mlp_gradient_f16(w, *parts[k], 4096, many[k], stream=stream)
            stream.synchronize()
        except Exception as e:  # reported below, on the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors
    assert torch.equal(one, many)
