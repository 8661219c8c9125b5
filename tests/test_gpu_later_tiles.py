"""Launches in which a wave takes several tiles, and the edges of the FP32 gradient's chunks.

FP8 inference: a workgroup's waves take the tiles of its range in turn, the operands of a layer and the
records of the next tile in two buffers each, so tiles of odd and even turn run different code.  FP32
inference deals 16-record tiles to 16 waves a CU (65,536 records a pass on 256 CUs), its gradient to 8
(32,768), and the weight gradient is summed over 512-record chunks (kPlainChunk)."""
import numpy as np
import pytest

import vknrc_amd as v
from oracle.fp8 import infer_fp8
from oracle.oracle import Oracle
from vknrc_amd import workloads as wl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"
KINDS = [(h, e) for h in (4, 5) for e in (v.ENCODING_TRI12, v.ENCODING_SINCOS6, v.ENCODING_UV_SINCOS16)]
ENCODINGS = [(5, v.ENCODING_TRI12), (5, v.ENCODING_SINCOS6), (4, v.ENCODING_UV_SINCOS16)]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def count(n):
    return dev(np.array([n], np.uint32).view(np.int32))


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def rel_err(y, ref):
    return float(np.linalg.norm(np.asarray(y, np.float64) - ref) / np.linalg.norm(ref))


def records(enc, n, seed):
    rng = np.random.default_rng(seed)
    r = wl.make_train_records(n, rng, wl.GaussianLights(7))
    if enc == v.ENCODING_UV_SINCOS16:
        r[:, :2] = rng.uniform(0, 1, (n, 2))
    return r


def fp8(state, q, live=None):
    out = torch.full((len(q), 3), 7.0, device=DEV)
    state.infer(q, out, count=None if live is None else count(live), path=v.PATH_FUSED_F8)
    return host(out)


@pytest.fixture
def workgroups():
    yield v.set_infer_workgroups_per_cu
    v.set_infer_workgroups_per_cu(2)


# 300,001 queries are 4,688 tiles: two or three a wave at two workgroups a CU, four or five at one.  The
# first FP8 inference of a cache has scales that do not depend on the queries, so the rows are those of
# calls small enough for one tile a wave, at device counts inside a tile and far below the size as well
@pytest.mark.parametrize("hidden,enc", KINDS)
def test_fp8_waves_with_several_tiles(hidden, enc, workgroups):
    n = 300001
    q = dev(records(enc, n, 50 + enc)[:, :14])
    cfg = v.NRCConfig(hidden_layers=hidden, encoding=enc, seed=4)

    def first(part, live=None):
        st = v.NRCState(cfg)
        y = fp8(st, part, live)
        st.close()
        return y

    assert 64 * 4 * 256 < n / 3  # one workgroup a CU on 256 CUs: more than three tiles a wave
    parts = np.concatenate([first(q[k:k + 60000]) for k in range(0, n, 60000)])
    st, results = v.NRCState(cfg), []
    for wg in (2, 1, 3):
        workgroups(wg)
        for live in (None, 299969, 200000, 131073, 1000, 0):
            y = first(q, live)
            m = n if live is None else live
            assert np.array_equal(y[:m], parts[:m]), (wg, live)
            assert (y[m:] == 7.0).all(), (wg, live)
        # the activation maxima of the sampled tiles, and with them the next scales and results, do not depend
        # on how the tiles are dealt
        st.close()
        st = v.NRCState(cfg)
        fp8(st, q)
        results.append((fp8(st, q), st.get_fp8_scales()))
    for y, sc in results[1:]:
        assert np.array_equal(y, results[0][0])
        assert np.array_equal(sc["layer_scales"], results[0][1]["layer_scales"]) and sc["out_scale"] == results[0][1]["out_scale"]
    y, sc = results[0]
    w = st.get_state()["weight"]
    rows = np.r_[0:300, 131000:131300, 262000:262300, n - 300:n]
    f = Oracle("f32").encode(host(q)[rows], enc)
    # 5e-2: an e4m3 step is 6-12 % of a value, and sums near a rounding boundary fall either way
    assert rel_err(y[rows], infer_fp8(f, w, hidden, sc["layer_scales"], sc["out_scale"], clamp0=True)) < 5e-2
    st.close()


# a workgroup whose range holds tiles of several caches copies each cache's weights to LDS in turn
@pytest.mark.parametrize("hidden,enc", KINDS)
def test_fp8_group_has_the_bits_of_each_cache_alone(hidden, enc):
    sizes = [(200001, 199000), (777, 777), (64, 0), (90001, 90001), (1000, 65), (63, 63)]

    def caches():
        return [dict(cache=v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc, seed=i)), queries=dev(records(enc, n, i)[:, :14]),
                     max_queries=n, query_count=count(live), rgb=torch.full((n, 3), 7.0, device=DEV)) for i, (n, live) in enumerate(sizes)]

    group, alone = caches(), caches()
    for _ in range(3):  # on first scales, then on measured ones
        v.group_infer(group, path=v.PATH_FUSED_F8)
        for e in alone:
            e["cache"].infer(e["queries"], e["rgb"], count=e["query_count"], path=v.PATH_FUSED_F8)
        for i, (g, a) in enumerate(zip(group, alone)):
            assert np.array_equal(host(g["rgb"]), host(a["rgb"])), i
            x, y = g["cache"].get_fp8_scales(), a["cache"].get_fp8_scales()
            assert np.array_equal(x["layer_scales"], y["layer_scales"]) and x["out_scale"] == y["out_scale"] and x["frames"] == y["frames"], i
    for e in group + alone:
        e["cache"].close()


# FP32 sums of 64 products over at most 6 layers are within 6 * 64 * 2^-24 = 2.3e-5 of their exact values
# relative to the largest terms
PLAIN_TOL = 2.3e-5


# a second tile for some waves, with a partial last one and a device count just past the first pass; a third
@pytest.mark.parametrize("hidden,enc", ENCODINGS)
@pytest.mark.parametrize("n,live", [(66000, 65553), (66001, 66001), (140001, 131089)])
def test_plain_inference_later_tiles(hidden, enc, n, live):
    r = records(enc, n, n + enc)
    st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc, seed=6))
    w = st.get_state()["weight"]
    out = torch.full((n, 3), 7.0, device=DEV)
    st.infer(dev(r[:, :14]), out, count=count(live), path=v.PATH_PLAIN_F32)
    y = host(out)
    f = Oracle("f32").encode(r[:live], enc).astype(np.float64)  # features rounded as FP32 computes them
    ref = np.maximum(Oracle("f64").infer_encoded(w.astype(np.float64), hidden, f), 0)
    assert rel_err(y[:live], ref) < PLAIN_TOL
    for a, b in ((0, 65536), (65536, 131072), (131072, live)):  # each pass by itself
        if a < live:
            assert rel_err(y[a:min(b, live)], ref[a:b]) < PLAIN_TOL, a
    assert (y[live:] == 7.0).all()
    st.close()


# Every record at an edge carries about a tenth of the gradient, so one that is dropped or counted twice
# moves it by several percent.  The bound leaves room for ReLU masks that FP32 rounding flips, a few of
# the up to 320 * 40,001 units: each changes one unit's delta of one ordinary record, an eighth of that
# record's part, and that part is 1 / sqrt(n) of the whole at most (1 / 22 for n = 511, where such a flip
# has a chance of 3 %; five of them at n = 40,001 are 1.4e-3).
EDGE_TOL = 6e-3


@pytest.mark.parametrize("hidden,enc", ENCODINGS)
@pytest.mark.parametrize("n,live,edges", [(511, 511, [0, 510]), (512, 512, [15, 16, 511]), (513, 513, [511, 512]),
                                          (1025, 1025, [511, 512, 1023, 1024]), (1100, 1024, [1022, 1023]),
                                          (40001, 40001, [32767, 32768, 40000]), (40001, 32769, [32752, 32767, 32768]),
                                          (65536, 65536, [32767, 32768, 65535])])
def test_plain_gradient_edges(hidden, enc, n, live, edges):
    r = records(enc, n, n + live)
    r[edges, 14:] = n / 10 * r[:, 14:].mean()
    r[live:, 14:] = 1e6  # nothing past the device count may enter
    st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc, loss=v.LOSS_L2, seed=8, train_batch_size=65536))
    w = st.get_state()["weight"].astype(np.float64)
    st.train(dev(r), count=count(live), path=v.PATH_PLAIN_F32)
    s = st.get_state()
    st.close()
    f = Oracle("f32").encode(r[:live], enc).astype(np.float64)
    o64 = Oracle("f64")
    G, loss = o64.gradient_encoded(w, hidden, f, r[:live, 14:].astype(np.float64), loss=1)
    for k in edges:
        Gk, _ = o64.gradient_encoded(w, hidden, f[k:k + 1], r[k:k + 1, 14:].astype(np.float64), loss=1)
        assert np.linalg.norm(Gk) > 4 * EDGE_TOL * np.linalg.norm(G), k
    assert rel_err(s["m"] / (1.0 - np.float32(0.9)), G / live) < EDGE_TOL
    assert abs(s["state"]["last_loss"] / (loss / live) - 1) < 7e-5
    assert s["state"]["last_count"] == live
