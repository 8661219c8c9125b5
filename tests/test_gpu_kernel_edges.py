"""Kernels at the sizes where their tiling can go wrong, through the C ABI.

The FP16 gradient is compared with the same network in float64 that rounds the
activations and the deltas of each layer to FP16, as the kernels store them (a float64
network without these roundings has other ReLU masks on a few records, which shows when
there are few records).  What is left is the FP32 order of sums, which moves a rounding
now and then: 1e-2 in norm holds a few such moves even on one record.
"""
import numpy as np
import pytest

import vknrc_amd as v
from oracle import frontend
from oracle.fp8 import infer_fp8
from oracle.oracle import Oracle
from vknrc_amd import workloads as wl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"
GRAD_F16_TOL = 1e-2


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def rel_err(y, ref):
    return float(np.linalg.norm(np.asarray(y, np.float64) - ref) / np.linalg.norm(ref))


def gradient_f16(w, hidden, x, t):
    """d(sum of squared errors)/dw in float64 with FP16 activations and deltas; w, x hold FP16 values."""
    r16 = lambda a: a.astype(np.float16).astype(np.float64)  # noqa: E731
    m = [w[4096 * l:4096 * (l + 1)].reshape(64, 64) for l in range(hidden)] + [w[4096 * hidden:].reshape(3, 64)]
    acts = [x]
    for l in range(hidden):
        acts.append(r16(np.maximum(acts[-1] @ m[l].T, 0)))
    g = r16(2 * (acts[-1] @ m[hidden].T - t))
    out = []
    for l in range(hidden, -1, -1):
        out.append((g.T @ acts[l]).ravel())
        if l:
            g = r16((g @ m[l]) * (acts[l] > 0))
    return np.concatenate(out[::-1])


# partial rows of 1, 16, 17, 64, 65 and 256 gradient workgroups: the edges of the three
# reductions, with full and partial last workgroups; an odd address for the weights
@pytest.mark.parametrize("hidden", [4, 5])
@pytest.mark.parametrize("n", [1, 64, 1024, 1025, 4096, 4097, 16384])
def test_mlp_gradient_reduction_edges(hidden, n):
    rng = np.random.default_rng(n + hidden)
    w = rng.normal(0, np.sqrt(2 / 64), v.weight_count(hidden)).astype(np.float16)
    x = rng.uniform(-1, 1, (n, 64)).astype(np.float16)
    t = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    buf = dev(np.concatenate([np.zeros(1, np.float16), w]))
    dw = torch.full((v.weight_count(hidden),), 7.0, device=DEV)
    v.mlp_gradient_f16(buf[1:], dev(x), dev(t), n, dw, hidden_layers=hidden)
    G = gradient_f16(w.astype(np.float64), hidden, x.astype(np.float64), t.astype(np.float64))
    assert rel_err(host(dw), G) < GRAD_F16_TOL


# more streams than kept scratch blocks, in flight together: each call has a block of its own
# or one ordered behind its last use, so the bits are those of the calls one at a time
def test_mlp_gradient_streams():
    rng = np.random.default_rng(11)
    w = dev(rng.normal(0, np.sqrt(2 / 64), v.weight_count(5)).astype(np.float16))
    x, t = dev(rng.uniform(-1, 1, (12 * 4096, 64)).astype(np.float16)), dev(rng.uniform(0, 1, (12 * 4096, 3)).astype(np.float32))
    calls = [(x[4096 * k:4096 * (k + 1)], t[4096 * k:4096 * (k + 1)]) for k in range(12)]
    one, many = (torch.zeros((12, v.weight_count(5)), device=DEV) for _ in range(2))
    for k, (xk, tk) in enumerate(calls):
        v.mlp_gradient_f16(w, xk, tk, 4096, one[k])
        torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(4)]
    for k, (xk, tk) in enumerate(calls):
        v.mlp_gradient_f16(w, xk, tk, 4096, many[k], stream=streams[k % 4])
    assert np.array_equal(host(many), host(one))


# the forward reads row-major weights with 16-byte loads at any alignment and puts them into LDS
# in fragment order: the same fragments, so the same bits
@pytest.mark.parametrize("hidden", [4, 5])
@pytest.mark.parametrize("n", [1, 63, 65, 4097])
def test_mlp_forward_weight_alignment(hidden, n):
    rng = np.random.default_rng(n + hidden)
    w = rng.normal(0, np.sqrt(2 / 64), v.weight_count(hidden)).astype(np.float16)
    x = dev(rng.uniform(-1, 1, (n, 64)).astype(np.float16))
    out = []
    for shift in (0, 1, 2, 4):
        buf = dev(np.concatenate([np.zeros(shift, np.float16), w]))
        out.append(torch.full((n, 3), 7.0, device=DEV))
        v.mlp_forward_f16(buf[shift:], x, n, out[-1], hidden_layers=hidden)
    m = [w.astype(np.float64)[4096 * l:4096 * (l + 1)].reshape(64, 64) for l in range(hidden)]
    a = host(x).astype(np.float64)
    for l in range(hidden):
        a = np.maximum(a @ m[l].T, 0).astype(np.float16).astype(np.float64)
    assert rel_err(host(out[0]), a @ w.astype(np.float64)[4096 * hidden:].reshape(3, 64).T) < GRAD_F16_TOL
    assert all(torch.equal(o, out[0]) for o in out)


# FP32 sums of 64 products over at most 6 layers are within 6 * 64 * 2^-24 = 2.3e-5 of their
# exact values relative to the largest terms; the gradient passes through three such chains.
PLAIN_TOL, PLAIN_GRAD_TOL = 2.3e-5, 7e-5
ENCODINGS = [(5, v.ENCODING_TRI12), (5, v.ENCODING_SINCOS6), (4, v.ENCODING_UV_SINCOS16)]


def plain_inputs(hidden, enc, n):
    rng = np.random.default_rng(100 * n + hidden + enc)
    r = wl.make_train_records(n, rng, wl.GaussianLights(7))
    if enc == v.ENCODING_UV_SINCOS16:
        r[:, :2] = rng.uniform(0, 1, (n, 2))
    return rng.normal(0, np.sqrt(2 / 64), v.weight_count(hidden)).astype(np.float32), r


# 16-record tiles over one workgroup a CU: partial tiles, one tile more than CUs, waves with
# no tile, and a device count that ends inside a tile
@pytest.mark.parametrize("hidden,enc", ENCODINGS)
@pytest.mark.parametrize("n,live", [(1, 1), (16, 16), (17, 17), (4112, 4097), (33000, 32769)])
def test_plain_inference_tiles(hidden, enc, n, live):
    w, r = plain_inputs(hidden, enc, n)
    st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc))
    st.set_state(weight=w)
    out = torch.full((n, 3), 7.0, device=DEV)
    st.infer(dev(r[:, :14]), out, count=dev(np.array([live], np.uint32).view(np.int32)), path=v.PATH_PLAIN_F32)
    y = host(out)
    f = Oracle("f32").encode(r[:live], enc).astype(np.float64)  # features rounded as FP32 computes them
    ref = np.maximum(Oracle("f64").infer_encoded(w.astype(np.float64), hidden, f), 0)
    assert rel_err(y[:live], ref) < PLAIN_TOL
    assert (y[live:] == 7.0).all()
    st.close()


# the FP32 weight gradient: inside one tile, at its edges, half a 512-record chunk and one record more,
# many chunks with a partial last one, and a device count below the size (the edges of a chunk are
# test_gpu_later_tiles.py's)
@pytest.mark.parametrize("hidden,enc", ENCODINGS)
@pytest.mark.parametrize("n,live", [(1, 1), (16, 16), (17, 17), (256, 256), (257, 257), (8193, 8100)])
def test_plain_gradient_chunks(hidden, enc, n, live):
    w, r = plain_inputs(hidden, enc, n)
    st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc, loss=v.LOSS_L2))
    st.set_state(weight=w)
    st.train(dev(r), count=dev(np.array([live], np.uint32).view(np.int32)), path=v.PATH_PLAIN_F32)
    s = st.get_state()
    f = Oracle("f32").encode(r[:live], enc).astype(np.float64)
    G, loss = Oracle("f64").gradient_encoded(w.astype(np.float64), hidden, f, r[:live, 14:].astype(np.float64), loss=1)
    assert rel_err(s["m"] / (1.0 - np.float32(0.9)), G / live) < PLAIN_GRAD_TOL
    assert abs(s["state"]["last_loss"] / (loss / live) - 1) < PLAIN_GRAD_TOL
    st.close()


# the FP8 tiles: one to a few records of a 32-record half, both halves, one tile and one more, and
# a workgroup's worth of tiles; every size gives the records the bits they have in a large call
# (whose parity with the FP8 oracle is tests/test_gpu_fp8.py's), and nothing past the count is written
@pytest.mark.parametrize("hidden,enc", ENCODINGS)
def test_fp8_inference_tiles(hidden, enc):
    w, r = plain_inputs(hidden, enc, 4097)
    r[:, 3:8] = np.linspace(-0.5, 1.5, r[:, 3:8].size, dtype=np.float32).reshape(-1, 5)  # every one-blob knot

    def first(n, live):
        st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc))
        st.set_state(weight=w)
        out = torch.full((n, 3), 7.0, device=DEV)
        st.infer(dev(r[:n, :14]), out, count=dev(np.array([live], np.uint32).view(np.int32)), path=v.PATH_FUSED_F8)
        y = host(out)
        st.close()
        return y

    whole = first(4097, 4097)
    f = Oracle("f32").encode(r, enc)
    st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc))
    st.set_state(weight=w)
    st.infer(dev(r[:, :14]), torch.zeros((4097, 3), device=DEV), path=v.PATH_FUSED_F8)
    sc = st.get_fp8_scales()
    st.close()
    # 5e-2: an e4m3 step is 6-12 % of a value, and sums near a rounding boundary fall either way
    assert rel_err(whole, infer_fp8(f, w, hidden, sc["layer_scales"], sc["out_scale"], clamp0=True)) < 5e-2
    for n, live in ((1, 1), (31, 31), (33, 33), (64, 63), (65, 65), (257, 257), (1025, 900)):
        y = first(n, live)
        assert np.array_equal(y[:live], whole[:live]), n
        assert (y[live:] == 7.0).all()


# a launch for many records takes a wave's 64 through LDS, one for few goes straight to memory:
# every lane of a partial wave, one wave and one record more, a device count inside a wave, odd
# record addresses; each prefix gives the rows of the whole, and nothing past the count is written
@pytest.mark.parametrize("room", [0, 70000])
@pytest.mark.parametrize("packed", [False, True])
def test_unpack_partial_waves(packed, room):
    s = wl.make_scene(5, primitives=300, vertices=200, instances=3, materials=5, textures=2, texture_size=16)
    ds = v.DeviceScene(torch, s["vertices"], s["vertex_indices"], s["texcoords"], s["texcoord_indices"], s["materials"],
                       s["material_ids"], s["transforms"], s["textures"])
    if packed:
        ds.pack_primitives()
    rng = np.random.default_rng(6)
    ev = np.zeros(700, v.EVAL_RECORD)
    ev["packed_input"] = wl.make_packed_inputs(s, 700, rng)
    tr = np.zeros(700, v.WIRE_TRAIN_RECORD)
    tr["packed_input"], tr["bias"] = ev["packed_input"], rng.uniform(0, 1, (700, 3))
    ref = frontend.unpack(s, ev["packed_input"])
    words = lambda a: dev(np.concatenate([np.zeros(1, np.int32), np.frombuffer(a.tobytes(), np.int32)]))[1:]  # noqa: E731

    def rows(fn, rec, width, n, live):
        rec = np.concatenate([rec[:n], np.zeros(max(room - n, 0), rec.dtype)])
        n = len(rec)
        out = torch.full((n, width), 7.0, device=DEV)
        fn(ds, words(rec), n, out, count=dev(np.array([live], np.uint32).view(np.int32)))
        y = host(out)
        assert (y[live:] == 7.0).all()
        return y[:live]

    whole = rows(v.unpack_eval_records, ev, 14, 700, 700)
    # 2e-5 is FP32 rounding of positions and colours of order 1; the sphere encoding's acos is steep at its poles
    assert np.abs(whole - ref)[:, [0, 1, 2, 3, 4, 7, 8, 9, 10, 11, 12, 13]].max() < 2e-5
    assert np.quantile(np.abs(whole - ref)[:, 5:7], 0.99) < 1e-5
    trained = rows(v.unpack_train_records, tr, 17, 700, 700)
    assert np.array_equal(trained[:, :14], whole) and np.array_equal(trained[:, 14:], tr["bias"])
    for n, live in ((1, 1), (3, 2), (63, 63), (64, 64), (65, 65), (256, 255), (257, 257), (600, 321)):
        assert np.array_equal(rows(v.unpack_eval_records, ev, 14, n, live), whole[:live]), n
        assert np.array_equal(rows(v.unpack_train_records, tr, 17, n, live), trained[:live]), n


# a group of multi-chunk rows in three rounds, which run one a workgroup on 256 CUs (two a workgroup:
# test_gpu_row_pairs.py): caches with an odd number of rows, a single row, a partial last chunk, device
# counts that leave a row's last chunk or whole rows empty, and a chunk whose deltas carry a scale, each with
# the bits that the cache has alone
@pytest.mark.parametrize("hidden,enc", ENCODINGS)
@pytest.mark.parametrize("loss", [v.LOSS_RELATIVE_L2_LUMINANCE, v.LOSS_L2])
def test_gradient_row_pairs(hidden, enc, loss):
    sizes = [(16384, 16384, 2), (16383, 16383, 2), (12000, 7001, 3), (64, 64, 2), (16384, 100, 2), (16000, 0, 4),
             (8257, 8257, 2)]
    assert sum(-(-n // (64 * c)) for n, _, c in sizes) > 256

    def caches():
        out = []
        for i, (n, live, chunks) in enumerate(sizes):
            w, r = plain_inputs(hidden, enc, n)
            if i == 1:
                r[200:230, 14:] *= 1e6
            st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc, loss=loss))
            st.set_state(weight=w)
            st.set_grad_chunks(chunks)
            out.append(dict(cache=st, batches=dev(r), max_batch_records=n,
                            batch_counts=dev(np.array([live], np.uint32).view(np.int32))))
        return out

    group, alone = caches(), caches()
    v.group_train(group, 0, write_use_weights=True)
    for e in alone:
        e["cache"].train(e["batches"], count=e["batch_counts"], max_count=e["max_batch_records"])
    for g, a in zip(group, alone):
        x, y = g["cache"].get_state(), a["cache"].get_state()
        for k in ("weight", "m", "v", "ema_weight", "weights_f16", "use_weights_f16"):
            assert np.array_equal(x[k], y[k]), k
        assert x["state"] == y["state"]
    for e in group + alone:
        e["cache"].close()


# one cache's inference deals the tiles of the device count if there are more than waves (2,048), else
# those of the maximum: counts around a tile, far below the maximum and zero give the rows of the whole
# and write nothing past the count
@pytest.mark.parametrize("n", [70001, 140001])
@pytest.mark.parametrize("hidden,enc", ENCODINGS)
def test_f16_inference_deals_the_counted_tiles(hidden, enc, n):
    w, r = plain_inputs(hidden, enc, n)
    st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc))
    st.set_state(weight=w)
    q = dev(r[:, :14])
    whole = torch.zeros((n, 3), device=DEV)
    st.infer(q, whole)
    whole = host(whole)
    for live in (0, 1, 63, 64, 65, 2048 * 64 // 4 + 1, n - 1):
        out = torch.full((n, 3), 7.0, device=DEV)
        st.infer(q, out, count=dev(np.array([live], np.uint32).view(np.int32)))
        y = host(out)
        assert np.array_equal(y[:live], whole[:live]), live
        assert (y[live:] == 7.0).all(), live
    st.close()
