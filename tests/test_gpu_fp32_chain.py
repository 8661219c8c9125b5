"""The FP32 inference and gradient bit for bit: a layer's sums are fused multiply-adds over k = 0 .. 63 in
order, and a weight's gradient over the records in order, with ordinary, subnormal, very large, infinite
and NaN weights and fields (restated in numpy on the features that nrc_encode gives)."""
import numpy as np
import pytest

import vknrc_amd as v
from vknrc_amd import workloads as wl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"
F32 = np.float32
ENCODINGS = [(5, v.ENCODING_TRI12), (5, v.ENCODING_SINCOS6), (4, v.ENCODING_UV_SINCOS16)]


def fma32(a, b, c):
    """fmaf on float32 arrays: the product is exact in float64, and the sum is rounded to odd there (by
    TwoSum's error), which rounds to float32 as the exact sum does."""
    p, c = a.astype(np.float64) * b.astype(np.float64), c.astype(np.float64)
    s = p + c
    bb = s - p
    err = (p - (s - bb)) + (c - bb)
    even = (err != 0) & np.isfinite(err) & (s.view(np.int64) & 1 == 0)
    return np.where(even, np.nextafter(s, np.where(err > 0, np.inf, -np.inf)), s).astype(F32)


def chain(m, x):
    """W x for rows of x, each sum one fused multiply-add after the other."""
    acc = np.zeros((len(x), len(m)), F32)
    for k in range(64):
        acc = fma32(np.broadcast_to(x[:, k:k + 1], acc.shape), np.broadcast_to(m[:, k], acc.shape), acc)
    return acc


def special_weights(rng, hidden, kind):
    w = rng.normal(0, np.sqrt(2 / 64), v.weight_count(hidden)).astype(F32)
    at = rng.integers(0, w.size, 40)
    if kind == "subnormal":  # products of two are zero, so only the first layer's sums are not
        w *= F32(3e-39)
    elif kind == "subnormal first layer":  # every sum after it is of subnormals
        w[:4096] *= F32(3e-39)
    elif kind == "some subnormal":
        w[rng.random(w.size) < 0.5] *= F32(3e-39)
    elif kind == "small":  # products of two of them are subnormal or zero
        w *= F32(1e-20)
    elif kind == "large":  # sums overflow after a few layers
        w *= F32(1e10)
    elif kind == "infinite":
        w[at[:20]], w[at[20:]] = np.inf, -np.inf
    elif kind == "nan":
        w[at[:3]] = np.nan
    return w


@pytest.mark.parametrize("hidden,enc", ENCODINGS)
@pytest.mark.parametrize("kind", ["ordinary", "fields", "subnormal", "subnormal first layer", "some subnormal", "small", "large", "infinite", "nan"])
def test_plain_inference_is_the_chain_of_fmas(hidden, enc, kind):
    rng = np.random.default_rng(3)
    n = 333
    q = wl.make_queries(n, rng)
    if kind == "fields":
        for value in (np.nan, np.inf, -np.inf, 1e30, 1e-40, -1e-40, 3e38, -0.0):
            q[rng.random(q.shape) < 0.02] = value
    w = special_weights(rng, hidden, kind)
    st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc))
    st.set_state(weight=w)
    dq = torch.from_numpy(q).to(DEV)
    feat, out = torch.zeros((n, 64), device=DEV), torch.full((n, 3), 7.0, device=DEV)
    v.encode(dq, n, feat, encoding=enc)
    st.infer(dq, out, path=v.PATH_PLAIN_F32)
    torch.cuda.synchronize()
    st.close()
    x = feat.cpu().numpy()
    with np.errstate(all="ignore"):
        for l in range(hidden):
            x = np.fmax(chain(w[4096 * l:4096 * (l + 1)].reshape(64, 64), x), F32(0))
        want = np.fmax(chain(w[4096 * hidden:].reshape(3, 64), x), F32(0))
    assert np.array_equal(out.cpu().numpy(), want, equal_nan=True)
    if kind in ("ordinary", "subnormal first layer", "some subnormal"):
        assert np.count_nonzero(want) > n / 2


def gradient(w, hidden, x, t):
    """dW of the squared error, as the optimizer gets it: ReLU masks of the stored activations, a NaN delta is
    0 and an infinite one passes (NN_nv.glsl:198-220)."""
    m = [w[4096 * l:4096 * (l + 1)].reshape(64, 64) for l in range(hidden)] + [w[4096 * hidden:].reshape(3, 64)]
    acts = [x]
    for l in range(hidden):
        acts.append(np.fmax(chain(m[l], acts[-1]), F32(0)))
    d = (F32(2) * (chain(m[hidden], acts[-1]) - t)).astype(F32)
    out = []
    for l in range(hidden, -1, -1):
        g = np.zeros((d.shape[1], 64), F32)
        for k in range(len(x)):
            g = fma32(np.broadcast_to(d[k][:, None], g.shape), np.broadcast_to(acts[l][k], g.shape), g)
        out.append(g.ravel())
        if l:
            y = np.zeros((len(x), 64), F32)
            for k in range(d.shape[1]):
                y = fma32(np.broadcast_to(m[l][k], y.shape), np.broadcast_to(d[:, k:k + 1], y.shape), y)
            d = np.where((acts[l] > 0) & ~np.isnan(y), y, F32(0))
    return np.concatenate(out[::-1])


# one partial row (at most 512 records), a partial last tile; the first moment of the first step is
# (1 - beta1) g with g = dW / count, or 0 where that is not finite, and a dynamic loss scale skips the step
# if any of it is not
@pytest.mark.parametrize("hidden,enc", ENCODINGS)
@pytest.mark.parametrize("kind", ["ordinary", "fields", "one field", "targets", "subnormal first layer", "some subnormal",
                                  "small", "large", "infinite", "nan"])
def test_plain_gradient_is_the_chain_of_fmas(hidden, enc, kind):
    rng = np.random.default_rng(13)
    n = 125
    r = wl.make_train_records(n, rng, wl.GaussianLights(7))
    if kind == "fields":
        for value in (np.nan, np.inf, -np.inf, 1e30, 1e-40, -1e-40, 3e38, -0.0):
            r[:, :14][rng.random((n, 14)) < 0.02] = value
    elif kind == "one field":
        r[70, 1] = np.nan
    elif kind == "targets":
        for value in (np.nan, np.inf, 1e-40, 3e38):
            r[:, 14:][rng.random((n, 3)) < 0.01] = value
    w = special_weights(rng, hidden, kind)
    dr, feat = torch.from_numpy(r).to(DEV), torch.zeros((n, 64), device=DEV)
    v.encode(dr[:, :14].contiguous(), n, feat, encoding=enc)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        G = gradient(w, hidden, feat.cpu().numpy(), r[:, 14:])
        g = (G / F32(n)).astype(F32)
        m = ((F32(1) - F32(0.9)) * np.where(np.isfinite(g), g, F32(0))).astype(F32)
    if kind in ("ordinary", "subnormal first layer", "some subnormal"):
        assert np.isfinite(G).all() and np.count_nonzero(G) > 100
    for dynamic in (False, True):
        st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc, loss=v.LOSS_L2, dynamic_loss_scale=dynamic))
        st.set_state(weight=w)
        st.train(dr, path=v.PATH_PLAIN_F32)
        s = st.get_state()
        st.close()
        if dynamic and not np.isfinite(G).all():
            assert s["state"]["skipped_steps"] == 1 and s["state"]["t"] == 0 and not s["m"].any()
            assert np.array_equal(s["weight"], w, equal_nan=True)
        else:
            assert s["state"]["skipped_steps"] == 0 and s["state"]["t"] == 1
            assert np.array_equal(s["m"], m)
