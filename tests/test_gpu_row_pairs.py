"""The gradient kernel that runs two rows a workgroup (fused_grad_dual_kernel) against the one that
runs one (fused_grad_small_kernel): the same bits, for every depth, encoding and loss.  Which of the
two a launch takes is asserted by the rule of csrc/nrc_grad_rows.hpp (grad_rows.py, which
test_gradient_rows_rule.py holds to the C++), with the CU count of the device."""
import numpy as np
import pytest

import grad_rows
import vknrc_amd as v
from vknrc_amd import workloads as wl

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda"
KINDS = [(h, e) for h in (4, 5) for e in (v.ENCODING_TRI12, v.ENCODING_SINCOS6, v.ENCODING_UV_SINCOS16)]
LOSSES = [v.LOSS_RELATIVE_L2_LUMINANCE, v.LOSS_L2]
DELTA_LIMIT = 8192.0  # largest output gradient of a chunk above which its deltas carry a scale


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def caches(hidden, enc, loss, sizes):
    """Caches with their records: sizes (records, device count, chunks a row); some records of the second
    have targets so large that the deltas of their chunks carry a scale."""
    out = []
    for i, (n, live, chunks) in enumerate(sizes):
        rng = np.random.default_rng(1000 * i + 10 * hidden + enc)
        r = wl.make_train_records(n, rng, wl.GaussianLights(7))
        if enc == v.ENCODING_UV_SINCOS16:
            r[:, :2] = rng.uniform(0, 1, (n, 2))
        if i == 1:
            r[200:230, 14:] = 1e6 * (1 + r[200:230, 14:])  # the relative loss divides by at most the output's square
        st = v.NRCState(v.NRCConfig(hidden_layers=hidden, encoding=enc, loss=loss, seed=i, train_batch_size=max(n, 16384)))
        st.set_grad_chunks(chunks)
        out.append(dict(cache=st, batches=dev(r), max_batch_records=n,
                        batch_counts=dev(np.array([live], np.uint32).view(np.int32))))
    return out


def same_state(a, b):
    x, y = a["cache"].get_state(), b["cache"].get_state()
    for k in ("weight", "m", "v", "ema_weight", "weights_f16", "use_weights_f16"):
        assert np.array_equal(x[k], y[k]), k
    assert x["state"] == y["state"] and x["state"]["skipped_steps"] == 0
    assert np.isfinite(x["m"]).all()


# caches with full rows, a partial last chunk, an odd number of rows, a single row of one chunk, a row
# of which one chunk has records, rows that the device count leaves empty beside a live one, and no record
# at all; in one launch of pairs, and each in a launch of single rows
@pytest.mark.parametrize("loss", LOSSES)
@pytest.mark.parametrize("hidden,enc", KINDS)
def test_group_of_pairs_has_the_bits_of_single_rows(hidden, enc, loss):
    sizes = [(16384, 16384, 2), (16383, 16383, 2), (12000, 7001, 3), (64, 64, 2), (8257, 8257, 2), (4096, 100, 2),
             (4000, 0, 3)]
    assert grad_rows.in_pairs([(n, c) for n, _, c in sizes], cus())
    assert not any(grad_rows.in_pairs([(n, c)], cus()) for n, _, c in sizes)
    group, alone = caches(hidden, enc, loss, sizes), caches(hidden, enc, loss, sizes)
    for _ in range(2):  # the second step runs on other weights and the other state buffer
        v.group_train(group, 0, write_use_weights=True)
        for e in alone:
            e["cache"].train(e["batches"], count=e["batch_counts"], max_count=e["max_batch_records"])
    for g, a in zip(group, alone):
        same_state(g, a)
    assert sum(e["cache"].get_state()["m"].any() for e in group) == len(sizes) - 1  # all but the empty one trained
    for e in group + alone:
        e["cache"].close()


# one cache with more rows than CUs runs in pairs alone, and as single rows in a group of three rounds
@pytest.mark.parametrize("live", [40000, 20001])
@pytest.mark.parametrize("loss", LOSSES)
@pytest.mark.parametrize("hidden,enc", KINDS)
def test_one_cache_in_pairs_has_the_bits_of_single_rows(hidden, enc, loss, live):
    sizes = [(40000, live, 2), (16384, 16384, 2), (16384, 9000, 2)]
    assert grad_rows.in_pairs([(40000, 2)], cus())
    assert not grad_rows.in_pairs([(n, c) for n, _, c in sizes], cus())
    group, alone = caches(hidden, enc, loss, sizes), caches(hidden, enc, loss, sizes[:1])
    v.group_train(group, 0, write_use_weights=True)
    alone[0]["cache"].train(alone[0]["batches"], count=alone[0]["batch_counts"], max_count=40000)
    same_state(group[0], alone[0])
    for e in group + alone:
        e["cache"].close()


# the scaled chunk of the second cache is one: its largest output gradient, 2 s e / d with the loss's
# denominator, is past the limit whatever the network's output
@pytest.mark.parametrize("loss", LOSSES)
def test_the_scaled_chunk_passes_the_limit(loss):
    e = caches(5, v.ENCODING_TRI12, loss, [(64, 64, 2), (16383, 16383, 2)])[1]
    st = e["cache"]
    q = e["batches"][:, :14].contiguous()
    out = torch.zeros((16383, 3), device=DEV)
    st.infer(q, out)
    torch.cuda.synchronize()
    o, t = out.cpu().numpy()[200:230], e["batches"].cpu().numpy()[200:230, 14:]
    d = 1.0 if loss == v.LOSS_L2 else (o @ np.array([0.299, 0.587, 0.114])) ** 2 + 0.01
    assert (np.abs(2 * (o - t)).max(1) / d).max() > DELTA_LIMIT
    st.close()


# a row without a record beside a live one runs on zeros where a single row is left out: no infinite or NaN
# weight, field or target may show the difference
@pytest.mark.parametrize("kind", ["infinite weights", "NaN weights", "infinite output weight", "fields", "targets"])
@pytest.mark.parametrize("hidden,enc", [(5, v.ENCODING_TRI12), (4, v.ENCODING_UV_SINCOS16)])
def test_pairs_and_single_rows_agree_on_special_values(hidden, enc, kind):
    sizes = [(16384, 16384, 2), (16383, 16383, 2), (12000, 7001, 3), (64, 64, 2), (8257, 8257, 2), (4096, 100, 2),
             (4000, 0, 3)]
    assert grad_rows.in_pairs([(n, c) for n, _, c in sizes], cus())
    sets = []
    for _ in range(2):
        sets.append(caches(hidden, enc, v.LOSS_L2, sizes))
        for i, e in enumerate(sets[-1]):
            rng = np.random.default_rng(i)
            w, r = e["cache"].get_state()["weight"].copy(), e["batches"].cpu().numpy()
            at = rng.integers(0, w.size, 6)
            if kind == "infinite weights":
                w[at[:3]], w[at[3:]] = np.inf, -np.inf
            elif kind == "NaN weights":
                w[at[:2]] = np.nan
            elif kind == "infinite output weight":
                w[w.size - 192 + at[0] % 192] = np.inf
            else:
                cols, rate = (slice(0, 14), 1e-3) if kind == "fields" else (slice(14, 17), 1e-4)
                for value in (np.nan, np.inf, 1e30, -1e30, 1e-40):
                    r[:, cols][rng.random((len(r), cols.stop - cols.start)) < rate] = value
            e["cache"].set_state(weight=w)
            e["batches"] = dev(r)
    group, alone = sets
    v.group_train(group, 0, write_use_weights=True)
    for e in alone:
        e["cache"].train(e["batches"], count=e["batch_counts"], max_count=e["max_batch_records"])
    for g, a in zip(group, alone):
        x, y = g["cache"].get_state(), a["cache"].get_state()
        for k in ("weight", "m", "v", "ema_weight", "weights_f16", "use_weights_f16"):
            assert np.array_equal(x[k], y[k], equal_nan=True), k
        for k, value in x["state"].items():
            assert value == y["state"][k] or (np.isnan(value) and np.isnan(y["state"][k])), k
    for e in group + alone:
        e["cache"].close()
