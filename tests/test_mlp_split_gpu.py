"""GPU: the MLP's hidden layers with every fp32 number in three bf16 pieces
(habitat_amd/csrc/mlp_split.h), at the sizes where its kernels change."""
import ctypes

import numpy as np
import pytest
import torch

from habitat_amd import _lib, synthetic
from habitat_amd.analysis.mlp.mlp import RuntimePredictor
from oracle import mlp as omlp

pytestmark = pytest.mark.gpu


def network(kind, hidden, seed=0):
    """Weights that keep the activations' size from layer to layer."""
    torch.manual_seed(seed)
    rp = RuntimePredictor(kind, hidden, 1024)
    with torch.no_grad():
        for name, p in rp.model.named_parameters():
            if name.endswith("weight") and not name.startswith("fc2"):
                p.mul_(6.0 ** 0.5)
    return rp


def without_pairs(rp):
    """Keeps `rp` from the fp16 pairs (mlp_pairs.h), from 1025 rows on: the last unit of the
    last hidden layer, which fc2 no longer reads, hangs on one of its inputs.  Returns a
    predictor without that weight, for which a batch of some rows gives the same numbers in
    other roundings if and only if one of the two runs in pairs and the other does not."""
    rp.model.fc2.weight.data[0, 1023] = 0.0
    other = RuntimePredictor(rp.model_name, rp.layers, 1024)
    other.model.load_state_dict(rp.model.state_dict())
    other.set_normalization(rp.mu, rp.sigma)
    rp.model.mlp.layers[2 * (rp.layers - 1)].weight.data[1023, 5] = 100.0
    rp.refresh()
    return other


def forward_fp64(rp, x):
    """oracle.mlp.forward_fp64 on the GPU (float64 matrix products)."""
    sd = {k: v.double().cuda() for k, v in rp.model.state_dict().items()}
    h = torch.from_numpy(omlp.standardise(x, rp.mu, rp.sigma)).cuda().double()
    layers = ["fc1"] + sorted({k[:-7] for k in sd if k.startswith("mlp") and k.endswith("weight")},
                              key=lambda k: int(k.split(".")[2]))
    for name in layers:
        h = torch.relu(h @ sd[name + ".weight"].t() + sd[name + ".bias"])
    return (h @ sd["fc2.weight"].t() + sd["fc2.bias"]).reshape(-1).cpu().numpy()


# around the 32-row tiles, the workgroups' 32 to 256 rows, the rounds of 256, 512,
# 1024, 1536, 2048, 3072, 4096, 6144 and 16 384 rows, and chunks of 16 384
@pytest.mark.parametrize("rows", [129, 160, 161, 255, 256, 257, 480, 511, 512, 513, 700, 1023, 1024,
                                  1025, 1500, 1536, 1537, 2048, 2049, 2080, 2177, 3071, 3072, 3073,
                                  4095, 4096, 4097, 4161, 4608, 4609, 5911, 6113, 6144, 6145, 7169,
                                  7200, 7424, 7425, 8193, 9217, 10241, 11000, 12288, 12289, 13000,
                                  16351, 16383, 16384, 16385, 24001, 32768, 32769, 40001])
@pytest.mark.parametrize("hidden", [1, 2])
def test_rows_around_the_kernels_edges(rows, hidden):
    rp = network("lstm", hidden)
    x, mu, sigma = synthetic.mlp_features("lstm", rows, seed=rows)
    rp.set_normalization(mu, sigma)
    check_against_fp64(rp, x)


def check_against_fp64(rp, x):
    hidden = rp.layers
    y = rp.predict_batch(x).cpu().numpy().astype(np.float64)
    want = forward_fp64(rp, x)
    # Per layer a sum of 1024 products in fp32: an error of at most 8 x 2^-24 of the
    # output's rms, as fp32 sums of that length have (7 on the fp32 matrix cores),
    # each layer's carried through the later ones at the same size; torch's own
    # float32 forward measures 3e-7 at the worst row here.
    rms = float(np.sqrt(np.mean((want - want.mean()) ** 2))) + abs(float(want.mean()))
    err = float(np.sqrt(np.mean((y - want) ** 2)))
    assert err <= (hidden + 1) * 8 * 2.0 ** -24 * rms
    assert float(np.max(np.abs(y - want))) <= 6 * (hidden + 1) * 8 * 2.0 ** -24 * rms
    assert np.array_equal(y, rp.predict_batch(x).cpu().numpy().astype(np.float64))


# The kernels of split_kernel_for from 1025 rows on, where other networks take the pairs.
@pytest.mark.parametrize("rows", [1025, 1500, 1536, 1537, 2048, 2049, 2177, 3071, 3072, 3073, 4000, 4096,
                                  4097, 4608, 4609, 5911, 6144, 6145, 7300, 8192, 8193, 9216, 9217,
                                  10240, 10241, 11000, 12288, 12289, 13000, 16384, 16385 + 1024, 32769])
@pytest.mark.parametrize("hidden", [1, 2])
def test_rows_around_the_kernels_edges_in_pieces(rows, hidden):
    rp = network("lstm", hidden)
    x, mu, sigma = synthetic.mlp_features("lstm", rows, seed=rows)
    rp.set_normalization(mu, sigma)
    pairs = without_pairs(rp)
    check_against_fp64(rp, x)
    assert not torch.equal(rp.predict_batch(x), pairs.predict_batch(x))
    assert torch.equal(rp.predict_batch(x[:1024]), pairs.predict_batch(x[:1024]))


@pytest.mark.parametrize("rows", [200, 400, 800, 1400, 2000, 3000, 4000, 6000, 9000, 20000])
def test_values_beyond_bf16(rows):
    """Activations beyond the largest bf16, up to infinity, and NaN: what fp32
    arithmetic gives."""
    rp = network("bmm", 1)
    big = np.float32(3.4028234663852886e38)
    finite = np.array([big, np.nextafter(big, np.float32(0)), 3.3961775e38, 3.39617e38, 3.3895e38,
                       1.0 / 3.0, 2.0 ** -100, 1e-30, 65537.0, -big, 0.0])
    x = np.zeros((rows, 8))
    # One unit of fc1 is the feature and one hidden unit an eighth of it, so every
    # result is exact; a NaN is handed on.
    with torch.no_grad():
        for p in rp.model.parameters():
            p.zero_()
        rp.model.fc1.weight[7, 2] = 1.0
        rp.model.mlp.layers[0].weight[100, 7] = 2.0 ** -3
        rp.model.fc2.weight[0, 100] = 1.0
    rp.set_normalization(np.zeros(8), np.ones(8))
    x[:, 2] = np.resize(np.append(finite, np.nan), rows)
    y = rp.predict_batch(x).cpu().numpy()
    v = x[:, 2].astype(np.float32)
    want = np.maximum(v, 0) * np.float32(2.0 ** -3)
    assert np.array_equal(y, want, equal_nan=True)
    # An infinite activation whose every weight is positive stays an infinity:
    # none of its pieces may meet a zero or a negative piece of a weight (0.3 and
    # 0.7 have both).
    with torch.no_grad():
        rp.model.fc1.weight[:, 2] = 1.0
        rp.model.mlp.layers[0].weight.fill_(0.3)
        rp.model.mlp.layers[0].weight[:, ::2] = 0.7
        rp.model.mlp.layers[0].weight[:, ::3] = 0.5
        rp.model.fc2.weight.fill_(2.0 ** -10)
    rp.refresh()
    x[:, 2] = np.resize(np.array([np.inf, 1.0, 1e300, -np.inf]), rows)
    y = rp.predict_batch(x).cpu().numpy()
    assert np.array_equal(np.isposinf(y), x[:, 2] > 1.0)
    assert np.all(y[x[:, 2] < 0] == 0) and np.all(np.isfinite(y[x[:, 2] == 1.0]))


@pytest.mark.parametrize("rows", [200, 400, 800, 1400, 2000, 3000, 4000, 6000, 9000, 11000, 13000,
                                  16351])
def test_values_beyond_bf16_among_dense_weights(rows):
    """As above where the network takes the pieces: one unit of fc1 is the feature,
    the others are zero, and the hidden weights are dense.  NaN and infinities too."""
    rp = network("bmm", 1)
    big = np.float32(3.4028234663852886e38)
    values = np.array([big, np.nextafter(big, np.float32(0)), 3.3961775e38, 3.39617e38, 3.3895e38,
                       1.0 / 3.0, 2.0 ** -100, 1e-30, 65537.0, -big, 0.0, np.nan, np.inf, -np.inf])
    with torch.no_grad():
        rp.model.fc1.weight.zero_()
        rp.model.fc1.bias.zero_()
        rp.model.fc1.weight[7, 2] = 1.0
        hidden = rp.model.mlp.layers[0]
        hidden.bias.zero_()
        hidden.weight[:, 7] = -0.7                 # the other units are dead
        hidden.weight[100, 7] = 2.0 ** -3
        rp.model.fc2.weight.fill_(1.0)
        rp.model.fc2.bias.zero_()
    rp.set_normalization(np.zeros(8), np.ones(8))
    x = np.zeros((rows, 8))
    x[:, 2] = np.resize(values, rows)
    v = x[:, 2].astype(np.float32)
    with np.errstate(invalid="ignore"):
        # a NaN or an infinity of the feature is NaN in every unit of fc1 (0 x inf)
        want = np.where(np.isfinite(v), np.maximum(v, 0) * np.float32(2.0 ** -3), np.nan)
    for y in (rp.predict_batch(x), rp.predict_batch_fp32(x)):
        assert np.array_equal(y.cpu().numpy(), want, equal_nan=True)


@pytest.mark.parametrize("rows", [200, 400, 800, 1400, 2000, 3000, 4000, 6000, 9000, 13000])
def test_infinite_and_huge_weights(rows):
    """One weight that is infinite, huge or tiny against activations that are
    infinite, huge and zero: infinities and NaN where fp32 has them."""
    rp = network("bmm", 1)
    x = np.abs(np.random.default_rng(rows).normal(size=(rows, 8)))
    x[:, 2] = np.resize([10.0, 1.0, 0.5, 0.0, -1.0], rows)
    rp.set_normalization(np.zeros(8), np.ones(8))
    with torch.no_grad():
        for p in rp.model.parameters():
            p.abs_()
        rp.model.fc1.weight[:, 2] = 0.0
        rp.model.fc1.weight[7] = torch.tensor([0, 0, 3e38, 0, 0, 0, 0, 0])   # unit 7 alone
        rp.model.fc1.bias[7] = 0.0
        rp.model.mlp.layers[0].weight[:, 7] = -0.3     # dead where unit 7 is large
        rp.model.fc2.weight.zero_()
        rp.model.fc2.weight[0, 100] = 1.0
        rp.model.fc2.bias.zero_()
    with np.errstate(all="ignore"):
        unit7 = np.maximum(np.float32(3e38) * x[:, 2].astype(np.float32), 0)
        assert np.isposinf(unit7[0]) and unit7[1] > 1e38 and unit7[4] == 0
        for special in (np.inf, -np.inf, 3e38, -3e38, 128.0, 127.0, -127.0, 2.0 ** -100,
                        -2.0 ** -100, 2.0 ** -120):
            with torch.no_grad():
                rp.model.mlp.layers[0].weight[100, 7] = special
            rp.refresh()
            big = np.float32(special) * unit7
            pieces, fp32 = rp.predict_batch(x).cpu().numpy(), rp.predict_batch_fp32(x).cpu().numpy()
            # a network with a weight that does not fit the pieces takes the fp32 kernels
            if abs(special) >= 128:
                assert np.array_equal(pieces, fp32, equal_nan=True)
            else:
                assert not np.array_equal(pieces, fp32, equal_nan=True)
            for y in (pieces, fp32):
                assert np.array_equal(np.isnan(y), np.isnan(big)), special
                assert np.array_equal(np.isposinf(y), np.isposinf(big)), special
                assert np.all(y[big < -1e8] == 0) and np.all(y[big == 0] > 0), special
                large = (big > 1e8) & np.isfinite(big)   # the other units give some hundreds
                assert np.all(np.abs(y[large] / big[large] - 1) < 1e-5), special


@pytest.mark.parametrize("tiny", ["weights", "activations"])
@pytest.mark.parametrize("rows", [200, 3000, 5911, 13000])
def test_numbers_below_the_third_piece(rows, tiny):
    """Weights or activations around 2^-115 lose at most 2^-134 of each product's
    other operand, beside the roundings of the sum."""
    rp = network("bmm", 1)
    x = np.random.default_rng(rows).normal(size=(rows, 8))
    rp.set_normalization(np.zeros(8), np.ones(8))
    with torch.no_grad():
        hidden = rp.model.mlp.layers[0]
        hidden.bias.zero_()
        for p in ((hidden.weight,) if tiny == "weights" else (rp.model.fc1.weight, rp.model.fc1.bias)):
            p.mul_(2.0 ** -115)
        rp.model.fc2.weight.zero_()
        rp.model.fc2.weight[0, 5] = 2.0 ** 100
        rp.model.fc2.bias.zero_()
    rp.refresh()
    y, want = rp.predict_batch(x).double().cpu().numpy(), forward_fp64(rp, x)
    sd = {k: v.double() for k, v in rp.model.state_dict().items()}
    act = torch.relu(torch.from_numpy(x) @ sd["fc1.weight"].t() + sd["fc1.bias"])
    weight = sd["mlp.layers.0.weight"][5].abs()
    other = float(act.sum(1).max()) if tiny == "weights" else float(weight.sum())
    # (the bound of test_rows_around_the_kernels_edges on the largest possible sum)
    size = float((act @ weight).max())
    assert 0 < size < 2.0 ** -100
    bound = 2.0 ** 100 * (2.0 ** -134 * other + 8 * 2.0 ** -24 * size)
    assert float(np.max(np.abs(y - want))) <= bound
    assert not torch.equal(rp.predict_batch(x), rp.predict_batch_fp32(x))


def static_forward(rp, x):
    """hbt_mlp_forward_static."""
    raw = torch.from_numpy(x).cuda()
    out = torch.empty((raw.shape[0],), dtype=torch.float32, device="cuda")
    assert _lib.lib().hbt_mlp_forward_static(
        rp._device_mlp().handle, ctypes.c_void_p(raw.data_ptr()), raw.shape[0],
        ctypes.c_void_p(out.data_ptr()),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    return out


@pytest.mark.parametrize("rows", [129, 1000, 3000, 13000])
def test_sparse_weights_keep_fp32_sums(rows):
    """One output with fewer nonzero weights than the pieces need: the fp32 kernels,
    also through the library's static scratch."""
    rp = network("linear", 2)
    x, mu, sigma = synthetic.mlp_features("linear", rows, seed=rows)
    rp.set_normalization(mu, sigma)
    weight = rp.model.mlp.layers[2].weight
    whole = weight.detach()[1023].clone()
    for nonzero, pieces in ((1024, True), (1, False), (191, False), (192, True), (0, True)):
        with torch.no_grad():
            weight[1023] = whole
            weight[1023, torch.randperm(1024)[nonzero:]] = 0.0
        rp.refresh()
        y, fp32 = rp.predict_batch(x), rp.predict_batch_fp32(x)
        assert torch.equal(y, fp32) != pieces, nonzero
        assert rows > 1024 or torch.equal(static_forward(rp, x), y)


def whole_numbers(seed):
    """Two dense hidden layers of sixteenths, 11 bits wide in the first, whose sums are exact
    in any order: below 2^24 sixteenths in every partial sum, activations of up to three
    pieces and weights of two."""
    rng = np.random.default_rng(seed)
    rp = RuntimePredictor("bmm", 2, 1024)
    first = rng.integers(1, 2048, (1024, 1024)) * rng.choice([-1, 1], (1024, 1024)) / 16
    second = rng.choice([-1, 1], (1024, 1024)) * (rng.random((1024, 1024)) < 0.3)
    last = np.zeros(1024)
    last[rng.choice(1023, 16, replace=False)] = rng.choice([-1, 1], 16)
    with torch.no_grad():
        for p in rp.model.parameters():
            p.zero_()
        rp.model.fc1.weight.copy_(torch.from_numpy(rng.integers(-1, 2, (1024, 8))))
        rp.model.mlp.layers[0].weight.copy_(torch.from_numpy(first))
        rp.model.mlp.layers[2].weight.copy_(torch.from_numpy(second))
        rp.model.mlp.layers[0].bias.copy_(torch.from_numpy(rng.integers(-2048, 2048, 1024) / 16))
        rp.model.mlp.layers[2].bias.copy_(torch.from_numpy(rng.integers(-2048, 2048, 1024) / 16))
        rp.model.fc2.weight.copy_(torch.from_numpy(last)[None])
    rp.set_normalization(np.zeros(8), np.ones(8))
    return rp, rng


# Every kernel of split_kernel_for (256 compute units) at the ends of its ranges and
# between: 1 x 1, 1 x 2, 2 x 2, 2 x 3, 2 x 4, 4 x 3 and 4 x 4 tiles, mid_kernel from 4609
# and 10 241 rows, large_kernel from 12 289; whole and partial last blocks of each.
@pytest.mark.parametrize("rows", [129, 191, 256, 257, 500, 513, 1000, 1025, 1505, 1537, 1950, 2049, 2900,
                                  3073, 4000, 4097, 4605, 4609, 5121, 5911, 6113, 6144, 6145, 7300,
                                  8193, 9100, 9217, 10200, 10241, 11000, 12288, 12289, 13000, 14433,
                                  16351, 16384, 16384 + 12500])
def test_every_weight_position_is_wired_in_pieces(rows):
    rp, rng = whole_numbers(rows)
    other = without_pairs(rp)     # (its last unit is not summed exactly, and not read)
    x = rng.integers(-1, 2, (rows, 8)).astype(np.float64)
    sd = {k: v.double().cuda() for k, v in rp.model.state_dict().items()}
    h = torch.relu(torch.from_numpy(x).cuda() @ sd["fc1.weight"].t())
    for name in ("mlp.layers.0", "mlp.layers.2", "fc2"):
        w = sd[name + ".weight"]
        assert 16 * float((h @ w.abs().t())[:, :1023].max()) + 2048 < 2 ** 24
        h = h @ w.t() + sd[name + ".bias"]
        h = torch.relu(h) if name != "fc2" else h
    pieces, fp32 = rp.predict_batch(x).double(), rp.predict_batch_fp32(x).double()
    assert torch.equal(fp32, h.reshape(-1))
    assert torch.equal(pieces, h.reshape(-1))
    # neither the fp32 kernels nor, from 1025 rows on, the pairs
    x = rng.normal(size=(rows, 8))
    pieces, fp32 = rp.predict_batch(x), rp.predict_batch_fp32(x)
    assert not torch.equal(pieces, fp32)
    if rows > 1024:
        # (the other one's second layer is near what the pairs ask of a sum's terms: it is one
        # of +-1 and 0; with every weight +-1 it takes them)
        with torch.no_grad():
            for m in (rp.model, other.model):
                w = m.mlp.layers[2].weight
                w[:1023][w[:1023] == 0] = 1.0
            other.model.mlp.layers[2].weight[1023] = 1.0
        rp.refresh(), other.refresh()
        assert not torch.equal(rp.predict_batch(x), other.predict_batch(x))


# hbt_mlp_forward_fp32 (device sweeps): around its per-layer path's end at 7168 rows, the
# fused kernel's rounds of 8192 and what such a round leaves over
@pytest.mark.parametrize("kind,rows", [("linear", r) for r in (2048, 2049, 7168, 7169, 8192, 8193,
                                                                16384, 20001)] +
                         [(("conv2d", "linear", "bmm", "lstm")[r % 4], r)
                          for r in (129, 160, 161, 255, 511, 512, 513, 1000, 1025, 1503, 2047,
                                    4095, 4096, 4097, 5002)])
def test_fp32_sums_at_any_row_count(kind, rows):
    rp = network(kind, 2)
    x, mu, sigma = synthetic.mlp_features(kind, rows, seed=rows)
    rp.set_normalization(mu, sigma)
    y = rp.predict_batch_fp32(x).cpu().numpy()
    want = forward_fp64(rp, x)
    rms = float(np.sqrt(np.mean(want ** 2)))
    # the bound of test_rows_around_the_kernels_edges
    assert float(np.sqrt(np.mean((y - want) ** 2))) <= 3 * 8 * 2.0 ** -24 * rms
    # a row's sums do not depend on the rows after it: whole rounds, then the rest
    whole = rows - rows % 8192 if rows % 8192 <= 7168 else rows
    if whole:
        assert np.array_equal(y[:whole], rp.predict_batch_fp32(x[:whole]).cpu().numpy())
    if whole < rows:
        assert np.array_equal(y[whole:], rp.predict_batch_fp32(x[whole:]).cpu().numpy())


@pytest.mark.parametrize("zero_sigma", [False, True])
def test_fp32_sums_hand_on_nan_and_infinities(zero_sigma):
    """test_nan_and_infinite_features_give_what_torch_gives for hbt_mlp_forward_fp32:
    K over workgroups, K in 4, 2 and 1 parts, and the fused kernel."""
    rp = network("conv2d", 4)
    x, mu, sigma = synthetic.mlp_features("conv2d", 9000, seed=2)
    rng, x = np.random.default_rng(1), x.copy()
    special = np.array([np.nan, np.inf, -np.inf, 1e300, -1e300, 3e38, 1e-300, 0.0])
    for r in rng.choice(9000, 900, replace=False):
        x[r, rng.integers(0, x.shape[1])] = rng.choice(special)
    if zero_sigma:
        sigma = np.where(np.arange(sigma.shape[0]) == 3, 0.0, sigma)
    rp.set_normalization(mu, sigma)
    with np.errstate(all="ignore"):
        every = omlp.forward_fp32(rp.model.state_dict(), x, mu, sigma)
    for rows in (20, 100, 300, 3000, 5000, 9000):
        want, got = every[:rows], rp.predict_batch_fp32(x[:rows]).cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(np.isposinf(got), np.isposinf(want))
        assert np.array_equal(np.isneginf(got), np.isneginf(want))
        fin = np.isfinite(want) & (np.abs(want) < 1e3)    # (a feature of 3e38 gives more)
        # the bound of test_rows_around_the_kernels_edges at the worst row, for each of
        # the two orders of fp32 sums
        rms = np.sqrt(np.mean(want[fin].astype(np.float64) ** 2)) if fin.any() else 0.0
        assert np.all(np.abs(got[fin] - want[fin]) <= 2 * 6 * 5 * 8 * 2.0 ** -24 * rms)
        assert not zero_sigma or np.all(np.isnan(want))


def test_a_sweep_divides_predictions_with_fp32_sums():
    from habitat_amd import Device
    from habitat_amd.analysis.predictor import Predictor
    preds = {kind: network(kind, 2) for kind in ("conv2d", "linear")}
    for kind, rp in preds.items():
        _, mu, sigma = synthetic.mlp_features(kind, 2048, seed=1)
        rp.set_normalization(mu, sigma)
        with torch.no_grad():
            rp.model.fc2.bias.fill_(4.0)
        rp.refresh()
    trace = synthetic.resnet50_trace(Device.V100, batch=32, seed=3)
    devices, feats = synthetic.device_sweep(120, seed=3)     # 2783 convolution rows
    features = {d.name: list(f) for d, f in zip(devices, feats)}
    features[Device.V100.name] = [16, 900, 80, 14.028]
    plan = Predictor(mlp_predictors=preds).plan_trace(trace)
    sweep = plan.prepare(devices, features)
    res = sweep.launch()
    for kind, (_, rp, op_feats, ms, op_row) in plan.special.items():
        y = rp.predict_batch_fp32(sweep.rows[kind]).double().view(121, -1)[:, op_row.long()]
        want = torch.clamp(ms * y[:120] / y[120], min=0.0)
        assert torch.equal(res.special_ms[kind], want)


def test_a_trace_divides_predictions_with_fp32_sums():
    """From 65 distinct operations of a kind on (129 rows) hbt_mlp_forward takes the
    pieces; a trace's quotients do not."""
    from habitat_amd import Device
    from habitat_amd.analysis.predictor import Predictor
    rp = network("conv2d", 2)
    _, mu, sigma = synthetic.mlp_features("conv2d", 2048, seed=1)
    rp.set_normalization(mu, sigma)
    with torch.no_grad():
        rp.model.fc2.bias.fill_(4.0)
    rp.refresh()
    predictor = Predictor(mlp_predictors={"conv2d": rp})
    ops = [op for b in (16, 32, 64)
           for op in synthetic.resnet50_trace(Device.V100, batch=b, seed=3).operations
           if op.name == "conv2d"]
    gpu, seen = rp._device_mlp(), []
    forward = gpu.forward
    gpu.forward = lambda raw, **kw: seen.append(raw) or forward(raw, **kw)
    y, pairs = predictor._special_enqueue("conv2d", ops, Device.T4)
    predicted = predictor.predict_operations(ops, Device.T4)
    assert seen[0].shape[0] == 138 and torch.equal(seen[0], seen[1])
    assert torch.equal(y, rp.predict_batch_fp32(seen[0]))
    assert not torch.equal(y, rp.predict_batch(seen[0]))
    pair = y.cpu().numpy().astype(np.float64).reshape(-1, 2)
    for op, i, got in zip(ops, pairs, predicted):
        assert got.run_time_ms == op.run_time_ms * pair[i, 0] / pair[i, 1]
