"""GPU: the MLP's hidden layers with every fp32 number as a pair of fp16 numbers
(habitat_amd/csrc/mlp_pairs.h): scales, and what has no scale."""
import numpy as np
import pytest
import torch

from habitat_amd import synthetic
from habitat_amd.analysis.mlp.mlp import RuntimePredictor
from tests.test_mlp_split_gpu import forward_fp64, network

pytestmark = pytest.mark.gpu

# 1 x 1 tiles in one round and in several, 1 x 2 in one and two, 1 x 3 in one and two, 2 x 4,
# a second chunk; whole and partial last blocks of each
ROWS = [1025, 1500, 2048, 4097, 4600, 9217, 10240, 2049, 3071, 4096, 4609, 5911, 6144, 6145, 8192, 8193, 10241, 12288, 12289, 13001, 16384,
        16384 + 2100]


def scaled(rp, units, rows):
    """The same network with everything 2^rows as large, the prediction too, and unit n of
    every layer 2^units[n] as large, which the next layer's weights undo."""
    sd = {k: v.clone() for k, v in rp.model.state_dict().items()}
    out = RuntimePredictor(rp.model_name, rp.layers, 1024)
    layers = ["fc1"] + ["mlp.layers.%d" % (2 * i) for i in range(rp.layers)] + ["fc2"]
    by = torch.ldexp(torch.ones(1024), units)
    for i, name in enumerate(layers):
        w, b = sd[name + ".weight"], sd[name + ".bias"]
        if i > 0:
            w /= by
        else:
            w *= 2.0 ** rows
        if i < len(layers) - 1:
            w *= by[:, None]
            b *= by * 2.0 ** rows
        else:
            b *= 2.0 ** rows
    out.model.load_state_dict(sd)
    out.set_normalization(rp.mu, rp.sigma)
    return out


@pytest.mark.parametrize("rows", ROWS)
def test_powers_of_two_change_no_bit(rows):
    rp = network("lstm", 3)
    x, mu, sigma = synthetic.mlp_features("lstm", rows, seed=rows)
    rp.set_normalization(mu, sigma)
    want = rp.predict_batch(x)
    units = torch.from_numpy(np.random.default_rng(rows).integers(-5, 5, 1024)).to(torch.int32)
    assert torch.equal(scaled(rp, units, 0).predict_batch(x), want)
    for size in (40, -40):
        assert torch.equal(scaled(rp, units, size).predict_batch(x), want * 2.0 ** size)


@pytest.mark.parametrize("rows", ROWS)
def test_rows_of_all_sizes_in_one_batch(rows):
    """Without biases a row 2^k as large gives 2^k the prediction, bit for bit, beside
    rows of any other size: every row has a scale of its own."""
    rp = network("bmm", 2)
    with torch.no_grad():
        for name, p in rp.model.named_parameters():
            if name.endswith("bias"):
                p.zero_()
    rp.set_normalization(np.zeros(8), np.ones(8))
    rng = np.random.default_rng(rows)
    x = rng.normal(size=(rows, 8)).astype(np.float32).astype(np.float64)
    size = rng.integers(-60, 60, rows)
    y = rp.predict_batch(x).cpu().numpy()
    assert np.array_equal(rp.predict_batch(np.ldexp(x, size[:, None])).cpu().numpy(), np.ldexp(y, size))
    want = forward_fp64(rp, x)
    # 8 x 2^-24 of the output's rms for each layer's sum (tests/test_mlp_split_gpu.py)
    assert np.sqrt(np.mean((y - want) ** 2)) <= \
        3 * 8 * 2.0 ** -24 * np.sqrt(np.mean(want ** 2))


@pytest.mark.parametrize("rows", ROWS)
def test_whole_numbers_are_exact(rows):
    """Weights of 11 bits in the first hidden layer and activations of up to 23 in the
    second, with sums below 2^24 in any order: every number is held and every position wired."""
    rng = np.random.default_rng(rows)
    rp = RuntimePredictor("bmm", 2, 1024)
    last = np.zeros(1024)
    last[rng.choice(1024, 16, replace=False)] = rng.choice([-1, 1], 16)
    with torch.no_grad():
        for p in rp.model.parameters():
            p.zero_()
        rp.model.fc1.weight.copy_(torch.from_numpy(rng.choice([-1, 1], (1024, 8))))
        rp.model.mlp.layers[0].weight.copy_(torch.from_numpy(
            rng.integers(1, 256, (1024, 1024)) * rng.choice([-1, 1], (1024, 1024)) / 4))
        rp.model.mlp.layers[2].weight.copy_(torch.from_numpy(rng.choice([-1, 1], (1024, 1024))))
        rp.model.mlp.layers[0].bias.copy_(torch.from_numpy(rng.integers(-2048, 2048, 1024)))
        rp.model.fc2.weight.copy_(torch.from_numpy(last)[None])
    rp.set_normalization(np.zeros(8), np.ones(8))
    x = rng.integers(-1, 2, (rows, 8)).astype(np.float64)
    assert np.array_equal(rp.predict_batch(x).double().cpu().numpy(), forward_fp64(rp, x))


@pytest.mark.parametrize("rows", [1500, 2100, 4500, 5000, 10000, 13000])
def test_infinities_and_nan_among_finite_rows(rows):
    """Where fp32 gives an infinity, zero or NaN for a row, and nothing in the rows beside it."""
    rp = network("conv2d", 3)
    x, mu, sigma = synthetic.mlp_features("conv2d", rows, seed=3)
    rp.set_normalization(mu, sigma)
    plain = rp.predict_batch(x).cpu().numpy()
    rng, x = np.random.default_rng(rows), x.copy()
    at = rng.choice(rows, rows // 10, replace=False)
    x[at, rng.integers(0, x.shape[1], at.size)] = np.resize(
        [np.nan, np.inf, -np.inf, 1e300, -1e300], at.size)
    got, want = rp.predict_batch(x).cpu().numpy(), rp.predict_batch_fp32(x).cpu().numpy()
    for of in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(of(got), of(want))
    others = np.setdiff1d(np.arange(rows), at)
    assert np.array_equal(got[others], plain[others])


def test_units_on_few_inputs_are_not_for_pairs():
    """A unit of which one input makes nearly all: what the pairs would lose of the others
    shows where that one is off.  The bf16 pieces take the network then, and give the same
    for its rows whether others with that input on are beside them."""
    rp = network("linear", 1)
    with torch.no_grad():
        for p in rp.model.parameters():
            p.zero_() if p.dim() == 1 else p.abs_()
        rp.model.fc1.weight[:, 0] = 0.0
        rp.model.fc1.weight[7] = 0.0
        rp.model.fc1.weight[7, 0] = 1.0            # unit 7 is feature 0 alone
        hidden = rp.model.mlp.layers[0].weight
        hidden.mul_(2.0 ** -24)
        hidden[:, 7] = 1.0
    rp.set_normalization(np.zeros(8), np.ones(8))
    x = np.abs(np.random.default_rng(1).normal(size=(6000, 8)))
    x[:, 0] = 0.0
    want = forward_fp64(rp, x)
    y = rp.predict_batch(x).double().cpu().numpy()
    assert np.max(np.abs(y / want - 1)) <= 6 * 2 * 8 * 2.0 ** -24


@pytest.mark.parametrize("features", [1, 16, 17, 60])
@pytest.mark.parametrize("rows", [1500, 3000, 5000, 13000])
def test_any_number_of_features(rows, features):
    """fc1 of 5 to 64 inputs: its two kernels, and the bound on what it makes of them."""
    from habitat_amd.analysis.mlp.mlp import _OperationMLP, _DeviceMLP

    class Network(_OperationMLP):
        features = ["f%d" % i for i in range(60)]

    Network.features = Network.features[:features]
    torch.manual_seed(features)
    model = Network(2, 1024)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("weight") and not name.startswith("fc2"):
                p.mul_(6.0 ** 0.5)
    x = np.random.default_rng(rows).normal(size=(rows, features + 4))
    x[::7] *= 2.0 ** 30
    handle = _DeviceMLP(model, np.zeros(features + 4), np.ones(features + 4))
    y = handle.forward(torch.from_numpy(x).cuda()).double().cpu().numpy()
    rp = RuntimePredictor("bmm", 2, 1024)
    rp.model, rp.mu, rp.sigma = model, np.zeros(features + 4), np.ones(features + 4)
    want = forward_fp64(rp, x)
    for part in (slice(0, None, 7), np.arange(rows) % 7 != 0):
        # the bound of tests/test_mlp_split_gpu.py, for rows of each size
        assert np.sqrt(np.mean((y[part] - want[part]) ** 2)) <= \
            3 * 8 * 2.0 ** -24 * np.sqrt(np.mean(want[part] ** 2))


@pytest.mark.parametrize("rows", [1500, 5911, 16384 + 3000])
def test_replays_of_a_captured_forward(rows):
    rp = network("linear", 3)
    x, mu, sigma = synthetic.mlp_features("linear", rows, seed=4)
    rp.set_normalization(mu, sigma)
    raw, out = torch.from_numpy(x).cuda(), torch.empty(rows, device="cuda")
    want = rp.predict_batch(raw).clone()
    other = rp.predict_batch(raw * 1.5).clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rp.predict_batch(raw, out=out)
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(rp.predict_batch(raw * 1.5), other)   # eager work between the replays


def layers_of(rp):
    """(weight, bias) of fc1 and the hidden layers."""
    names = ["fc1"] + ["mlp.layers.%d" % (2 * i) for i in range(rp.layers)]
    params = dict(rp.model.named_parameters())
    return [(params[n + ".weight"], params[n + ".bias"]) for n in names]


@pytest.mark.parametrize("rows", [1024, 1025, 3000, 5911, 13000])
@pytest.mark.parametrize("exponents", [(40, 40), (60, 60), (76, 80), (100, 100), (120, 120)])
def test_collapsed_layers(rows, exponents):
    """Two layers that make next to nothing of their inputs, one after the other: the
    prediction is what the biases after them make, at any number of rows."""
    rp = network("lstm", 4)
    with torch.no_grad():
        for (weight, bias), e in zip(layers_of(rp)[1:], exponents + (0, 0)):
            weight.mul_(2.0 ** -e)
            bias.zero_()
        layers_of(rp)[0][1].zero_()
        rp.model.fc2.bias.fill_(4.0)
    x, mu, sigma = synthetic.mlp_features("lstm", rows, seed=rows)
    rp.set_normalization(mu, sigma)
    assert np.allclose(rp.predict_batch(x).double().cpu().numpy(), forward_fp64(rp, x), rtol=2.0 ** -22)


@pytest.mark.parametrize("rows", [1500, 3000, 5911, 13000])
@pytest.mark.parametrize("size", [0, -20, -30, -40])
def test_units_of_zeros_beside_small_ones(rows, size):
    """Units without weights or bias, as pruning leaves them, beside units of any size: their
    outgoing weights, which meet nothing but zeros, take no bits of the others'."""
    rp = network("lstm", 3)
    with torch.no_grad():
        for weight, bias in layers_of(rp):
            bias.mul_(2.0 ** size)
        layers_of(rp)[0][0].mul_(2.0 ** size)
        for (weight, bias), unit in zip(layers_of(rp)[:2], (3, 700)):
            weight[unit], bias[unit] = 0.0, 0.0
        rp.model.fc2.bias.zero_()
    x, mu, sigma = synthetic.mlp_features("lstm", rows, seed=rows)
    rp.set_normalization(mu, sigma)
    y, want = rp.predict_batch(x).double().cpu().numpy(), forward_fp64(rp, x)
    rms = np.sqrt(np.mean((want - want.mean()) ** 2)) + abs(want.mean())
    # the bound of tests/test_mlp_split_gpu.py
    assert np.sqrt(np.mean((y - want) ** 2)) <= 4 * 8 * 2.0 ** -24 * rms
    x[::5, 2] = np.nan                        # a unit of zeros hands a NaN on
    x[1::5, 3] = np.inf
    got, fp32 = rp.predict_batch(x).cpu().numpy(), rp.predict_batch_fp32(x).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(fp32)) and np.isnan(got).sum() >= 2 * (rows // 5)


@pytest.mark.parametrize("signs", ["either", "positive"])
@pytest.mark.parametrize("rows", [1025, 1500, 2048, 2500, 4500, 5911, 10000, 13000])
def test_sums_beyond_fp32_are_infinite(rows, signs):
    """A hidden layer's output of 2^128 and more is an infinity, at any number of rows, and
    does not come back as a number where the next layer's weights are small."""
    rp = network("bmm", 3)
    with torch.no_grad():
        for (weight, bias), e in zip(layers_of(rp), (0, 6, 6, -40)):
            if signs == "positive":
                weight.abs_()
            weight.mul_(2.0 ** e)
        if signs == "positive":
            rp.model.fc2.weight.abs_()
    rp.set_normalization(np.zeros(8), np.ones(8))
    x = np.abs(np.random.default_rng(rows).normal(size=(rows, 8))) + 0.1
    plain = rp.predict_batch(x).cpu().numpy()
    x[::7] *= 2.0 ** (110 if signs == "positive" else 118)
    h = torch.from_numpy(x[::7]).cuda()
    with torch.no_grad():
        for weight, bias in layers_of(rp)[:3]:
            h = torch.relu(h @ weight.double().cuda().t() + bias.double().cuda())
    assert bool(((h > 2.0 ** 129).sum(1) > 100).all())      # far beyond, in every such row
    got = rp.predict_batch(x).cpu().numpy()
    assert np.all(np.isposinf(got[::7]) if signs == "positive" else np.isnan(got[::7]))
    others = np.arange(rows) % 7 != 0
    assert np.array_equal(got[others], plain[others])


@pytest.mark.parametrize("rows", [1025, 2048, 3000, 4500, 5911, 10000, 13001, 16384 + 3001])
def test_rows_that_some_units_dominate(rows):
    """Two networks of 512 units side by side, of which fc2 reads the second and feature 0
    feeds the first: where that one is large, what the second makes is held as fp32 holds it,
    and the rows beside such a row are left alone."""
    rp = network("conv2d", 3)
    inputs = rp.model.fc1.weight.shape[1]
    with torch.no_grad():
        for weight, bias in layers_of(rp):
            bias.zero_()
            if weight.shape[1] == 1024:
                weight[:512, 512:] = 0.0
                weight[512:, :512] = 0.0
                weight.mul_(2.0 ** 0.5)
            else:
                weight[:512, 1:] = 0.0
                weight[512:, 0] = 0.0
        rp.model.fc2.weight[0, :512] = 0.0
        rp.model.fc2.bias.zero_()
    rp.set_normalization(np.zeros(inputs), np.ones(inputs))
    rng = np.random.default_rng(rows)
    x = rng.normal(size=(rows, inputs))
    plain = rp.predict_batch(x).cpu().numpy()
    want = forward_fp64(rp, x)                              # (feature 0 is no part of it)
    rms = np.sqrt(np.mean(want ** 2))
    at = np.sort(rng.choice(rows, rows // 40, replace=False))
    others = np.setdiff1d(np.arange(rows), at)
    for k in (4, 8, 10, 12, 16, 20, 32):
        x[at, 0] = 2.0 ** k
        y = rp.predict_batch(x).cpu().numpy()
        # the bound of tests/test_mlp_split_gpu.py
        assert np.sqrt(np.mean((y[at] - want[at]) ** 2)) <= 4 * 8 * 2.0 ** -24 * rms, k
        assert np.array_equal(y[others], plain[others]), k
        if k >= 12:   # (whole rounds of the fused fp32 kernel)
            whole = np.resize(x[at], (8192, inputs))
            assert np.array_equal(y[at], rp.predict_batch_fp32(whole).cpu().numpy()[:at.size])
    graph, out = torch.cuda.CUDAGraph(), torch.empty(rows, device="cuda")
    raw = torch.from_numpy(x).cuda()
    with torch.cuda.graph(graph):
        rp.predict_batch(raw, out=out)
    raw[:, 0] = 0.5                          # what was marked in one pass is not in the next
    want = rp.predict_batch(raw).cpu().numpy()
    assert not np.array_equal(want[at], y[at])
    for _ in range(2):
        out.zero_()
        graph.replay()
        assert np.array_equal(out.cpu().numpy(), want)
        assert np.array_equal(rp.predict_batch(x).cpu().numpy(), y)


@pytest.mark.parametrize("rows", [1500, 3000, 4500, 5911, 13000])
def test_rows_in_which_few_units_are_on(rows):
    """Features that switch all but twenty units off, whatever they would have made of them,
    and the others' activations far below what the features bound them by."""
    rp = network("linear", 2)
    with torch.no_grad():
        for _, bias in layers_of(rp):
            bias.zero_()
        rp.model.fc2.bias.zero_()
        first = rp.model.fc1.weight
        first.copy_(-first.abs())
        first[:, 0] = 0.0
        first[300:320] = 0.0
        first[300:320, 0] = torch.rand(20) + 0.5
    rp.set_normalization(np.zeros(8), np.ones(8))
    x = np.abs(np.random.default_rng(rows).normal(size=(rows, 8))) + 0.1
    x[::3, 1:] *= 2.0 ** 30
    y, want = rp.predict_batch(x).double().cpu().numpy(), forward_fp64(rp, x)
    # All rows are multiples of one, so one sum's chance is all rows'; the bound of
    # tests/test_mlp_split_gpu.py on the last sum's terms (sums of 20 products have less)
    h = torch.from_numpy(x).cuda()
    with torch.no_grad():
        for weight, _ in layers_of(rp):
            h = torch.relu(h @ weight.double().cuda().t())
        size = (h * rp.model.fc2.weight.double().cuda()).norm(dim=1).cpu().numpy()
    for part in (slice(0, None, 3), slice(1, None, 3)):
        assert np.max(np.abs(y[part] - want[part]) / size[part]) <= 6 * 3 * 8 * 2.0 ** -24


@pytest.mark.parametrize("rows", [1500, 3000, 4500, 5911, 13000])
def test_an_input_of_tiny_weights_alone(rows):
    """A unit whose outgoing weights are 2^-60 of the others', large, and alone in being on:
    its weights are not for pairs, and the network is not."""
    rp = network("linear", 2)
    with torch.no_grad():
        for _, bias in layers_of(rp):
            bias.zero_()
        rp.model.fc2.bias.zero_()
        first = rp.model.fc1.weight
        first.copy_(-first.abs())
        first[:, 0] = 0.0
        first[40] = 0.0
        first[40, 0] = 1.0
        layers_of(rp)[1][0][:, 40] *= 2.0 ** -60
    rp.set_normalization(np.zeros(8), np.ones(8))
    x = np.abs(np.random.default_rng(rows).normal(size=(rows, 8))) + 0.1
    x[:, 0] *= 2.0 ** 32
    y, want = rp.predict_batch(x).double().cpu().numpy(), forward_fp64(rp, x)
    h = torch.from_numpy(x).cuda()
    with torch.no_grad():
        for weight, _ in layers_of(rp):
            h = torch.relu(h @ weight.double().cuda().t())
        size = (h * rp.model.fc2.weight.double().cuda()).norm(dim=1).cpu().numpy()
    # as above
    assert np.max(np.abs(y - want) / size) <= 6 * 3 * 8 * 2.0 ** -24


@pytest.mark.parametrize("rows", [1500, 3000, 5911, 13000])
def test_small_weights_that_are_all_that_counts(rows):
    """Half of the inputs with ordinary weights, the other half with 2^-24 of them, and rows
    in which the first half is off."""
    rp = network("linear", 2)
    with torch.no_grad():
        for _, bias in layers_of(rp):
            bias.zero_()
        rp.model.fc2.bias.zero_()
        rp.model.fc1.weight.abs_()
        rp.model.fc1.weight[::2, 0] = 0.0
        rp.model.fc1.weight[1::2, 1:] = 0.0               # every second unit is feature 0 alone
        layers_of(rp)[1][0][:, ::2] *= 2.0 ** -24
    rp.set_normalization(np.zeros(8), np.ones(8))
    x = np.abs(np.random.default_rng(rows).normal(size=(rows, 8)))
    x[::2, 0] = 0.0
    y, want = rp.predict_batch(x).double().cpu().numpy(), forward_fp64(rp, x)
    h = torch.from_numpy(x).cuda()
    with torch.no_grad():
        for weight, _ in layers_of(rp):
            h = torch.relu(h @ weight.double().cuda().t())
        size = (h * rp.model.fc2.weight.double().cuda()).norm(dim=1).cpu().numpy()
    for part in (slice(0, None, 2), slice(1, None, 2)):
        # The bound of tests/test_mlp_split_gpu.py, for either kind of row.  All activations of
        # a second row are multiples of one feature, so that what the last sum cancels to is
        # the same part of it in all of them: its terms' root sum of squares stands for it.
        assert np.sqrt(np.mean((y[part] - want[part]) ** 2)) <= \
            3 * 8 * 2.0 ** -24 * np.sqrt(np.mean(size[part] ** 2))
