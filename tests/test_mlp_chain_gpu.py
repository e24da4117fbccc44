"""GPU: a few rows through the whole network in one launch
(habitat_amd/csrc/mlp_chain.h)."""
import ctypes
import os

import numpy as np
import pytest
import torch

from habitat_amd import _lib, synthetic
from habitat_amd.analysis.mlp import mlp as mlp_module
from habitat_amd.analysis.mlp.mlp import RuntimePredictor
from oracle import mlp as omlp

pytestmark = pytest.mark.gpu

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "_build",
                      "libmlp_chain.so")


def network(kind, hidden, seed=0):
    torch.manual_seed(seed)
    rp = RuntimePredictor(kind, hidden, 1024)
    with torch.no_grad():
        for name, p in rp.model.named_parameters():
            if name.endswith("weight") and not name.startswith("fc2"):
                p.mul_(6.0 ** 0.5)
    x, mu, sigma = synthetic.mlp_features(kind, 64, seed=seed)
    rp.set_normalization(mu, sigma)
    return rp, x


# 5 rows and more take a launch per layer, whose sums the one launch repeats: the
# same bits.  Every row count of it, between other counts.
@pytest.mark.parametrize("kind,hidden", [("conv2d", 8), ("lstm", 1), ("bmm", 3), ("linear", 20)])
def test_the_bits_of_the_launches_per_layer(kind, hidden):
    rp, x = network(kind, hidden)
    x[3] = 0.0
    x[5, 1] = np.inf        # NaN and infinities travel as in the per-layer kernels
    x[7, 0] = np.nan
    x[11] *= 1e-3
    want = rp.predict_batch(x[:16]).cpu().numpy()
    exact = omlp.forward_fp64(rp.model.state_dict(), x[:16], rp.mu, rp.sigma)
    ok = np.isfinite(exact)
    # fp32 sums of 1024 products: at most 8 x 2^-24 of the output's size per layer
    size = np.sqrt(np.mean(exact[ok] ** 2))
    assert np.max(np.abs(want[ok] - exact[ok])) <= 6 * (hidden + 1) * 8 * 2.0 ** -24 * size
    for rows in (1, 4, 3, 2, 5, 4, 2, 3, 1):
        for first in (0, 16 - rows):
            got = rp.predict_batch(x[first:first + rows]).cpu().numpy()
            assert np.array_equal(got, want[first:first + rows], equal_nan=True), (rows, first)
    gpu = rp._device_mlp()
    raw = torch.from_numpy(x).cuda()
    for rows in (1, 3):
        out = torch.empty((rows,), dtype=torch.float32, device="cuda")
        assert _lib.lib().hbt_mlp_forward_static(
            gpu.handle, ctypes.c_void_p(raw.data_ptr()), rows, ctypes.c_void_p(out.data_ptr()),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        assert np.array_equal(out.cpu().numpy(), want[:rows], equal_nan=True)
    assert gpu.predict_one(np.ascontiguousarray(x[11])) == want[11]


def test_more_input_features_than_32():
    class Wide(mlp_module._OperationMLP):
        features = ["f%d" % i for i in range(36)]
    torch.manual_seed(3)
    rp = RuntimePredictor("conv2d", 2, 1024)
    rp.model = Wide(2, 1024)
    rp.set_normalization(np.arange(40) / 10.0, np.ones(40))
    x = np.random.default_rng(3).normal(size=(12, 40))
    want = rp.predict_batch(x).cpu().numpy()
    for rows in (1, 2, 4):
        assert np.array_equal(rp.predict_batch(x[:rows]).cpu().numpy(), want[:rows])


def test_two_networks_on_two_streams():
    """Launches that share the GPU: each waits only for its own workgroups."""
    nets = [network("conv2d", 8, seed=s) for s in (1, 2)]
    want = [rp.predict_batch(x[:12]).cpu().numpy() for rp, x in nets]
    raw = [torch.from_numpy(x).cuda() for _, x in nets]
    streams = [torch.cuda.Stream() for _ in nets]
    torch.cuda.synchronize()
    got = []
    for i in range(40):
        for (rp, _), r, s, w in zip(nets, raw, streams, want):
            rows = 1 + i % 5
            with torch.cuda.stream(s):
                got.append((rp.predict_batch(r[:rows]), w[:rows]))
    torch.cuda.synchronize()
    for y, w in got:
        assert np.array_equal(y.cpu().numpy(), w)


def test_replayed_from_a_graph():
    rp, x = network("linear", 8)
    rows = torch.from_numpy(x).cuda()
    raw, out = rows[:3].clone(), torch.zeros((3,), dtype=torch.float32, device="cuda")
    rp.predict_batch(raw, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rp.predict_batch(raw, out=out)
    for i in range(6):
        raw.copy_(rows[3 * i:3 * i + 3])
        graph.replay()
        torch.cuda.synchronize()
        replayed = out.clone()
        assert torch.equal(replayed, rp.predict_batch(rows[3 * i:3 * i + 3]))
        torch.cuda.synchronize()


class Chain:
    """A network of eight features and up to 16 for hbt::chain::launch, with the
    hand-over's counter and words in tensors of the test's."""

    def __init__(self, rp):
        if not os.path.exists(NATIVE):
            pytest.fail("tests/native/_build/libmlp_chain.so is not built: run "
                        "`make -C tests/native` (or __graft_entry__.build()) first")
        lib = ctypes.CDLL(NATIVE)
        P, I, F = ctypes.c_void_p, ctypes.c_int32, ctypes.c_float
        lib.chain_forward.argtypes = [P, I, I, P, P, P, F, P, P, P, I, I, P, P, P, I, P]
        self.lib, self.max_rows = lib, lib.chain_max_rows()
        sd = {k: v.numpy() for k, v in rp.model.state_dict().items()}
        names = ["fc1"] + sorted({k[:-7] for k in sd if k.startswith("mlp") and "weight" in k},
                                 key=lambda k: int(k.split(".")[2]))
        self.hidden = len(names) - 1
        self.blocks = 32 * self.hidden + 1
        fc1 = sd["fc1.weight"]
        self.f = fc1.shape[1]
        assert self.f <= 16
        packed, first_t = [], np.zeros((16, 1024), np.float32)
        first_t[:self.f] = fc1.T
        for name in names:
            w = sd[name + ".weight"]
            w = np.pad(w, ((0, 0), (0, (-w.shape[1]) % 32)))
            # [stream][k-group][n-tile % 8][half][row][4]
            packed.append(w.reshape(4, 8, 32, -1, 2, 4).transpose(0, 3, 1, 4, 2, 5))
        up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
        self.w, self.first_t = up(np.concatenate(packed, axis=1)), up(first_t)
        self.bias = up(np.stack([sd[n + ".bias"] for n in names]))
        self.w_last, self.b_last = up(sd["fc2.weight"].reshape(-1)), float(sd["fc2.bias"][0])
        self.mu, self.sigma = up(rp.mu), up(rp.sigma)
        self.tickets = torch.zeros(1, dtype=torch.int64, device="cuda")
        self.words = torch.zeros((self.hidden, self.max_rows, 1024), dtype=torch.int64,
                                 device="cuda")

    def __call__(self, raw, looks=None):
        looks = self.lib.chain_max_looks() if looks is None else looks
        out = torch.full((raw.shape[0],), -1.0, dtype=torch.float32, device="cuda")
        p = lambda t: ctypes.c_void_p(t.data_ptr())
        rc = self.lib.chain_forward(
            p(self.w), 4, self.hidden, p(self.first_t), p(self.bias), p(self.w_last), self.b_last,
            p(raw), p(self.mu), p(self.sigma), self.f, raw.shape[0], p(out), p(self.tickets),
            p(self.words), looks, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        return out.cpu().numpy()


def test_words_of_older_calls_are_never_taken():
    """A word counts when it carries this call's number: not one that was never
    written, or by a call 2^31 numbers ago, nor where the number's 32 bits turn over."""
    rp, x = network("conv2d", 3)
    want = rp.predict_batch(x[:20]).cpu().numpy()
    chain, raw = Chain(rp), torch.from_numpy(x).cuda()
    assert np.array_equal(chain(raw[:4]), want[:4])
    for before in (2 ** 31 - 2, 2 ** 31 + 5, 2 ** 32 - 3, 3 * 2 ** 31):
        for left in (0, 0x7fc00000, (7 << 32) + 0x3f800000):   # unwritten, NaN, call 7's 1.0
            chain.tickets.fill_(before * chain.blocks)
            chain.words.fill_(left)
            for i, rows in enumerate((4, 1, 1, 3, 1, 2, 4)):
                got = chain(raw[i:i + rows])
                assert np.array_equal(got, want[i:i + rows]), (before, left, i)
                call = (before + i + 1) % 2 ** 32
                numbered = ((chain.words >> 32) & 0xffffffff) == call
                assert bool(torch.all(numbered[:, :rows]))
                if call % 2 ** 16 == 0:    # every so often all rows', so that none gets old
                    assert bool(torch.all(numbered))
                else:
                    assert not bool(torch.any(numbered[:, rows:]))


@pytest.mark.parametrize("kind,hidden", [("conv2d", 1), ("lstm", 4), ("bmm", 8)])
def test_a_wait_that_is_given_up_changes_no_bit(kind, hidden):
    """The bound on a wait at nothing (every workgroup computes its input by itself)
    and at a few looks (some do): the results of calls that wait, NaN handed on."""
    rp, x = network(kind, hidden)
    x[3] = 0.0
    x[5, 1] = np.inf
    x[7, 0] = np.nan
    want = rp.predict_batch(x[:16]).cpu().numpy()
    chain, raw = Chain(rp), torch.from_numpy(x).cuda()
    for looks in (0, 1, 2, 5, 20, 0):
        for rows, first in ((1, 0), (4, 2), (3, 9), (2, 6), (1, 7), (4, 12)):
            got = chain(raw[first:first + rows], looks=looks)
            assert np.array_equal(got, want[first:first + rows], equal_nan=True), (looks, rows)
