"""GPU router front end and the graph-captured layer stack against the oracle.

Routing parity: the GPU's logits match float64 x . W_r to 1e-5 relative; top-k
ids are bit-exact and weights match to 1e-6 when the oracle routes the GPU's
own logits (the selection is then decided by the same values); the drop rules
follow oracle/routing.py.  Stack parity: every layer's expert-FFN output
against the oracle on that layer's GPU input (rel-L2 <= 2e-3), and graph
replays equal the eager run bit for bit.
"""

import numpy as np
import pytest

from oracle import latent_ref as ref
from oracle import routing, synth
from tests._layers import to_device

pytestmark = pytest.mark.gpu

TOL = 2e-3


def _cuda(a, dtype=None):
    import torch

    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    return t if dtype is None else t.to(dtype)


@pytest.mark.parametrize("T,d,E,k,x_dtype,r_dtype", [
    (1, 7168, 256, 8, "bf16", "f32"),
    (32, 7168, 256, 8, "bf16", "f32"),
    (37, 300, 64, 6, "f32", "bf16"),
    (5, 1000, 1024, 64, "f16", "f32"),
])
def test_route_from_x_matches_oracle(gpu, T, d, E, k, x_dtype, r_dtype):
    import torch

    tdt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    rng = np.random.default_rng(T * 1000 + E)
    x = _cuda(rng.standard_normal((T, d)).astype(np.float32), tdt[x_dtype])
    W = _cuda((rng.standard_normal((d, E)) / np.sqrt(d)).astype(np.float32), tdt[r_dtype])
    logits = torch.empty((T, E), dtype=torch.float32, device="cuda")
    ids, w = gpu.route(k, x=x, router=W, logits_out=logits)
    torch.cuda.synchronize()
    want_lg = routing.router_logits(x.float().cpu().numpy(), W.float().cpu().numpy())
    got_lg = logits.cpu().numpy()
    assert np.abs(got_lg - want_lg).max() <= 1e-5 * max(1.0, np.abs(want_lg).max())
    want_ids, want_w = routing.softmax_topk(got_lg, k)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    np.testing.assert_allclose(w.cpu().numpy(), want_w, rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("T,d,E,k,x_dtype,r_dtype,shift", [
    (220, 7168, 256, 8, "bf16", "f32", 0),    # 128-token tiles, last one ragged
    (137, 7168, 256, 8, "bf16", "f32", 0),    # the fewest tokens of this shape it takes
    (2049, 7168, 256, 8, "f16", "f32", 0),    # 256-token tiles, one token over
    (1500, 2080, 130, 6, "f32", "f32", 0),    # two experts in the last tile, 65 steps of 32 rows
    (4096, 2048, 64, 6, "bf16", "bf16", 0),
    (300, 1408, 1000, 64, "bf16", "f32", 0),  # 16 experts a lane in the selection
    (1300, 1280, 257, 8, "f16", "bf16", 1),   # x rows not 16-byte aligned
    (12600, 32, 1000, 1, "f32", "bf16", 1),   # a slice is one step
])
def test_route_long_batches_against_float64(gpu, T, d, E, k, x_dtype, r_dtype, shift):
    """The split-operand logits: fp32 sums of exact bf16 products, so the error
    of a logit stays a few 2^-24 of sum |x w| (|x| |w| sqrt(d) here), and the
    selection is the oracle's on the same logits."""
    import torch

    tdt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    x = torch.randn(T * d + shift, generator=gen, device="cuda").to(tdt[x_dtype])[shift:].view(T, d)
    W = (torch.randn((d, E), generator=gen, device="cuda") / d ** 0.5).to(tdt[r_dtype])
    logits = torch.empty((T, E), dtype=torch.float32, device="cuda")
    ids, w = gpu.route(k, x=x, router=W, logits_out=logits)
    want = x.double() @ W.double()
    scale = x.double().abs() @ W.double().abs()
    assert float(((logits.double() - want).abs() / scale).max()) <= 8 * 2.0 ** -24
    assert float((logits.double() - want).norm() / want.norm()) <= 3e-7
    want_ids, want_w = routing.softmax_topk(logits.cpu().numpy(), k)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    np.testing.assert_allclose(w.cpu().numpy(), want_w, rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("x_dtype", ["f32", "f16"])
@pytest.mark.parametrize("lo,hi", [(2 ** -7 - 2 ** -12, 2 ** -7), (2 ** -8 - 2 ** -12, 2 ** -8), (0.0, 2 ** -7), (-1.0, 0.0)])
def test_route_long_batches_have_no_bias_on_positive_data(gpu, x_dtype, lo, hi):
    """Positive operands 1 + u, u in [lo, hi): what the split leaves out of a
    product has either sign, so the mean error over all logits is far below one
    rounding (2^-24); parts cut off instead of rounded had 2^-22 of it."""
    import torch

    T, d, E = 1536, 2048, 128
    gen = torch.Generator(device="cuda").manual_seed(5)

    def draw(*shape):
        return 1 + lo + (hi - lo) * torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64)

    x = draw(T, d).to({"f32": torch.float32, "f16": torch.float16}[x_dtype])
    W = draw(d, E).float()
    logits = torch.empty((T, E), dtype=torch.float32, device="cuda")
    gpu.route(6, x=x, router=W, logits_out=logits)
    want = x.double() @ W.double()
    err = (logits.double() - want) / want
    # f16 values in [1 + 2^-7 - 2^-12, 1 + 2^-7) are one or two numbers: their
    # sums repeat, and so does the sums' own rounding.
    assert float(err.mean().abs()) <= 2.0 ** -26
    assert float(err.abs().max()) <= 8 * 2.0 ** -24


def test_route_in_the_documented_workspace(gpu):
    """A workspace of T E 4 ceil(d / 64) bytes holds a long batch of a small d
    (its query once asked for more)."""
    import torch

    T, d, E = 3052, 1024, 128
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn((T, d), generator=gen, device="cuda")
    W = torch.randn((d, E), generator=gen, device="cuda") / d ** 0.5
    logits = torch.empty((T, E), dtype=torch.float32, device="cuda")
    ws = torch.empty(T * E * 4 * -(-d // 64), dtype=torch.uint8, device="cuda")
    gpu.route(6, x=x, router=W, logits_out=logits, workspace=ws)
    want = x.double() @ W.double()
    assert float((logits.double() - want).norm() / want.norm()) <= 3e-7


def test_route_long_batches_non_finite(gpu):
    """A non-finite operand spoils its own tokens or experts only, as a plain
    fp32 sum has it: inf stays inf, inf - inf and NaN are NaN and never chosen."""
    import torch

    T, d, E, k = 230, 7168, 256, 8
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((T, d), generator=gen, device="cuda")
    W = torch.randn((d, E), generator=gen, device="cuda") / d ** 0.5
    W[:, 17] = W[:, 17].abs()
    x[5, 100] = float("inf")
    x[7, 3] = float("nan")
    W[9, 40] = float("-inf")
    logits = torch.empty((T, E), dtype=torch.float32, device="cuda")
    ids, _ = gpu.route(k, x=x, router=W, logits_out=logits)
    want = x.double() @ W.double()
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(logits), nan) and float(logits[5, 17]) == float("inf")
    fin = torch.isfinite(want)
    assert torch.equal(torch.isfinite(logits), fin)
    assert float((logits.double() - want)[fin].abs().max()) <= 1e-5
    got = ids.cpu().numpy()
    chosen = torch.gather(nan, 1, ids.long().clamp(min=0)).cpu().numpy()
    rows = nan.sum(1).cpu().numpy() < E - k
    assert not chosen[rows].any() and (got[rows] >= 0).all()


@pytest.mark.parametrize("T,d,E,k,x_dtype,r_dtype", [
    (1534, 2080, 130, 6, "f32", "f32"),    # two tokens in the last workgroup, d ends in half a slice
    (301, 1408, 1000, 9, "bf16", "bf16"),  # 16 experts a lane
    (2049, 3072, 64, 6, "f16", "f32"),
])
def test_route_long_batches_recompute(gpu, T, d, E, k, x_dtype, r_dtype):
    """Logits without bf16 parts come from the fp32 sum: tokens of inf and NaN
    beside finite ones, a router value that rounds to infinity in bf16 (finite
    logits), one that is infinite."""
    import torch

    tdt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    gen = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((T, d), generator=gen, device="cuda").to(tdt[x_dtype])
    W = (torch.randn((d, E), generator=gen, device="cuda") / d ** 0.5).to(tdt[r_dtype])
    x[2, 5] = float("nan")
    x[3, d - 1] = float("inf")
    x[T - 1, 0] = float("-inf")
    W[d - 1, E - 1] = torch.finfo(W.dtype).max
    x[:, d - 1] = x[:, d - 1].clamp(-0.5, 0.5)
    x[3, d - 1] = float("inf")
    W[7, 3] = float("inf")
    logits = torch.empty((T, E), dtype=torch.float32, device="cuda")
    ids, _ = gpu.route(k, x=x, router=W, logits_out=logits)
    want = x.double() @ W.double()
    assert torch.equal(torch.isnan(logits), torch.isnan(want))
    assert torch.equal(torch.isinf(logits), torch.isinf(want))
    inf = torch.isinf(want)
    assert torch.equal(logits[inf].double(), want[inf])
    fin = torch.isfinite(want)
    scale = x.double().abs() @ W.double().abs()
    assert float(((logits.double() - want).abs() / scale)[fin].max()) <= 8 * 2.0 ** -24
    rows = torch.isnan(want).sum(1) < E - k
    assert not torch.gather(torch.isnan(want), 1, ids.long().clamp(min=0))[rows].any()


def test_route_of_nan_tokens_stays_bounded(gpu):
    """A batch with a NaN in every token takes some 8 times a finite one's time
    (140 times when a lane summed a token alone)."""
    import torch

    T, d, E = 4096, 7168, 256
    gen = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn((T, d), generator=gen, device="cuda").bfloat16()
    r = gpu.Router(torch.randn((d, E), generator=gen, device="cuda") / d ** 0.5, 8)

    def best(x):
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                r(x)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    finite = best(x)
    x[:, -1] = float("nan")
    assert best(x) < 30 * finite


@pytest.mark.parametrize("drop,param", [("none", 0.0), ("below", 0.05), ("below", 0.2), ("inclusive", 0.95),
                                        ("inclusive", 0.5)])
def test_route_from_logits_drop_rules(gpu, drop, param):
    rng = np.random.default_rng(11)
    lg = routing.zipf_logits(rng, 257, 256, gamma=0.11)
    ids, w = gpu.route(8, logits=_cuda(lg), drop=drop, drop_param=param)
    want_ids, want_w = routing.route(lg, 8, drop, param)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    np.testing.assert_allclose(w.cpu().numpy(), want_w, rtol=2e-6, atol=1e-7)


def test_route_ties_go_to_lower_expert(gpu):
    lg = np.zeros((4, 200), np.float32)
    lg[0, [5, 150, 7]] = 1.0          # equal maxima: 5, 7, 150 then zeros from id 0
    lg[1, :] = -np.inf                 # all -inf: lowest ids first
    lg[2, 199] = np.nan                # NaN never wins
    lg[3, :] = -1.0
    lg[3, [64, 3]] = -0.0              # -0 and +0 are equal: lower id first
    lg[3, [130, 9]] = 0.0
    ids, w = gpu.route(4, logits=_cuda(lg))
    got = ids.cpu().numpy()
    assert got[0].tolist() == [5, 7, 150, 0]
    assert got[1].tolist() == [0, 1, 2, 3]
    assert 199 not in got[2].tolist()
    assert got[3].tolist() == [3, 9, 64, 130]


def test_route_rejects_bad_arguments(gpu):
    import torch

    from latent_amd import LatentError

    lg = torch.zeros((2, 8), dtype=torch.float32, device="cuda")
    with pytest.raises(LatentError):
        gpu.route(9, logits=lg)  # k > E
    with pytest.raises(LatentError):
        gpu.route(2, logits=lg, drop="inclusive", drop_param=0.0)
    with pytest.raises(ValueError):
        gpu.route(2, logits=lg, drop="nope")


@pytest.mark.parametrize("T", [2, 8])
def test_graph_stack_matches_eager_and_oracle(gpu, T):
    """Three small layers (8 routed pairs: multi-kernel path; 32: fp32 chain)."""
    import torch

    E, d, ff, R, k, n_layers = 16, 256, 256, 64, 4, 3
    hosts = [synth.make_layer(seed=40 + l, n_expert=E, d=d, ff=ff, max_rank=R) for l in range(n_layers)]
    layers = [to_device(h) for h in hosts]
    rng = np.random.default_rng(5)
    routers = [gpu.Router(_cuda((rng.standard_normal((d, E)) / np.sqrt(d)).astype(np.float32)), k)
               for _ in range(n_layers)]
    stack = gpu.DecodeStack(layers, routers, T)
    x0 = _cuda(rng.standard_normal((T, d)).astype(np.float32))
    eager = stack.forward(x0).clone()
    xs = [t.clone() for t in stack.x]
    ys = [t.clone() for t in stack.y]
    lgs = [t.clone() for t in stack.logits]
    ids_l = [t.clone() for t in stack.ids]
    torch.cuda.synchronize()
    # Per layer: routing and expert FFN against the oracle on the GPU's layer input.
    for l in range(n_layers):
        x_l = xs[l].cpu().numpy()
        lg = lgs[l].cpu().numpy()
        want_lg = routing.router_logits(x_l, routers[l].weight.cpu().numpy())
        assert np.abs(lg - want_lg).max() <= 1e-5 * max(1.0, np.abs(want_lg).max())
        want_ids, want_w = routing.softmax_topk(lg, k)
        assert np.array_equal(ids_l[l].cpu().numpy(), want_ids)
        want_y = ref.moe_forward(x_l, want_ids, want_w, hosts[l])
        err = ref.rel_l2(want_y, ys[l].cpu().numpy())
        print(f"T={T} layer {l}: rel_l2={err:.3e}")
        assert err <= TOL
        np.testing.assert_array_equal(xs[l + 1].cpu().numpy(), x_l + ys[l].cpu().numpy())
    # Graph replays, with eager work and synchronisations between them.
    # The fp32 chain (>= 32 pairs) sums in a fixed order; the multi-kernel
    # path adds workgroup partials with float atomics (order not fixed).
    exact = gpu.moe_path(layers[0], x0, k) == "fused"
    assert exact == (T * k >= 32)
    stack.capture()
    for rep in range(3):
        stack.load(x0)
        out = stack.replay()
        torch.cuda.synchronize()
        _same(out, eager, exact, f"replay {rep}")
        stack.forward(x0)  # eager run between replays
        torch.cuda.synchronize()
        _same(stack.output, eager, exact, f"eager run after replay {rep}")


def _same(got, want, exact, what):
    import torch

    if exact:
        assert torch.equal(got, want), f"{what} differs from the first eager run"
    else:
        err = ref.rel_l2(want.cpu().numpy(), got.cpu().numpy())
        assert err <= 1e-6, f"{what}: rel_l2 {err:.3e} against the first eager run"
