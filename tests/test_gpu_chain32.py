"""The fp32 matrix-core chain over the row layout (chain32.hip, path "fused").

Sizes at the edges of its split: 32 and 512 routed pairs, experts of 16, 17
and many pairs (several units), ranks 32 to 512 (64-, 128-, 256- and twice
256-column tiles, true ranks below them and ranks that are no multiple of 32),
ff and d that end inside a 256- and a 512-column item, INT8 groups, every x
type, both output modes, weighting before down, dropped and out-of-range ids.

Bar: rel-L2 1e-5 against the oracle: both sum in fp32, and a sum of K terms
rounds to about sqrt(K) 2^-24 (5e-6 at 7168, the deepest here 2e-6), four of
them in a chain.  Sums run in a fixed order, so two calls agree bit for bit.
"""

import numpy as np
import pytest

from oracle import latent_ref as ref
from oracle import routing, synth
from tests.test_gpu_rows import _rows_layer

pytestmark = pytest.mark.gpu

TOL = 1e-5

LAYERS = {
    "r32": dict(seed=81, n_expert=40, d=544, ff=288, max_rank=32),
    "r128": dict(seed=82, n_expert=6, d=1056, ff=1408, max_rank=128),
    "r192": dict(seed=83, n_expert=9, d=512, ff=256, max_rank=192, ranks=[192, 64, 1, 100, 33, 191, 129, 160, 0]),
    "r512": dict(seed=84, n_expert=5, d=768, ff=544, max_rank=512, ranks=[512, 64, 257, 300, 128]),
    "int8": dict(seed=85, n_expert=7, d=1088, ff=320, max_rank=256, ranks=[256, 64, 100, 200, 32, 128, 250],
                 int8_fraction=0.2),
}


@pytest.fixture(scope="module", params=sorted(LAYERS))
def layers(request, gpu):
    spec = dict(LAYERS[request.param])
    host = synth.make_layer(**spec)
    return host, _rows_layer(host)


@pytest.mark.parametrize("T,k,x_dtype,mode,wbd", [
    (8, 4, "bf16", 0, False), (32, 1, "f16", 1, True), (17, 3, "f32", 0, True), (128, 4, "bf16", 1, False),
    (512, 1, "f32", 0, False),
])
def test_chain32_matches_oracle(gpu, layers, monkeypatch, T, k, x_dtype, mode, wbd):
    import torch

    monkeypatch.setenv("LATENT_MOE_PATH", "fused")
    host, dev = layers
    rng = np.random.default_rng(T * 10 + k)
    tdt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[x_dtype]
    xt = torch.from_numpy(rng.standard_normal((T, host.d)).astype(np.float32)).cuda().to(tdt)
    ids, w = routing.softmax_topk(rng.standard_normal((T, host.n_expert)), k)
    ids[rng.random(ids.shape) < 0.1] = -1
    ids[0, 0] = host.n_expert + 3
    if T == 32:
        ids[:17] = 2  # one unit of 16 pairs and one of a single pair
    it, wt = torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w.astype(np.float32)).cuda()
    assert gpu.moe_path(dev, xt, k) == "fused"
    got = gpu.moe_forward(xt, it, wt, dev, weight_before_down=wbd, out_mode=mode)
    again = gpu.moe_forward(xt, it, wt, dev, weight_before_down=wbd, out_mode=mode)
    want = ref.moe_forward(xt.float().cpu().numpy(), np.where(ids >= host.n_expert, -1, ids), w, host,
                           weight_before_down=wbd, out_mode=mode)
    assert torch.equal(got, again)
    assert ref.rel_l2(want, got.cpu().numpy()) <= TOL
    if mode == 1:
        assert not got[torch.from_numpy((ids < 0) | (ids >= host.n_expert)).cuda()].any()
