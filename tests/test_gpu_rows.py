"""Row-layout MFMA phases (rows.hip, latent_moe_path 4) against the oracle.

LATENT_MOE_PATH=rows selects them for every call here.  Layers in the row
layout: uniform rank 256 pure NF4; heterogeneous per-expert ranks (multiples
of 32 and not, so chunks of 1 to 16 groups and partial groups) with 10 % INT8
groups; the config-0 expert shape (d 512, ff 1408: partial 256-column items
of ff, one 512-column item of d).  Batches from one token to experts with
more than 16 pairs (several passes), both output modes, weighting before
down, f32 / f16 / bf16 x, dropped and out-of-range slots.  Bar: rel-L2 <= 2e-3
against the oracle's fp32 result on the same packed factors (fp16 operands,
fp32 accumulation).
"""

import numpy as np
import pytest

from oracle import latent_ref as ref
from oracle import routing, synth

pytestmark = pytest.mark.gpu

TOL = 2e-3

LAYERS = {
    "uniform": dict(seed=71, n_expert=12, d=1024, ff=1024, max_rank=256),
    "hetero": dict(seed=72, n_expert=12, d=1024, ff=1536, max_rank=512,
                   ranks=[64, 128, 256, 512, 96, 320, 100, 512, 128, 256, 32, 448], int8_fraction=0.1),
    "config0": dict(seed=73, n_expert=4, d=512, ff=1408, max_rank=64),
}


def _rows_layer(layer):
    import torch

    from latent_amd import DeviceFactor, StackedLayer

    facs = {}
    for name in ref.FACTOR_NAMES:
        f = layer.factors[name]
        ext = None if f.int8 is None else (f.int8.bitmap, f.int8.row_offset, f.int8.data)
        facs[name] = DeviceFactor.from_numpy(f.codes, f.scales, ext)
    ranks = None if layer.ranks is None else torch.from_numpy(layer.ranks.astype(np.int32)).cuda()
    return StackedLayer(**facs, ranks=ranks, layout="rows")


@pytest.fixture(autouse=True)
def rows_path(monkeypatch):
    monkeypatch.setenv("LATENT_MOE_PATH", "rows")


@pytest.fixture(scope="module", params=sorted(LAYERS))
def layers(request, gpu):
    host = synth.make_layer(**LAYERS[request.param])
    return request.param, host, _rows_layer(host)


def _run(gpu, host, dev, x, ids, w, x_dtype="bf16", wbd=False, mode=0):
    import torch

    tdt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[x_dtype]
    xt = torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda().to(tdt)
    it = torch.from_numpy(np.ascontiguousarray(ids, np.int32)).cuda()
    wt = torch.from_numpy(np.ascontiguousarray(w, np.float32)).cuda()
    assert gpu.moe_path(dev, xt, ids.shape[1]) == "rows"
    out = gpu.moe_forward(xt, it, wt, dev, weight_before_down=wbd, out_mode=mode, check_timeout=True)
    torch.cuda.synchronize()
    E = host.n_expert
    want = ref.moe_forward(xt.float().cpu().numpy(), np.where(ids >= E, -1, ids), w, host,
                           weight_before_down=wbd, out_mode=mode)
    got = out.cpu().numpy()
    return got, want


@pytest.mark.parametrize("T,k", [(1, 8), (4, 4), (16, 8), (40, 8)])
@pytest.mark.parametrize("mode", [0, 1])
def test_rows_shapes(gpu, layers, T, k, mode):
    name, host, dev = layers
    E = host.n_expert
    k = min(k, E)
    rng = np.random.default_rng(1000 * T + 10 * k + mode)
    x = rng.standard_normal((T, host.d)).astype(np.float32)
    ids, w = routing.softmax_topk(rng.standard_normal((T, E)), k)
    got, want = _run(gpu, host, dev, x, ids, w, mode=mode)
    err = ref.rel_l2(want, got)
    print(f"rows {name} T={T} k={k} mode={mode} rel_l2={err:.3e}")
    assert np.isfinite(got).all() and err <= TOL


@pytest.mark.parametrize("x_dtype,wbd", [("f32", True), ("f16", False), ("bf16", True)])
def test_rows_dtypes_weighting_and_drops(gpu, layers, x_dtype, wbd):
    name, host, dev = layers
    E = host.n_expert
    rng = np.random.default_rng(9)
    T, k = 6, 4
    # Rows of very different magnitude, dropped and out-of-range slots, a
    # token with every slot dropped.
    x = (rng.standard_normal((T, host.d)) * np.array([[1e-3], [40.0], [1.0], [1.0], [3.0], [1.0]])).astype(np.float32)
    ids, w = routing.softmax_topk(rng.standard_normal((T, E)), k)
    ids[1, 2] = -1
    ids[2, 3] = E + 3
    ids[5, :] = -1
    for mode in (0, 1):
        got, want = _run(gpu, host, dev, x, ids, w, x_dtype=x_dtype, wbd=wbd, mode=mode)
        err = ref.rel_l2(want, got)
        print(f"rows {name} {x_dtype} wbd={wbd} mode={mode} rel_l2={err:.3e}")
        assert err <= TOL
        if mode == 1:
            assert not got[1, 2].any() and not got[2, 3].any() and not got[5].any()
        else:
            assert not got[5].any()


@pytest.mark.parametrize("T,k,mode,wbd", [(70, 4, 0, False), (100, 4, 1, True), (9, 3, 0, True)])
def test_rows_pair_blocks(gpu, T, k, mode, wbd):
    """Passes of one, two and four blocks of 16 pairs (the pairs per expert
    decide), with experts far below and above the average, ranks 192 (a tile of
    128 columns and half of one), ff and d that end inside an item."""
    host = synth.make_layer(seed=91, n_expert=9, d=1056, ff=1184, max_rank=192,
                            ranks=[192, 64, 32, 160, 192, 128, 191, 96, 0])
    dev = _rows_layer(host)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, host.d)).astype(np.float32)
    ids, w = routing.softmax_topk(rng.standard_normal((T, host.n_expert)) + np.linspace(2, 0, host.n_expert), k)
    ids[rng.random(ids.shape) < 0.05] = -1
    got, want = _run(gpu, host, dev, x, ids, w, wbd=wbd, mode=mode)
    assert ref.rel_l2(want, got) <= TOL


@pytest.mark.parametrize("R", [288, 416, 512])
@pytest.mark.parametrize("T", [60, 79, 80])
def test_rows_pair_blocks_of_high_ranks(gpu, R, T):
    """Pure NF4 layers above rank 256: 48, 63 and 64 pairs an expert (one block of
    pairs a pass, then four, whose latents and sums take up to 149 KB of LDS)."""
    host = synth.make_layer(seed=R, n_expert=5, d=544, ff=576, max_rank=R, ranks=[R, R - 31, 100, R, 260])
    dev = _rows_layer(host)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, host.d)).astype(np.float32)
    ids, w = routing.softmax_topk(rng.standard_normal((T, 5)), 4)
    for mode in (0, 1):
        got, want = _run(gpu, host, dev, x, ids, w, mode=mode)
        assert ref.rel_l2(want, got) <= TOL


@pytest.mark.parametrize("E,T,k", [
    (512, 700, 3),   # rounds of 1024 pairs: two and a part, the most experts they take
    (512, 256, 4),   # exactly one of them
    (513, 260, 4),   # rounds of 512 pairs: two and 16 pairs
    (1024, 128, 4),  # one whole round, the most experts placed in order
    (1025, 129, 4),  # more experts: placed as the threads come
])
def test_rows_grouping_rounds(gpu, E, T, k):
    """The grouping's placement rounds at their edges, a hot expert over every
    round, dropped slots, ids past the last expert and a repeated expert."""
    host = synth.make_layer(seed=E, n_expert=E, d=64, ff=64, max_rank=32)
    dev = _rows_layer(host)
    rng = np.random.default_rng(E + T)
    x = rng.standard_normal((T, host.d)).astype(np.float32)
    ids = rng.integers(0, E, (T, k)).astype(np.int32)
    w = rng.random((T, k)).astype(np.float32)
    ids[::3, 0] = E - 1
    ids[1::7, 1] = -1
    ids[2::11, 1] = E
    ids[5::13, 1] = ids[5::13, 0]
    for mode in (0, 1):
        got, want = _run(gpu, host, dev, x, ids, w, mode=mode)
        assert ref.rel_l2(want, got) <= TOL


@pytest.mark.parametrize("T,E,d,ff,R,mode", [
    (2050, 7, 288, 544, 128, 0),   # y rows and the per-token combine; passes shared by workgroups
    (2050, 7, 384, 640, 128, 1),   # also a shape of the GEMMs
    (1400, 5, 1056, 256, 64, 0),   # three pairs a token: 4200 pairs, the multi-workgroup grouping
])
def test_rows_large_batches(gpu, monkeypatch, T, E, d, ff, R, mode):
    """Batches from 2048 pairs (y rows) and 4096 (grouping in several
    workgroups), one hot expert; a sample of the tokens against the oracle,
    every token of the two output modes and of the GEMM engine (where the rank
    allows it) against each other."""
    import torch

    host = synth.make_layer(seed=95, n_expert=E, d=d, ff=ff, max_rank=R)
    dev = _rows_layer(host)
    rng = np.random.default_rng(T + R)
    k = 3 if R == 64 else 2
    x = torch.from_numpy(rng.standard_normal((T, d)).astype(np.float32)).cuda()
    logits = rng.standard_normal((T, E))
    logits[:, 3] += 1.5
    ids, w = routing.softmax_topk(logits, k)
    ids[rng.random(ids.shape) < 0.03] = -1
    it, wt = torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w.astype(np.float32)).cuda()
    got = gpu.moe_forward(x, it, wt, dev, out_mode=mode).cpu().numpy()
    pick = np.array(sorted(set(range(0, T, T // 40)) | {T - 1}))
    want = ref.moe_forward(x.cpu().numpy()[pick], ids[pick], w[pick], host, out_mode=mode)
    assert ref.rel_l2(want, got[pick]) <= TOL
    other = gpu.moe_forward(x, it, wt, dev, out_mode=1 - mode).cpu().numpy().astype(np.float64)
    slots, red = (other, got) if mode == 0 else (got.astype(np.float64), other)
    assert ref.rel_l2((slots * np.where(ids >= 0, w, 0.0)[..., None]).sum(1), red) <= 1e-4
    if R % 128 == 0 and d % 128 == 0:
        monkeypatch.setenv("LATENT_MOE_PATH", "prefill")
        gemm = gpu.moe_forward(x, it, wt, dev, out_mode=mode).cpu().numpy()
        assert ref.rel_l2(gemm, got) <= TOL


@pytest.mark.parametrize("T,E,d,ff,R,k,mode", [
    (300, 12, 256, 640, 128, 2, 0),    # four pair blocks, three planes of down latents, one of gate and up
    (130, 16, 1024, 256, 256, 2, 0),   # two pair blocks, four planes of gate and up, one of down latents
    (130, 16, 1024, 896, 384, 2, 1),   # the same with planes of both, per-slot output
    (2100, 7, 640, 512, 512, 2, 0),    # several workgroups group 4200 pairs
])
def test_row_layout_prefill_repeats_bit_for_bit(gpu, monkeypatch, T, E, d, ff, R, k, mode):
    """Row-layout prefill in these kernels: every sum has a fixed order, so calls
    repeat their bits (their latents used to meet in atomics), also on a
    workspace that another call left full of its own sums."""
    import torch

    monkeypatch.delenv("LATENT_MOE_PATH")
    ranks = [max(1, R - 37 * (i % 5)) for i in range(E)]
    host = synth.make_layer(seed=R, n_expert=E, d=d, ff=ff, max_rank=R, ranks=ranks)
    dev = _rows_layer(host)
    rng = np.random.default_rng(T + R)
    x = torch.from_numpy(rng.standard_normal((T, d)).astype(np.float32)).cuda()
    ids, w = routing.softmax_topk(rng.standard_normal((T, E)) + np.linspace(1.5, 0, E), k)
    ids[rng.random(ids.shape) < 0.03] = -1
    it, wt = torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w.astype(np.float32)).cuda()
    assert gpu.moe_path(dev, x, k) == "prefill"
    got = gpu.moe_forward(x, it, wt, dev, out_mode=mode)
    for _ in range(4):
        gpu.moe_forward(x.flip(0), it, wt, dev, out_mode=mode)
        assert torch.equal(got, gpu.moe_forward(x, it, wt, dev, out_mode=mode))
    pick = np.array(sorted(set(range(0, T, T // 30)) | {T - 1}))
    want = ref.moe_forward(x.cpu().numpy()[pick], ids[pick], w[pick], host, out_mode=mode)
    assert ref.rel_l2(want, got.cpu().numpy()[pick]) <= TOL


def test_row_layout_prefill_in_less_workspace(gpu, monkeypatch):
    """Given less than the queried size, row-layout prefill runs the GEMMs, whose
    need is that of a call in which they were chosen."""
    import torch

    from latent_amd._lib import LatentError

    monkeypatch.delenv("LATENT_MOE_PATH")
    host = synth.make_layer(seed=5, n_expert=8, d=512, ff=384, max_rank=128)
    dev = _rows_layer(host)
    rng = np.random.default_rng(8)
    T, k = 400, 2
    x = torch.from_numpy(rng.standard_normal((T, 512)).astype(np.float32)).cuda()
    ids, w = routing.softmax_topk(rng.standard_normal((T, 8)), k)
    it, wt = torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w.astype(np.float32)).cuda()
    full = gpu.workspace_size(dev, T, k)
    ws = torch.zeros(full, dtype=torch.uint8, device="cuda")
    phases = gpu.moe_forward(x, it, wt, dev, workspace=ws)
    monkeypatch.setenv("LATENT_MOE_PATH", "prefill")
    gemms = gpu.moe_forward(x, it, wt, dev, workspace=ws)
    monkeypatch.delenv("LATENT_MOE_PATH")
    assert not torch.equal(phases, gemms)
    assert torch.equal(gemms, gpu.moe_forward(x, it, wt, dev, workspace=ws[:full - 256]))
    with pytest.raises(LatentError):
        gpu.moe_forward(x, it, wt, dev, workspace=ws[:full // 3])


def test_rows_in_less_workspace(gpu):
    """Given less than the queried size, a call of 2048 pairs or more adds into its
    output instead of combining y rows; INT8 word offsets (two bitmap words a row)
    follow whichever scratch it has."""
    import torch

    from latent_amd._lib import LatentError

    host = synth.make_layer(seed=6, n_expert=6, d=1056, ff=1088, max_rank=96, int8_fraction=0.1)
    dev = _rows_layer(host)
    rng = np.random.default_rng(9)
    T, k = 700, 3
    x = rng.standard_normal((T, host.d)).astype(np.float32)
    ids, w = routing.softmax_topk(rng.standard_normal((T, 6)), k)
    xt, wt = torch.from_numpy(x).cuda(), torch.from_numpy(w.astype(np.float32)).cuda()
    it = torch.from_numpy(ids.astype(np.int32)).cuda()
    full = gpu.workspace_size(dev, T, k)
    ws = torch.zeros(full, dtype=torch.uint8, device="cuda")
    y_rows = gpu.moe_forward(xt, it, wt, dev, workspace=ws)
    least = full - T * k * (host.d + 1) * 4 // 256 * 256  # without y rows and their positions
    added = gpu.moe_forward(xt, it, wt, dev, workspace=ws[:least + 256])
    pick = np.arange(0, T, 17)
    want = ref.moe_forward(x[pick], ids[pick], w[pick], host)
    for got in (y_rows, added):
        assert ref.rel_l2(want, got.cpu().numpy()[pick]) <= TOL
    # The latents' sums differ in their last bits from call to call (atomics, a few
    # 2^-24); about 2^-11 of them then round to another fp16 value, 2^-11 away:
    # 2^-11 sqrt(2^-11) = 1e-5 of a row, ten times that allowed.
    assert ref.rel_l2(y_rows.cpu().numpy(), added.cpu().numpy()) <= 1e-4
    with pytest.raises(LatentError):
        gpu.moe_forward(xt, it, wt, dev, workspace=ws[:least // 2])


def test_rows_more_tokens_than_a_grid_dimension(gpu):
    """70,000 tokens, y rows and their combine: beyond the 65,535 workgroups of a
    launch's second dimension."""
    import torch

    host = synth.make_layer(seed=4, n_expert=3, d=64, ff=64, max_rank=32)
    dev = _rows_layer(host)
    rng = np.random.default_rng(1)
    T = 70000
    x = rng.standard_normal((T, host.d)).astype(np.float32)
    ids = rng.integers(-1, 3, (T, 1)).astype(np.int32)
    w = rng.random((T, 1)).astype(np.float32)
    got = gpu.moe_forward(torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda(), torch.from_numpy(w).cuda(), dev)
    got = got.cpu().numpy()
    pick = np.array([0, 1, 65534, 65535, 65536, T - 1])
    assert ref.rel_l2(ref.moe_forward(x[pick], ids[pick], w[pick], host), got[pick]) <= TOL
    assert not got[ids[:, 0] < 0].any() and got[ids[:, 0] >= 0].any(1).all()
