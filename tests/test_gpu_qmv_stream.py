"""Streaming form of the batched-decode GEMV (qmv_tile.hip,
qmv_stream_kernel): a workgroup owns its weight rows over a run of K slices,
with the next slices' codes and activations in flight while it works on the
current one.  Forced onto small shapes through MLXQ_QMV_TILE_STREAM (waves,
Q4 chunks per wave, K parts, K splits) and checked against the f64 CPU
oracle; the default dispatch is checked at the Llama-3-8B shapes it is chosen
for.  Bar: max|y - ref| / max|ref| <= 4e-3 (bf16 output rounding)."""
import numpy as np
import pytest

import oracle as orc
from helpers import bf16_acts, rel_err
from test_gpu_qmatmul import TIGHT, make_layer, run

pytestmark = pytest.mark.gpu


@pytest.fixture
def stream(monkeypatch):
    monkeypatch.setenv("MLXQ_QMV_TILE_ALL", "1")
    monkeypatch.delenv("MLXQ_QMV_TILE", raising=False)
    return monkeypatch


# (config, K): K slices of 512 (Q4 chunks x K parts x 128 codes) give 1, 2,
# 3, 4 and 8 steps per workgroup; splits divide the steps
CASES = [
    ("8,2,2,1", 512),    # one step
    ("8,2,2,1", 1536),   # three steps (odd: the loop's second half skipped at the end)
    ("8,2,2,1", 4096),   # eight steps
    ("8,4,2,1", 2048),   # two steps of 1024
    ("8,4,2,1", 3072),   # three steps of 1024
    ("8,2,4,1", 2048),   # K parts of 4 (two row groups)
    ("4,2,1,1", 1024),   # one K part
    ("4,4,1,1", 1536),
    ("8,2,1,1", 2048),   # eight row groups
    ("8,4,1,1", 1024),
    ("8,2,2,2", 4096),   # two splits of four steps
    ("8,2,2,4", 4096),   # four splits of two steps
    ("8,2,2,4", 2048),   # four splits of one step
    ("4,4,1,4", 4096),
    ("8,2,8,1", 2048),   # eight K parts: one step (M blocks of 16 above 16 rows)
    ("8,2,8,1", 6144),   # three steps
    ("8,2,8,2", 8192),   # two splits of two steps
]


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("cfg,k", CASES)
@pytest.mark.parametrize("m", [5, 16, 17, 32])
def test_stream_configs(torch_gpu, stream, bits, cfg, k, m):
    stream.setenv("MLXQ_QMV_TILE_STREAM", cfg)
    n = 200  # not a multiple of the row group (rows past N repeat N-1, dropped)
    wq, s, b = make_layer(90 + bits, n, k, 64, bits)
    x = bf16_acts(91 + m, m, k)
    ref = orc.qmatmul_f64(x, wq, s, b, 64, bits)
    assert rel_err(run(x, wq, s, b, 64, bits), ref) <= TIGHT


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("cfg,k", [("4,2,1,8", 2048), ("4,2,1,8", 2816), ("4,2,1,8", 3840), ("4,4,1,8", 6656),
                                   ("8,2,2,3", 4096), ("8,2,4,2", 3072)])
@pytest.mark.parametrize("m", [5, 16, 17, 32])
def test_stream_uneven_splits(torch_gpu, stream, bits, cfg, k, m):
    """K splits that do not divide the slices: 8 over 8, 11, 13 and 15 slices
    (K a multiple of 256 only), 3 over 8, 2 over 3."""
    stream.setenv("MLXQ_QMV_TILE_STREAM", cfg)
    n = 200
    wq, s, b = make_layer(110 + bits, n, k, 64, bits)
    x = bf16_acts(111 + m, m, k)
    ref = orc.qmatmul_f64(x, wq, s, b, 64, bits)
    assert rel_err(run(x, wq, s, b, 64, bits), ref) <= TIGHT


# (bits, M, N, K, the kernel's name up to its activation-row blocks)
ROUTES = [
    (4, 3, 5120, 13824, "stream<4,64,1,4,4,1"), (4, 17, 5120, 13824, "stream<4,64,2,4,2,1"),
    (8, 3, 5120, 13824, "stream<8,64,1,4,8,1"), (4, 4, 4096, 11008, "qmv_kernel"),
    (4, 5, 4096, 11008, "stream<4,64,1,4,2,1"), (8, 8, 4096, 11008, "qmv_kernel"),
    (8, 9, 4096, 11008, "stream<8,64,1,4,4,1"), (4, 5, 2048, 5632, "stream<4,64,1,4,2,1"),
    (8, 32, 2048, 5632, "stream<8,64,2,4,4,1"), (8, 5, 2049, 5632, "qmv_kernel"),
    (4, 15, 512, 2816, "qmv_kernel"), (4, 16, 512, 2816, "stream<4,64,1,4,2,1"),
    (4, 3, 8192, 3072, "stream<4,64,1,8,2,4"), (4, 32, 8192, 3072, "stream<4,64,2,8,2,4"),
    (8, 5, 8192, 3072, "qmv_kernel"), (8, 6, 8192, 3072, "stream<8,64,1,8,4,4"),
    (8, 16, 4097, 2048, "stream<8,64,1,8,4,4"), (8, 17, 4097, 2048, "tile<8,64,2"),
    (4, 5, 5120, 5120, "tile<4,64,1,8,8,1"), (8, 6, 5120, 5120, "tile<8,64,1,8,8,2"),
    (4, 5, 5632, 2048, "tile<4,64,1,8,4,4"), (4, 32, 3072, 8192, "tile<4,64,2,8,8,2"),
    (8, 6, 4096, 6144, "qmv_kernel"), (4, 8, 8192, 28672, "tile<4"),
]


@pytest.mark.parametrize("bits,m,n,k,kernel", ROUTES)
def test_stream_and_tile_routes(torch_gpu, monkeypatch, bits, m, n, k, kernel):
    """Both sides of each line of the default dispatch of batched decode away
    from the Llama-3-8B shapes: the kernel's name, and sampled rows against
    the oracle (above 2^25 codes: random codes, scales and biases)."""
    import mlxq
    for v in ("MLXQ_QMV_TILE_STREAM", "MLXQ_QMV_TILE", "MLXQ_QMV_TILE_ALL"):
        monkeypatch.delenv(v, raising=False)
    mlxq.reload_overrides()
    assert kernel in mlxq.qmatmul_route(m, n, k, 64, bits).replace(" ", "").replace("_kernel<", "<").replace(
        "qmv<", "qmv_kernel<")
    if n * k > 1 << 25:
        rng = np.random.default_rng(0x120 + bits)
        wq = rng.integers(0, 1 << 32, (n, k * bits // 32), dtype=np.uint32)
        s = orc.f32_to_bf16(rng.uniform(0.001, 0.01, (n, k // 64)).astype(np.float32)).reshape(n, -1)
        b = orc.f32_to_bf16(-(orc.bf16_to_f32(s).reshape(n, -1) * 2.0 ** (bits - 1)).astype(np.float32)).reshape(n, -1)
    else:
        wq, s, b = make_layer(0x120 + bits, n, k, 64, bits)
    x = bf16_acts(0x121 + m, m, k)
    y = run(x, wq, s, b, 64, bits)
    rows = np.unique(np.concatenate([np.random.default_rng(0x122).choice(n, 128, replace=False), np.arange(n - 16, n)]))
    assert rel_err(y[:, rows], orc.qmatmul_f64(x, wq[rows], s[rows], b[rows], 64, bits)) <= TIGHT


@pytest.mark.parametrize("bits,m,n,k", [r[:4] for r in ROUTES if "stream" in r[4] or "tile" in r[4]] + [
    (4, 16, 4096, 4096), (4, 32, 4096, 4096), (8, 16, 1024, 4096), (4, 96, 14336, 4096)])
def test_group_sums_keep_f32(torch_gpu, monkeypatch, bits, m, n, k):
    """The affine term's group sums of the activations hold all 24 bits of an
    f32: every group of a row sums to 189.5, one to 189.5 + 2^-12, and biases
    of alternating sign (scales of 2^-60, codes 0) cancel all but +-2^-12.  A
    group sum cut to 16 bits gives 0.  Q8: an infinite activation under
    weights of one sign gives an infinity in every output of its row."""
    import torch

    import mlxq
    for v in ("MLXQ_QMV_TILE_STREAM", "MLXQ_QMV_TILE", "MLXQ_QMV_TILE_ALL"):
        monkeypatch.delenv(v, raising=False)
    mlxq.reload_overrides()
    route = mlxq.qmatmul_route(m, n, k, 64, bits)
    assert "stream" in route or "tile" in route, route
    G = k // 64
    x = torch.full((m, G, 64), 3.0)
    x[:, :, 0] = 3.5
    x[:, :, 1] = 0.0
    hit = (torch.arange(m) * (G - 1) // max(m - 1, 1)).tolist()  # spread over the groups
    for i, g in enumerate(hit):
        x[i, g, 1] = 2.0**-12
    x = x.view(m, k).to(torch.bfloat16).cuda()
    sign = 1.0 - 2.0 * (torch.arange(G) % 2)
    wq = torch.zeros((n, k * bits // 32), dtype=torch.int32, device="cuda")
    s = torch.full((n, G), 2.0**-60, dtype=torch.bfloat16, device="cuda")
    b = sign.to(torch.bfloat16).cuda().expand(n, G).contiguous()
    want = (sign[hit] * 2.0**-12 + 189.5 * float(sign.sum()))[:, None].expand(m, n)
    got = mlxq.qmatmul(x, wq, s, b, 64, bits).float().cpu()
    assert torch.all((got - want).abs() <= 2.0**-8 * want.abs()), (got[:, 0], want[:, 0])
    if bits == 8:
        x[m // 2, k // 2 + 1] = float("inf")
        got = mlxq.qmatmul(x, wq + 0x01010101, s.fill_(1), s, 64, bits).float()
        assert torch.isinf(got[m // 2]).all() and torch.isfinite(got[m // 2 + 1:]).all()


def test_stream_splits_without_workspace(torch_gpu):
    """Shapes whose default form splits K run on another kernel when the
    workspace has no room for the partials."""
    import mlxq
    for bits, m, n, k in ((4, 8, 5120, 13824), (4, 8, 2048, 5632), (8, 16, 512, 2816), (4, 8, 5120, 5120)):
        assert "split_reduce" in mlxq.qmatmul_route(m, n, k, 64, bits)
        alone = mlxq.qmatmul_route(m, n, k, 64, bits, workspace_bytes=0)
        assert "split_reduce" not in alone and "qmv" in alone, alone


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("cfg", ["8,4,2,1", "8,2,2,4"])
def test_stream_bias_and_outliers(torch_gpu, stream, bits, cfg):
    stream.setenv("MLXQ_QMV_TILE_STREAM", cfg)
    n, k, m = 640, 4096, 24
    wq, s, b = make_layer(95 + bits, n, k, 64, bits, outlier_cols=8)
    x = bf16_acts(96, m, k)
    bias = orc.f32_to_bf16(np.random.default_rng(97).normal(0, 1, n).astype(np.float32))
    ref = orc.qmatmul_f64(x, wq, s, b, 64, bits) + orc.bf16_to_f32(bias)[None, :].astype(np.float64)
    assert rel_err(run(x, wq, s, b, 64, bits, bias=bias), ref) <= TIGHT


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("proj,m", [("gate_up", 8), ("gate_up", 16), ("gate_up", 32), ("down", 12), ("down", 16), ("down", 32)])
def test_stream_default_llama(torch_gpu, monkeypatch, bits, proj, m):
    """The shapes the default dispatch streams (no overrides), sampled rows
    against the oracle."""
    for v in ("MLXQ_QMV_TILE_STREAM", "MLXQ_QMV_TILE", "MLXQ_QMV_TILE_ALL"):
        monkeypatch.delenv(v, raising=False)
    k, n = {"gate_up": (4096, 14336), "down": (14336, 4096)}[proj]
    wq, s, b = make_layer(98 + bits, n, k, 64, bits)
    x = bf16_acts(99 + m, m, k)
    y = run(x, wq, s, b, 64, bits)
    rows = np.random.default_rng(100).choice(n, 256, replace=False)
    ref = orc.qmatmul_f64(x, wq[rows], s[rows], b[rows], 64, bits)
    assert rel_err(y[:, rows], ref) <= TIGHT


def test_stream_graph_replay_bit_exact(torch_gpu, stream):
    """HIP-graph replays of the streaming form (with K splits and without)
    equal the eager call bit for bit, with eager work between replays."""
    import torch

    import mlxq
    from helpers import dev

    stream.setenv("MLXQ_QMV_TILE_STREAM", "8,2,2,2")
    n, k, m = 512, 4096, 32
    wq, s, b = make_layer(101, n, k, 64, 4)
    x = bf16_acts(102, m, k)
    xd, wd, sd, bd = dev(x, bf16=True), dev(wq), dev(s, bf16=True), dev(b, bf16=True)
    y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    call = mlxq.bind_qmatmul(xd, wd, sd, bd, 64, 4, out=y)
    call()
    torch.cuda.synchronize()
    eager = y.clone()
    g = torch.cuda.CUDAGraph()
    st = torch.cuda.Stream()  # its workspace is the graph's
    with torch.cuda.graph(g, stream=st):
        call()
    for i in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager), i
        with torch.cuda.stream(st):
            mlxq.qmatmul(xd, wd, sd, bd, 64, 4)  # eager work on the same workspace in between
        torch.cuda.synchronize()


@pytest.fixture(scope="module")
def tall_layers():
    """A ragged very tall gate/up-like matrix (65544 rows, an lm_head's
    shape class) per bit width, quantized once by the oracle."""
    return {bits: make_layer(0x7A11 + bits, 65544, 4096, 64, bits) for bits in (4, 8)}


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m", [4, 16, 32])
def test_stream_default_very_tall(torch_gpu, monkeypatch, tall_layers, bits, m):
    """Very tall matrices (N >= 65536) stream in 4-wave workgroups under the
    default dispatch; sampled rows (the ragged last ones included) against
    the oracle."""
    for v in ("MLXQ_QMV_TILE_STREAM", "MLXQ_QMV_TILE", "MLXQ_QMV_TILE_ALL"):
        monkeypatch.delenv(v, raising=False)
    n, k = 65544, 4096
    wq, s, b = tall_layers[bits]
    x = bf16_acts(0x7A12 + m, m, k)
    y = run(x, wq, s, b, 64, bits)
    rows = np.concatenate([np.random.default_rng(0x7A13).choice(n - 8, 248, replace=False), np.arange(n - 8, n)])
    ref = orc.qmatmul_f64(x, wq[rows], s[rows], b[rows], 64, bits)
    assert rel_err(y[:, rows], ref) <= TIGHT


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,force", [(65, False), (96, False), (128, False), (33, True), (200, True)])
def test_stream64_short_prefill(torch_gpu, monkeypatch, bits, m, force):
    """Short prefills of gate/up-like matrices on the 64-row streaming form
    (grid z = blocks of 64 activation rows, ragged last block): taken by
    default at 65..128 rows (no workspace), forced outside that range with
    MLXQ_QMV_STREAM64=1; sampled rows with a bias against the oracle."""
    import mlxq
    for v in ("MLXQ_QMV_TILE_STREAM", "MLXQ_QMV_TILE", "MLXQ_QMV_TILE_ALL", "MLXQ_QMV_STREAM64"):
        monkeypatch.delenv(v, raising=False)
    if force:
        monkeypatch.setenv("MLXQ_QMV_STREAM64", "1")
    mlxq.reload_overrides()
    k, n = 4096, 14336
    if not force:
        assert mlxq.workspace_size(m, n, k, 64, bits) == 0
    wq, s, b = make_layer(0x6400 + bits, n, k, 64, bits)
    x = bf16_acts(0x6401 + m, m, k)
    bias = orc.f32_to_bf16(np.linspace(-1, 1, n, dtype=np.float32))
    y = run(x, wq, s, b, 64, bits, bias=bias)
    rows = np.concatenate([np.random.default_rng(0x6402).choice(n - 8, 120, replace=False), np.arange(n - 8, n)])
    ref = orc.qmatmul_f64(x, wq[rows], s[rows], b[rows], 64, bits) + orc.bf16_to_f32(bias[rows]).astype(np.float64)
    assert rel_err(y[:, rows], ref) <= TIGHT
    monkeypatch.delenv("MLXQ_QMV_STREAM64", raising=False)
    mlxq.reload_overrides()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m", [40, 100])
def test_stream64_down_like_forced(torch_gpu, monkeypatch, bits, m):
    """The 64-row streaming form on a down-like matrix (four K splits through
    the workspace, then the reduction launch), forced with
    MLXQ_QMV_STREAM64=1 (not the default there); against the oracle."""
    import mlxq
    monkeypatch.setenv("MLXQ_QMV_STREAM64", "1")
    mlxq.reload_overrides()
    k, n = 14336, 4096
    assert mlxq.workspace_size(m, n, k, 64, bits) == 4 * m * n * 4
    wq, s, b = make_layer(0x6410 + bits, n, k, 64, bits)
    x = bf16_acts(0x6411 + m, m, k)
    y = run(x, wq, s, b, 64, bits)
    rows = np.random.default_rng(0x6412).choice(n, 128, replace=False)
    assert rel_err(y[:, rows], orc.qmatmul_f64(x, wq[rows], s[rows], b[rows], 64, bits)) <= TIGHT
    monkeypatch.delenv("MLXQ_QMV_STREAM64")
    mlxq.reload_overrides()

