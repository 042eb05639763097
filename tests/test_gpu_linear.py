"""GPU tests of the caller layer: packed-weight file, registered torch operators on a side
stream, and the linear layer, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import mx_oracle as mo
from tests import helpers as H

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def linear():
    from mixedgemm_amd import abi, linear as l
    abi.lib()
    return l


def _oracle_linear(x, w, idx, split):
    qx = mo.reorder_quantize_x(H.bf16_f32(x), idx.numpy(), *split)
    qw = mo.reorder_quantize_w(H.bf16_f32(w), idx.numpy(), *split)
    ref = mo.mixed_matmul(qx, qw)
    slack = (np.abs(mo.dequantize_x(qx)).astype(np.float64) @ np.abs(mo.dequantize_w(qw)).astype(np.float64).T) * 2.0 ** -20
    return ref, slack


def _close(d, ref, slack):
    err = np.abs(d.float().cpu().numpy() - mo.bf16_rne(ref))
    assert np.all(err <= H.bf16_ulp(ref) + slack), f"max err {err.max()}"


@pytest.mark.parametrize("m,n,k", [(24, 64, 4096), (3, 32, 3584), (256, 256, 5120)])
def test_linear_layer_matches_oracle(linear, m, n, k):
    print("linear layer", m, n, k, flush=True)
    split = linear.default_split(k)
    x = H.make_activations(m, k, 900 + m)
    w = H.make_weights(n, k, 901 + m)
    layer = linear.MixedLinear.from_float(w.to(DEV), calibration_x=x.to(DEV))
    idx = H.absmax_sort_index(x)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(layer.reorder_index.cpu().numpy(), idx.numpy())
    y = layer(x.to(DEV).reshape(1, m, k))
    torch.cuda.synchronize()
    assert y.shape == (1, m, n)
    ref, slack = _oracle_linear(x, w, idx, split)
    _close(y[0], ref, slack)


def test_pack_file_round_trip_through_the_gpu(linear, tmp_path):
    m, n, k = 16, 48, 4096
    split = linear.default_split(k)
    x = H.make_activations(m, k, 77)
    w = H.make_weights(n, k, 78)
    idx = H.absmax_sort_index(x)
    pw = linear.PackedWeights.from_float(w.to(DEV), idx.to(DEV), split)
    assert not pw.tiled          # 48 features: not a multiple of 256
    torch.cuda.synchronize()
    path = str(tmp_path / "layer.mgw")
    pw.save(path)
    back = linear.PackedWeights.load(path, device=DEV)
    assert not back.tiled
    for a, b in zip((*pw.tensors(), pw.reorder_index), (*back.tensors(), back.reorder_index)):
        assert torch.equal(a, b)
    y0 = linear.MixedLinear(pw)(x.to(DEV))
    y1 = linear.MixedLinear(back)(x.to(DEV))
    torch.cuda.synchronize()
    assert torch.equal(y0, y1)
    ref, slack = _oracle_linear(x, w, idx, split)
    _close(y1, ref, slack)


def test_operators_run_on_the_current_stream_without_synchronizing(linear):
    """The three reference calls as registered operators on a side stream: results are complete
    after waiting for that stream only, and equal those of the default stream."""
    m, n, k = 40, 64, 4096
    kn, ks, ko = linear.default_split(k)
    x = H.make_activations(m, k, 5).to(DEV)
    w = H.make_weights(n, k, 6).to(DEV)
    idx = torch.ops.mixedgemm_amd.calibrate_reorder_index(x)
    ops = torch.ops.mixedgemm_amd
    a = ops.reorder_quantize_x(x, idx, kn, ks, ko)
    b = ops.reorder_quantize_w(w, idx, kn, ks, ko)
    d0 = ops.matmul(a[0], b[0], a[1], b[1], a[2], b[2], a[3], b[3], a[4], b[4], a[5], b[5])
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        a1 = ops.reorder_quantize_x(x, idx, kn, ks, ko)
        d1 = ops.matmul(a1[0], b[0], a1[1], b[1], a1[2], b[2], a1[3], b[3], a1[4], b[4], a1[5], b[5])
        d2 = ops.fused_linear(x, idx, *b, kn, ks, ko)
    side.synchronize()
    assert torch.equal(d0, d1) and torch.equal(d0, d2)
    for t0, t1 in zip(a[:3], a1[:3]):
        assert torch.equal(t0, t1)


@pytest.mark.parametrize("m", [8, 300])
def test_tiled_pack_round_trip_and_layer(linear, tmp_path, m):
    """Default packing of a tileable layer is tile-major; the file keeps the layout and the layer gives
    the row-major result bit for bit."""
    n, k = 512, 4096
    split = linear.default_split(k)
    x = H.make_activations(m, k, 81)
    w = H.make_weights(n, k, 82)
    idx = H.absmax_sort_index(x)
    tiled = linear.PackedWeights.from_float(w.to(DEV), idx.to(DEV), split)
    plain = linear.PackedWeights.from_float(w.to(DEV), idx.to(DEV), split, tile=False)
    assert tiled.tiled and not plain.tiled and not torch.equal(tiled.wn, plain.wn)
    path = str(tmp_path / "tiled.mgw")
    tiled.save(path)
    assert linear.read_header(path)[0]["code_layout"] == "tile-major-256x128"
    back = linear.PackedWeights.load(path, device=DEV)
    assert back.tiled and torch.equal(back.wn, tiled.wn) and torch.equal(back.ws, tiled.ws)
    y0 = linear.MixedLinear(plain)(x.to(DEV))
    y1 = linear.MixedLinear(back)(x.to(DEV))
    torch.cuda.synchronize()
    assert torch.equal(y0, y1)
    ref, slack = _oracle_linear(x, w, idx, split)
    _close(y1, ref, slack)


def test_layer_with_fused_rmsnorm(linear):
    m, n, k, eps = 70, 256, 4096, 1e-5
    split = linear.default_split(k)
    x = H.make_activations(m, k, 91)
    w = H.make_weights(n, k, 92)
    g = torch.Generator().manual_seed(93)
    gamma = (torch.randn(k, generator=g) * 0.3 + 1.0).to(torch.bfloat16)
    y = torch.from_numpy(mo.rmsnorm_bf16(H.bf16_bits(x), H.bf16_bits(gamma), eps).view(np.int16)).view(torch.bfloat16)
    idx = H.absmax_sort_index(y)
    pw = linear.PackedWeights.from_float(w.to(DEV), idx.to(DEV), split)
    layer = linear.MixedLinear(pw, norm_weight=gamma.to(DEV), eps=eps)
    out = layer(x.to(DEV))
    torch.cuda.synchronize()
    ref, slack = _oracle_linear(y, w, idx, split)
    _close(out, ref, slack)


def test_layer_replayed_as_a_hip_graph(linear):
    """The whole layer (RMSNorm + reorder-quantize + GEMM: three of our launches, nothing else) captured once
    and replayed with new inputs in the same buffers; every replay must equal the eager result."""
    m, n, k = 300, 512, 4096
    split = linear.default_split(k)
    g = torch.Generator().manual_seed(7)
    gamma = (torch.randn(k, generator=g) * 0.3 + 1.0).to(torch.bfloat16).to(DEV)
    xs = [H.make_activations(m, k, 200 + i).to(DEV) for i in range(3)]
    w = H.make_weights(n, k, 210).to(DEV)
    from mixedgemm_amd import abi
    idx = abi.calibrate_reorder_index(xs[0])
    pw = linear.PackedWeights.from_float(w, idx, split)
    x_buf = xs[0].clone()
    ws = torch.empty(abi.fused_workspace_bytes(m, *split), dtype=torch.uint8, device=DEV)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)

    def run():
        abi.fused_linear(x_buf, idx, *pw.tensors(), *split, workspace=ws, out=out, w_tiled=pw.tiled,
                         norm_weight=gamma, eps=1e-5)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        run()                                # warm-up outside the capture (first-call setup)
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            run()
    torch.cuda.synchronize()
    for i in (1, 2, 0, 1):
        x_buf.copy_(xs[i])
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        eager = abi.fused_linear(xs[i], idx, *pw.tensors(), *split, w_tiled=pw.tiled, norm_weight=gamma, eps=1e-5)
        torch.cuda.synchronize()
        assert torch.equal(got, eager), f"replay with input {i} differs from the eager result"


@pytest.mark.parametrize("m,n", [(300, 1000), (8, 300)])
def test_layer_pads_odd_feature_counts_to_whole_tiles(linear, tmp_path, m, n):
    """N that is not a multiple of 256: the packer appends zero rows so that the whole-tile kernel and
    tile-major weights apply; the layer returns the real N columns, and the file keeps both counts."""
    k = 4096
    split = linear.default_split(k)
    x = H.make_activations(m, k, 95)
    w = H.make_weights(n, k, 96)
    idx = H.absmax_sort_index(x)
    pw = linear.PackedWeights.from_float(w.to(DEV), idx.to(DEV), split)
    assert pw.out_features == n and pw.rows % 256 == 0 and pw.rows >= n and pw.tiled
    path = str(tmp_path / "odd.mgw")
    pw.save(path)
    back = linear.PackedWeights.load(path, device=DEV)
    assert back.out_features == n and back.rows == pw.rows and back.tiled
    y = linear.MixedLinear(back)(x.to(DEV))
    torch.cuda.synchronize()
    assert y.shape == (m, n)
    ref, slack = _oracle_linear(x, w, idx, split)
    _close(y, ref, slack)


@pytest.mark.parametrize("split", [(512, 0, 0), (384, 0, 128), (384, 128, 0)])
def test_layer_with_a_plan_that_has_no_e3m2_or_e4m3_segment(linear, tmp_path, split):
    """All-MXFP4 activations, MXFP4 + MXFP8 outliers, MXFP4 + MXFP6: packed tile-major, saved, loaded, run."""
    m, n, k = 300, 512, sum(split)
    x = H.make_activations(m, k, 97, n_out=8)
    w = H.make_weights(n, k, 98)
    idx = H.absmax_sort_index(x)
    pw = linear.PackedWeights.from_float(w.to(DEV), idx.to(DEV), split)
    assert pw.tiled
    path = str(tmp_path / "partial.mgw")
    pw.save(path)
    back = linear.PackedWeights.load(path, device=DEV)
    assert back.split == tuple(split) and back.tiled
    y = linear.MixedLinear(back)(x.to(DEV))
    torch.cuda.synchronize()
    ref, slack = _oracle_linear(x, w, idx, split)
    _close(y, ref, slack)


@pytest.mark.parametrize("m", [1, 16, 40, 300])
@pytest.mark.parametrize("n", [24, 1001, 1004, 1280])
@pytest.mark.parametrize("bias", [False, True])
def test_layer_stores_the_real_features_and_adds_the_bias(linear, m, n, bias):
    """The kernels' own slice and bias against the operators' result, sliced and added to by torch: the same roundings in
    the same order, so the same bits.  Feature counts with whole, half and odd 16-byte pieces in the last tile."""
    k = 1088                                     # (640, 320, 128): two blocks past the last whole step of a segment
    split = linear.default_split(k)
    x = H.make_activations(m, k, 300 + m).to(DEV)
    w = H.make_weights(n, k, 301 + n).to(DEV)
    b = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(torch.bfloat16).to(DEV) if bias else None
    pw = linear.PackedWeights.from_float(w, torch.ops.mixedgemm_amd.calibrate_reorder_index(x), split)
    want = torch.ops.mixedgemm_amd.fused_linear(x, pw.reorder_index, *pw.tensors(), *split, pw.tiled)[:, :n]
    want = want + b if bias else want
    got = linear.MixedLinear(pw, bias=b)(x.view(m, 1, k))
    torch.cuda.synchronize()
    assert got.shape == (m, 1, n) and got.is_contiguous()
    assert torch.equal(got[:, 0], want)


# A few tokens in one launch against the quantizer and the GEMM one after the other: the same bits.  One to eight tokens on
# both sides of the largest count it takes, with and without RMSNorm, all three feature group counts, ragged features, one
# and several rounds of blocks per lane, a last step of 1 to 3 blocks, an index with entries out of range.
@pytest.mark.parametrize("n,split", [(256, (128, 128, 128)), (4096, (2560, 1408, 128)), (8192, (1024, 480, 160)), (14336, (2560, 1408, 128)),
                                     (1000, (416, 224, 96)), (40, (32, 32, 32)), (520, (5120, 2560, 512)), (264, (0, 1056, 0)),
                                     (300, (96, 0, 672)), (256, (512, 384, 128)), (264, (640, 320, 96))])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("tiled", [False, True])
def test_few_tokens_in_one_launch(linear, n, split, norm, tiled):
    from mixedgemm_amd import abi
    k = sum(split)
    if tiled and not (n % 256 == 0 and abi.weights_tileable(n, *split)):
        pytest.skip("shape cannot be tiled")
    g = torch.Generator().manual_seed(n + k)
    idx = torch.randperm(k, generator=g).to(torch.int16)
    idx[3], idx[k - 1] = -5, 32767   # read as channel K - 1 on both ways
    idx, w = idx.to(DEV), H.make_weights(n, k, 7).to(DEV)
    b = abi.reorder_quantize_w(w, idx, *split)
    if tiled:
        b = abi.tile_weights(*b[:3]) + tuple(b[3:])
    gamma = (1 + 0.1 * torch.randn(k, generator=g)).to(torch.bfloat16).to(DEV) if norm else None
    for m in (1, 2, 3, 5, 8):
        x = H.make_activations(m, k, 100 + m, n_out=max(1, k // 32)).to(DEV)
        got = abi.fused_linear(x, idx, *b, *split, w_tiled=tiled, norm_weight=gamma, eps=1e-5)
        a = abi.rmsnorm_reorder_quantize_x(x, gamma, 1e-5, idx, *split) if norm else abi.reorder_quantize_x(x, idx, *split)
        want = abi.matmul(a[0], b[0], a[1], b[1], a[2], b[2], a[3], b[3], a[4], b[4], a[5], b[5], w_tiled=tiled)
        torch.cuda.synchronize()
        assert torch.equal(got, want), m


# Rings of five slots and steps two at a time with one and two feature groups, four slots with four: 2 ... 16 steps per wave, odd and even, the
# segments' borders at either step of a pair, with and without partial last steps.
@pytest.mark.parametrize("n,split", [(264, (640, 256, 128)), (264, (1216, 480, 96)), (264, (1920, 896, 256)), (264, (4096, 3072, 1024)),
                                     (6144, (640, 256, 128)), (6144, (1216, 480, 96)), (6144, (2688, 1024, 384)), (14336, (1216, 480, 96))])
@pytest.mark.parametrize("tiled", [False, True])
def test_few_tokens_take_steps_in_pairs(linear, n, split, tiled):
    test_few_tokens_in_one_launch(linear, n, split, False, tiled)


# The same with rows that no random draw gives: zeros of both signs, the smallest subnormals, the largest finite values, one
# infinity, one NaN.  A block that holds an infinity or a NaN has no specified codes, but both ways run the same arithmetic.
@pytest.mark.parametrize("n,split", [(256, (128, 128, 128)), (1000, (416, 224, 96)), (4096, (1280, 640, 128))])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("tiled", [False, True])
def test_special_rows_in_one_launch(linear, n, split, norm, tiled):
    from mixedgemm_amd import abi
    k = sum(split)
    if tiled and not (n % 256 == 0 and abi.weights_tileable(n, *split)):
        pytest.skip("shape cannot be tiled")
    g = torch.Generator().manual_seed(n)
    idx, w = torch.randperm(k, generator=g).to(torch.int16).to(DEV), H.make_weights(n, k, 8).to(DEV)
    b = abi.reorder_quantize_w(w, idx, *split)
    if tiled:
        b = abi.tile_weights(*b[:3]) + tuple(b[3:])
    gamma = (1 + 0.1 * torch.randn(k, generator=g)).to(torch.bfloat16).to(DEV) if norm else None
    signs = torch.where(torch.arange(k) % 2 == 0, 1.0, -1.0)
    ordinary = H.make_activations(1, k, 9)[0].float()
    one = lambda v: torch.where(torch.arange(k) == 77, torch.tensor(v), ordinary)
    rows = torch.stack([torch.zeros(k) * signs, signs * 2.0 ** -133, signs * 2.0 ** -126, signs * 3.38953139e38, one(float("inf")),
                        one(float("-inf")), one(float("nan")), ordinary]).to(torch.bfloat16).to(DEV)
    for m in (1, 2, 4):
        for first in range(0, 8, m):
            x = rows[first:first + m].contiguous()
            got = abi.fused_linear(x, idx, *b, *split, w_tiled=tiled, norm_weight=gamma, eps=1e-5)
            a = abi.rmsnorm_reorder_quantize_x(x, gamma, 1e-5, idx, *split) if norm else abi.reorder_quantize_x(x, idx, *split)
            want = abi.matmul(a[0], b[0], a[1], b[1], a[2], b[2], a[3], b[3], a[4], b[4], a[5], b[5], w_tiled=tiled)
            torch.cuda.synchronize()
            torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)


# Views of a fused weight where the packer appends rows: the bits of the same weight packed from a tensor of its own.
@pytest.mark.parametrize("view", ["transposed", "columns", "offset"])
def test_a_view_packs_as_its_copy_does(linear, view):
    n, k = 1000, 1088                            # 1000 features are stored as 1024
    w = H.make_weights(n, k, 17).to(DEV)
    idx = H.random_index(k, 18).to(DEV)
    if view == "transposed":
        strided = w.t().contiguous().t()
    elif view == "columns":
        strided = w.repeat_interleave(2, dim=1)[:, ::2]
    else:                                        # rows start 2 bytes past a 16-byte line
        strided = torch.cat([w.new_zeros(1), w.reshape(-1)])[1:].view(n, k)
    got, want = linear.PackedWeights.from_float(strided, idx), linear.PackedWeights.from_float(w, idx)
    assert got.tiled and got.features == n
    for a, b in zip(got.tensors()[:3], want.tensors()[:3]):
        assert torch.equal(a, b)
    x = H.make_activations(300, k, 19).to(DEV)
    assert torch.equal(linear.MixedLinear(got)(x), linear.MixedLinear(want)(x))


# An error that the HIP runtime holds when a call launches reaches the caller, once, from every way into the library, and the
# next call works.  (hipSetDevice of a device that is not there leaves one: the kernel itself is launched as ever.)
@pytest.mark.parametrize("call", ["layer", "layer with RMSNorm", "fused_linear", "reorder_quantize_x", "reorder_quantize_w",
                                  "reorder_quantize_w_tiled", "matmul", "calibrate", "operator", "quantizer operator",
                                  "calibration operator"])
def test_a_hip_error_is_raised_not_retried(linear, call):
    from mixedgemm_amd import abi
    m, n, k = 40, 256, 1088
    split = linear.default_split(k)
    x, w = H.make_activations(m, k, 1).to(DEV), H.make_weights(n, k, 2).to(DEV)
    idx = H.random_index(k, 3).to(DEV)
    a, b = abi.reorder_quantize_x(x, idx, *split), abi.reorder_quantize_w(w, idx, *split)
    packed = linear.PackedWeights.from_float(w, idx)
    layer = linear.MixedLinear(packed)
    norm_layer = linear.MixedLinear(packed, norm_weight=torch.ones(k, dtype=torch.bfloat16, device=DEV))
    ops = torch.ops.mixedgemm_amd
    run = {"layer": lambda: layer(x), "layer with RMSNorm": lambda: norm_layer(x),
           "fused_linear": lambda: abi.fused_linear(x, idx, *b, *split),
           "reorder_quantize_x": lambda: abi.reorder_quantize_x(x, idx, *split),
           "reorder_quantize_w": lambda: abi.reorder_quantize_w(w, idx, *split),
           "reorder_quantize_w_tiled": lambda: abi.reorder_quantize_w_tiled(w, idx, *split),
           "matmul": lambda: abi.matmul(a[0], b[0], a[1], b[1], a[2], b[2], a[3], b[3], a[4], b[4], a[5], b[5]),
           "calibrate": lambda: abi.calibrate_reorder_index(x),
           "operator": lambda: ops.fused_linear(x, idx, *b, *split),
           "quantizer operator": lambda: ops.reorder_quantize_x(x, idx, *split),
           "calibration operator": lambda: ops.calibrate_reorder_index(x)}[call]
    run()                                        # what a first call sets up, and the allocator's blocks
    torch.cuda.synchronize()
    assert abi.lib().hipSetDevice(9999) != 0
    with pytest.raises(abi.MixedGemmError, match="invalid device"):
        run()
    got = run()
    torch.cuda.synchronize()
    assert got is not None


# The queue of a stream takes so many launches; the next one waits on the host until the GPU has worked some off.  Behind a
# kernel that spins for a second, layer calls fill the queue in a fraction of it, and while the one that waits does, a second
# Python thread goes on.
def test_other_threads_run_while_a_launch_waits(linear):
    import threading
    import time
    n, k = 256, 1088
    x = H.make_activations(1, k, 1).to(DEV)
    layer = linear.MixedLinear(linear.PackedWeights.from_float(H.make_weights(n, k, 2).to(DEV), H.random_index(k, 3).to(DEV)))
    want = layer(x)
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda._sleep(1_000_000)
    a.record(); torch.cuda._sleep(10_000_000); b.record()
    torch.cuda.synchronize()
    cycles_per_s = 10_000_000 / (a.elapsed_time(b) * 1e-3)

    ticks, done = [], threading.Event()

    def tick():
        while not done.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.002)

    thread = threading.Thread(target=tick)
    thread.start()
    torch.cuda._sleep(int(1.0 * cycles_per_s))
    start, waited = time.perf_counter(), 0.0
    while waited < 0.1 and time.perf_counter() - start < 1.5:
        t = time.perf_counter()
        got = layer(x)
        waited = time.perf_counter() - t
    torch.cuda.synchronize()
    done.set()
    thread.join()
    gap = max(b - a for a, b in zip(ticks, ticks[1:]))
    print(f"a launch waited {waited:.3f} s, the other thread stood still for {gap:.3f} s", flush=True)
    assert torch.equal(got, want)
    assert waited >= 0.1, "no launch waited: nothing was tested"
    assert gap < waited / 2


# Layer calls of several threads run side by side, each on its own stream: the bits of the same calls one after the other.
def test_layer_calls_from_several_threads(linear):
    import threading
    k, n = 1088, 512
    layer = linear.MixedLinear(linear.PackedWeights.from_float(H.make_weights(n, k, 2).to(DEV), H.random_index(k, 3).to(DEV)))
    xs = [H.make_activations(m, k, m).to(DEV) for m in (1, 7, 40, 300)]
    want = [layer(x) for x in xs]
    torch.cuda.synchronize()
    wrong = []

    def work(x, y):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            got = [layer(x) for _ in range(50)]
        stream.synchronize()
        wrong.extend(i for i, g in enumerate(got) if not torch.equal(g, y))

    threads = [threading.Thread(target=work, args=pair) for pair in zip(xs, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong

# ------------------------------------------------------------------ what observes or intercepts a layer call
def _small_layer(linear, norm=False, m=4, n=300, k=1088):
    x = H.make_activations(m, k, 1).to(DEV)
    pw = linear.PackedWeights.from_float(H.make_weights(n, k, 2).to(DEV), H.random_index(k, 3).to(DEV))
    bias = torch.linspace(-1, 1, n).to(torch.bfloat16).to(DEV)
    gamma = torch.linspace(0.5, 1.5, k).to(torch.bfloat16).to(DEV) if norm else None
    return linear.MixedLinear(pw, bias=bias, norm_weight=gamma), x


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("shapes", [False, True])
def test_a_profiler_sees_the_layer_as_its_operator(linear, norm, shapes):
    layer, x = _small_layer(linear, norm)
    layer(x)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=shapes) as prof:
        layer(x)
    name = "mixedgemm_amd::fused_norm_linear" if norm else "mixedgemm_amd::fused_linear"
    events = [e for e in prof.events() if e.name == name]
    assert len(events) == 1
    if shapes:
        assert list(events[0].input_shapes[0]) == list(x.shape)


@pytest.mark.parametrize("norm", [False, True])
def test_the_native_layer_call_is_the_one_that_runs(linear, norm):
    """Taken as it stands for a plain tensor -- and then the same bits as through the operators --, left to them where
    something intercepts the call or the tensor is not plain bf16."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from mixedgemm_amd import abi
    layer, x = _small_layer(linear, norm)
    args = (layer._buffers, layer.split, layer.tiled, layer.out_features, layer.eps)
    got = abi.host().layer(x, *args)
    assert got is not None

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(func.name())
            return func(*args, **(kwargs or {}))

    with Seen() as seen:
        assert abi.host().layer(x, *args) is None
        through_operators = layer(x)
    assert f"mixedgemm_amd::fused_{'norm_' if norm else ''}linear" in seen.names
    assert torch.equal(got, through_operators)
    assert abi.host().layer(x.float(), *args) is None and torch.equal(layer(x.float()), got)
    strided = torch.stack([x, x], dim=-1)[..., 0]
    assert abi.host().layer(strided, *args) is None and torch.equal(layer(strided), got)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(layer(x), got)


@pytest.mark.parametrize("norm", [False, True])
def test_a_gradient_through_the_layer_is_an_error(linear, norm):
    layer, x = _small_layer(linear, norm)
    y = layer(x.clone().requires_grad_())
    assert y.requires_grad and torch.equal(y.detach(), layer(x))
    with pytest.raises((RuntimeError, NotImplementedError)):
        y.sum().backward()
    with torch.no_grad():
        assert not layer(x.clone().requires_grad_()).requires_grad
