"""The GEMM on whole tiles (256 x 256 and 256 x 128): every instance of the kernel, bit for bit.

The kernel is compiled per set of segments, length of the last segment, tile, weight layout, and with or without segment boundaries in
the K loop and blocks past the whole stages.  Each of these runs here, on a shape that the dispatcher gives to it."""
import numpy as np
import pytest
import torch

from oracle import mx_oracle as mo

pytestmark = pytest.mark.gpu

DEV = "cuda"
FORMATS = ("e2m1", "e3m2", "e4m3")


@pytest.fixture(scope="module")
def abi():
    from mixedgemm_amd import abi as module
    module.lib()
    return module


# last segments of 1, 2 and 3 stages behind segments of fewer than 3 stages (2) and more; one, two and three segments; 1 to 3 blocks of
# 32 past the whole stages
SPLITS = (
    [s for a in (256, 512) for last in (128, 256, 384) for s in ((a, last, 0), (a, 0, last), (0, a, last))]
    + [(512, 0, 0), (0, 512, 0), (0, 0, 512)]
    + [(a, b, last) for a in (256, 512) for b in (256, 512) for last in (128, 256, 384)]
    + [s for last in (160, 288, 416) for s in ((544, 448, last), (416, 160, last))]
)
# 224 tiles of 256 x 128, half of them without their last token; 135 tiles of 256 x 256, 148 of which every other one has 44 tokens, 272 of
# which the last 16 run as half tiles; ragged tokens and features
SIZES = [(255, 28672), (2304, 3840), (300, 18944), (4352, 4096), (4300, 4104)]


def _table(fmt):
    """(codes, their values): all of a format, of E4M3 those up to 16 that are multiples of 1/16."""
    codes = np.arange(1 << mo.BITS[fmt])
    values = mo.decode_codes(codes, fmt).astype(np.float64)
    if fmt == "e4m3":
        keep = np.isfinite(values) & (np.abs(values) <= 16) & (np.mod(values * 16, 1) == 0)
        codes, values = codes[keep], values[keep]
    return torch.from_numpy(codes).to(DEV), torch.from_numpy(values).to(DEV)


def _operand(rows, kseg, fmt, operand, g):
    """Packed codes, scale buffer and values (fp64) of random codes with scales of 1/2, 1 and 2."""
    codes, values = _table(fmt)
    pick = torch.randint(0, len(codes), (rows, kseg), device=DEV, generator=g)
    c = codes[pick].int()
    if fmt == "e2m1":
        packed = c[:, 0::2] | c[:, 1::2] << 4
    elif fmt == "e3m2":   # a little-endian stream of 6-bit codes
        word = c[:, 0::4] | c[:, 1::4] << 6 | c[:, 2::4] << 12 | c[:, 3::4] << 18
        packed = torch.stack((word & 255, word >> 8 & 255, word >> 16), dim=2).flatten(1)
    else:
        packed = c
    scale = torch.randint(126, 129, (rows, kseg // 32), device=DEV, generator=g)
    buffer = torch.from_numpy(mo.sf_scatter(scale.to(torch.uint8).cpu().numpy(), kseg, operand)).to(DEV)
    return packed.to(torch.uint8).contiguous(), buffer, values[pick] * torch.exp2((scale - 127).double()).repeat_interleave(32, dim=1)


def _check(abi, m, n, kn, ks, ko):
    """Products are multiples of 2^-7 and their absolute values sum up to less than 2^17, so that every fp32 sum in any order is the
    exact one: the result is the fp64 product rounded once.  The activation buffers end with row m."""
    print("whole tiles", m, n, kn, ks, ko, flush=True)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tileable = abi.weights_tileable(n, kn, ks, ko)
    assert abi.gemm_kernel(m, n, kn, ks, ko, False, cus)[0] == "whole" and (not tileable or abi.gemm_kernel(m, n, kn, ks, ko, True, cus)[0] == "whole")
    g = torch.Generator(device=DEV).manual_seed(m + 3 * kn + 5 * ks + 7 * ko)
    a = [_operand(m, k, fmt, "a", g) for k, fmt in zip((kn, ks, ko), FORMATS)]
    b = [_operand(n, k, "e2m1", "b", g) for k in (kn, ks, ko)]
    av, bv = torch.cat([x[2] for x in a], dim=1), torch.cat([x[2] for x in b], dim=1)
    assert float((av.abs() @ bv.abs().T.contiguous()).max()) < 2 ** 17
    want = (av @ bv.T.contiguous()).to(torch.float32).to(torch.bfloat16)
    scales = (a[0][1], b[0][1], a[1][1], b[1][1], a[2][1], b[2][1])
    layouts = [([x[0] for x in b], False)]
    if tileable:
        layouts.append((abi.tile_weights(*(x[0] for x in b)), True))
    for w, w_tiled in layouts:
        d = abi.matmul(a[0][0], w[0], a[1][0], w[1], a[2][0], w[2], *scales, w_tiled=w_tiled)
        torch.cuda.synchronize()
        assert torch.equal(d.view(torch.int16), want.view(torch.int16)), f"w_tiled={w_tiled}: {int((d != want).sum())} of {d.numel()} differ"


@pytest.mark.parametrize("m,n", SIZES)
@pytest.mark.parametrize("kn,ks,ko", SPLITS)
def test_every_instance_of_the_whole_tile_kernel(abi, m, n, kn, ks, ko):
    _check(abi, m, n, kn, ks, ko)


# around the lengths of the runs of rows that a lane copies (2, 4, 8), the copy blocks of 16 rows and the second scale atom: tiles of 256 x 128
# (16384 features; fewer than 256 tokens) and of 256 x 256
@pytest.mark.parametrize("m,n", [(m, n) for m in (257, 258, 261, 263, 271, 272, 273, 384, 385, 511) for n in (16384, 28672)] + [(129, 28672), (200, 28672)])
@pytest.mark.parametrize("kn,ks,ko", [(480, 448, 160), (384, 384, 256)])
def test_rows_up_to_the_last_one_on_whole_tiles(abi, m, n, kn, ks, ko):
    _check(abi, m, n, kn, ks, ko)


# A layer call hands the codes of its tokens to whole tiles stage by stage, matmul gets them row by row: the same bits.  Ragged tokens and features, 256 x 256,
# 256 x 128 and both in one launch; one to three segments, 1 to 3 blocks past the whole stages; one lane per block from 16416 channels on.
@pytest.mark.parametrize("m,n", [(2304, 3840), (300, 18944), (511, 28672), (4300, 4104)])
@pytest.mark.parametrize("kn,ks,ko", [(512, 0, 0), (0, 512, 0), (0, 0, 512), (1024, 0, 128), (544, 448, 416), (480, 416, 160), (384, 384, 256), (10272, 5120, 1024),
                                      (12832, 6400, 1280)])
@pytest.mark.parametrize("norm", [False, True])
def test_layer_calls_on_whole_tiles_equal_quantize_then_gemm(abi, m, n, kn, ks, ko, norm):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert abi.gemm_kernel(m, n, kn, ks, ko, False, cus)[0] == "whole" or (m == 300 and kn > 10000)   # (small tiles)
    _check_layer_call(abi, m, n, kn, ks, ko, norm)


# The same on small tiles of tile-major weights: every tile, fewer and more than 256 tokens (two quantizers), one to three segments that begin and end
# inside a batch, 1 to 3 blocks past the whole stages, few and many stages.
@pytest.mark.parametrize("tf,tt,m,n", [(64, 64, 262, 256), (64, 64, 70, 5632), (128, 64, 145, 5632), (128, 64, 460, 2304), (128, 128, 399, 4864)])
@pytest.mark.parametrize("kn,ks,ko", [(1664, 640, 384), (1632, 736, 544), (2432, 0, 256), (0, 2176, 384), (2560, 1408, 128), (4160, 2144, 288)])
@pytest.mark.parametrize("norm", [False, True])
def test_layer_calls_on_small_tiles_equal_quantize_then_gemm(abi, tf, tt, m, n, kn, ks, ko, norm):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert abi.gemm_kernel(m, n, kn, ks, ko, True, cus)[0] == "tile"
    _check_layer_call(abi, m, n, kn, ks, ko, norm)


# Codes stage by stage out of every instance of the quantizer for many rows: its workgroup sizes with two lanes per block and with one, without RMSNorm
# and with it, one row per workgroup and two; the last stage of every segment is not whole.
@pytest.mark.parametrize("m", [256, 261, 531])
@pytest.mark.parametrize("k", [1024 * i - 32 for i in range(1, 17)] + [18400, 20448, 20512, 32736])
@pytest.mark.parametrize("norm", [False, True])
def test_layer_calls_of_every_width_equal_quantize_then_gemm(abi, m, k, norm):
    kn, ko = k * 5 // 8 // 128 * 128 + 32, max(k // 8 // 128, 1) * 128 + 96
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert abi.weights_tileable(256, kn, k - kn - ko, ko) and abi.gemm_kernel(m, 256, kn, k - kn - ko, ko, True, cus)[0] == "tile"
    _check_layer_call(abi, m, 256, kn, k - kn - ko, ko, norm)


# Codes stage by stage out of every instance of the quantizer for fewer rows than CUs: parts of 256 lanes, one to four of a row, and of 512, three and
# four (more than 256 parts of more than 16384 channels), with RMSNorm where that takes the kernel; on small tiles of each size and on whole ones; segments
# that end in a whole stage and 1 to 3 blocks behind one.
@pytest.mark.parametrize("kernel,m,n,kn,ks,ko", [
    (("tile", 64, 64), 52, 8448, 11808, 6496, 640), (("tile", 64, 64), 52, 12544, 11776, 6560, 608), (("tile", 128, 64), 100, 12544, 12832, 6400, 1280),
    (("tile", 128, 64), 100, 12544, 12800, 6720, 992), (("tile", 64, 64), 190, 2816, 20448, 10240, 2048), (("tile", 64, 64), 51, 8448, 11808, 6496, 640),
    (("tile", 64, 64), 64, 8448, 8960, 4928, 448), (("tile", 64, 64), 60, 8448, 8992, 4896, 448), (("tile", 64, 64), 200, 2816, 2560, 1408, 128),
    (("tile", 128, 64), 200, 4352, 2592, 1376, 160), (("tile", 128, 128), 255, 8448, 1632, 736, 544), (("tile", 64, 64), 255, 2816, 1248, 608, 192),
    (("whole", 256, 256), 200, 16640, 2560, 1408, 128), (("whole", 256, 256), 255, 16640, 1120, 544, 384)])
@pytest.mark.parametrize("norm", [False, True])
def test_layer_calls_of_few_rows_equal_quantize_then_gemm(abi, kernel, m, n, kn, ks, ko, norm):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert abi.weights_tileable(n, kn, ks, ko) and abi.gemm_kernel(m, n, kn, ks, ko, True, cus) == kernel
    _check_layer_call(abi, m, n, kn, ks, ko, norm)


# The tiles that the layer calls above are meant for.
@pytest.mark.parametrize("tf,tt,m,n", [(64, 64, 262, 256), (64, 64, 70, 5632), (128, 64, 145, 5632), (128, 64, 460, 2304), (128, 128, 399, 4864)])
@pytest.mark.parametrize("kn,ks,ko", [(1664, 640, 384), (1632, 736, 544), (2432, 0, 256), (0, 2176, 384), (2560, 1408, 128), (4160, 2144, 288)])
def test_layer_calls_take_their_small_tile(abi, tf, tt, m, n, kn, ks, ko):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert abi.gemm_kernel(m, n, kn, ks, ko, True, cus) == ("tile", tf, tt)


def _check_layer_call(abi, m, n, kn, ks, ko, norm):
    print("staged codes", m, n, kn, ks, ko, norm, flush=True)
    k, g = kn + ks + ko, torch.Generator(device=DEV).manual_seed(m + kn)
    x = torch.randn(m, k, device=DEV, generator=g)
    x[:, ::37] *= 30
    x, w = x.to(torch.bfloat16), (torch.randn(n, k, device=DEV, generator=g) * 0.02).to(torch.bfloat16)
    idx = torch.randperm(k, device=DEV, generator=g).to(torch.int16)
    gamma = (1 + 0.1 * torch.randn(k, device=DEV, generator=g)).to(torch.bfloat16)
    b = abi.reorder_quantize_w(w, idx, kn, ks, ko)
    a = abi.rmsnorm_reorder_quantize_x(x, gamma, 1e-5, idx, kn, ks, ko) if norm else abi.reorder_quantize_x(x, idx, kn, ks, ko)
    kw = dict(norm_weight=gamma, eps=1e-5) if norm else {}
    want = abi.matmul(a[0], b[0], a[1], b[1], a[2], b[2], *[t for pair in zip(a[3:], b[3:]) for t in pair])
    assert torch.equal(abi.fused_linear(x, idx, *b, kn, ks, ko, **kw), want)
    if abi.weights_tileable(n, kn, ks, ko):
        assert torch.equal(abi.fused_linear(x, idx, *abi.tile_weights(*b[:3]), *b[3:], kn, ks, ko, w_tiled=True, **kw), want)
