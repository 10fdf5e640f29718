"""Q8_0 product on the GPU vs the oracle (tests/matrix_test.cu strategy): tolerance
1e-2 of max(|want|, rms) at small shapes in full, spot checks at the benchmark shapes,
the transposed-operand control, fp16 output, and bit-exact dequantisation."""
import ctypes

import numpy as np
import pytest

from tests.gpu_util import dev, p, rel_rms

pytestmark = pytest.mark.gpu
TOL = 1e-2


@pytest.fixture(scope="module")
def torch():
    import torch
    return torch


def make(torch, lib, n, k, seed):
    w = torch.empty(n * (k // 32) * 34, dtype=torch.uint8, device="cuda")
    assert lib.aotx_synth_q8(p(w), n, k, 0.02, seed, None) == 0
    return w


@pytest.mark.parametrize("n,k", [(64, 256), (128, 704), (80, 128), (1000, 4096), (256, 14336)])
@pytest.mark.parametrize("m", [1, 3, 8, 17, 32, 40])
def test_gemv_small_full(torch, lib, orc, n, k, m):
    w = make(torch, lib, n, k, 7 + n + k)
    rng = np.random.default_rng(n * 131 + m)
    x = rng.normal(0, 1, (m, k)).astype(np.float16)
    xd = dev(x, torch)
    y = torch.zeros(m * n, dtype=torch.float32, device="cuda")
    assert lib.aotx_q8_gemv(p(w), n, k, p(xd), m, p(y), None) == 0
    torch.cuda.synchronize()
    want = orc.q8_gemv_f64(w.cpu().numpy(), n, k, x.view(np.uint16))
    assert rel_rms(y.cpu().numpy().reshape(m, n), want) < TOL


@pytest.mark.parametrize("n,k", [(4096, 4096), (14336, 4096), (4096, 14336), (128256, 4096)])
@pytest.mark.parametrize("m", [1, 4, 8, 32])
def test_gemv_benchmark_shapes_spot(torch, lib, orc, n, k, m):
    """64 spot checks against a double dot product of the same bytes
    (tests/matrix_test.cu:279-312) plus an fp16-output run."""
    w = make(torch, lib, n, k, 1234)
    rng = np.random.default_rng(m)
    x = rng.normal(0, 1, (m, k)).astype(np.float16)
    xd = dev(x, torch)
    y = torch.zeros(m * n, dtype=torch.float32, device="cuda")
    y16 = torch.zeros(m * n, dtype=torch.float16, device="cuda")
    assert lib.aotx_q8_gemv(p(w), n, k, p(xd), m, p(y), None) == 0
    assert lib.aotx_q8_gemv_f16(p(w), n, k, p(xd), m, p(y16), None) == 0
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    got16 = y16.cpu().numpy().reshape(m, n)
    wn = w.cpu().numpy().reshape(n, -1)
    rows = rng.integers(0, n, 64)
    want = orc.q8_gemv_f64(np.ascontiguousarray(wn[rows]), 64, k, x.view(np.uint16))
    rms = np.sqrt((want ** 2).mean())
    err = np.abs(got[:, rows] - want) / np.maximum(np.abs(want), rms)
    assert err.max() < TOL
    assert np.array_equal(got16, got.astype(np.float16))


def test_gemv_transposed_control(torch, lib, orc):
    n = k = 256
    w = make(torch, lib, n, k, 77)
    x = np.random.default_rng(1).normal(0, 1, (2, k)).astype(np.float16)
    y = torch.zeros(2 * n, dtype=torch.float32, device="cuda")
    assert lib.aotx_q8_gemv(p(w), n, k, p(dev(x, torch)), 2, p(y), None) == 0
    torch.cuda.synchronize()
    wn = w.cpu().numpy()
    right = orc.q8_gemv_f64(wn, n, k, x.view(np.uint16))
    swapped = orc.q8_gemv_f64(wn, n, k, x.view(np.uint16), swap=True)
    got = y.cpu().numpy().reshape(2, n)
    assert rel_rms(got, right) < TOL
    assert rel_rms(got, swapped) > 0.1


def test_dequant_bit_exact(torch, lib, orc):
    """Dequantised rows equal half(q * scale) of the host reading bit for bit
    (tests/matrix_test.cu:331-345)."""
    n, k = 40, 512
    w = make(torch, lib, n, k, 5)
    out = torch.zeros(10 * k, dtype=torch.float16, device="cuda")
    assert lib.aotx_q8_dequant(p(w), k, 7, 10, p(out), None) == 0
    torch.cuda.synchronize()
    from aotx_amd.model import dequant_q8
    want = dequant_q8(w.cpu().numpy().reshape(n, -1)[7:17], k).astype(np.float16)
    assert np.array_equal(out.cpu().numpy().reshape(10, k).view(np.uint16), want.view(np.uint16))


def test_device_synth_equals_host(torch, lib):
    n, k = 333, 4096
    w = make(torch, lib, n, k, 0xABCDEF)
    host = np.empty(n * (k // 32) * 34, dtype=np.uint8)
    lib.aotx_synth_q8_host(host.ctypes.data_as(ctypes.c_void_p), n, k, 0.02, 0xABCDEF, 4)
    assert np.array_equal(w.cpu().numpy(), host)


def repack(torch, lib, w, n, k):
    size = lib.aotx_q8r_size(n, k)
    assert size > 0
    wr = torch.empty(size, dtype=torch.uint8, device="cuda")
    assert lib.aotx_q8_repack(p(w), n, k, p(wr), None) == 0
    return wr


@pytest.mark.parametrize("n,k", [(64, 256), (128, 704), (80, 128), (1000, 4096), (256, 14336),
                                 (17, 96)])
@pytest.mark.parametrize("m", [1, 3, 6, 8, 16, 17, 32, 40, 33, 128, 300])
def test_repacked_gemv_small_full(torch, lib, orc, n, k, m):
    """The streaming product over repacked weights (the model path) vs the oracle."""
    w = make(torch, lib, n, k, 11 + n + k)
    wr = repack(torch, lib, w, n, k)
    rng = np.random.default_rng(n * 7 + m)
    x = rng.normal(0, 1, (m, k)).astype(np.float16)
    y = torch.zeros(m * n, dtype=torch.float32, device="cuda")
    assert lib.aotx_q8r_gemv(p(wr), n, k, p(dev(x, torch)), m, p(y), None) == 0
    torch.cuda.synchronize()
    want = orc.q8_gemv_f64(w.cpu().numpy(), n, k, x.view(np.uint16))
    assert rel_rms(y.cpu().numpy().reshape(m, n), want) < TOL


@pytest.mark.parametrize("n,k", [(4096, 4096), (14336, 4096), (4096, 14336), (128256, 4096)])
@pytest.mark.parametrize("m", [1, 4, 8, 32, 128, 512])
def test_repacked_gemv_benchmark_shapes(torch, lib, orc, n, k, m):
    w = make(torch, lib, n, k, 4321)
    wr = repack(torch, lib, w, n, k)
    rng = np.random.default_rng(m + 100)
    x = rng.normal(0, 1, (m, k)).astype(np.float16)
    xd = dev(x, torch)
    y = torch.zeros(m * n, dtype=torch.float32, device="cuda")
    y2 = torch.zeros(m * n, dtype=torch.float32, device="cuda")
    assert lib.aotx_q8r_gemv(p(wr), n, k, p(xd), m, p(y), None) == 0
    assert lib.aotx_q8_gemv(p(w), n, k, p(xd), m, p(y2), None) == 0
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    wn = w.cpu().numpy().reshape(n, -1)
    rows = rng.integers(0, n, 64)
    want = orc.q8_gemv_f64(np.ascontiguousarray(wn[rows]), 64, k, x.view(np.uint16))
    rms = np.sqrt((want ** 2).mean())
    assert (np.abs(got[:, rows] - want) / np.maximum(np.abs(want), rms)).max() < TOL
    # both kernels sum the same fp16 products in fp32: they agree far inside the tolerance
    assert rel_rms(got, y2.cpu().numpy().reshape(m, n)) < 1e-4


def test_repack_layout(torch, lib):
    """Repacked bytes: lane l = r + 16 g of (tile t, quad q) holds row 16t + r, block 4q + g;
    its quants 0..15 sit in the first 1 KB half of the (t, q) record, 16..31 in the second,
    each stored as q + 128 (the byte XOR 0x80); padding is q = 0 with scale 0."""
    n, k = 40, 384
    w = make(torch, lib, n, k, 3)
    wr = repack(torch, lib, w, n, k).cpu().numpy()
    src = w.cpu().numpy().reshape(n, k // 32, 34)
    tiles, quads = (n + 15) // 16, (k + 127) // 128
    quant = wr[:tiles * quads * 64 * 32].reshape(tiles, quads, 2, 64, 16).transpose(0, 1, 3, 2, 4)
    quant = quant.reshape(tiles, quads, 64, 32)
    scale = wr[tiles * quads * 64 * 32:].view(np.uint16).reshape(tiles, quads, 64)
    for t in range(tiles):
        for q in range(quads):
            for lane in range(64):
                r, g = lane % 16, lane // 16
                row, blk = 16 * t + r, 4 * q + g
                if row < n and blk < k // 32:
                    assert np.array_equal(quant[t, q, lane], src[row, blk, 2:] ^ 0x80)
                    assert scale[t, q, lane] == src[row, blk, :2].view(np.uint16)[0]
                else:
                    assert (quant[t, q, lane] == 0x80).all() and scale[t, q, lane] == 0


@pytest.mark.parametrize("n,k,shift", [(17, 96, 0), (33, 160, 2), (48, 32, 0), (300, 4128, 2), (130, 416, 0), (64, 512, 6),
                                       (200, 6304, 2), (2100, 416, 2), (8200, 416, 0)])
@pytest.mark.parametrize("m", [1, 4, 5, 9, 32, 33, 64, 100])
def test_product_ends_and_alignment(torch, lib, orc, n, k, shift, m):
    """Products over the file's layout whose blocks start at odd multiples of two bytes (an odd
    number of blocks a row, a tensor at any even address), and of both layouts where k ends
    inside 128 and rows inside 16, by every kernel (1-4, 5-32, 33 rows and more). What lies
    after x and the weights is never used: it holds NaN and scales of infinity here. The fp32
    sums agree with the fp64 product to 1e-5 of the result's rms (of 1 where that is smaller) times
    the square root of the 32-value blocks added up."""
    w = make(torch, lib, n, k, 3 + n + k)
    buf = torch.full((shift + w.numel() + 512,), 0x7C, dtype=torch.uint8, device="cuda")
    buf[shift:shift + w.numel()] = w
    rng = np.random.default_rng(n + m)
    x = rng.normal(0, 1, (m, k)).astype(np.float16)
    xb = torch.full((m * k + 256,), float("nan"), dtype=torch.float16, device="cuda")
    xb[:m * k] = torch.from_numpy(x).cuda().reshape(-1)
    want = orc.q8_gemv_f64(w.cpu().numpy(), n, k, x.view(np.uint16))
    rms = np.sqrt((want ** 2).mean())
    wr = repack(torch, lib, w, n, k)
    for fn, at in ((lib.aotx_q8_gemv, buf.data_ptr() + shift), (lib.aotx_q8r_gemv, wr.data_ptr())):
        y = torch.zeros(m * n, dtype=torch.float32, device="cuda")
        assert fn(ctypes.c_void_p(at), n, k, p(xb), m, p(y), None) == 0
        torch.cuda.synchronize()
        assert np.abs(y.cpu().numpy().reshape(m, n) - want).max() < 1e-5 * max(rms, 1.0) * np.sqrt(k / 32.0)


def test_product_rows_past_32_bit_offsets(torch, lib, orc):
    """x of more than 2^32 values: the rows past them are read where they are (both layouts, by
    the GEMM: 544 rows of 14336 are too many workgroups for passes of the 32-row kernel)."""
    n, k = 544, 14336
    m = 586 * 512                          # the last pass is a whole one
    assert (m - 100) * k > 1 << 32
    w = make(torch, lib, n, k, 77)
    wr = repack(torch, lib, w, n, k)
    rng = np.random.default_rng(77)
    last = rng.normal(0, 1, (8, k)).astype(np.float16)
    x = torch.zeros(m, k, dtype=torch.float16, device="cuda")
    x[:64] = 1.0
    x[m - 8:] = torch.from_numpy(last).cuda()
    want = orc.q8_gemv_f64(w.cpu().numpy(), n, k, last.view(np.uint16))
    rms = np.sqrt((want ** 2).mean())
    y = torch.zeros(m, n, dtype=torch.float32, device="cuda")
    for fn, at in ((lib.aotx_q8_gemv, w), (lib.aotx_q8r_gemv, wr)):
        y.fill_(7.0)
        assert fn(p(at), n, k, p(x), m, p(y), None) == 0
        torch.cuda.synchronize()
        assert np.abs(y[m - 8:].cpu().numpy() - want).max() < 1e-5 * max(rms, 1.0) * np.sqrt(k / 32.0)
        assert float(y[64:m - 8].abs().max()) == 0.0
    del x, y
    torch.cuda.empty_cache()


def _product64(w, n, k, x):
    """The fp64 product over the fp16 weights the kernels multiply with, on many rows at once."""
    rows = w.cpu().numpy().reshape(n, k // 32, 34)
    scale = rows[:, :, :2].copy().view(np.float16).astype(np.float32)
    wide = (scale * rows[:, :, 2:].view(np.int8)).astype(np.float16).astype(np.float64).reshape(n, k)
    return x.astype(np.float64) @ wide.T


@pytest.mark.parametrize("n,k", [(544, 4128), (2064, 512), (100, 96)])
@pytest.mark.parametrize("m", [512, 513, 580, 1024, 1100])
def test_product_of_more_rows_than_a_pass(torch, lib, orc, n, k, m):
    """Products run in passes of 512 rows: every row of the later ones is written, by the GEMM and
    by passes of the 32-row kernel, in both layouts."""
    w = make(torch, lib, n, k, m)
    wr = repack(torch, lib, w, n, k)
    rng = np.random.default_rng(n + m)
    x = rng.normal(0, 1, (m, k)).astype(np.float16)
    want = _product64(w, n, k, x)
    assert np.abs(want[-2:] - orc.q8_gemv_f64(w.cpu().numpy(), n, k, x[-2:].view(np.uint16))).max() < 1e-9
    rms = np.sqrt((want ** 2).mean())
    for fn, at in ((lib.aotx_q8_gemv, w), (lib.aotx_q8r_gemv, wr)):
        y = torch.full((m, n), 7.0, dtype=torch.float32, device="cuda")
        assert fn(p(at), n, k, p(dev(x, torch)), m, p(y), None) == 0
        torch.cuda.synchronize()
        assert np.abs(y.cpu().numpy() - want).max() < 1e-5 * max(rms, 1.0) * np.sqrt(k / 32.0)


@pytest.mark.parametrize("n,k", [(48, 160), (300, 4128), (1000, 1056), (8200, 416), (4096, 4096)])
@pytest.mark.parametrize("m", [1, 4, 8, 32, 64, 100])
def test_file_product_of_infinities(torch, lib, n, k, m):
    """An infinity in a row of x gives infinities of its weights' signs (NaN where the weight is
    0, as in any sum of products), wherever it lies: at k that does not divide evenly among
    waves, k splits or pairs of 128, by every kernel over the file's layout and, from 33 rows on,
    over the repacked one."""
    w = make(torch, lib, n, k, n + k)
    wr = repack(torch, lib, w, n, k)
    rows = w.cpu().numpy().reshape(n, k // 32, 34)
    quant = rows[:, :, 2:].view(np.int8).reshape(n, k).astype(np.float32)
    rng = np.random.default_rng(m + k)
    for base in range(0, max(1, k // 32), max(1, m)):
        x = rng.normal(0, 1, (m, k)).astype(np.float16)
        at = np.array([((base + i) * 32 + rng.integers(32)) % k for i in range(m)])
        x[np.arange(m), at] = np.where(rng.random(m) < 0.5, np.inf, -np.inf)
        with np.errstate(invalid="ignore"):
            want = quant[:, at].T * x[np.arange(m), at].astype(np.float32)[:, None]
        for fn, weights in ((lib.aotx_q8_gemv, w), (lib.aotx_q8r_gemv, wr))[:2 if m > 32 else 1]:
            y = torch.zeros(m, n, dtype=torch.float32, device="cuda")
            assert fn(p(weights), n, k, p(dev(x, torch)), m, p(y), None) == 0
            torch.cuda.synchronize()
            assert np.array_equal(y.cpu().numpy(), want, equal_nan=True)


@pytest.mark.parametrize("n,k,m", [(6144, 4128, 64), (6144, 4096, 40), (20000, 416, 300), (2064, 14336, 512)])
def test_product_large_forms(torch, lib, orc, n, k, m):
    """Both layouts through the 64-row form with k in two splits (96 groups of 4 tiles), the GEMM of
    more workgroups than CUs where k ends inside 128 (79 groups of 16 tiles x 5 row blocks), and
    its split merge (9 groups x 8 row blocks x 2 splits)."""
    w = make(torch, lib, n, k, n + m)
    wr = repack(torch, lib, w, n, k)
    x = np.random.default_rng(n + m).normal(0, 1, (m, k)).astype(np.float16)
    want = _product64(w, n, k, x)
    assert np.abs(want[-1:] - orc.q8_gemv_f64(w.cpu().numpy(), n, k, x[-1:].view(np.uint16))).max() < 1e-9
    rms = np.sqrt((want ** 2).mean())
    for fn, at in ((lib.aotx_q8_gemv, w), (lib.aotx_q8r_gemv, wr)):
        y = torch.full((m, n), 7.0, dtype=torch.float32, device="cuda")
        assert fn(p(at), n, k, p(dev(x, torch)), m, p(y), None) == 0
        torch.cuda.synchronize()
        assert np.abs(y.cpu().numpy() - want).max() < 1e-5 * max(rms, 1.0) * np.sqrt(k / 32.0)
