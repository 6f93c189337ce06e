"""GPU quantizer (pe_quantize) against the oracle's quantize_tensor and the
reference's golden codes (quantizer.py:206-257).

Codes are integers but come from an argmin over fp32 distances: the kernel's
butterfly transform and the reference's fp32 matmul round differently, so a
code may differ where the rotated value sits within fp32 rounding of the
midpoint between two centroids. The tests accept exactly those cases (and
count them); every other code, and every fp16 norm, must be equal."""

import math

import numpy as np
import pytest
import torch

import polar_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TIE_TOL = 1e-5  # |d_a - d_b| of a tolerated flip, relative to the centroid scale


def _say(msg):
    print(f"[case] {msg}", flush=True)


def rotated(w: np.ndarray) -> np.ndarray:
    """float64 statement of the rotated unit blocks (r in quantizer.py:235-241)."""
    w = np.asarray(w, dtype=np.float64)
    n, k = w.shape
    kp = (k + 127) // 128 * 128
    w = np.pad(w, ((0, 0), (0, kp - k))).reshape(n, kp // 128, 128)
    nrm = np.maximum(np.sqrt((w ** 2).sum(-1)), 1e-10)
    return ((w / nrm[..., None]) @ (O.hadamard(128).astype(np.float64) * math.sqrt(128))).reshape(n, kp)


def check_codes(got: np.ndarray, want: np.ndarray, w: np.ndarray, bits: int, what: str) -> int:
    got = np.asarray(got).astype(np.int64)
    want = np.asarray(want).astype(np.int64)
    assert got.shape == want.shape, what
    bad = np.argwhere(got != want)
    if len(bad):
        r = rotated(w)
        ct = O.get_centroids(bits).astype(np.float64)
        for i, j in bad:
            da = abs(r[i, j] - ct[got[i, j]])
            db = abs(r[i, j] - ct[want[i, j]])
            assert abs(da - db) <= TIE_TOL, (f"{what}: code ({i},{j}) {got[i, j]} vs {want[i, j]} "
                                             f"is not a near-tie (|d| {da:.3e} vs {db:.3e})")
    assert len(bad) <= max(2, got.size // 10000), f"{what}: {len(bad)} near-tie flips"
    return len(bad)


def check_norms(got: np.ndarray, want: np.ndarray, what: str) -> None:
    g = np.asarray(got).view(np.uint16).astype(np.int64)
    w = np.asarray(want).view(np.uint16).astype(np.int64)
    diff = np.abs(g - w)
    assert diff.max() <= 1, f"{what}: fp16 norm off by {diff.max()} ulp"
    assert (diff != 0).mean() <= 1e-3, f"{what}: {(diff != 0).sum()} norms off by 1 ulp"


@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6])
def test_quantizer_matches_reference_golden(golden, bits):
    from polarengine_vllm.quantizer import PolarQuantizer
    _say(f"quantize golden bits={bits}")
    w = golden["quant_w"]
    q = PolarQuantizer(128).quantize_tensor(torch.from_numpy(w).to(DEV), bits)
    torch.cuda.synchronize()
    check_codes(q["codes"].cpu().numpy(), golden[f"quant_codes_b{bits}"], w.astype(np.float32),
                bits, f"golden b{bits}")
    check_norms(q["norms"].cpu().numpy(), golden[f"quant_norms_b{bits}"], f"golden b{bits}")
    assert np.array_equal(q["ct_scaled"].cpu().numpy(), golden[f"quant_ct_scaled_b{bits}"])


@pytest.mark.parametrize("n,k,bits,dt", [(64, 4096, 4, torch.float16), (333, 1000, 3, torch.float32),
                                         (128, 384, 5, torch.bfloat16), (96, 2048, 6, torch.float16),
                                         (17, 130, 2, torch.float32), (512, 1408, 8, torch.float16)])
def test_quantizer_matches_oracle(n, k, bits, dt):
    from polarengine_vllm.quantizer import PolarQuantizer
    _say(f"quantize n={n} k={k} bits={bits} dt={dt}")
    w16 = O.seeded_normal((n, k), 0.02, n + k + bits)
    wt = torch.from_numpy(w16.astype(np.float32)).to(dt)
    w = wt.float().numpy()  # the values the kernel sees
    q = PolarQuantizer(128).quantize_tensor(wt.to(DEV), bits)
    torch.cuda.synchronize()
    want = O.quantize_tensor(w, bits)
    flips = check_codes(q["codes"].cpu().numpy(), want["codes"], w, bits, f"{n}x{k} b{bits}")
    check_norms(q["norms"].cpu().numpy(), want["norms"], f"{n}x{k} b{bits}")
    np.testing.assert_array_equal(q["ct_scaled"].cpu().numpy(), want["ct_scaled"])
    print(f"near-tie flips: {flips}")


@pytest.mark.parametrize("bits", [2, 3, 4])
def test_quantizer_packed_output(bits):
    """pack=True writes exactly the nibbles of the int8 codes."""
    from polarengine_vllm.quantizer import PolarQuantizer
    _say(f"quantize packed bits={bits}")
    w = torch.from_numpy(O.seeded_normal((200, 1536), 0.02, 5 + bits)).to(DEV)
    qz = PolarQuantizer(128)
    q = qz.quantize_tensor(w, bits)
    qp = qz.quantize_tensor(w, bits, pack=True)
    torch.cuda.synchronize()
    assert qp["codes"].dtype == torch.uint8 and tuple(qp["codes"].shape) == (200, 768)
    assert np.array_equal(qp["codes"].cpu().numpy(), O.pack_nibble(q["codes"].cpu().numpy()))
    assert torch.equal(qp["norms"], q["norms"])


def test_quantizer_roundtrip_quality_and_plugin():
    """Quantize on the GPU, run the plugin's linear, compare with the dense
    product (the format's approximation) and with the oracle (the kernels)."""
    from polarengine_vllm.linear_method import PolarQuantLinearMethod
    from polarengine_vllm.quantizer import PolarQuantizer
    _say("quantize -> linear")
    w = O.seeded_normal((768, 2048), 0.02, 77).astype(np.float32)
    q = PolarQuantizer(128).quantize_tensor(torch.from_numpy(w).to(DEV), 4)
    deq = O.dequant_weight(q["codes"].cpu().numpy(), q["norms"].cpu().numpy(),
                           q["ct_scaled"].cpu().numpy())
    cos = float((deq * w).sum() / (np.linalg.norm(deq) * np.linalg.norm(w)))
    assert cos > 0.99, f"Q4 reconstruction cosine {cos}"
    meth = PolarQuantLinearMethod(bits=4)
    layer = torch.nn.Module()
    meth.create_weights(layer, 2048, [768], 2048, 768, torch.float16)
    layer.to(DEV)
    layer.codes.copy_(q["codes"])
    layer.norms.copy_(q["norms"])
    meth.process_weights_after_loading(layer)
    x = O.seeded_normal((5, 2048), 1.0, 78)
    y = meth.apply(layer, torch.from_numpy(x).to(DEV)).float().cpu().numpy()
    want = O.linear_apply(x, q["codes"].cpu().numpy(), q["norms"].cpu().numpy(),
                          q["ct_scaled"].cpu().numpy(), 2048)
    err = np.abs(y - want).max() / np.abs(want).max()
    assert err <= 1e-2, err


def test_quantize_rejects_bad_arguments():
    from polarengine_vllm import _lib
    L = _lib.lib()
    w = torch.zeros(4, 256, device=DEV, dtype=torch.float16)
    ct = torch.zeros(32, device=DEV)
    c = torch.zeros(4, 256, dtype=torch.int8, device=DEV)
    nr = torch.zeros(4, 2, dtype=torch.float16, device=DEV)
    st = _lib.stream_ptr(torch.device(DEV))
    assert L.pe_quantize(w.data_ptr(), 0, 4, 256, 256, ct.data_ptr(), 32, 1, c.data_ptr(),
                         nr.data_ptr(), st) == _lib.PE_ERR_BITS  # nibbles need <= 16 levels
    assert L.pe_quantize(w.data_ptr(), 0, 4, 256, 100, ct.data_ptr(), 32, 0, c.data_ptr(),
                         nr.data_ptr(), st) == _lib.PE_ERR_DIMS  # ldw < K
    assert L.pe_quantize(w.data_ptr(), 7, 4, 256, 256, ct.data_ptr(), 32, 0, c.data_ptr(),
                         nr.data_ptr(), st) == _lib.PE_ERR_DTYPE
    assert L.pe_quantize(None, 0, 4, 256, 256, ct.data_ptr(), 32, 0, c.data_ptr(),
                         nr.data_ptr(), st) == _lib.PE_ERR_NULL


def _by_cell(ct: np.ndarray) -> bool:
    """Whether every two thresholds (midpoints of neighbouring levels) lie in
    cells of their own: the kernel's 1024-cell table, cells of a power of two w
    such that the outermost threshold is at most 510 cells out."""
    thr = (ct[1:].astype(np.float64) + ct[:-1]) / 2
    w = 2.0 ** math.frexp(np.abs(thr).max() / 510)[1]
    return len(set(np.rint(thr / w))) == len(thr)


@pytest.mark.parametrize("levels", [2, 4, 8, 16, 64, 100, 128, 255])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,k,pad", [(67, 1024, 0), (33, 1000, 8), (5, 131, 0), (40, 260, 3)])
def test_quantize_by_cell_equals_scan(levels, dt, n, k, pad):
    """The codes by cell against the scan over the centroids (which a codebook
    that repeats its last level takes: the repeated level is never the first
    nearest): codes and norms bit for bit, with zero blocks, tiny and huge
    values, infinities and NaN, aligned and unaligned rows."""
    from polarengine_vllm import _lib
    _say(f"quantize by cell levels={levels} {dt} {n}x{k} ld +{pad}")
    g = torch.Generator().manual_seed(levels * 7 + k)
    w = torch.randn(n, k + pad, generator=g, dtype=torch.float64) * 0.02
    w[0], w[1, :5] = 0.0, float("nan")
    w[2, 3], w[3] = float("inf"), w[3] * 1e-30
    w[4] = w[4] * 1e6
    w[4, 64:], w[4, 7] = 1e-39, 3e-25
    if n > 8:
        w[5] = w[5] * 1e30 if dt != torch.float16 else w[5] * 1e6
        w[6] = torch.randint(-2, 3, (k + pad,), generator=g).double()  # many ties
        w[7] = w[7] * 1e-8
    w = w.to(dt).to(DEV)
    ct = torch.sort(torch.randn(levels, generator=g) * 1.5).values
    if levels not in (2, 8):  # the first levels of the smallest codebook that has so many
        ct = torch.from_numpy(O.get_centroids(math.ceil(math.log2(levels))).astype(np.float32))[:levels]
    assert _by_cell(ct.numpy())  # and one more level, a repeated one, takes the scan
    nb = (k + 127) // 128
    dtc = {torch.float16: 0, torch.bfloat16: 1, torch.float32: 2}[dt]
    out = []
    for c in (ct, torch.cat([ct, ct[-1:]])):
        c = c.to(DEV).contiguous()
        for pack in ([0, 1] if c.numel() <= 16 else [0]):
            codes = torch.full((n, nb * (64 if pack else 128)), 255, dtype=torch.uint8, device=DEV)
            norms = torch.empty(n, nb, dtype=torch.float16, device=DEV)
            _lib.check(_lib.lib().pe_quantize(w.data_ptr(), dtc, n, k, w.stride(0), c.data_ptr(),
                                              c.numel(), pack, codes.data_ptr(), norms.data_ptr(),
                                              _lib.stream_ptr(torch.device(DEV))), "pe_quantize")
            if pack:
                lo, hi = codes.view(n, nb, 64) & 15, codes.view(n, nb, 64) >> 4
                codes = torch.cat([lo, hi], -1).reshape(n, -1)
            out.append((codes.cpu(), norms.view(torch.int16).cpu()))
    for codes, norms in out[1:]:
        assert torch.equal(norms, out[0][1])
        assert torch.equal(codes, out[0][0])


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,k", [(32769, 128), (98400, 128), (17001, 384), (7003, 1160), (9001, 500),
                                 (2049, 5000)])
def test_quantize_more_blocks_than_one_step(dt, n, k):
    """More blocks than the grid takes in one step (32768 on 256 CUs), block
    counts that do not divide the step, a ragged last step: rows that repeat
    give the codes and norms of the rows, bit for bit."""
    from polarengine_vllm.quantizer import PolarQuantizer
    _say(f"quantize strided {dt} {n}x{k}")
    g = torch.Generator().manual_seed(n + k)
    base = (torch.randn(97, k, generator=g) * 0.02).to(dt).to(DEV)
    rows = torch.arange(n, device=DEV) % 97
    want = PolarQuantizer(128).quantize_tensor(base, 4)
    got = PolarQuantizer(128).quantize_tensor(base[rows], 4)
    for key in ("codes", "norms"):
        assert torch.equal(got[key], want[key][rows]), key
