"""Several-row GEMM over Q8_G64, MARLIN Q4, ternary, affine and GGUF 2-bit codes against the float64 product of the
decoded codes.

Code products are exact and sums fp32, so the result is the float64 one to the fp16 rounding of the output: 2^-11 of
each value at most, plus fp32 sums whose error (2^-24 of the sum of magnitudes per add) matters only where a row's
terms cancel; 1.05 x 2^-11 in the 2-norm covers both."""

import numpy as np
import pytest
import torch

from oracle import formats as fm

pytestmark = pytest.mark.gpu
REL = 1.05 * 2.0 ** -11


def _decode_marlin(p, s, K):
    """float64 rows of the 8-row tiles, padding rows included."""
    q = fm.unpack_marlin_codes(p).astype(np.float64).reshape(-1, K // 64, 64)
    sb = s.transpose(0, 2, 1, 3).reshape(-1, K // 64, 2).astype(np.float64)
    return (q * sb[..., 0:1] + sb[..., 1:2]).reshape(-1, K)


def _packed(fmt, rng, N, K):
    """(device arrays, float64 weights)"""
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float16)
    if fmt == "q8":
        p, s = fm.pack_linear_q8_g64(w)
        q = p.reshape(N, K // 64, 64).astype(np.float64)
        return (p.view(np.int32).reshape(N, K // 4), s), (q * s[..., 0:1] + s[..., 1:2].astype(np.float64)).reshape(N, K)
    if fmt == "marlin":
        p, s = fm.pack_linear_q4_marlin(w, clip_search=False)
        return (p, s), _decode_marlin(p, s, K)[:N]
    if fmt == "ternary":
        p, s = fm.pack_linear_ternary(w)
        q = fm.ternary_decode_bytes(p).reshape(N, K // 64, 64).astype(np.float64)
        return (p, s), (q * s[..., None]).reshape(N, K)
    if fmt == "gguf":
        b = fm.pack_q2_k_gguf(w)
        at, shift, sub = fm.q2k_element_maps()
        q = ((b[:, :, 16:80][:, :, at] >> shift) & 3).astype(np.float64)
        sc = b[:, :, :16][:, :, sub]
        d, dmin = (b[:, :, o:o + 2].copy().view(np.float16).astype(np.float64) for o in (80, 82))
        return (b, b), (d * (sc & 15) * q - dmin * (sc >> 4)).reshape(N, K)
    p, s = fm.pack_linear_q2_k(w)
    q = ((p[..., None] >> (2 * np.arange(4))) & 3).reshape(N, K // 64, 64).astype(np.float64)
    return (p, s), (q * s[..., 0:1] + s[..., 1:2].astype(np.float64)).reshape(N, K)


def _run(fmt, x, packs, N, bias=None, ws=True):
    """The several-row entry itself (the Python wrappers choose by size)."""
    from axiomlm_amd import _lib

    L = _lib.lib()
    M, K = x.shape
    fn = {"q8": L.axm_qmm_q8_g64, "marlin": L.axm_qmm_q4_marlin, "ternary": L.axm_qmm_ternary, "q2": L.axm_qmm_q2_k,
          "gguf": L.axm_qmm_q2_k_gguf}[fmt]
    weights = [_lib.ptr(p) for p in (packs[:1] if fmt == "gguf" else packs)]
    y = torch.empty((M, N), dtype=torch.float16, device=x.device)
    n = L.axm_qmm_codes_workspace_bytes({"q8": 0, "q2": 1, "ternary": 2, "gguf": 3, "marlin": 4}[fmt], M, K, N) if ws else 0
    buf = torch.empty(max(n, 1), dtype=torch.uint8, device=x.device)
    _lib.check(fn(_lib.ptr(x), *weights, _lib.ptr(bias), _lib.ptr(y), M, K, N,
                  _lib.ptr(buf) if n else None, n, _lib.stream_of(x.device)), fmt)
    return y


# Row tiles of 16 - 64 with remainders, two and four weight tiles per wave (the last: four), several row blocks, weight
# tiles past N, one and two stages, odd and even counts, half a stage, split and unsplit K; 2-bit sizes beyond what their
# GEMV launches take.
SHAPES = [(5, 16, 64), (7, 24, 192), (16, 1000, 704), (33, 72, 128), (48, 264, 4096), (64, 96, 8192), (70, 130, 320),
          (129, 2056, 1024), (17, 40, 192),
          (930, 12280, 128)]


@pytest.mark.parametrize("fmt", ["q8", "marlin", "ternary", "q2", "gguf"])
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("ws", [True, False])
def test_codes_gemm_matches_float64(dev, fmt, M, N, K, ws):
    if fmt not in ("q8", "marlin"):
        M += 64  # four launches of 16 rows and more
    if fmt == "gguf":
        K = (K + 255) // 256 * 256
    rng = np.random.default_rng(M + N + K)
    packs, w = _packed(fmt, rng, N, K)
    packs = [torch.from_numpy(a).to(dev) for a in packs]
    x = rng.standard_normal((M, K)).astype(np.float16)
    x[:, : K // 2] += 1  # group sums far from zero: the bias term counts
    bad = M // 3
    x[bad, :64] = np.inf  # this row only: row bad - 1's last half stage is followed by it in memory
    buf = torch.full((M * K + 256,), float("inf"), dtype=torch.float16, device=dev)
    buf[: M * K] = torch.from_numpy(x.reshape(-1)).to(dev)
    bias = rng.standard_normal(N).astype(np.float16)
    keep = np.arange(M) != bad
    ref = x[keep].astype(np.float64) @ w.T
    got = _run(fmt, buf[: M * K].view(M, K), packs, N, None, ws).cpu().numpy()[keep].astype(np.float64)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - ref) <= REL * np.linalg.norm(ref)
    got = _run(fmt, buf[: M * K].view(M, K), packs, N, torch.from_numpy(bias).to(dev), ws).cpu().numpy()[keep]
    # a second fp16 rounding
    assert np.linalg.norm(got.astype(np.float64) - (ref + bias)) <= 2 * REL * np.linalg.norm(ref + bias)


@pytest.mark.parametrize("fmt", ["ternary", "q2", "gguf"])
@pytest.mark.parametrize("N", [64, 70])
@pytest.mark.parametrize("ws", [True, False])
def test_codes_gemm_bias_joins_the_fp32_sum(dev, fmt, N, ws):
    """A bias that cancels the fp16 product leaves what that rounding would have dropped: the 2-bit formats round
    once, after the bias.  Rounding before it would leave about 2^-13 of the product (its own rounding, rms); the
    bound is the final rounding and the fp32 sums: K / 32 matrix-core adds and eight more, rounding at random, each
    2^-24 of at most the sum of magnitudes, a weight's code and bias parts taken as three times the weight."""
    M, K = 80, 512
    rng = np.random.default_rng(N)
    packs, w = _packed(fmt, rng, N, K)
    x = rng.standard_normal((M, K)).astype(np.float16)
    ref = x.astype(np.float64) @ w.T
    bias = -ref[7].astype(np.float16)
    got = _run(fmt, torch.from_numpy(x).to(dev), [torch.from_numpy(a).to(dev) for a in packs], N,
               torch.from_numpy(bias).to(dev), ws).cpu().numpy()[7].astype(np.float64)
    want = ref[7] + bias
    sums = 3 * np.abs(x[7].astype(np.float64)) @ np.abs(w).T
    bound = 2.0 ** -11 * np.linalg.norm(want) + np.sqrt(K / 32 + 8) * 2.0 ** -24 * np.linalg.norm(sums)
    assert bound < 2.0 ** -14 * np.linalg.norm(ref[7])  # below what the extra rounding would leave
    assert np.linalg.norm(got - want) <= bound


@pytest.mark.parametrize("fmt", ["q8", "marlin", "q2", "gguf"])
def test_codes_gemm_bias_term_over_the_fp16_range(dev, fmt):
    """Group sums beyond the fp16 range and activations near its bottom keep 24 bits in the bias term."""
    rng = np.random.default_rng(1)
    N, K, M = 32, 512, 80
    packs, w = _packed(fmt, rng, N, K)
    packs = [torch.from_numpy(a).to(dev) for a in packs]
    for scale in (3000.0, 2.0 ** -18):
        x = (np.abs(rng.standard_normal((M, K))) * scale).astype(np.float16)
        wn = w
        if scale > 1 and fmt == "gguf":  # smaller d and dmin
            b = packs[0].cpu().numpy()
            d = (b[:, :, 80:84].copy().view(np.float16).astype(np.float32) * 2.0 ** -6).astype(np.float16)
            b[:, :, 80:84] = d.view(np.uint8)
            packs = [torch.from_numpy(b).to(dev)] * 2
            at, shift, sub = fm.q2k_element_maps()
            sc = b[:, :, :16][:, :, sub]
            d = d.astype(np.float64)
            wn = (d[:, :, :1] * (sc & 15) * ((b[:, :, 16:80][:, :, at] >> shift) & 3) - d[:, :, 1:] * (sc >> 4)).reshape(N, K)
        elif scale > 1:  # keep the results in range: smaller scales and biases, same codes
            packs[1] = (packs[1].double() * 2.0 ** -6).half()
            s = packs[1].cpu().numpy().astype(np.float64)
            p = packs[0].cpu().numpy()
            if fmt == "marlin":
                wn = _decode_marlin(p, s, K)
            else:
                codes = (p.view(np.uint8).reshape(N, K // 64, 64) if fmt == "q8" else
                         ((p[..., None] >> (2 * np.arange(4))) & 3).reshape(N, K // 64, 64)).astype(np.float64)
                wn = (codes * s[..., 0:1] + s[..., 1:2]).reshape(N, K)
        ref = x.astype(np.float64) @ wn.T
        got = _run(fmt, torch.from_numpy(x).to(dev), packs, N).cpu().numpy().astype(np.float64)
        # fp16 results: half a unit of the last place, which near the bottom of the range is 2^-25
        tol = np.maximum(np.abs(ref) * 2.0 ** -11, 2.0 ** -25) * 1.05 + 2.0 ** -20 * (np.abs(x.astype(np.float64)) @ np.abs(wn).T)
        assert np.isfinite(got).all() and (np.abs(got - ref) <= tol).all()
        packs, w = _packed(fmt, np.random.default_rng(1), N, K)
        packs = [torch.from_numpy(a).to(dev) for a in packs]


def test_wrappers_choose_the_same_result_on_both_sides(dev):
    """The Python products just below and above the rows at which the launch changes."""
    from axiomlm_amd.kernels import qmv_q2_k, qmv_q4_marlin, qmv_q8_g64, qmv_ternary

    rng = np.random.default_rng(5)
    for fmt, fn, rows, N, K in (("q8", qmv_q8_g64, (4, 5), 96, 320), ("q8", qmv_q8_g64, (5, 6, 7), 96, 1024),
                                ("ternary", qmv_ternary, (32, 33), 96, 320),
                                ("q2", qmv_q2_k, (32, 33), 96, 320), ("ternary", qmv_ternary, (8, 9), 8192, 4096),
                                ("marlin", qmv_q4_marlin, (4, 5), 96, 320),
                                ("marlin", qmv_q4_marlin, (1, 2, 4), 8192, 4096)):
        packs, w = _packed(fmt, rng, N, K)
        packs = [torch.from_numpy(a).to(dev) for a in packs]
        x = rng.standard_normal((rows[-1], K)).astype(np.float16)
        ref = x.astype(np.float64) @ w.T
        for M in rows:
            got = fn(torch.from_numpy(x[:M]).to(dev), *packs).cpu().numpy().astype(np.float64)
            assert np.linalg.norm(got - ref[:M]) <= REL * np.linalg.norm(ref[:M])


@pytest.mark.parametrize("fmt", ["ternary", "q2", "gguf"])
def test_codes_gemm_few_rows_of_a_large_matrix(dev, fmt):
    """2-bit row tiles of 16 and 32, taken where one GEMV launch no longer pays; N ends inside a tile."""
    N, K = 8200, 4096
    rng = np.random.default_rng(3)
    packs, w = _packed(fmt, rng, N, K)
    packs = [torch.from_numpy(a).to(dev) for a in packs]
    x = rng.standard_normal((40, K)).astype(np.float16)
    ref = x.astype(np.float32) @ w.astype(np.float32).T
    for M in (9, 16, 17, 31, 40):
        for ws in (True, False):
            got = _run(fmt, torch.from_numpy(x[:M]).to(dev), packs, N, None, ws).cpu().numpy()
            assert np.linalg.norm(got.astype(np.float32) - ref[:M]) <= REL * np.linalg.norm(ref[:M]), (M, ws)


def test_affine_2bit_infinite_activations(dev):
    """An infinite activation gives what the few-row kernel gives: infinity where its code is not zero and the group's
    bias has the code term's sign, else NaN (a zero code, or two infinities of opposite sign)."""
    rng = np.random.default_rng(8)
    N, K = 96, 256
    w = (np.abs(rng.standard_normal((N, K))) * 0.02 + 0.01).astype(np.float16)
    w[N // 2:] -= np.float16(0.03)  # biases below zero
    packs = [torch.from_numpy(a).to(dev) for a in fm.pack_linear_q2_k(w)]
    x = rng.standard_normal((80, K)).astype(np.float16)
    x[3, 70], x[5, 200], x[64, 1], x[79, 255] = np.inf, -np.inf, np.inf, np.inf
    xd = torch.from_numpy(x).to(dev)
    got = _run("q2", xd, packs, N).cpu().numpy()
    few = np.concatenate([_run("q2", xd[m:m + 16], packs, N).cpu().numpy() for m in range(0, 80, 16)])
    bad = np.array([3, 5, 64, 79])
    assert np.isinf(few[bad, :N // 2]).any() and np.isnan(few[bad]).any()
    assert np.array_equal(np.isnan(got), np.isnan(few))
    inf = np.isinf(few)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], few[inf])
    keep = np.setdiff1d(np.arange(80), bad)
    assert np.isfinite(got[keep]).all()


def test_infinite_scale_of_a_last_half_stage(dev):
    """K % 128 == 64: the half stage past K adds nothing, also to rows whose last scale is infinite."""
    rng = np.random.default_rng(9)
    N, K = 40, 320
    packs = list(_packed("ternary", rng, N, K)[0])
    packs[1] = packs[1].copy()
    packs[1].reshape(N, K // 64)[7, -1] = np.inf
    packs = [torch.from_numpy(a).to(dev) for a in packs]
    xd = torch.from_numpy(rng.standard_normal((80, K)).astype(np.float16)).to(dev)
    got = _run("ternary", xd, packs, N).cpu().numpy()
    few = np.concatenate([_run("ternary", xd[m:m + 16], packs, N).cpu().numpy() for m in range(0, 80, 16)])
    assert np.isinf(few[:, 7]).all() and np.array_equal(got[:, 7], few[:, 7])
    assert np.isfinite(np.delete(got, 7, 1)).all()


def test_gguf_infinite_activations(dev):
    """The same of GGUF blocks, whose two terms have one sign only where d and dmin have opposite ones."""
    rng = np.random.default_rng(10)
    N, K = 96, 512
    blocks = fm.pack_q2_k_gguf((rng.standard_normal((N, K)) * 0.02).astype(np.float16))
    blocks[N // 2:, :, 83] ^= 0x80  # dmin < 0
    packs = [torch.from_numpy(blocks).to(dev)]
    x = rng.standard_normal((80, K)).astype(np.float16)
    x[3, 70], x[5, 200], x[64, 300], x[79, 511] = np.inf, -np.inf, np.inf, np.inf
    xd = torch.from_numpy(x).to(dev)
    got = _run("gguf", xd, packs, N).cpu().numpy()
    few = np.concatenate([_run("gguf", xd[m:m + 16], packs, N).cpu().numpy() for m in range(0, 80, 16)])
    bad = np.array([3, 5, 64, 79])
    assert np.isinf(few[bad, N // 2:]).any() and np.isnan(few[bad]).any()
    assert np.array_equal(np.isnan(got), np.isnan(few))
    inf = np.isinf(few)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], few[inf])
    assert np.isfinite(np.delete(got, bad, 0)).all()
