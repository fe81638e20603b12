"""Many-row tile16 GEMM (more than 64 rows) against the float64 product of the oracle's decoded weights.

Tolerance: each weight is rounded once to fp16 (at most 2^-11 of it) and each output once (2^-11 of it), so the
2-norm of the error stays below 2^-10 of the result's."""

import numpy as np
import pytest

from oracle import formats as fm

pytestmark = pytest.mark.gpu
REL = 2.0 ** -10


def _pack(rng, N, K, group):
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float16)
    if group == 128:
        p, s = fm.pack_linear_q4_marlin_g128(w)
    else:
        p, s = fm.pack_linear_q4_marlin(w, clip_search=False)
    q = fm.unpack_marlin_codes(p).astype(np.float64).reshape(p.shape[0] * 8, K // group, group)
    sb = s.transpose(0, 2, 1, 3).reshape(p.shape[0] * 8, K // group, 2).astype(np.float64)
    return p, s, (q * sb[..., 0:1] + sb[..., 1:2]).reshape(-1, K)[:N]


def _tile16(dev, p, s, N, K):
    import torch

    from axiomlm_amd.kernels import repack_q4_marlin_tile16

    return repack_q4_marlin_tile16(torch.from_numpy(p).to(dev), torch.from_numpy(s).to(dev), N, K)


# Tile edges: 64- and 128-row tiles with remainders, weight tiles that do not fill a wave (16 rows) or a workgroup,
# N not a multiple of 16 / 4, one stage, half a stage, odd and even stage counts, split and unsplit K.
@pytest.mark.parametrize("M,N,K,group", [(65, 16, 64, 64), (65, 1000, 704, 64), (96, 264, 4096, 64),
                                         (128, 72, 128, 128), (129, 2056, 384, 128), (200, 1002, 320, 64),
                                         (1031, 520, 512, 64)])
def test_rows_gemm_matches_oracle(dev, M, N, K, group):
    import torch

    from axiomlm_amd.kernels import qmv_q4_tile16

    rng = np.random.default_rng(M + N + K)
    p, s, w = _pack(rng, N, K, group)
    # What follows the rows in memory, and each row's successor, must not reach a row's sums
    # (K % 128 == 64 reads half a stage past the row).
    buf = torch.full((M * K + 256,), float("inf"), dtype=torch.float16, device=dev)
    x = rng.standard_normal((M, K)).astype(np.float16)
    x[M // 2, :64] = np.inf
    buf[: M * K] = torch.from_numpy(x.reshape(-1)).to(dev)
    bias = rng.standard_normal(N).astype(np.float16)
    y = qmv_q4_tile16(buf[: M * K].view(M, K), *_tile16(dev, p, s, N, K), N, torch.from_numpy(bias).to(dev))
    keep = np.arange(M) != M // 2
    ref = x[keep].astype(np.float64) @ w.T + bias.astype(np.float64)
    got = y.cpu().numpy()[keep].astype(np.float64)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - ref) <= REL * np.linalg.norm(ref) * 2  # the bias is a second fp16 rounding


@pytest.mark.parametrize("M,H,K,group", [(65, 16, 64, 64), (100, 720, 704, 64), (130, 1040, 256, 128), (70, 48, 4096, 64)])
def test_rows_gemm_swiglu_matches_oracle(dev, M, H, K, group):
    import torch

    from axiomlm_amd.kernels import qmv_q4_tile16_swiglu

    rng = np.random.default_rng(M + H + K)
    p, s, w = _pack(rng, 2 * H, K, group)
    x = rng.standard_normal((M, K)).astype(np.float16)
    y = qmv_q4_tile16_swiglu(torch.from_numpy(x).to(dev), None, 1e-5, *_tile16(dev, p, s, 2 * H, K), H)
    g, u = np.split(x.astype(np.float64) @ w.T, 2, axis=1)
    ref = g / (1 + np.exp(-g)) * u
    # gate, up, silu and the product each round to fp16, weights as above (silu's slope is below 1.1)
    assert np.linalg.norm(y.cpu().numpy().astype(np.float64) - ref) <= 4 * REL * np.linalg.norm(ref)


def test_rows_gemm_workspace_is_optional(dev):
    """Less workspace than preferred means fewer K splits (none without it), never an error."""
    import torch

    from axiomlm_amd import _lib

    rng = np.random.default_rng(3)
    M, N, K = 70, 64, 4096
    p, s, w = _pack(rng, N, K, 64)
    w16, sb16 = _tile16(dev, p, s, N, K)
    x = rng.standard_normal((M, K)).astype(np.float16)
    xd = torch.from_numpy(x).to(dev)
    want = _lib.lib().axm_qmm_q4_tile16_rows_workspace_bytes(M, K, N, 0)
    one = M * N * 4
    assert want >= 2 * one
    ref = x.astype(np.float64) @ w.T
    for size in (0, one, 2 * one + 12, want):
        ws = torch.empty(max(size, 16), dtype=torch.uint8, device=dev)
        y = torch.empty(M, N, dtype=torch.float16, device=dev)
        _lib.check(_lib.lib().axm_qmm_q4_tile16(xd.data_ptr(), w16.data_ptr(), sb16.data_ptr(), None, y.data_ptr(), M, K,
                                                N, 64, ws.data_ptr() if size else None, size, _lib.stream_of(dev)),
                   "qmm_q4_tile16")
        assert np.linalg.norm(y.cpu().numpy().astype(np.float64) - ref) <= REL * np.linalg.norm(ref)


@pytest.mark.parametrize("skip", [4, 1])
@pytest.mark.parametrize("swiglu", [False, True])
def test_rows_of_a_misaligned_view(dev, skip, swiglu):
    """Rows that start 8 or 2 bytes past a 16-byte boundary (contiguous: nothing copies them) run in passes of 64, also
    where the many-row GEMM would want no workspace (unsplit) and the passes split K."""
    import torch

    from axiomlm_amd import _lib
    from axiomlm_amd.kernels import qmv_q4_tile16, qmv_q4_tile16_swiglu

    M, N, K = 130, 4096, 1024
    L = _lib.lib()
    assert L.axm_qmm_q4_tile16_rows_workspace_bytes(M, K, N, 0) >= L.axm_qmm_q4_tile16_workspace_bytes(K, N, 0) > 0
    rng = np.random.default_rng(skip)
    p, s, w = _pack(rng, N, K, 64)
    x = rng.standard_normal((M, K)).astype(np.float16)
    buf = torch.empty(skip + M * K, dtype=torch.float16, device=dev)
    buf[skip:] = torch.from_numpy(x.reshape(-1)).to(dev)
    xd = buf[skip:].view(M, K)
    assert xd.data_ptr() % 16 == 2 * skip
    y = x.astype(np.float64) @ w.T
    if swiglu:
        got = qmv_q4_tile16_swiglu(xd, None, 1e-5, *_tile16(dev, p, s, N, K), N // 2)
        g, u = np.split(y, 2, axis=1)
        y = g / (1 + np.exp(-g)) * u
    else:
        got = qmv_q4_tile16(xd, *_tile16(dev, p, s, N, K), N)
    # bounds as for the aligned rows
    assert np.linalg.norm(got.cpu().numpy().astype(np.float64) - y) <= (4 if swiglu else 1) * REL * np.linalg.norm(y)
