"""GPU parity of the many-token dense GEMMs: the resident linear and the MX
shared expert over a prompt's tokens (DeferredLinear.__call__, layers.py:38-70;
DenseMLP, layers.py:160-171) against the oracle, at the edges of their tiles:
token tiles of 32 to 128, weight rows in 16-row blocks that do not fill a
64-, 128- or 256-row tile, and one to many K chunks (fewer than the stages of
the LDS ring, odd counts, bf16's 64-wide chunks)."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import moe_oracle as O
from livglm_amd import native

pytestmark = pytest.mark.gpu

REL_L2 = 2e-3  # the layer bar: one bf16 rounding of an f32 sum
FMTS = [native.GLM_FMT_MXFP8, native.GLM_FMT_MXFP4, native.GLM_FMT_BF16]


@pytest.fixture(scope="module")
def gu():
    import gpu_util
    native.load()
    return gpu_util


def _weights(gu, rng, rows, cols, fmt):
    """(f32 values, device codes or bf16, device scales or None)"""
    w = O.f32_to_bf16_bits(rng.normal(0, 0.02, (rows, cols)).astype(np.float32))
    if fmt == native.GLM_FMT_BF16:
        return O.bf16_bits_to_f32(w), gu.to_dev(w), None
    c, s = O.quantize_mx(w, 8 if fmt == native.GLM_FMT_MXFP8 else 4, O.MX_RULE_NEAREST)
    deq = O.dequant_mxfp8 if fmt == native.GLM_FMT_MXFP8 else O.dequant_mxfp4
    return deq(c, s), gu.to_dev(c), gu.to_dev(s)


def _check(got, want):
    assert O.rel_l2(got, want) < REL_L2
    assert np.mean(got == want) > 0.97


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("T,N,K", [
    (65, 16, 128), (65, 272, 256), (96, 144, 384), (127, 528, 512), (128, 256, 640),
    (129, 304, 896), (300, 2064, 128), (520, 1040, 1152),
    # tiles of 256 rows x 96 and 128 tokens: grids near one workgroup per CU
    (1500, 4096, 256), (2100, 4000, 384),
    # 64-row weight tiles of 32 and 64 tokens (MXFP8 from 49 tokens on, bf16)
    (49, 1040, 256), (64, 80, 1152), (100, 2048, 512), (128, 4064, 128), (190, 3984, 256),
    # no K split for the streaming tiles: few tokens come here too
    (5, 256, 640), (16, 80, 3328),
])
def test_dense_linear_parity(gu, fmt, T, N, K):
    import torch
    rng = np.random.default_rng(900 + T + N + K)
    mat, codes, scales = _weights(gu, rng, N, K, fmt)
    x = O.f32_to_bf16_bits(rng.normal(0, 1, (T, K)).astype(np.float32))
    # guard rows around the output: nothing outside it may be written
    y = torch.full((T + 2, N), 7.0, dtype=torch.bfloat16, device="cuda")
    gu.call("glm_linear", gu.stream(), gu.p(gu.to_dev(x)), T, K, gu.p(codes), gu.p(scales), fmt, N,
            y[1:].data_ptr())
    got = O.bf16_bits_to_f32(gu.bf16_bits(y))
    _check(got[1:-1], O.linear_bf16(O.bf16_bits_to_f32(x), mat))
    assert np.all(got[0] == 7.0) and np.all(got[-1] == 7.0)


@pytest.mark.parametrize("fmt", [native.GLM_FMT_BF16, native.GLM_FMT_MXFP8])
def test_dense_linear_bf16_half_chunks_and_unaligned_scales(gu, fmt):
    # K = 192 is whole 64-wide chunks (bf16); MXFP8 scales that start off a
    # 4-byte boundary stay on the streaming tiles and give the same result
    import torch
    rng = np.random.default_rng(77)
    T, N, K = 70, 96, 192 if fmt == native.GLM_FMT_BF16 else 256
    mat, codes, scales = _weights(gu, rng, N, K, fmt)
    if scales is not None:
        moved = torch.empty(scales.numel() + 1, dtype=torch.uint8, device="cuda")[1:]
        moved.copy_(scales.reshape(-1))
        scales = moved
    x = O.f32_to_bf16_bits(rng.normal(0, 1, (T, K)).astype(np.float32))
    y = torch.empty((T, N), dtype=torch.bfloat16, device="cuda")
    gu.call("glm_linear", gu.stream(), gu.p(gu.to_dev(x)), T, K, gu.p(codes), gu.p(scales), fmt, N,
            gu.p(y))
    _check(O.bf16_bits_to_f32(gu.bf16_bits(y)), O.linear_bf16(O.bf16_bits_to_f32(x), mat))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("T,d,I", [(65, 384, 160), (130, 512, 640), (200, 640, 1024), (3, 640, 640)])
def test_dense_mlp_many_tokens_parity(gu, fmt, T, d, I):
    import torch
    rng = np.random.default_rng(40 + T)
    ws = [_weights(gu, rng, *s, fmt) for s in ((I, d), (I, d), (d, I))]
    x = O.f32_to_bf16_bits(rng.normal(0, 1, (T, d)).astype(np.float32))
    h = torch.empty((T, I), dtype=torch.bfloat16, device="cuda")
    out = torch.empty((T, d), dtype=torch.bfloat16, device="cuda")
    gu.call("glm_dense_mlp", gu.stream(), gu.p(gu.to_dev(x)), T, d, I, fmt,
            *(gu.p(t) for w in ws for t in w[1:]), 10.0, gu.p(h), gu.p(out))
    _check(O.bf16_bits_to_f32(gu.bf16_bits(out)),
           O.dense_mlp(O.bf16_bits_to_f32(x), *(w[0] for w in ws), 10.0))
