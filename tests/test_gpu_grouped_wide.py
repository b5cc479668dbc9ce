"""GPU parity of whole layers on the wide grouped GEMMs (many rows per expert,
native_expert_ssd.py:726-743) against the oracle: row tiles partial and full,
experts of several tiles, widths that leave half of the last gate/up feature
tile empty (I an odd multiple of 128, so the down GEMM has an odd count of K
chunks), the bf16 shared expert's tiles behind the routed ones in one launch,
shared experts that run by themselves, and none.  Every test says which path
its layer takes, so that a line of the dispatch that moves does not take the
tests along."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import moe_oracle as O
from livglm_amd import native
from livglm_amd.workloads import MoEShape, make_layer

from test_gpu_grouped_stream import REL_L2, _oracle, _shared_weights, gu  # noqa: F401 (fixture)
from test_gpu_parity import _check_indices

pytestmark = pytest.mark.gpu

BF16, MXFP8, MXFP4 = native.GLM_FMT_BF16, native.GLM_FMT_MXFP8, native.GLM_FMT_MXFP4


def _check(gu, shape, layer, fmt, path="wide"):  # noqa: F811
    """Runs the layer and compares it; returns (its output, the oracle's, the
    rows whose route agrees, the oracle's indices)."""
    how = dict(shared=fmt is not None, shared_fmt=BF16 if fmt is None else fmt)
    assert gu.layer_path(shape, **how) == path
    want, inter = _oracle(layer, shape, _shared_weights(layer, fmt))
    out, w, idx = gu.run_layer(gu.upload_layer(layer), shape, **how)
    got_idx = gu.host(idx).astype(np.uint32)
    _check_indices(got_idx, inter["indices"], inter["choice"], shape.k)
    same = np.all(got_idx == inter["indices"], axis=1)
    assert same.mean() > 0.99
    np.testing.assert_allclose(gu.host(w)[same], inter["weights"][same], rtol=2e-6, atol=1e-7)
    return gu.host(out), want, same, inter["indices"]


def _close(got, want, same):
    assert O.rel_l2(got[same], want[same]) < REL_L2
    # no row of any tile is off on its own
    rows = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert rows[same].max() < 5 * REL_L2


@pytest.mark.parametrize("T,d,E,k,I,Is,fmt", [
    # I 896 and 640: the last feature tile half empty; the shared expert riding
    # (partial in tokens; Is as wide and narrow), none, and in MX by itself
    (720, 512, 64, 8, 896, 896, BF16), (720, 512, 64, 8, 896, 128, BF16), (720, 512, 64, 8, 896, 0, None),
    (720, 512, 64, 8, 896, 256, MXFP8), (980, 512, 88, 8, 640, 640, BF16), (980, 512, 88, 8, 640, 0, None),
    (980, 512, 88, 8, 640, 384, MXFP4),
    # I 128: the first feature tile too
    (2850, 512, 256, 8, 128, 128, BF16), (2850, 512, 256, 8, 128, 0, None), (2850, 512, 256, 8, 128, 128, MXFP4),
    # whole feature tiles; a shared width that cannot ride
    (1450, 512, 128, 8, 512, 512, BF16), (1450, 512, 128, 8, 512, 96, BF16), (1450, 1024, 128, 8, 384, 256, MXFP8),
    # 200 rows an expert: two tiles of most
    (1600, 512, 64, 8, 896, 256, BF16),
])
def test_wide_layer(gu, T, d, E, k, I, Is, fmt):  # noqa: F811
    shape = MoEShape("wide", T, d, E, k, I, Is)
    _close(*_check(gu, shape, make_layer(shape, 7700 + T + I + Is), fmt)[:3])


@pytest.mark.parametrize("I,fmt", [(896, BF16), (768, None)])
def test_wide_layer_skewed_routing(gu, I, fmt):  # noqa: F811
    # Zipf-biased routing: experts of several full row tiles beside experts of
    # one partial tile
    shape = MoEShape("skew", 1500, 512, 88, 8, I, 256, routing="zipf")
    got, want, same, idx = _check(gu, shape, make_layer(shape, 7800 + I), fmt)
    counts = np.bincount(idx.reshape(-1).astype(np.int64), minlength=shape.E)
    assert counts.max() > 3 * 160 and counts.min() < 100
    _close(got, want, same)


@pytest.mark.parametrize("I,fmt", [(896, BF16), (768, None)])
def test_wide_layer_nan_gate_scale(gu, I, fmt):  # noqa: F811
    # a NaN scale byte in one expert's gate row: every output of the tokens
    # routed to it is NaN (through the split that the gate/up epilogue writes),
    # no other is
    shape = MoEShape("nan", 1000, 512, 88, 8, I, 128)
    layer = make_layer(shape, 7900 + I)
    layer["gate_proj.weight_scale"][3, I - 3, 1] = 255
    got, want, same, idx = _check(gu, shape, layer, fmt)
    hit = (idx == 3).any(axis=1)
    assert hit.any() and not hit.all() and np.array_equal(np.isnan(want).all(axis=1), hit)
    assert np.array_equal(np.isnan(got[same]), np.isnan(want[same]))
    _close(got, want, same & ~hit)


def test_router_behind_its_own_weight_split(gu):  # noqa: F811
    # from 256 tokens and 96 M products on the router multiplies bf16 parts of
    # its weights; on the bf16 streaming path no split of x carries theirs along
    shape = MoEShape("router", 400, 1024, 256, 8, 128, 128)
    assert shape.T * shape.d * shape.E > 96 << 20
    _close(*_check(gu, shape, make_layer(shape, 8000), BF16, path="stream_bf16")[:3])
