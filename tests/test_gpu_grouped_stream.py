"""GPU parity of the layer's streaming grouped GEMMs (few rows per expert,
native_expert_ssd.py:726-743) against the oracle, at the edges of their row
tiles (experts of 0, 1, 15, 16, 17, 63, 64, 65 and 130 rows) and of their K
loops (1 to 12 chunks of 128: fewer than the stages of the ring, every
remainder), with the shared expert's tiles riding in the same launches in
every storage format, partial in tokens and in weight rows, and not riding."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import moe_oracle as O
from livglm_amd import native
from livglm_amd.workloads import BANK_KEYS, MoEShape, make_layer

pytestmark = pytest.mark.gpu

REL_L2 = 2e-3  # the layer bar
COUNTS = (0, 1, 15, 16, 17, 63, 64, 65, 130)


@pytest.fixture(scope="module")
def gu():
    import gpu_util
    native.load()
    return gpu_util


def _routed_layer(d, I, Is, k):
    """A layer whose token rows go to the experts COUNTS times (and, for k = 2,
    to the next expert too): the first E features of x name the experts."""
    E = len(COUNTS)
    first = np.repeat(np.arange(E), COUNTS)
    shape = MoEShape("rows", len(first), d, E, k, I, Is)
    layer = make_layer(shape, 7100 + d + I + k)
    rng = np.random.default_rng(d + I)
    first = rng.permutation(first)
    x = O.bf16_bits_to_f32(layer["x"]).copy()
    x[:, :E] = 0.0
    x[np.arange(len(first)), first] = 1.0
    if k == 2:
        x[np.arange(len(first)), (first + 1) % E] = 0.5
    layer["x"] = O.f32_to_bf16_bits(x)
    layer["router_weight"] = np.zeros((E, d), dtype=np.float32)
    layer["router_weight"][np.arange(E), np.arange(E)] = 4.0
    return layer, shape


def _shared_weights(layer, fmt):
    """The shared expert's f32 matrices in format fmt (None: no shared expert),
    its codes and scales put into the layer."""
    if fmt is None:
        return None
    shared = []
    for key in ("shared.gate", "shared.up", "shared.down"):
        if fmt == native.GLM_FMT_BF16:
            shared.append(O.bf16_bits_to_f32(layer[key]))
            continue
        bits, deq = (8, O.dequant_mxfp8) if fmt == native.GLM_FMT_MXFP8 else (4, O.dequant_mxfp4)
        layer[key], layer[key + ".scales"] = O.quantize_mx(layer[key], bits, O.MX_RULE_NEAREST)
        shared.append(deq(layer[key], layer[key + ".scales"]))
    return tuple(shared)


def _oracle(layer, shape, shared):
    return O.moe_layer(O.bf16_bits_to_f32(layer["x"]), layer["router_weight"], layer["router_bias"],
                       O.Bank(*(layer[key] for key in BANK_KEYS)), shared, top_k=shape.k, n_group=1,
                       topk_group=1, norm_topk_prob=True,
                       routed_scaling_factor=shape.routed_scaling_factor,
                       swiglu_limit=shape.swiglu_limit, return_intermediates=True)


@pytest.mark.parametrize("fmt", [None, native.GLM_FMT_BF16, native.GLM_FMT_MXFP8, native.GLM_FMT_MXFP4])
@pytest.mark.parametrize("d,I,Is,k", [
    # 41 rows an expert on average: bf16 activations
    (512, 128, 128, 1), (1536, 384, 640, 1), (512, 512, 1280, 1), (1024, 640, 160, 1),
    # 82: their FP8 split
    (1024, 256, 384, 2), (1024, 640, 160, 2), (512, 128, 128, 2), (1536, 384, 640, 2),
])
def test_stream_layer_row_and_chunk_edges(gu, d, I, Is, k, fmt):
    layer, shape = _routed_layer(d, I, Is, k)
    shared = _shared_weights(layer, fmt)
    want, inter = _oracle(layer, shape, shared)
    counts = np.bincount(inter["indices"].reshape(-1).astype(np.int64), minlength=shape.E)
    assert k > 1 or tuple(counts) == COUNTS
    out, w, idx = gu.run_layer(gu.upload_layer(layer), shape, shared=fmt is not None,
                               shared_fmt=native.GLM_FMT_BF16 if fmt is None else fmt)
    assert np.array_equal(gu.host(idx).astype(np.uint32), inter["indices"])
    got = gu.host(out)
    assert O.rel_l2(got, want) < REL_L2
    # no row of any tile is off on its own
    rows = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert rows.max() < 5 * REL_L2


@pytest.mark.parametrize("T,d,E,k,I,Is,fmt", [
    # decode batches: the smallest and largest of its range, an expert with a
    # row of every token (64 in a tile), few bytes but an MX shared expert, no
    # shared expert, one that cannot ride (I_shared 96)
    (16, 1024, 64, 8, 512, 512, native.GLM_FMT_MXFP8), (64, 2048, 32, 8, 768, 768, native.GLM_FMT_BF16),
    (64, 1024, 8, 8, 1280, 128, native.GLM_FMT_MXFP4), (33, 512, 16, 2, 128, 128, native.GLM_FMT_MXFP8),
    (33, 2560, 48, 6, 640, 0, None), (40, 2048, 24, 8, 1024, 96, native.GLM_FMT_BF16),
    # small layers that neither the decode kernels nor the GEMV tiles split
    (32, 1024, 8, 2, 1408, 1408, native.GLM_FMT_BF16), (16, 512, 8, 2, 1664, 0, None),
    (20, 6656, 8, 2, 256, 0, None),
    # too few work items: the decode kernels
    (17, 2560, 48, 6, 640, 0, None),
])
def test_stream_decode_batches(gu, T, d, E, k, I, Is, fmt):
    shape = MoEShape("decode", T, d, E, k, I, Is)
    assert gu.layer_path(shape, shared=fmt is not None, shared_fmt=fmt or 0) == \
        ("decode" if T == 17 else "stream_bf16")
    layer = make_layer(shape, 7300 + T + d)
    shared = _shared_weights(layer, fmt)
    want, inter = _oracle(layer, shape, shared)
    out, w, idx = gu.run_layer(gu.upload_layer(layer), shape, shared=fmt is not None,
                               shared_fmt=native.GLM_FMT_BF16 if fmt is None else fmt)
    same = np.all(gu.host(idx).astype(np.uint32) == inter["indices"], axis=1)
    assert same.sum() >= T - 1  # at most one near-tie
    assert O.rel_l2(gu.host(out)[same], want[same]) < REL_L2


@pytest.mark.parametrize("T,d,E,k,I,path,otherwise", [
    (3, 1024, 16, 2, 512, "few_tokens", "few_tokens"),
    (64, 1024, 64, 8, 512, "stream_bf16", "decode"),
    (100, 1024, 8, 2, 256, "stream_bf16", "work_list"),
    (100, 512, 8, 8, 256, "stream_split", "work_list"),
])
def test_routed_scales_off_a_4_byte_boundary(gu, T, d, E, k, I, path, otherwise):
    # scales that start off a 4-byte boundary are read by other kernels and give
    # the same layer
    shape = MoEShape("scales", T, d, E, k, I, 0)
    layer = make_layer(shape, 7500 + T + d)
    want, inter = _oracle(layer, shape, None)
    dl = gu.upload_layer(layer)
    names = [key for key in BANK_KEYS if key.endswith("scale")]
    assert gu.layer_path(shape, scales=[dl[key].data_ptr() for key in names]) == path
    for i, key in enumerate(names):
        moved = torch_bytes(gu, dl[key].numel() + 4)[i + 1:][:dl[key].numel()]
        moved.copy_(dl[key].reshape(-1))
        dl[key] = moved
    assert gu.layer_path(shape, scales=[dl[key].data_ptr() for key in names]) == otherwise
    out, w, idx = gu.run_layer(dl, shape, shared=False)
    same = np.all(gu.host(idx).astype(np.uint32) == inter["indices"], axis=1)
    assert same.sum() >= T - 1
    assert O.rel_l2(gu.host(out)[same], want[same]) < REL_L2


def torch_bytes(gu, n):
    return gu.to_dev(np.zeros(n, dtype=np.uint8))


def test_bank_keeps_scales_on_aligned_memory(gu):
    # load_bank takes a view that starts off the kernels' alignment by copying it
    from glm53flash.expert_ssd import HBMExpertBank
    shape = MoEShape("bank", 1, 512, 4, 2, 128, 0)
    layer = make_layer(shape, 7600)
    bank = HBMExpertBank(layer=0, num_experts=4, hidden_size=512, intermediate_size=128,
                         swiglu_limit=10.0, device="cuda")
    tensors = {key: gu.to_dev(layer[key]) for key in BANK_KEYS}
    kept = {}
    for key in BANK_KEYS:
        if key.endswith("scale"):
            n = tensors[key].numel()
            kept[key] = tensors[key]
            tensors[key] = torch_bytes(gu, n + 1)[1:].copy_(kept[key].reshape(-1)).reshape(kept[key].shape)
    bank.load_bank(tensors)
    for key, scales in kept.items():
        assert bank.tensors[key].data_ptr() % 16 == 0
        assert np.array_equal(gu.host(bank.tensors[key]), gu.host(scales))
    bank.load_bank({**tensors, **kept})  # aligned scales are not copied
    assert all(bank.tensors[key].data_ptr() == kept[key].data_ptr() for key in kept)


def test_stream_gemms_equal_the_wide_forms(gu):
    """Bit for bit: the layer's routed output against the wide grouped GEMMs
    called by themselves on the same split, tiles and weights."""
    import torch
    d, I, k, E = 1024, 512, 2, len(COUNTS)
    layer, shape = _routed_layer(d, I, 0, k)
    dl = gu.upload_layer(layer)
    out, w, idx = gu.run_layer(dl, shape, shared=False)
    T = shape.T
    P = T * k
    i32 = dict(dtype=torch.int32, device="cuda")
    counts, offsets, perm, inv, tok, act, nact, status = (
        torch.empty(n, **i32) for n in (E, E + 1, P, P, P, E, 1, 1))
    work = torch.empty((E, 4), **i32)
    gu.call("glm_moe_dispatch", gu.stream(), idx.data_ptr(), T, k, E,
            *(t.data_ptr() for t in (counts, offsets, perm, inv, tok, act, nact, work, status)))
    cap = P // 160 + 1 + E
    tiles, ntiles = torch.zeros((cap, 4), **i32), torch.zeros(1, **i32)
    gu.call("glm_moe_tiles", gu.stream(), work.data_ptr(), E, tiles.data_ptr(), ntiles.data_ptr())
    lib = native.load()

    def split(rows, t, K):
        s = torch.empty(lib.glm_act_split_bytes(rows, K), dtype=torch.uint8, device="cuda")
        gu.call("glm_act_split_fp8", gu.stream(), t.data_ptr(), rows, K, s.data_ptr())
        return s

    h = torch.empty((P, I), dtype=torch.bfloat16, device="cuda")
    y = torch.empty((P, d), dtype=torch.bfloat16, device="cuda")
    limit = shape.swiglu_limit
    gu.call("glm_expert_gate_up_grouped", gu.stream(), split(T, dl["x"], d).data_ptr(), T, d, I,
            *(gu.p(dl[key]) for key in BANK_KEYS[:4]), tok.data_ptr(), tiles.data_ptr(),
            ntiles.data_ptr(), cap, limit, h.data_ptr())
    gu.call("glm_expert_down_grouped", gu.stream(), split(P, h, I).data_ptr(), P, I, d,
            *(gu.p(dl[key]) for key in BANK_KEYS[4:]), tiles.data_ptr(), ntiles.data_ptr(), cap,
            y.data_ptr())
    wide = torch.empty((T, d), dtype=torch.float32, device="cuda")
    gu.call("glm_moe_combine", gu.stream(), y.data_ptr(), inv.data_ptr(), w.data_ptr(), None, T, k,
            d, wide.data_ptr())
    assert torch.equal(out, wide)
