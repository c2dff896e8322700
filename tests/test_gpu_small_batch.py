"""Batches of at most 64 routes run a layer as two launches (route + W13, W2 + merge). W8A8 bit for bit
against the oracle; BF16 and W8A16 bit for bit against the same tokens inside a larger batch, which takes
the route, W13, W2 and combine launches (16-row tiles: the same K order per product). Both merges (tree for
2, 4, 6, 8 slots, ordered otherwise), dropped ids, an appended shared expert, biases, ragged channels."""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests import helpers as H  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,E,hd,f,shared", [(2, 3, 5, 96, 48, False), (7, 8, 20, 1040, 528, True),
                                               (64, 1, 9, 512, 256, False), (4, 15, 16, 160, 80, True)])
def test_w8a8_small_batch_bit_exact(gpu, oracle_lib, T, k, E, hd, f, shared):
    x, ids, w, q13, s13, q2, s2 = H.w8a8_case(T * 100 + k, T, hd, f, E, k)
    ids[0, 0] = -1
    ids[T - 1, k - 1] = E + 3
    if shared:
        ids[ids == E - 1] = 0
    sid = E - 1 if shared else -1
    got = H.gpu_w8a8_forward(x, ids, w, q13, s13, q2, s2, gpu, shared_id=sid, scale=1.5,
                             valid_experts=E - 1 if shared else None)
    ref_ids = np.where((ids < 0) | (ids >= (E - 1 if shared else E)), -1, ids)
    np.testing.assert_array_equal(got, oracle_lib.w8a8_forward(x, ref_ids, w, q13, s13, q2, s2, shared_id=sid,
                                                               routed_scale=1.5))


@pytest.mark.parametrize("kind,T,k,E,hd,f,act,bias,shared", [
    ("bf16", 1, 2, 4, 64, 32, "silu", False, False), ("bf16", 5, 4, 6, 1056, 544, "gelu", True, False),
    ("bf16", 9, 6, 7, 256, 96, "silu", False, True), ("bf16", 64, 1, 3, 128, 64, "silu", True, False),
    ("w8a16", 3, 8, 9, 1088, 576, "silu", False, False), ("w8a16", 16, 2, 5, 128, 64, "gelu", False, False),
    ("w8a16", 6, 9, 12, 192, 128, "silu", False, True)])
def test_bf16_small_batch_equals_larger_batch(gpu, monkeypatch, kind, T, k, E, hd, f, act, bias, shared):
    from fused_cpp_amd import moe

    monkeypatch.setenv("FUSED_CPP_AMD_VALIDATE_IDS", "0")  # dropped ids contribute nothing
    rng = np.random.default_rng(T + 10 * k)
    big = 70  # over 64 routes at any k
    g = lambda *s: torch.from_numpy((rng.standard_normal(s) * 0.1).astype(np.float32)).to(gpu)  # noqa: E731
    x = (g(big, hd) * 10).to(torch.bfloat16)
    w13, w2 = g(E + shared, 2 * f, hd).to(torch.bfloat16), g(E + shared, hd, f).to(torch.bfloat16)
    ids = torch.from_numpy(np.stack([rng.permutation(E)[:k] for _ in range(big)])).to(gpu)
    ids[0, 0] = -1
    ids[T - 1, k - 1] = E + 1
    w = torch.rand((big, k), device=gpu)
    if shared:
        if kind == "bf16":
            packed = moe.prepare_routed_shared_moe_bf16_tiled_weights(w13[:E], w2[:E], w13[E], w2[E])
        else:
            q13, q2 = torch.round(w13.float() * 200).clamp(-127, 127), torch.round(w2.float() * 200).clamp(-127, 127)
            s13, s2 = torch.rand(E + 1, 2 * f, device=gpu) / 200, torch.rand(E + 1, hd, device=gpu) / 200
            i8 = torch.int8
            packed = moe.prepare_routed_shared_moe_w8a16_tiled_quantized_weights(
                q13[:E].to(i8), s13[:E], q2[:E].to(i8), s2[:E], q13[E].to(i8), s13[E], q2[E].to(i8), s2[E])
        fn = getattr(moe, f"fused_moe_{kind}_tiled_with_shared")
        call = lambda n: fn(x[:n], packed, w[:n], ids[:n], routed_scaling_factor=1.5, swiglu_limit=10.0)  # noqa: E731
    else:
        if kind == "bf16":
            packed = moe.prepare_fused_moe_bf16_tiled_weights(w13, w2, fuse_silu=act == "silu")
        else:
            packed = moe.prepare_fused_moe_w8a16_tiled_weights(w13, w2)
        kw = {"w13_bias": g(E, 2 * f), "w2_bias": g(E, hd)} if bias else {}
        call = lambda n: moe.fused_moe_tiled(x[:n], packed, w[:n], ids[:n], activation=act, **kw)  # noqa: E731
    assert T * (k + shared) <= 64 < big * (k + shared)
    assert torch.equal(call(T).view(torch.int16), call(big)[:T].view(torch.int16))
