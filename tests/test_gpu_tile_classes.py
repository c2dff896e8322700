"""Every tile class of the MoE forwards at the edges of its tiles: experts of
1, 15, 16, 17, 63, 64, 65, 128, 129 and 260 rows, K of fewer chunks than a ring,
whole rings and a ring with a remainder, channel counts that leave the last
block part empty. FCMOE_TILE_CLASSES picks the class set at sizes whose rule
would take another. W8A8 is compared bit for bit with the oracle; BF16 and
W8A16 against the fp32 reference on the same bf16 values.
Reference semantics: csrc/moe/arm/i8mm_w8a8/kernels.cpp:463-694,
csrc/moe/arm/common/fused_moe_bf16_tiled.cpp:6376-7218."""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tests import helpers as H  # noqa: E402

pytestmark = pytest.mark.gpu

ROWS = (1, 15, 16, 17, 63, 64, 65, 128, 129, 260)
# 3 / 6, 16 / 32 and 10 / 20 chunks of K in W13 (int8 / bf16); 1 to 8 / 2 to 16 in W2
SHAPES = [(192, 48), (1024, 512), (640, 208)]


def _ids(rng):
    ids = np.repeat(np.arange(len(ROWS)), ROWS)
    rng.shuffle(ids)
    return ids[:, None].astype(np.int64)


@pytest.mark.parametrize("hd,f", SHAPES)
@pytest.mark.parametrize("classes", ["16", "64", "128", "256", "128,192,256", "16,32,64,128,192,256"])
def test_w8a8_tile_edges_bit_exact(gpu, oracle_lib, monkeypatch, classes, hd, f):
    ids = _ids(np.random.default_rng(hd + f))
    x, _, w, q13, s13, q2, s2 = H.w8a8_case(hd * 3 + f, ids.shape[0], hd, f, len(ROWS), 1)
    monkeypatch.setenv("FCMOE_TILE_CLASSES", classes)
    got = H.gpu_w8a8_forward(x, ids, w, q13, s13, q2, s2, gpu)
    np.testing.assert_array_equal(got, oracle_lib.w8a8_forward(x, ids, w, q13, s13, q2, s2))


@pytest.mark.parametrize("hd,f", SHAPES)
@pytest.mark.parametrize("kind,classes", [("bf16", "64"), ("bf16", "128,192,256"), ("w8a16", "64"),
                                          ("w8a16", "128,192,256"), ("bf16", "16,32,64,128,192,256"),
                                          ("w8a16", "16,32,64,128,192,256")])
def test_bf16_family_tile_edges(gpu, oracle_lib, monkeypatch, kind, classes, hd, f):
    from fused_cpp_amd import moe

    rng = np.random.default_rng(7 * hd + f)
    E, ids = len(ROWS), _ids(rng)
    x = H.bits_to_f32(H.bf16_bits(rng.standard_normal((ids.shape[0], hd)).astype(np.float32)))
    b13 = H.bf16_bits((rng.standard_normal((E, 2 * f, hd)) * 0.05).astype(np.float32))
    b2 = H.bf16_bits((rng.standard_normal((E, hd, f)) * 0.05).astype(np.float32))
    w = rng.uniform(0.2, 1.0, (ids.shape[0], 1)).astype(np.float32)
    bf = lambda b: torch.from_numpy(b.view(np.int16)).to(gpu).view(torch.bfloat16)  # noqa: E731
    if kind == "bf16":
        packed, call = moe.prepare_fused_moe_bf16_tiled_weights(bf(b13), bf(b2), fuse_silu=True), moe.fused_moe_bf16_tiled
        f13, f2 = H.bits_to_f32(b13), H.bits_to_f32(b2)
    else:
        (q13, s13), (q2, s2) = oracle_lib.quant_weight_rows(b13), oracle_lib.quant_weight_rows(b2)
        packed = moe.prepare_fused_moe_w8a16_tiled_quantized_weights(*map(torch.from_numpy, (q13, s13, q2, s2)))
        call = moe.fused_moe_w8a16_tiled
        f13, f2 = q13.astype(np.float32) * s13[..., None], q2.astype(np.float32) * s2[..., None]
    monkeypatch.setenv("FCMOE_TILE_CLASSES", classes)
    out = call(bf(H.bf16_bits(x)), packed, torch.from_numpy(w).to(gpu), torch.from_numpy(ids).to(gpu))
    got = out.float().cpu().numpy().astype(np.float64)
    ref = oracle_lib.bf16_moe_reference(x, f13, f2, w, ids, round_intermediate=True).astype(np.float64)
    # fp32 sums in another order leave the intermediate y within a few 2^-24 of the reference's, so a
    # value next to a rounding boundary may fall on bf16's other side: one ulp, at most 2^-7 |y|, times
    # its W2 weight and the route's. The chance is ~1e-4 a value, so two of a row's F values at most.
    # On top of the result's own rounding (half a bf16 ulp) and fp32 sums over F terms.
    ymax = np.empty((ids.shape[0], 1))
    for e in range(E):
        sel = ids[:, 0] == e
        gate, up = np.split(x[sel].astype(np.float64) @ f13[e].T.astype(np.float64), 2, axis=1)
        ymax[sel, 0] = np.abs(gate / (1.0 + np.exp(-gate)) * up).max(1)
    step = ymax * np.abs(f2).max() * w
    bound = H.bf16_half_ulp(ref) + 2 * 2.0 ** -7 * step + f * 2.0 ** -24 * step
    assert (np.abs(got - ref) <= bound).all(), float((np.abs(got - ref) / bound).max())


def test_w8a8_weights_read_once_bit_exact(gpu, oracle_lib):
    """Enough experts that the 64-row tiles load weights nontemporal (over 300 MB), a few rows each."""
    T, hd, f, E, k = 150, 1024, 512, 220, 8
    x, ids, w, q13, s13, q2, s2 = H.w8a8_case(5, T, hd, f, E, k)
    got = H.gpu_w8a8_forward(x, ids, w, q13, s13, q2, s2, gpu)
    tok = np.array([0, 1, 74, T - 1])
    np.testing.assert_array_equal(got[tok], oracle_lib.w8a8_forward(x[tok], ids[tok], w[tok], q13, s13, q2, s2))


@pytest.mark.parametrize("kind,T,classes", [("bf16", 70, "64"), ("w8a16", 70, "64"), ("bf16", 70, "128,192,256"),
                                            ("w8a16", 70, "128,192,256"), ("bf16", 70, "16"), ("w8a16", 3, ""),
                                            ("mlp", 40, ""), ("mlp", 300, "")])
@pytest.mark.parametrize("offset", [1, 4])
def test_rows_that_start_off_16_bytes(gpu, monkeypatch, kind, T, classes, offset):
    """The same rows 2 or 8 bytes off a 16-byte start: bit for bit the aligned rows' result on every
    tile (the LDS tiles load 16-byte pieces)."""
    from fused_cpp_amd import moe

    E, hd, f, k = 9, 256, 192, 2
    g = torch.Generator(device="cuda").manual_seed(T + offset)
    bf = lambda *s: (torch.randn(s, generator=g, device=gpu) * 0.1).to(torch.bfloat16)  # noqa: E731
    x = bf(T, hd) * 10
    buf = torch.zeros(T * hd + offset, dtype=torch.bfloat16, device=gpu)
    shifted = buf[offset:].view(T, hd)
    shifted.copy_(x)
    assert shifted.is_contiguous() and shifted.data_ptr() % 16 == 2 * offset
    if kind == "mlp":
        packed = moe.prepare_shared_mlp_bf16_tiled_weights(bf(2 * f, hd), bf(hd, f))
        call = lambda v: moe.shared_mlp_bf16_tiled(v, packed)  # noqa: E731
    else:
        packed = getattr(moe, f"prepare_fused_moe_{kind}_tiled_weights")(bf(E, 2 * f, hd), bf(E, hd, f))
        ids = torch.randint(0, E, (T, k), generator=g, device=gpu)
        w = torch.rand((T, k), generator=g, device=gpu)
        call = lambda v: getattr(moe, f"fused_moe_{kind}_tiled")(v, packed, w, ids)  # noqa: E731
    if classes:
        monkeypatch.setenv("FCMOE_TILE_CLASSES", classes)
    assert torch.equal(call(shifted).view(torch.int16), call(x).view(torch.int16))


@pytest.mark.parametrize("family,T,hd,f,experts,k,shared,classes", [
    # work from 80 GOP leaves the 64-row tiles (64 against 128 rows, us: 331 / 222, 536 / 334, 152 / 132), of few
    # experts from 91 (284 / 275), W8A16's from 111
    ("bf16", 1600, 4096, 1536, 8, 2, False, "128"), ("bf16", 600, 2880, 2880, 32, 4, False, "128"),
    ("bf16", 1100, 7168, 2048, 2, 1, False, "128"), ("w8a8", 1600, 1024, 2048, 32, 4, False, "128"),
    ("bf16", 800, 4096, 1536, 8, 2, False, "64"), ("w8a8", 1000, 7168, 2048, 1, 1, False, "64"),
    ("bf16", 1000, 7168, 2048, 1, 1, False, "64"),
    ("w8a16", 1200, 4096, 1536, 8, 2, False, "64"),
    # at most 48 rows per expert: W8A8's from 120 GOP (908 / 730), W8A16's not
    ("w8a8", 800, 5120, 1536, 160, 6, True, "128"), ("w8a8", 400, 5120, 1536, 160, 6, True, "128"),
    ("w8a8", 350, 5120, 1536, 160, 6, True, "64"), ("w8a16", 300, 7168, 2048, 64, 8, True, "64"),
    # over 2 GiB of weights and 128 to 256 rows per expert: three classes (128 rows against them: 1070 / 828)
    ("w8a8", 1200, 7168, 2048, 64, 8, True, "128,192,256"), ("w8a16", 1600, 7168, 2048, 64, 8, True, "128,192,256"),
    ("w8a8", 900, 7168, 2048, 64, 8, True, "128"), ("w8a8", 2400, 7168, 2048, 64, 8, True, "128"),
    ("w8a8", 2400, 4096, 1536, 64, 4, True, "128"), ("bf16", 4096, 7168, 256, 256, 8, True, "128"),
    # 16-row tiles of BF16 layers of few experts (us on 16 / 64 rows: 91 / 98, 54 / 60, 211 / 240)
    ("bf16", 24, 2048, 1024, 40, 4, False, "16"), ("bf16", 16, 1024, 768, 48, 6, True, "16"),
    ("bf16", 24, 6144, 2048, 16, 2, True, "16"), ("bf16", 48, 2048, 1024, 40, 4, False, "64"),
    ("bf16", 48, 6144, 2048, 16, 2, True, "64"), ("bf16", 40, 2048, 768, 128, 8, False, "64"),
    ("w8a16", 24, 6144, 2048, 16, 2, True, "64")])
def test_tile_class_rule(gpu, family, T, hd, f, experts, k, shared, classes):
    """The class set on both sides of the rule's lines, from the stages that ran (weights of zeros)."""
    import ctypes

    from fused_cpp_amd import cabi

    L = cabi.lib()
    size = 2 if family == "bf16" else 1
    total = experts + shared
    keep = {
        "x": torch.zeros((T, hd), dtype=torch.bfloat16, device=gpu),
        "topk_ids": torch.randint(0, experts, (T, k), device=gpu),
        "topk_weights": torch.ones((T, k), device=gpu),
        "w13": torch.zeros(total * L.fcmoe_packed_expert_bytes(size, 2 * f, hd, 2), dtype=torch.uint8, device=gpu),
        "w2": torch.zeros(total * L.fcmoe_packed_expert_bytes(size, hd, f, 1), dtype=torch.uint8, device=gpu),
        "out": torch.ones((T, hd), dtype=torch.bfloat16, device=gpu)}
    if size == 1:
        keep["w13_scale"], keep["w2_scale"] = torch.ones((total, 2 * f), device=gpu), torch.ones((total, hd), device=gpu)
    a = cabi.MoeArgs()
    a.tokens, a.hidden, a.inter, a.top_k, a.ids_is_i64, a.routed_scaling = T, hd, f, k, 1, 1.0
    a.experts, a.valid_experts, a.shared_expert_id = total, experts, experts if shared else -1
    a.activation = cabi.FCMOE_ACT_SILU_CLAMP10
    a.workspace_bytes = getattr(L, f"fcmoe_{family}_workspace_bytes")(ctypes.byref(a))
    keep["workspace"] = torch.empty(a.workspace_bytes, dtype=torch.uint8, device=gpu)
    for name, t in keep.items():
        setattr(a, name, t.data_ptr())
    cabi.stage_timing_read()
    cabi.stage_timing_enable(True)
    try:
        cabi.check(getattr(L, f"fcmoe_{family}_forward")(ctypes.byref(a), cabi.stream_handle()), "forward")
        ran = cabi.stage_timing_read()
    finally:
        cabi.stage_timing_enable(False)
    assert {s for s in ran if "bm" in s} == {f"{w}_bm{c}" for w in ("w13", "w2") for c in classes.split(",")}
    assert not keep["out"].any()
