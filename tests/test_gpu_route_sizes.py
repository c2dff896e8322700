"""The route build around its workgroups' 1024 routes, over many of them and past the size where three
launches take over, with a hot expert, dropped ids and an appended shared slot: counts, offsets and the
stable per-expert order against a stable sort.
Reference semantics: csrc/moe/arm/i8mm_w8a8/kernels.cpp:583-592."""

from __future__ import annotations

import numpy as np
import pytest

pytest.importorskip("torch")

from tests import helpers as H  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,k,experts,shared", [
    (1, 1, 1, False), (63, 1, 5, False), (341, 3, 1024, False), (128, 8, 257, True), (1024, 1, 2, False),
    (1025, 1, 1000, False), (114, 8, 257, True), (5000, 6, 21, True), (32768, 8, 384, False), (32769, 8, 129, False),
    # both sides of the line that depends on the experts, and of the line for all
    (16339, 2, 8, False), (16340, 2, 8, False), (9416, 8, 385, True), (9417, 8, 385, True), (32768, 8, 1024, False),
    (32769, 8, 1024, False)])
def test_route_build_sizes(gpu, tokens, k, experts, shared):
    rng = np.random.default_rng(tokens + k)
    valid = experts - 1 if shared else experts
    ids = rng.integers(0, max(valid, 1), (tokens, k))
    ids[rng.random((tokens, k)) < 0.4] = 0  # a hot expert
    bad = rng.random((tokens, k)) < 0.05
    ids[bad] = rng.choice([-1, experts, 1 << 20], int(bad.sum()))
    counts, offsets, order, invalid = H.gpu_route_build(ids, experts, experts - 1 if shared else -1, gpu)
    flat = np.concatenate([ids, np.full((tokens, 1), experts - 1)], 1).reshape(-1) if shared else ids.reshape(-1)
    ok = (flat >= 0) & (flat < experts)
    ref = np.argsort(np.where(ok, flat, experts), kind="stable")[: int(ok.sum())]
    assert invalid == int((~ok).sum())
    np.testing.assert_array_equal(counts, np.bincount(flat[ok], minlength=experts))
    np.testing.assert_array_equal(offsets, np.concatenate([[0], np.cumsum(counts)]))
    np.testing.assert_array_equal(order[: ref.size], ref)
