"""fcmoe_quantize_rows over the forms its kernels split by: fp32 rows of whole
16-byte pieces and others, bf16 rows of any width, the register pieces' edges
(512 .. 16384 columns per row), rows past the registers, and row strides that
are no multiple of 4. The bytes and the scales' bits are those of
csrc/i8gemm.cpp:368-392 exactly."""
from __future__ import annotations

import numpy as np
import pytest

pytest.importorskip("torch")

from tests import helpers as H  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("cols,ldq", [(1, 64), (31, 31), (33, 35), (512, 512), (513, 576), (1024, 1024), (1028, 1030),
                                      (2047, 2112), (4100, 4160), (8191, 8192), (16384, 16384), (16383, 16384),
                                      (16385, 16448), (16388, 16448)])
def test_quant_rows_of_any_width_match_the_oracle(gpu, oracle_lib, f32, cols, ldq):
    rng = np.random.default_rng(cols)
    x = (rng.standard_normal((3, cols)) * 5).astype(np.float32)
    x[1] = 0  # scale 1, bytes 0
    x[2, cols - 1] = -400.0  # the maximum is the last element
    xin = x if f32 else H.bf16_bits(x)
    q, s = H.gpu_quant_rows(xin, 1, gpu, ldq)
    rq, rs = oracle_lib.quant_rows_even(xin)
    np.testing.assert_array_equal(q[:, :cols], rq)
    assert (q[:, cols:] == 0).all()
    np.testing.assert_array_equal(s.view(np.uint32), rs.view(np.uint32))


@pytest.mark.parametrize("rows,cols", [(1024, 320), (1025, 320), (1025, 321)])
def test_quant_rows_of_many_narrow_rows_match_the_oracle(gpu, oracle_lib, rows, cols):
    x = np.random.default_rng(rows + cols).standard_normal((rows, cols)).astype(np.float32)
    q, s = H.gpu_quant_rows(x, 1, gpu)
    rq, rs = oracle_lib.quant_rows_even(x)
    np.testing.assert_array_equal(q, rq)
    np.testing.assert_array_equal(s.view(np.uint32), rs.view(np.uint32))


def test_quant_rows_of_fp32_off_16_bytes(gpu, oracle_lib):
    import torch

    from fused_cpp_amd import cabi

    rng = np.random.default_rng(7)
    x = rng.standard_normal((4, 64)).astype(np.float32)
    buf = torch.zeros(4 * 64 + 1, device=gpu)
    buf[1:] = torch.from_numpy(x).flatten()
    q = torch.zeros(4 * 64 + 1, dtype=torch.int8, device=gpu)
    s = torch.zeros(4, device=gpu)
    cabi.check(cabi.lib().fcmoe_quantize_rows(buf.data_ptr() + 4, 1, 4, 64, 1, q.data_ptr() + 1, 64, s.data_ptr(),
                                              cabi.stream_handle()), "quantize_rows")
    rq, rs = oracle_lib.quant_rows_even(x)
    np.testing.assert_array_equal(q[1:].cpu().numpy().reshape(4, 64), rq)
    np.testing.assert_array_equal(s.cpu().numpy().view(np.uint32), rs.view(np.uint32))


def test_quant_rows_past_one_launch_of_row_workgroups(gpu, oracle_lib):
    """2^24 rows: a workgroup of 256 threads per row would be 2^32 threads, more than a launch may have."""
    import torch

    from fused_cpp_amd import cabi

    rows, cols = 1 << 24, 321
    x = torch.zeros((rows, cols), dtype=torch.bfloat16, device=gpu)
    at = [0, 1, 4095, rows // 2, rows - 2, rows - 1]
    xr = H.bits_to_f32(H.bf16_bits(np.random.default_rng(3).standard_normal((len(at), cols)).astype(np.float32)))
    x[at] = torch.from_numpy(xr).to(gpu).to(torch.bfloat16)
    q = torch.full((rows, cols), 99, dtype=torch.int8, device=gpu)
    s = torch.zeros(rows, device=gpu)
    cabi.check(cabi.lib().fcmoe_quantize_rows(x.data_ptr(), 0, rows, cols, 1, q.data_ptr(), cols, s.data_ptr(),
                                              cabi.stream_handle()), "quantize_rows")
    rq, rs = oracle_lib.quant_rows_even(H.bf16_bits(xr))
    np.testing.assert_array_equal(q[at].cpu().numpy(), rq)
    np.testing.assert_array_equal(s[at].cpu().numpy().view(np.uint32), rs.view(np.uint32))
    assert int((s == 1).sum()) == rows - len(at)  # rows of zeros: scale 1, bytes 0
    assert not q[2:4095].any()
