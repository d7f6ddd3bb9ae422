"""Every packed code as an MFMA operand, exactly.

Products with one-hot rows pick single weights out: y = scale * (code - centre),
one non-zero product and an exact one (an fp16 scale times a half-integer below
32), so it equals altxs_dequant's value, which unpacks a field at a time, in every
bit.  Random bytes bring all codes of each width; the row counts run the 16-row tasks and
both heights of the row bands, the x types all operand conversions.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("bits", [2, 3, 4, 6])
@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,count,K", [(16, 1, 256), (32, 65, 512), (64, 130, 512), (64, 130, 256)])
def test_one_hot_rows_give_the_weights(bits, xdt, rows, count, K):
    from altxs_amd import _lib, ops

    print(f"[gpu-case] codes bits={bits} {xdt} rows={rows} count={count} K={K}", flush=True)
    N = 256
    g = torch.Generator(device=DEV).manual_seed(bits)
    cs, ss = N * K * bits // 8, N * K // 64 * 2
    codes = torch.randint(0, 256, (count * cs,), dtype=torch.uint8, device=DEV, generator=g)
    scales = (torch.rand(count * ss // 2, device=DEV, generator=g) * 0.05 + 0.001).half().view(torch.int16)
    out = torch.empty(count, rows, N, device=DEV)
    want = torch.empty(N, K, device=DEV)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    eye = torch.eye(K, device=DEV).to(xdt)
    got = torch.empty(count, N, K, device=DEV)
    for c0 in range(0, K, rows):
        ops.qgemm_stream(codes, scales, count, N, K, bits, cs, ss, eye[c0:c0 + rows].contiguous(), out)
        got[:, :, c0:c0 + rows] = out.transpose(1, 2)
    for i in sorted({0, count // 2, count - 1}):
        qt = _lib.QTensor(codes.data_ptr() + i * cs, scales.data_ptr() + i * ss, N, K, bits, 0)
        _lib.check(_lib.load().altxs_dequant(ctypes.byref(qt), want.data_ptr(), stream), "altxs_dequant")
        assert torch.equal(got[i], want), i
