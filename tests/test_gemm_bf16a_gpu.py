"""The bf16-activation products at the sizes where their tile changes (one round
of 32 x 64, 64 x 64 and 64 x 128 blocks on 256 CUs) and at ragged ones, plain and
gated, against the oracle; C filled with NaN and guarded by NaN."""
import numpy as np
import pytest

import oracle
from n550_qwen3_bringup_handover_amd import abi, runtime
from tests import numerics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,gated,plan", [
    (1, 128, 1, False, "pb32x64k128"), (65, 1024, 4096, False, "pb32x64k128"), (128, 128, 4095, False, "pb32x64k128"),
    (129, 1024, 4096, False, "pb64x64k128"), (256, 256, 4033, False, "pb64x64k128"), (511, 3072, 1024, False, "pb32x64k128"),
    (513, 2048, 1024, False, "pb64x64k128"), (1023, 384, 1000, False, "pb64x64k128"), (257, 1024, 4096, False, "xb64x128"),
    (1025, 3072, 1024, False, "xb64x128"), (2049, 640, 1024, False, "xb128x128"), (33, 192, 200, False, "xb64x128"),
    (70, 64, 77, False, "xb64x128"), (65, 1024, 3072, True, "pb64x64k128"), (128, 512, 3071, True, "pb64x64k128"),
    (129, 1024, 3072, True, "xb64x128"), (50, 192, 333, True, "xb64x128"), (321, 1024, 3072, True, "xb128x128"),
    (3, 896, 33, True, "pb64x64k128")])
def test_bf16a_tiles(M, K, N, gated, plan):
    runtime.init()
    a = oracle.round_bf16(oracle.f32_bf16_normal(M * K, 5500 + M + K + N, 1.0))
    b = oracle.bf16_normal((2 if gated else 1) * N * K, 5501 + M + K + N, 0.02)
    ad = abi.DeviceBuffer.from_array((a.view(np.uint32) >> 16).astype(np.uint16))
    bd = abi.DeviceBuffer.from_array(b)
    cd = abi.DeviceBuffer.from_array(np.full(M * N + 64, np.nan, np.float32))
    if gated:
        abi.gemm_gate_up_silu_bf16a_dev(cd.ptr, ad.ptr, bd.ptr, bd.ptr + 2 * N * K, M, K, N)
    else:
        abi.gemm_bf16a_dev(cd.ptr, ad.ptr, bd.ptr, M, K, N)
    abi.sync()
    assert abi.last_plan() == plan
    c = cd.download(np.float32, M * N + 64)
    assert np.isnan(c[M * N:]).all()
    rows = numerics.pick_rows(M, 40)
    if gated:
        numerics.compare_gated(c[:M * N], a, b[:N * K], b[N * K:], M, K, N, rows=rows)
    else:
        numerics.compare(c[:M * N], a, b, M, K, N, rows=rows)
