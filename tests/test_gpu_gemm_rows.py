"""Row GEMM (mc_model_gemm_rows) at the edges of its activation row groups and
of the W row counts where its workgroups and LDS stages change, against float64
products. Bounds as in test_gpu_gemm_tiles.py (a K-term fp32 sum in any order
and the bf16 roundings)."""
import ctypes as C

import numpy as np
import pytest

from _util import to_dev

pytestmark = pytest.mark.gpu


def P(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("N,K,swi", [(16, 2048, 0), (2048, 2048, 0), (2064, 2048, 0),
                                     (4096, 2048, 0), (4112, 2048, 0), (48, 6144, 0),
                                     (2064, 6144, 0), (4112, 6144, 0), (16, 2048, 1),
                                     (2048, 2048, 1), (2064, 2048, 1), (4112, 2048, 1),
                                     (8208, 2048, 1)])
def test_row_groups_and_stage_counts(pkg, orc, dev, N, K, swi):
    import torch
    lib = pkg._native.lib()
    rng = np.random.default_rng(N + K + swi)
    rows = 2 * N if swi else N
    w = orc.f32_to_bf16(rng.standard_normal((rows, K), dtype=np.float32) / np.float32(K ** 0.5))
    x = orc.f32_to_bf16(rng.standard_normal((32, K + 8), dtype=np.float32))
    dw, dx = to_dev(w, dev), to_dev(x, dev)
    xf, wf = (orc.bf16_to_f32(a).astype(np.float64) for a in (x[:, :K], w))
    ref = xf @ wf.T
    bound = K * 2.0 ** -24 * (np.abs(xf) @ np.abs(wf).T) + 2.0 ** -8 * np.abs(ref)
    if swi:
        g, u, eg, eu = ref[:, :N], ref[:, N:], bound[:, :N], bound[:, N:]
        s = g / (1.0 + np.exp(-g))
        ref = s * u
        bound = 1.1 * eg * (np.abs(u) + eu) + np.abs(s) * eu + 2.0 ** -8 * np.abs(ref)
    for M in (9, 16, 17, 24, 25, 32):
        y = torch.full((M + 1, N + 4), -1, dtype=torch.int16, device=dev)
        st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert lib.mc_model_gemm_rows(P(dw), P(dx), K + 8, P(y), N + 4, M, N, K, swi, st) == 0
        torch.cuda.synchronize()
        y = y.cpu().numpy().view(np.uint16)
        err = np.abs(orc.bf16_to_f32(y[:M, :N]) - ref[:M]) / (bound[:M] + 1e-30)
        assert err.max() <= 1.0, (M, N, K, swi, err.max())
        assert np.all(y[M] == 0xFFFF) and np.all(y[:, N:] == 0xFFFF), (M, N, K, swi)
