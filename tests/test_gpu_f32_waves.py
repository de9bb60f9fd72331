"""GPU parity of the fp32 kernel whose eight wavefronts share a 32-row block's
key tiles, against the oracle on the same inputs."""

from __future__ import annotations

import math

import numpy as np
import pytest

from gpu_helpers import THREADS, assert_bars, make_inputs, norm_error
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("B,H,M,N,D,Dv,causal", [
    # ragged last block and key tile, wavefronts without a tile, M != N both
    # ways, widths inside one or two 64-column blocks, several rounds of blocks
    (1, 17, 257, 131, 64, 64, False), (2, 10, 300, 300, 64, 64, True), (1, 43, 97, 300, 36, 64, False),
    (1, 32, 200, 1030, 64, 40, True), (1, 8, 1000, 129, 64, 64, True), (1, 64, 225, 289, 64, 64, False),
    (3, 8, 193, 257, 128, 128, False), (1, 12, 513, 513, 128, 128, True), (1, 16, 300, 200, 100, 80, False),
    (1, 20, 300, 290, 64, 128, True), (1, 16, 300, 290, 128, 4, False), (2, 10, 330, 250, 100, 124, True)])
def test_f32_waves(ofh, B, H, M, N, D, Dv, causal):
    F = ofh
    p = F.make_params(B, H, M, N, D, Dv, causal=causal)
    info = F.launch_info(p)
    width = 64 if max(D, Dv) <= 64 else 128
    assert info.kernel_name.decode() == f"flash_fwd_f32_waves_kernel<{width}>"
    assert info.block_m == 32 and info.workgroups == B * H * ((M + 31) // 32) and F.workspace_bytes(p) == 0
    dev, host = make_inputs("f32", B, H, M, N, D, Dv, seed=M + D)
    # later keys score higher: running maxima rise against live accumulators
    # and differ between the wavefronts
    dev[1][:, :, N // 3:] *= 4
    host[1][:, :, N // 3:] *= 4
    dev = tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in dev)
    out = F.attention_fwd(*dev, causal=causal).cpu().numpy()
    prob = O.Problem(B, H, M, N, D, Dv, scale=1.0 / math.sqrt(D), causal=causal)
    heads = np.array([0, B * H // 2, B * H - 1], dtype=np.uint64)
    ref = O.standard_attention_rows(*host, prob, np.repeat(heads, M), np.tile(np.arange(M, dtype=np.uint64), 3),
                                    threads=THREADS).reshape(3, M, Dv)
    err, _ = norm_error(out.reshape(B * H, M, Dv)[heads.astype(int)], ref)
    assert_bars(err, "f32", f"M{M} N{N} D{D} Dv{Dv} causal={causal}")


def test_f32_waves_special_values(ofh):
    """What the 128-row tiles answer (max_key_splits=1 keeps them) for
    infinities and NaN in the inputs: the same rows and columns are not finite."""
    F = ofh
    g = torch.Generator(device="cpu").manual_seed(3)
    q, k, v = (torch.randn(2, 16, 200, 64, generator=g).cuda() for _ in range(3))
    q[0, 0, 5, 1] = float("nan")
    k[0, 1, 7, 2] = float("nan")
    k[0, 2, 9, 3] = float("inf")
    v[0, 3, 150, 4] = float("nan")
    v[1, 4, 0, 5] = float("inf")
    a, b = F.attention_fwd(q, k, v), F.attention_fwd(q, k, v, max_key_splits=1)
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())
    keep = a.isfinite()
    assert (a[keep] - b[keep]).abs().max().item() < 1e-5
