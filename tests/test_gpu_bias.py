"""GPU parity of the dense-bias kernel (bias tiles staged through LDS) at the
edges of its 64-key steps and 32-row slices, and of the calls it leaves to the
score_mod kernel (bias rows that are not 16-byte aligned), against the oracle on
the same rounded inputs."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from gpu_helpers import assert_bars, make_inputs, norm_error
from oracle import oracle as O
from test_gpu_parity import oracle_full

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DTYPE = {"bf16": 1, "f16": 2}


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("D", [32, 64, 72, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("splits", [1, 0])
def test_dense_bias_edges(ofh, dt, D, causal, splits):
    """One chunk of keys, steps and slices less and more than full; a masked (-inf) and a lowest-value column, which take
    weight 0; large late biases, so that running maxima rise; a soft-cap."""
    F = ofh
    for i, (M, N) in enumerate([(1, 4), (33, 64), (64, 63), (31, 68), (300, 260), (257, 321)]):
        p = F.make_params(1, 3, M, N, D, dtype=DTYPE[dt], causal=causal, bias_kind=F.BIAS_DENSE, bias=16,
                          max_key_splits=splits)
        staged = F.launch_info(p).kernel_name.decode().startswith("flash_fwd_bias_kernel<")
        assert staged == (N % 4 == 0)
        dev, host = make_inputs(dt, 1, 3, M, N, D, seed=i + D)
        bias = O.normal(41 + i, (M, N), std=2.0)
        bias[:, N // 2:] += 6.0
        if N > 3:
            bias[:, 2] = -np.inf
            bias[:, 3] = np.finfo(np.float32).min
        t = torch.from_numpy(bias).cuda()
        ref = oracle_full(host, causal=causal, bias=bias)
        out = F.attention_fwd(*dev, causal=causal, bias=t, out_dtype=torch.float32, max_key_splits=splits)
        assert_bars(norm_error(out.cpu().numpy(), ref)[0], dt, f"{dt} D{D} M{M} N{N} causal={causal}")
        # the same values behind an odd offset and a wider row, per head
        wide = torch.zeros(1, 3, M, N + 5, device="cuda")
        view = wide[:, :, :, 1:N + 1]
        view.copy_(t.expand(1, 3, M, N))
        again = F.attention_fwd(*dev, causal=causal, bias=view, out_dtype=torch.float32, max_key_splits=splits)
        assert_bars(norm_error(again.cpu().numpy(), ref)[0], dt, f"{dt} D{D} M{M} N{N} causal={causal} strided bias")
        cap = F.attention_fwd(*dev, causal=causal, bias=t.clamp(min=-50), softcap=20.0, out_dtype=torch.float32,
                              max_key_splits=splits)
        ref = oracle_full(host, causal=causal, bias=bias.clip(min=-50), softcap=20.0)
        assert_bars(norm_error(cap.cpu().numpy(), ref)[0], dt, f"{dt} D{D} M{M} N{N} causal={causal} soft-cap")


@pytest.mark.parametrize("D", [64, 128])
def test_bias_rows_in_reverse(ofh, D):
    """The C entry takes bias strides of either sign: rows stored last to first."""
    F = ofh
    M, N = 300, 260
    dev, host = make_inputs("f16", 1, 3, M, N, D, seed=D)
    bias = O.normal(77, (M, N), std=2.0)
    t = torch.from_numpy(bias[::-1].copy()).cuda()
    out = torch.empty(1, 3, M, D, device="cuda")
    p = F.make_params(1, 3, M, N, D, dtype=F.DTYPE_F16, out_dtype=F.DTYPE_F32, scale=D ** -0.5,
                      bias_kind=F.BIAS_DENSE, bias=t.data_ptr() + 4 * (M - 1) * N)
    p.bias_strides[:] = (0, 0, -N)
    assert F.launch_info(p).kernel_name.decode().startswith("flash_fwd_lockstep_kernel<f16,")
    F.check(F.lib().ofh_attention_fwd(ctypes.byref(p), dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr(),
                                      out.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream))
    assert_bars(norm_error(out.cpu().numpy(), oracle_full(host, bias=bias))[0], "f16", f"D{D} reversed bias rows")
