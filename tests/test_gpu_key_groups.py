"""GPU parity of the kernel whose wavefront groups split the keys inside a
workgroup (two or four groups), against the oracle on the same rounded inputs."""

from __future__ import annotations

import math

import numpy as np
import pytest

from gpu_helpers import THREADS, alibi_slopes, assert_bars, make_inputs, norm_error
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DTYPE = {"bf16": 1, "f16": 2}


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("D,Dv,shapes", [
    # (B, H, M, N, causal, groups): ragged ends of row slices and staged tiles,
    # groups without a key of their own, M != N, more workgroups than CUs
    (32, 32, [(1, 24, 257, 300, False, 4), (1, 9, 1001, 1001, True, 4)]),
    (64, 64, [(2, 6, 300, 129, False, 4), (1, 64, 500, 500, True, 2), (1, 8, 1025, 1100, False, 4)]),
    (80, 72, [(2, 8, 290, 290, True, 4), (2, 16, 1000, 1000, False, 2)]),
    (128, 128, [(1, 32, 1000, 1000, True, 2), (3, 8, 513, 700, True, 4), (1, 16, 700, 400, True, 4)]),
    (48, 128, [(2, 6, 300, 290, False, 4)])])
def test_key_groups(ofh, dt, D, Dv, shapes):
    F = ofh
    for i, (B, H, M, N, causal, groups) in enumerate(shapes):
        p = F.make_params(B, H, M, N, D, Dv, dtype=DTYPE[dt], causal=causal)
        name = F.launch_info(p).kernel_name.decode()
        assert name.startswith("flash_fwd_keygroups_kernel<") and name.endswith(f",{groups}groups>"), (name, i)
        assert F.workspace_bytes(p) == 0
        dev, host = make_inputs(dt, B, H, M, N, D, Dv, seed=i + D)
        # later keys score higher: running maxima rise against live accumulators
        # and differ between the groups
        dev[1][:, :, N // 3:] *= 4
        host[1][:, :, N // 3:] *= 4
        if i % 2:
            dev = tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in dev)
        out = F.attention_fwd(*dev, causal=causal, out_dtype=torch.float32).cpu().numpy()
        prob = O.Problem(B, H, M, N, D, Dv, scale=1.0 / math.sqrt(D), causal=causal)
        heads = np.array([0, B * H // 2, B * H - 1], dtype=np.uint64)
        ref = O.standard_attention_rows(*host, prob, np.repeat(heads, M), np.tile(np.arange(M, dtype=np.uint64), 3),
                                        threads=THREADS).reshape(3, M, Dv)
        err, _ = norm_error(out.reshape(B * H, M, Dv)[heads.astype(int)], ref)
        assert_bars(err, dt, f"{dt} {name} M{M} N{N} causal={causal}")
        low = F.attention_fwd(*dev, causal=causal)
        assert torch.equal(low, torch.from_numpy(out).cuda().to(low.dtype))


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("D,Dv,H,M,N,causal,mod", [
    (64, 64, 12, 300, 333, False, "alibi+cap"), (128, 128, 32, 500, 500, True, "alibi"),
    (96, 96, 32, 700, 700, True, "cap"), (64, 64, 16, 777, 777, False, "dense"),
    (128, 72, 16, 513, 300, True, "dense+cap"), (32, 32, 64, 129, 200, False, "dense")])
def test_key_groups_score_mod(ofh, dt, D, Dv, H, M, N, causal, mod):
    """The same kernel with every kind of score modification."""
    F = ofh
    cap = 20.0 if "cap" in mod else 0.0
    kind = F.BIAS_ALIBI if "alibi" in mod else F.BIAS_DENSE if "dense" in mod else F.BIAS_NONE
    p = F.make_params(1, H, M, N, D, Dv, dtype=DTYPE[dt], causal=causal, softcap=cap, bias_kind=kind,
                      alibi_slopes=16 if kind == F.BIAS_ALIBI else None, bias=16 if kind == F.BIAS_DENSE else None)
    name = F.launch_info(p).kernel_name.decode()
    assert name.startswith("flash_fwd_keygroups_kernel<") and ",mod," in name, name
    dev, host = make_inputs(dt, 1, H, M, N, D, Dv, seed=M)
    slopes = alibi_slopes(H) if kind == F.BIAS_ALIBI else None
    bias = O.normal(5, (M, N), std=2.0) if kind == F.BIAS_DENSE else None
    kw = {} if slopes is None else {"alibi_slopes": torch.from_numpy(slopes).cuda()}
    if bias is not None:
        kw["bias"] = torch.from_numpy(bias).cuda()
    out = F.attention_fwd(*dev, causal=causal, softcap=cap, out_dtype=torch.float32, **kw).cpu().numpy()
    prob = O.Problem(1, H, M, N, D, Dv, scale=1.0 / math.sqrt(D), causal=causal, alibi_slopes=slopes,
                     dense_bias=bias, softcap=cap)
    heads = np.array([0, H // 2, H - 1], dtype=np.uint64)
    ref = O.standard_attention_rows(*host, prob, np.repeat(heads, M), np.tile(np.arange(M, dtype=np.uint64), 3),
                                    threads=THREADS).reshape(3, M, Dv)
    err, _ = norm_error(out.reshape(H, M, Dv)[heads.astype(int)], ref)
    assert_bars(err, dt, f"{dt} {name} M{M} N{N} causal={causal} {mod}")
