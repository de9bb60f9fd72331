"""GPU parity of the decode kernel (a few query rows against many keys) at the
edges of its key groups, row widths and row counts, against the oracle on the
same rounded inputs. Probabilities and sums are fp32 there, so the fp32 bar
holds for every input dtype with fp32 output."""

from __future__ import annotations

import math

import numpy as np
import pytest

from gpu_helpers import THREADS, assert_bars, make_inputs, norm_error
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DTYPE = {"f32": 0, "bf16": 1, "f16": 2}


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def oracle_rows(host):
    uq, uk, uv = host
    B, H, M, D = uq.shape
    prob = O.Problem(B, H, M, uk.shape[2], D, uv.shape[3], scale=1.0 / math.sqrt(D))
    heads = np.repeat(np.arange(B * H, dtype=np.uint64), M)
    rows = np.tile(np.arange(M, dtype=np.uint64), B * H)
    return O.standard_attention_rows(uq, uk, uv, prob, heads, rows, threads=THREADS).reshape(B, H, M, uv.shape[3])


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("D,Dv", [(8, 8), (64, 64), (80, 72), (128, 128), (64, 120), (256, 32)])
def test_decode_kernel(ofh, dt, D, Dv):
    """The fewest keys, a step less and more than full, several steps with a ragged
    end; each row count of the kernel; unsplit, split with both merges; rows
    in [B,T,H,D] storage; keys with large scores late, so that the running max
    is raised against live accumulators."""
    F = ofh
    if dt != "f32" and D > 128:
        D, Dv = 128, 32  # the 16-bit kernel ends at 128
    rows = (1, 2, 3, 8) if dt == "f32" else (1, 2)
    for i, (M, N, splits) in enumerate([(m, n, s) for m in rows for n, s in ((64, 0), (191, 0), (513, 1), (2081, 3), (2081, 0))]):
        # (fp32 calls of three rows or more with few heads and keys take other kernels)
        H = 64 if dt == "f32" and M > 2 and max(D, Dv) <= 64 else 3
        p = F.make_params(2, H, M, N, D, Dv, dtype=DTYPE[dt], max_key_splits=splits)
        info = F.launch_info(p)
        assert info.kernel_name.decode().startswith("flash_fwd_decode_kernel<"), info.kernel_name
        dev, host = make_inputs(dt, 2, H, M, N, D, Dv, seed=i)
        dev[1][:, :, N // 2:] *= 4
        host[1][:, :, N // 2:] *= 4
        dev = tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in dev) if i % 2 else dev
        out = F.attention_fwd(*dev, out_dtype=torch.float32, max_key_splits=splits).cpu().numpy()
        err, _ = norm_error(out, oracle_rows(host))
        assert_bars(err, "f32", f"{dt} decode M{M} N{N} D{D} Dv{Dv} splits {info.key_splits}")
        if dt != "f32":  # 16-bit output: the fp32 result rounded once
            low = F.attention_fwd(*dev, max_key_splits=splits)
            assert torch.equal(low, torch.from_numpy(out).cuda().to(low.dtype))


@pytest.mark.parametrize("splits", [1, 3, 0])
def test_decode_infinite_value_in_the_last_key(ofh, splits):
    """The keys past the end of a ragged group repeat the last one with
    probability 0: an infinity in its V row stays an infinity."""
    F = ofh
    dev, _ = make_inputs("bf16", 1, 2, 1, 1000, 64, seed=3)
    dev[2][0, 0, 999, 5] = float("inf")
    out = F.attention_fwd(*dev, max_key_splits=splits).float().cpu().numpy()
    assert out[0, 0, 0, 5] == np.inf
    out[0, 0, 0, 5] = 0
    assert np.isfinite(out).all()


@pytest.mark.parametrize("dt,D", [("f32", 8), ("f32", 80), ("f32", 100), ("f32", 160), ("bf16", 32), ("f16", 96), ("bf16", 72)])
@pytest.mark.parametrize("splits", [1, 0])
def test_decode_infinite_key(ofh, dt, D, splits):
    """Keys whose score is -inf through an infinity in the last chunk of their
    row take weight 0, also where lanes past the row's width repeat that chunk."""
    F = ofh
    M = 3 if D > 96 else 2
    dev, host = make_inputs(dt, 1, 2, M, 700, D, seed=D)
    for q, k in [(dev[0], dev[1]), (host[0], host[1])]:
        q[..., D - 2:] = 1.5
        k[0, :, 3::7, D - 1] = -float("inf")
        k[0, 1, 690:, D - 2] = -float("inf")
    out = F.attention_fwd(*dev, out_dtype=torch.float32, max_key_splits=splits).cpu().numpy()
    assert np.isfinite(out).all()
    assert_bars(norm_error(out, oracle_rows(host))[0], "f32", f"{dt} D{D} infinite keys")
