"""Attention over tiles of 32 keys (knx_flash.hip): tile edges, head sizes, unequal query and key counts, scales and values
that have no finite bf16 parts, against float64."""
import ctypes
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from kernix_amd import hipabi  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    lib = hipabi.lib()
    hipabi.check(lib.knx_hip_init())
    return lib


def run(L, q, k, v, scale, causal, scores=True):
    B, H, Rq, d = q.shape
    S = k.shape[2]
    rows = lambda t: t.permute(0, 2, 1, 3).reshape(-1, H * d).contiguous().cuda()  # noqa: E731
    dq, dk, dv = rows(q), rows(k), rows(v)
    ctx = torch.full((B * Rq, H * d), 7.0, device="cuda")
    sc = torch.empty(B * H * Rq * S, device="cuda")
    hipabi.check(L.knx_hip_attention_core_ex(hipabi.ptr(dq), H * d, hipabi.ptr(dk), H * d, hipabi.ptr(dv), H * d, None,
                                             hipabi.ptr(ctx), hipabi.ptr(sc) if scores else None, B, H, Rq, S, d, d,
                                             ctypes.c_float(scale), int(causal), hipabi.stream()))
    return ctx.cpu().reshape(B, Rq, H, d).permute(0, 2, 1, 3).double().numpy()


def exact(q, k, v, scale, causal):
    s = (q.double() @ k.double().transpose(2, 3).contiguous()) * float(np.float32(scale))
    if causal:
        i, j = torch.arange(s.shape[2])[:, None], torch.arange(s.shape[3])[None]
        s = s.masked_fill(j > i, -math.inf)
    return (torch.softmax(s, -1) @ v.double()).numpy(), s


def bound(q, k, v, scale, s):
    """a score's error (six roundings per 16 of d, taken as truncations, of sums below Σ|q||k|) moves a probability by as
    much; the exponent's and the exponential's roundings; the 12 roundings per 32 keys and the rescalings of the context"""
    d, S = q.shape[3], k.shape[2]
    e = (6 * -(-d // 16) + 4) * 2.0 ** -23 * abs(scale) * float((q.abs().double() @ k.abs().double().transpose(2, 3).contiguous()).max())
    finite = s[torch.isfinite(s)].abs().max()
    e += 2.0 ** -22 * (float(finite) + 4) + (14 * -(-S // 32) + 16) * 2.0 ** -23
    return 2 * e * float(v.abs().max())


@pytest.mark.parametrize("B,H,Rq,S,d", [(1, 1, 1, 1, 4), (1, 2, 31, 33, 16), (2, 3, 128, 32, 32), (1, 8, 129, 127, 48),
                                        (2, 2, 130, 257, 64), (1, 3, 64, 500, 80), (1, 2, 300, 300, 96), (1, 2, 40, 289, 128),
                                        (1, 1, 7, 64, 100)])
@pytest.mark.parametrize("causal", [False, True])
def test_flash(L, B, H, Rq, S, d, causal, monkeypatch):
    monkeypatch.setenv("KNX_ATTN_KERNEL", "flash")
    g = torch.Generator().manual_seed(B + Rq + S + d)
    q, k, v = (torch.randn((B, H, n, d), generator=g) for n in (Rq, S, S))
    scale = 1 / math.sqrt(d)
    want, s = exact(q, k, v, scale, causal)
    assert np.max(np.abs(run(L, q, k, v, scale, causal) - want)) <= bound(q, k, v, scale, s)


@pytest.mark.parametrize("scale", [-0.3, 0.0, 3.0])
def test_scales(L, scale, monkeypatch):
    """also without scratch for the scores, which these shapes never needed"""
    monkeypatch.setenv("KNX_ATTN_KERNEL", "flash")
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn((2, 2, 100, 64), generator=g) for _ in range(3))
    want, s = exact(q, k, v, scale, True)
    assert np.max(np.abs(run(L, q, k, v, scale, True, scores=False) - want)) <= bound(q, k, v, scale, s)


def test_values_without_finite_parts(L, monkeypatch):
    """-inf scores leave a key out, NaN and +inf scores and infinite values give what fp32 arithmetic gives"""
    monkeypatch.setenv("KNX_ATTN_KERNEL", "flash")
    g = torch.Generator().manual_seed(11)
    q, k, v = (torch.randn((3, 2, 150, 64), generator=g) for _ in range(3))
    q[..., 0] = q[..., 0].abs() + 1.5
    k[0, 0, :40, 0] = -float("inf")   # the first 40 keys score -inf for every query of this head
    k[0, 1, 77, 3] = float("nan")
    v[1, 0, 20, 5] = float("inf")
    k[2, 0, 0, 0] = 3.4e38            # 1.5 · 3.4e38 and more: past the largest float, 3.4028e38, for every query
    q[1, 1, 9] = q[1, 1, 9] * 1e-39   # subnormal queries: equal weights
    want, s = exact(q, k, v, 0.125, False)
    want[2, 0] = np.nan               # (inf − inf in fp32)
    got = run(L, q, k, v, 0.125, False)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf, ok = np.isinf(want), np.isfinite(want)
    assert np.array_equal(got[inf], want[inf])
    kk = torch.nan_to_num(k, posinf=0.0, neginf=0.0)
    kk[2, 0, 0, 0] = 0.0
    lim = bound(q, kk, torch.nan_to_num(v, posinf=0.0), 0.125, torch.nan_to_num(s, posinf=0.0, neginf=0.0).clamp(-50, 50))
    assert np.max(np.abs(got[ok] - want[ok])) <= 4 * lim  # fp32 chains round every value
