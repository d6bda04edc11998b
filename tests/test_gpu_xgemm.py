"""fp32 products on the bf16 matrix cores (knx_xgemm.hip): every tile at its edges, odd strides and addresses, values
that have no finite bf16 parts; depthwise convolutions; rows of any width and alignment."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from kernix_amd import hipabi  # noqa: E402
from kernix_amd.hipabi import ptr  # noqa: E402

pytestmark = pytest.mark.gpu

TILES = ["t256", "t128", "t128w8", "t64", "t64x64", "t64x64k2"]


@pytest.fixture(scope="module")
def L():
    lib = hipabi.lib()
    hipabi.check(lib.knx_hip_init())
    return lib


def bound(A, B, K):
    """six products of bf16 parts per value, summed in fp32 16 at a time: a rounding (taken as a truncation, 2^-23) of
    partial sums that are at most Σ|a||b| per addition, the parts left out below 2^-24 of it, and the result's rounding"""
    return (6 * -(-K // 16) + 4) * 2.0 ** -23 * (np.abs(A) @ np.abs(B).T) + 1e-30


def nt(L, A, lda, B, ldb, C, ldc, M, N, K, act=-1, bias=None, R=None):
    if R is None:
        hipabi.check(L.knx_hip_sgemm_nt_ep(M, N, K, A, lda, B, ldb, bias, act, 0.0, C, ldc, hipabi.stream()))
    else:
        hipabi.check(L.knx_hip_sgemm_nt_ep_res(M, N, K, A, lda, B, ldb, bias, act, 0.0, R, ldc, C, ldc, hipabi.stream()))
    torch.cuda.synchronize()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (63, 65, 17), (64, 128, 31), (129, 127, 32), (257, 63, 33), (255, 257, 100),
                                   (300, 520, 48), (513, 260, 277)])
def test_tiles(L, M, N, K, tile, monkeypatch):
    """rows of odd stride at addresses that are no multiple of 16 bytes; nothing outside M × N is written"""
    monkeypatch.setenv("KNX_SGEMM_KERNEL", tile)
    rng = np.random.default_rng(M + N + K)
    lda, ldb, ldc = K + 3, K + 1, N + 5
    A = rng.standard_normal((M, lda)).astype(np.float32)
    B = rng.standard_normal((N, ldb)).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    a = torch.cat([torch.zeros(1), torch.from_numpy(A).flatten()]).cuda()
    w = torch.cat([torch.zeros(3), torch.from_numpy(B).flatten()]).cuda()
    bias = torch.from_numpy(b).cuda()
    C = torch.full((M, ldc), 7.0, device="cuda")
    nt(L, a.data_ptr() + 4, lda, w.data_ptr() + 12, ldb, ptr(C), ldc, M, N, K, bias=ptr(bias))
    got, A, B = C.cpu().numpy(), A[:, :K].astype(np.float64), B[:, :K].astype(np.float64)
    want = A @ B.T + b
    assert np.all(np.abs(got[:, :N] - want) <= bound(A, B, K) + 2.0 ** -23 * np.abs(want))
    assert np.all(got[:, N:] == 7.0)


@pytest.mark.parametrize("tile", TILES)
def test_residual_in_place(L, tile, monkeypatch):
    monkeypatch.setenv("KNX_SGEMM_KERNEL", tile)
    M, N, K = 200, 133, 65
    g = torch.Generator().manual_seed(3)
    A, B, R = (torch.randn(s, generator=g) for s in ((M, K), (N, K), (M, N)))
    want = torch.relu(A.double() @ B.double().t()).numpy() + R.double().numpy()
    a, w, C = A.cuda(), B.cuda(), R.cuda()
    nt(L, ptr(a), K, ptr(w), K, ptr(C), N, M, N, K, act=0, R=ptr(C))
    assert np.all(np.abs(C.cpu().numpy() - want) <= bound(A.double().numpy(), B.double().numpy(), K) + 2.0 ** -22 * np.abs(want))


@pytest.mark.parametrize("tile", TILES)
def test_values_without_finite_parts(L, tile, monkeypatch):
    """infinities, NaN and values next to the largest float: the fp32 products' results"""
    monkeypatch.setenv("KNX_SGEMM_KERNEL", tile)
    M, N, K = 290, 270, 50
    g = torch.Generator().manual_seed(5)
    A, B = torch.randn((M, K), generator=g), torch.randn((N, K), generator=g)
    top = float(np.finfo(np.float32).max)
    A[3, 7], A[40, 0], A[70, 49], A[200, 5] = float("inf"), float("nan"), -float("inf"), top
    B[100, 3], B[269, 49] = float("inf"), -top
    B[:, 5] *= 2.0 ** -3  # top · B stays finite
    A[:, 49] *= 2.0 ** -3
    A[70, 49] = -float("inf")
    want = (A.double() @ B.double().t()).numpy()
    with np.errstate(over="ignore"):
        w32 = want.astype(np.float32)
    a, w, C = A.cuda(), B.cuda(), torch.empty((M, N), device="cuda")
    nt(L, ptr(a), K, ptr(w), K, ptr(C), N, M, N, K)
    got = C.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(w32))
    inf = np.isinf(w32)
    assert np.array_equal(got[inf], w32[inf])
    ok = np.isfinite(w32)
    assert ok.mean() > 0.9
    A0, B0 = (np.nan_to_num(t.double().numpy(), nan=0.0, posinf=0.0, neginf=0.0) for t in (A, B))
    # (an fp32 chain rounds every value)
    lim = bound(A0, B0, 16 * K)
    assert np.all(np.abs(got[ok] - want[ok]) <= lim[ok])


@pytest.mark.parametrize("C,Co,k,stride,dil,groups", [(24, 80, 3, 2, 1, 1), (7, 20, 5, 1, 1, 1), (91, 62, 1, 1, 1, 1),
                                                      (64, 130, 3, 1, 2, 1), (36, 24, 3, 1, 1, 2), (30, 22, 3, 1, 1, 2)])
@pytest.mark.parametrize("tile", ["256x128", "256x64", "128x128", "128x64", "64x128", "64x64k2"])
def test_convolution(L, C, Co, k, stride, dil, groups, tile, monkeypatch):
    """channel counts that are multiples of 4 and that are not, an infinite and a NaN pixel; against a direct sum"""
    monkeypatch.setenv("KNX_CONV_TILE", tile)
    Bn, H, W = 3, 13, 11
    p = dil * (k // 2)
    Ho, Wo = (H + 2 * p - dil * (k - 1) - 1) // stride + 1, (W + 2 * p - dil * (k - 1) - 1) // stride + 1
    g = torch.Generator().manual_seed(C + Co)
    x, w = torch.randn((Bn, H, W, C), generator=g), torch.randn((Co, k * k * C // groups), generator=g)
    x[1, 4, 5, 2], x[2, 12, 10, C - 1] = float("nan"), float("inf")
    xp = torch.zeros((Bn, H + 2 * p, W + 2 * p, C), dtype=torch.float64)
    xp[:, p:p + H, p:p + W] = x
    cols = torch.stack([xp[:, ky * dil:ky * dil + (Ho - 1) * stride + 1:stride, kx * dil:kx * dil + (Wo - 1) * stride + 1:stride]
                        for ky in range(k) for kx in range(k)], 3).reshape(Bn * Ho * Wo, k * k, groups, C // groups)
    K, n = k * k * C // groups, Co // groups
    geom = hipabi.ConvGeom(Bn, H, W, C, Ho, Wo, Co, k, k, stride, stride, dil, dil, p, p, groups)
    dx, dw, y = x.cuda(), w.cuda(), torch.empty((Bn * Ho * Wo, Co), device="cuda")
    hipabi.check(L.knx_hip_conv_t(ctypes.byref(geom), ptr(dx), ptr(dw), None, -1, 0.0, ptr(y), hipabi.stream()))
    got = y.cpu().numpy()
    for j in range(groups):
        A, B = cols[:, :, j].reshape(-1, K), w[j * n:(j + 1) * n].double()
        want, part = (A @ B.t()).numpy(), got[:, j * n:(j + 1) * n]
        assert np.array_equal(np.isnan(part), np.isnan(want))
        inf, ok = np.isinf(want), np.isfinite(want)
        assert np.array_equal(part[inf], want[inf])
        lim = bound(torch.nan_to_num(A, posinf=0.0).numpy(), B.numpy(), 16 * K)
        assert np.all(np.abs(part[ok] - want[ok]) <= lim[ok])


@pytest.mark.parametrize("B,H,W,C,k,stride,dil,pad", [(2, 9, 7, 4, 3, 1, 1, 1), (3, 14, 14, 174, 3, 2, 1, 1), (1, 5, 6, 3, 3, 1, 2, 2),
                                                      (2, 12, 11, 64, 5, 1, 1, 2), (1, 8, 8, 6, 7, 2, 1, 3), (2, 3, 3, 2, 1, 1, 1, 0),
                                                      (40, 33, 31, 132, 3, 1, 1, 1)])
@pytest.mark.parametrize("transposed,act,res", [(True, 0, False), (True, -1, True), (False, 1, False)])
def test_depthwise(L, B, H, W, C, k, stride, dil, pad, transposed, act, res):
    """one filter per channel, four channels per thread or one, both weight layouts, the residual in place; a rounding per
    multiply-add and a few for the epilogue (GELU: its polynomial's 1.5e-7 and the hardware exp2 and reciprocal)"""
    Ho, Wo = (H + 2 * pad - dil * (k - 1) - 1) // stride + 1, (W + 2 * pad - dil * (k - 1) - 1) // stride + 1
    g = torch.Generator().manual_seed(B + H + C + k)
    x, w, b = torch.randn((B, H, W, C), generator=g), torch.randn((C, k * k), generator=g), torch.randn(C, generator=g)
    R = torch.randn((B, Ho, Wo, C), generator=g)
    xp = torch.zeros((B, H + 2 * pad, W + 2 * pad, C), dtype=torch.float64)
    xp[:, pad:pad + H, pad:pad + W] = x
    want, mag = b.double().expand(B, Ho, Wo, C).clone(), b.abs().double().expand(B, Ho, Wo, C).clone()
    for t in range(k * k):
        ky, kx = t // k * dil, t % k * dil
        part = xp[:, ky:ky + (Ho - 1) * stride + 1:stride, kx:kx + (Wo - 1) * stride + 1:stride] * w[:, t].double()
        want, mag = want + part, mag + part.abs()
    if act == 0:
        want = torch.relu(want)
    elif act == 1:
        want = 0.5 * want * (1 + torch.erf(want / 2 ** 0.5))
    if res:
        want = want + R.double()
    geom = hipabi.ConvGeom(B, H, W, C, Ho, Wo, C, k, k, stride, stride, dil, dil, pad, pad, C)
    dx, dw, db, y = x.cuda(), (w if transposed else w.t().contiguous()).cuda(), b.cuda(), R.cuda()
    if res:
        rc = L.knx_hip_conv_t_res(ctypes.byref(geom), ptr(dx), ptr(dw), ptr(db), act, 0.0, ptr(y), ptr(y), hipabi.stream())
    else:
        entry = L.knx_hip_conv_t if transposed else L.knx_hip_conv
        rc = entry(ctypes.byref(geom), ptr(dx), ptr(dw), ptr(db), act, 0.0, ptr(y), hipabi.stream())
    hipabi.check(rc)
    lim = (k * k + 4) * 2.0 ** -24 * (mag + R.abs().double()) + (1e-6 * mag if act == 1 else 0)
    assert torch.all((y.cpu().double() - want).abs() <= lim)


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 2), (5, 63), (17, 65), (9, 127), (4, 130), (6, 257), (3, 513), (2, 1001), (2, 2047),
                                       (3, 2051), (2, 4094), (2, 4095), (2, 4096), (2, 4097)])
@pytest.mark.parametrize("offset", [0, 1])
def test_rows_of_any_width(L, rows, cols, offset):
    """layer_norm and softmax at every lanes-per-row choice, with a ragged last quad or a row address that is no multiple of
    16 bytes; masked entries and a masked row as the definition has them; nothing past a row is written.  Sums of n values
    in fp32 trees and chains of at most 64 per lane: 70 roundings and the exponential's."""
    g = torch.Generator().manual_seed(rows + cols)
    x, ga, be = torch.randn((rows, cols), generator=g) * 2, 1 + torch.randn(cols, generator=g) * 0.05, torch.randn(cols, generator=g)
    buf = torch.zeros(rows * cols + offset + 1)
    buf[offset:offset + rows * cols] = x.flatten()
    dx, y = buf.cuda(), torch.full((rows * cols + offset + 1,), 7.0, device="cuda")
    dg, db = ga.cuda(), be.cuda()
    at = lambda t: ctypes.c_void_p(t.data_ptr() + 4 * offset)  # noqa: E731
    hipabi.check(L.knx_hip_layernorm(at(dx), at(y), rows, cols, ptr(dg), ptr(db), 1e-5, hipabi.stream()))
    got = y.cpu()
    assert got[-1] == 7.0 and torch.all(got[:offset] == 7.0)
    xd = x.double()
    m = xd.mean(1, keepdim=True)
    sd = torch.sqrt(((xd - m) ** 2).mean(1, keepdim=True) + 1e-5)
    want = (xd - m) / sd * ga.double() + be.double()
    lim = 70 * 2.0 ** -24 * ((xd.abs() + m.abs() + xd.abs().mean(1, keepdim=True)) / sd * ga.abs().double() * 2 + be.abs().double())
    assert torch.all((got[offset:-1].double().reshape(rows, cols) - want).abs() <= lim)
    if cols > 2:
        x[0, 1], x[-1, cols - 1] = -float("inf"), -float("inf")
        buf[offset:offset + rows * cols] = x.flatten()
        dx = buf.cuda()
    hipabi.check(L.knx_hip_softmax(at(dx), at(y), rows, cols, hipabi.stream()))
    got = y.cpu()
    assert got[-1] == 7.0 and torch.all(got[:offset] == 7.0)
    want = torch.softmax(x.double(), 1)
    assert torch.all((got[offset:-1].double().reshape(rows, cols) - want).abs() <= (70 + 24) * 2.0 ** -24 * want)
