"""The chunk GEMM's launcher (q35_mlx4_xprep, q35_mlx4_gemm) against a float64
product, at the edges of its kernels' tiles and of the rule that picks them.

Bound, elementwise.  The kernel adds the terms x q s and b x; R is the 2-norm
of terms at least as large (x 16 s (1 + q / 16) and x (b - 16 s)), the size of a
partial sum of inputs of random sign.  The digits lose at most 2^-24 of a
block's largest |x|, for normal x at most 2^-22 of the block's rms: 2^-22 R.  A
group's 5 digits are added in partial sums of size R / sqrt(G), the G groups in
about 3 G sums of size R, each rounding 2^-24 of the sum it makes:
sqrt(128 + 3 G) 2^-24 R as a random walk.  Both times 4 for the tail over the
outputs.  A group left out or taken twice is off by R / sqrt(G).
"""
import ctypes

import numpy as np
import pytest

from ds4f_hip import lib as PL

pytestmark = pytest.mark.gpu
vp, ci = ctypes.c_void_p, ctypes.c_int


class Job(ctypes.Structure):
    _fields_ = [("vals", vp), ("sb", vp), ("y", vp), ("N", ci), ("ldy", ci)]


class Gemm(ctypes.Structure):
    _fields_ = [("xw", vp), ("xsum", vp), ("jobs", Job * 4), ("njobs", ci), ("M", ci), ("Mpad", ci),
                ("K", ci), ("accumulate", ci)]


class Xprep(ctypes.Structure):
    _fields_ = [("x", vp), ("norm_w", vp), ("xw", vp), ("xsum", vp), ("M", ci), ("Mpad", ci), ("K", ci),
                ("ldx", ci), ("status", vp)]


# (M, rows of the jobs, K): 32 x 32 tiles (one token, one group; an odd group
# count; a ragged width), 32 x 64 (a layer's rows; half-empty last tiles at 96
# and 160 tokens), 64 x 64, the general kernel by work (one and two groups
# among them) and by a row count that is not a multiple of 4; K past 2048 and
# 4096 and M past 256 and 2048 for the X prep's forms
@pytest.mark.parametrize("M,Ns,K", [
    (1, (32,), 64), (2, (100, 32), 192), (33, (64,), 320), (128, (2048,), 4096),
    (7, (8192, 4096, 32, 32), 2048), (96, (8192, 512, 512), 2048), (160, (2048,), 4096),
    (64, (8192, 4096, 32, 32), 2048), (63, (8192, 512, 512), 1984),
    (129, (8192, 512, 512), 2048), (1000, (2048,), 2112), (449, (8192, 4096, 32, 32), 2048),
    (5, (99, 64), 128), (9, (68,), 8192), (66, (35,), 64), (3, (257, 5), 192),
    (257, (64,), 2048), (258, (32,), 8192), (2049, (32,), 2048), (2055, (32,), 4096), (2050, (32,), 8192)])
@pytest.mark.parametrize("accumulate", [0, 1])
def test_gemm_matches_float64(M, Ns, K, accumulate):
    import torch

    lib = PL.load()
    PL.check(lib.ds4f_gpu_init(), "init")
    print(f"gemm M={M} N={Ns} K={K} accumulate={accumulate}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M * 10007 + K)
    G, Mpad = K // 64, (M + 63) // 64 * 64
    nan = float("nan")
    ldx = K + 8
    xbuf = torch.full((M, ldx), nan, device="cuda")
    xbuf[:, :K] = torch.randn((M, K), generator=g, device="cuda")
    x = xbuf[:, :K].double()
    xw = torch.full((Mpad * K * 2,), nan, device="cuda", dtype=torch.float16)
    xsum = torch.full((G * Mpad,), nan, device="cuda")
    xp = Xprep(xbuf.data_ptr(), None, xw.data_ptr(), xsum.data_ptr(), M, Mpad, K, ldx, None)
    keep, refs, mags, outs, y0s = [], [], [], [], []
    p = Gemm(xw.data_ptr(), xsum.data_ptr(), (Job * 4)(), len(Ns), M, Mpad, K, accumulate)
    for j, N in enumerate(Ns):
        vals = torch.randint(-2**31, 2**31, (N, K // 8), generator=g, device="cuda", dtype=torch.int32)
        sc = (torch.rand((N, G), generator=g, device="cuda") * 0.007 + 0.003).bfloat16()
        bi = (-sc.float() * (torch.rand((N, G), generator=g, device="cuda") * 3 + 6)).bfloat16()
        npad = (N + 255) // 256 * 256
        sb = torch.full((npad * G * 2,), nan, device="cuda")
        wt = torch.empty(npad * K // 8, device="cuda", dtype=torch.int32)
        torch.cuda.synchronize()
        assert lib.q35_mlx4_sb(vp(sc.data_ptr()), vp(bi.data_ptr()), vp(sb.data_ptr()), N, G, None) == 0
        assert lib.q35_mlx4_wt(vp(vals.data_ptr()), vp(wt.data_ptr()), N, K, None) == 0
        sh = 4 * torch.arange(8, device="cuda", dtype=torch.int32)
        q = ((vals.view(-1, 1) >> sh) & 15).view(N, G, 64).double()
        s64, b64 = sc.double()[..., None], bi.double()[..., None]
        refs.append(x @ (q * s64 + b64).view(N, K).T)
        mags.append(((x * x) @ ((16 * s64 * (1 + q / 16)) ** 2 + (b64 - 16 * s64) ** 2).view(N, K).T).sqrt())
        ldy = N + 4                           # a column past the rows must stay as it is
        y = torch.randn((M + 1, ldy), generator=g, device="cuda")
        y0s.append(y.clone())
        outs.append(y)
        p.jobs[j] = Job(wt.data_ptr(), sb.data_ptr(), y.data_ptr(), N, ldy)
        keep.append((vals, sc, bi, sb, wt))
    torch.cuda.synchronize()
    assert lib.q35_mlx4_xprep(ctypes.byref(xp), None) == 0
    assert lib.q35_mlx4_gemm(ctypes.byref(p), None) == 0
    torch.cuda.synchronize()
    for N, ref, mag, y, y0 in zip(Ns, refs, mags, outs, y0s):
        want = ref + (y0[:M, :N].double() if accumulate else 0)
        eps = 4 * (2.0 ** -22 + np.sqrt(128 + 3 * G) * 2.0 ** -24)
        bound = eps * mag + 2.0 ** -24 * want.abs()
        worst = float(((y[:M, :N].double() - want).abs() / bound).max())
        print(f"  N={N}: {worst:.3f} of the bound", flush=True)
        assert worst <= 1.0
        assert torch.equal(y[M:], y0[M:]) and torch.equal(y[:, N:], y0[:, N:])


def _product(lib, x, norm_w, vals, sc, bi):
    """Y = X W^T through the launchers for one weight; and the status word."""
    import torch

    (M, K), N = x.shape, vals.shape[0]
    G, Mpad, npad = K // 64, (M + 63) // 64 * 64, (N + 255) // 256 * 256
    xw = torch.zeros(Mpad * K * 2, device="cuda", dtype=torch.float16)
    xsum = torch.zeros(G * Mpad, device="cuda")
    status = torch.zeros(1, device="cuda", dtype=torch.int32)
    sb = torch.empty(npad * G * 2, device="cuda")
    wt = torch.empty(npad * K // 8, device="cuda", dtype=torch.int32)
    y = torch.empty((M, N), device="cuda")
    torch.cuda.synchronize()
    xp = Xprep(x.data_ptr(), norm_w, xw.data_ptr(), xsum.data_ptr(), M, Mpad, K, K, status.data_ptr())
    p = Gemm(xw.data_ptr(), xsum.data_ptr(), (Job * 4)(), 1, M, Mpad, K, 0)
    p.jobs[0] = Job(wt.data_ptr(), sb.data_ptr(), y.data_ptr(), N, N)
    assert lib.q35_mlx4_sb(vp(sc.data_ptr()), vp(bi.data_ptr()), vp(sb.data_ptr()), N, G, None) == 0
    assert lib.q35_mlx4_wt(vp(vals.data_ptr()), vp(wt.data_ptr()), N, K, None) == 0
    assert lib.q35_mlx4_xprep(ctypes.byref(xp), None) == 0
    assert lib.q35_mlx4_gemm(ctypes.byref(p), None) == 0
    torch.cuda.synchronize()
    return y, int(status.item())


@pytest.mark.parametrize("M,N", [(40, 96), (70, 35)])     # K split over waves; the general kernel
def test_gemm_digit_exponents(M, N):
    """Rows whose blocks' exponents lie at the ends of what the digits take: zeros, the
    smallest normals, 65519, a single large column among small ones (an error of
    2^-24 of the block's largest value times the weights), values past fp16
    (flagged), infinities and NaN (NaN through the row, and no other row)."""
    import torch

    lib = PL.load()
    PL.check(lib.ds4f_gpu_init(), "init")
    K = 256
    g = torch.Generator(device="cuda").manual_seed(N)
    vals = torch.randint(-2**31, 2**31, (N, K // 8), generator=g, device="cuda", dtype=torch.int32)
    sc = (torch.rand((N, K // 64), generator=g, device="cuda") * 0.007 + 0.003).bfloat16()
    bi = (-sc.float() * 7.5).bfloat16()
    sh = 4 * torch.arange(8, device="cuda", dtype=torch.int32)
    q = ((vals.view(-1, 1) >> sh) & 15).view(N, K // 64, 64).double()
    w = (q * sc.double()[..., None] + bi.double()[..., None]).view(N, K)
    mag = (16 * sc.double()[..., None] + bi.double().abs()[..., None]).expand(N, K // 64, 64).reshape(N, K)
    x = torch.randn((M, K), generator=g, device="cuda")
    x[1] = 0
    x[2] *= 2.0 ** -120
    x[3] = 65519.0 * x[3].sign()
    x[4, 33] = 3.0e4
    x[5, :32] *= 2.0 ** -60
    x[6, 0] = 1.0e-38
    y, status = _product(lib, x, None, vals, sc, bi)
    assert status == 0
    blockmax = x.double().abs().view(M, K // 32, 32).amax(-1, keepdim=True).expand(M, K // 32, 32).reshape(M, K)
    # 2^-24 of a block's largest value (an absolute 2^-126 below the exponents' range) per
    # term, and fp32 rounding of sums of at most the terms' magnitudes
    bound = (2.0 ** -22 * blockmax + 2.0 ** -126) @ mag.T
    err = (y.double() - x.double() @ w.T).abs()
    print("worst of the bound", float((err / bound).max()), flush=True)
    assert bool((err <= bound).all()) and bool((y[1] == 0).all())
    for bad, flagged in ((65520.0, 2), (1e30, 2), (float("inf"), 2), (float("nan"), 0)):
        xb = x.clone()
        xb[7, 100] = bad
        yb, status = _product(lib, xb, None, vals, sc, bi)
        assert status == flagged
        if not np.isfinite(bad):
            assert bool(torch.isnan(yb[7]).all())
        keep = [r for r in range(M) if r != 7]
        assert torch.equal(yb[keep], y[keep])
