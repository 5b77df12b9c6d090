"""The chunk GEMM's launcher (q35_mlx4_xprep, q35_mlx4_gemm) against a float64
product, at the edges of its kernels' tiles and of the rule that picks them.

Bound, elementwise.  The kernel adds the terms x w' with w' = 16 s (1 + q / 16)
and b - 16 s; R is their 2-norm, the size of a partial sum of inputs of random
sign.  The fp16 hi + lo split loses at most 2^-22 of each term: 2^-22 R.  A
group's 2 x 64 products are added in partial sums of size R / sqrt(G), the G
groups in about 3 G sums of size R, each rounding 2^-24 of the sum it makes:
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
# and 160 tokens), 64 x 64 with 8 waves and with 4, the general kernel by work
# and by a row count that is not a multiple of 4; K past 2048 and 4096 and M past
# 256 and 2048 for the X prep's forms
@pytest.mark.parametrize("M,Ns,K", [
    (1, (32,), 64), (2, (100, 32), 192), (33, (64,), 320), (128, (2048,), 4096),
    (7, (8192, 4096, 32, 32), 2048), (96, (8192, 512, 512), 2048), (160, (2048,), 4096),
    (64, (8192, 4096, 32, 32), 2048), (63, (8192, 512, 512), 1984),
    (129, (8192, 512, 512), 2048), (1000, (2048,), 2112), (449, (8192, 4096, 32, 32), 2048),
    (5, (99, 64), 128), (9, (68,), 8192),
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
