"""Performance cases of the denoiser: the calls that users of this package
make, over the sizes and options they make them with.

Every case runs through the public entry points of ``vbm3d_amd`` on
synthetic clips of moving rectangles over oriented sinusoids plus Gaussian
noise (the content of ``vbm3d_amd.synth``, generated on the GPU).  ``exact``
holds a 64-bit model of the same computations in plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import vbm3d_amd as V
from vbm3d_amd import api

DEV = "cuda:0"


# ---------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------
def _denoise(name, width, height, frames, channels, sigma, nb=1, flow=False, kt=1):
    return dict(name=name, kind="denoise", width=width, height=height, frames=frames, channels=channels,
                sigma=sigma, nb=nb, flow=flow, kt=kt)


def listed():
    return [
        # a thumbnail-size grey clip: launches and host work show here
        _denoise("gray_qcif", 176, 144, 10, 1, 20.0),
        # the mid-size colour clip of the test configurations
        _denoise("rgb_540p", 960, 540, 30, 3, 20.0),
        # the headline workload: a full-HD colour clip, resident on the GPU
        _denoise("rgb_1080p", 1920, 1080, 60, 3, 20.0),
        # strong noise, and the reference grid of a 16-thread run
        _denoise("gray_720p_tiled", 1280, 720, 16, 1, 40.0, nb=16),
        # optical-flow guided denoising (-fflow / -bflow), odd sizes
        _denoise("rgb_flow_odd", 637, 357, 12, 3, 30.0, flow=True),
        # temporal patches, two frames deep
        _denoise("rgb_kt2", 320, 240, 8, 3, 20.0, kt=2),
        # the drop-in entry on host buffers, as the command line calls it
        dict(name="host_rgb_540p", kind="host", width=960, height=540, frames=20, channels=3, sigma=20.0),
        # several clips of mixed size, colour and noise in one call
        dict(name="batch_mixed", kind="batch", clips=10, seed=100),
        # TV-L1 flow of one full-HD pair, and of a small odd-sized one
        dict(name="flow_1080p", kind="flow", width=1920, height=1080, sigma=20.0),
        dict(name="flow_small_odd", kind="flow", width=317, height=241, sigma=10.0),
        # multiscale denoising of a host clip (three DCT levels)
        dict(name="multiscale_360p", kind="multiscale", width=640, height=360, frames=4, channels=3, sigma=30.0,
             levels=3),
        # step 2 forward and backward: the gradient with respect to the noisy clip
        dict(name="adjoint_360p", kind="adjoint", width=640, height=360, frames=32, channels=1, sigma=25.0),
    ]


def _size(rng, lo, hi):
    """An area spread over its logarithm, with any aspect from 1:1 to 16:9
    and odd widths and heights."""
    area = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    asp = rng.uniform(1.0, 16.0 / 9.0)
    return max(48, round(math.sqrt(area * asp))), max(48, round(math.sqrt(area / asp)))


def draw(rng):
    kind = rng.choice(["denoise"] * 4 + ["host", "batch", "flow", "flow", "multiscale", "adjoint"])
    sigma = float(rng.choice([10, 20, 25, 30, 40, 50]))
    ch = rng.choice([1, 3])
    if kind == "denoise":
        opt = rng.choice(["plain", "plain", "tiled", "flow", "kt"])
        w, h = _size(rng, 100 * 80, 1920 * 1080 if opt == "plain" else (320 * 240 if opt == "kt" else 1280 * 720))
        f = rng.randint(5, 30) if opt != "kt" else rng.randint(4, 8)
        c = _denoise("", w, h, f, ch, sigma, nb=rng.choice([2, 4, 8, 16]) if opt == "tiled" and w * h > 40000 else 1,
                     flow=opt == "flow", kt=rng.choice([2, 3]) if opt == "kt" else 1)
        del c["name"]
        return c
    if kind == "batch":
        return dict(kind="batch", clips=rng.randint(2, 12), seed=rng.randint(0, 10000))
    if kind == "flow":
        w, h = _size(rng, 160 * 120, 1920 * 1080)
        return dict(kind="flow", width=w, height=h, sigma=float(rng.choice([5, 10, 20])))
    if kind == "host":
        w, h = _size(rng, 100 * 80, 960 * 540)
        return dict(kind="host", width=w, height=h, frames=rng.randint(5, 20), channels=ch, sigma=sigma)
    if kind == "multiscale":
        w, h = _size(rng, 200 * 150, 640 * 360)
        return dict(kind="multiscale", width=w, height=h, frames=rng.randint(2, 4), channels=ch, sigma=sigma, levels=3)
    w, h = _size(rng, 100 * 80, 640 * 360)
    return dict(kind="adjoint", width=w, height=h, frames=rng.randint(5, 32), channels=ch, sigma=25.0)


def _batch_specs(case):
    """(width, height, frames, channels, sigma) of each clip of a batch."""
    r = np.random.default_rng(case["seed"])
    sizes, sigmas = ((320, 240), (640, 360), (961, 541), (1280, 720)), (10.0, 20.0, 30.0, 50.0)
    return [sizes[int(r.integers(0, 4))] + (int(r.integers(8, 25)), 3 if int(r.integers(0, 2)) else 1,
                                            sigmas[int(r.integers(0, 4))]) for _ in range(case["clips"])]


# ---------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------
def _clip(width, height, frames, channels, sigma, seed):
    """Noisy clip [F][C][H][W] on the GPU: six static sinusoids, twelve
    rectangles moving up to 4 px a frame, clipped, plus white noise."""
    r = np.random.default_rng(seed)
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 1)
    yy = torch.arange(height, device=DEV, dtype=torch.float32)[:, None]
    xx = torch.arange(width, device=DEV, dtype=torch.float32)[None, :]
    off = r.uniform(64.0, 192.0, channels)
    bg = torch.empty(channels, height, width, device=DEV)
    for c in range(channels):
        bg[c] = off[c]
    for _ in range(6):
        th, per, ph = r.uniform(0, np.pi), r.uniform(8, 64), r.uniform(0, 2 * np.pi)
        wave = torch.sin((xx * math.cos(th) + yy * math.sin(th)) * (2 * np.pi / per) + ph)
        for c in range(channels):
            bg[c] += float(r.uniform(10, 30)) * wave
    rect = [(int(r.integers(-30, width)), int(r.integers(-30, height)), int(r.integers(10, 61)),
             int(r.integers(10, 61)), int(r.integers(-4, 5)), int(r.integers(-4, 5)), r.uniform(0, 255, channels))
            for _ in range(12)]
    out = torch.empty(frames, channels, height, width, device=DEV)
    for t in range(frames):
        out[t] = bg
        for x, y, w, h, vx, vy, col in rect:
            x0, y0 = x + vx * t, y + vy * t
            xa, xb, ya, yb = max(0, x0), min(width, x0 + w), max(0, y0), min(height, y0 + h)
            if xa < xb and ya < yb:
                for c in range(channels):
                    out[t, c, ya:yb, xa:xb] = float(col[c])
        out[t].clamp_(0, 255)
        out[t] += sigma * torch.randn(channels, height, width, generator=g, device=DEV)
    return out


def _flows(width, height, frames, seed):
    """Smooth forward and backward flows of up to about 3 px a frame."""
    r = np.random.default_rng(seed + 7)
    yy = torch.arange(height, device=DEV, dtype=torch.float32)[:, None]
    xx = torch.arange(width, device=DEV, dtype=torch.float32)[None, :]
    ff = torch.empty(max(frames - 1, 1), 2, height, width, device=DEV)
    for t in range(ff.shape[0]):
        for k in range(2):
            a, b, p, q = r.uniform(0.3, 1.5), r.uniform(0.3, 1.5), r.uniform(30, 90), r.uniform(30, 90)
            ff[t, k] = a * torch.sin(xx / p + t) + b * torch.cos(yy / q - t)
    return ff, -ff


def _params(case, sigma=None):
    s = case["sigma"] if sigma is None else sigma
    kt = case.get("kt", 1)
    opt = dict(kt=kt) if kt > 1 else {}
    return V.initialize_parameters_1(s, **opt), V.initialize_parameters_2(s, **opt)


def _case_clip(case, seed):
    return _clip(case["width"], case["height"], case["frames"], case["channels"], case["sigma"], seed)


def _pair(case, seed):
    z = _clip(case["width"], case["height"], 2, 1, case["sigma"], seed)
    return z[0, 0].contiguous(), z[1, 0].contiguous()


def _adjoint_inputs(case, seed):
    z = _case_clip(case, seed)
    noise = torch.Generator(device=DEV).manual_seed(int(seed) + 2)
    # a pilot estimate: the clip with most of its noise averaged away
    k = torch.ones(case["channels"], 1, 5, 5, device=DEV) / 25
    basic = torch.nn.functional.conv2d(z, k, padding=2, groups=case["channels"]).contiguous()
    grad = torch.randn(z.shape, generator=noise, device=DEV)
    return z, basic, grad


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "denoise":
        st["pristine"] = _case_clip(case, seed)
        # a grey clip is left as it was; a colour clip goes through the
        # colour round trip in place, so a program that keeps it copies it
        st["noisy"] = st["pristine"] if case["channels"] == 1 else torch.empty_like(st["pristine"])
        st["basic"], st["final"] = torch.empty_like(st["pristine"]), torch.empty_like(st["pristine"])
        st["ff"], st["bf"] = _flows(case["width"], case["height"], case["frames"], seed) if case["flow"] else (None, None)
        st["p1"], st["p2"] = _params(case)
    elif kind == "host":
        st["pristine"] = _case_clip(case, seed).cpu().numpy()
        st["noisy"], st["basic"], st["final"] = (np.empty_like(st["pristine"]) for _ in range(3))
        st["p1"], st["p2"] = _params(case)
    elif kind == "batch":
        st["items"], st["pristine"] = [], []
        for i, (w, h, f, c, s) in enumerate(_batch_specs(case)):
            z = _clip(w, h, f, c, s, 1000 * seed + i)
            st["pristine"].append(z)
            st["items"].append(V.BatchItem(s, z if c == 1 else z.clone()))
    elif kind == "flow":
        st["I0"], st["I1"] = _pair(case, seed)
        st["u"], st["v"] = torch.empty_like(st["I0"]), torch.empty_like(st["I0"])
        st["p"] = V.tvl1_params()
        st["p"].nscales = V.tvl1_nscales(case["width"], case["height"], st["p"].zfactor, st["p"].nscales)
    elif kind == "multiscale":
        st["noisy"] = _case_clip(case, seed).cpu().numpy()
    else:
        st["noisy"], st["basic"], st["grad"] = _adjoint_inputs(case, seed)
        st["final"] = torch.empty_like(st["noisy"])
        st["p2"] = V.initialize_parameters_2(case["sigma"])
    torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "denoise":
        if case["channels"] == 3:
            st["noisy"].copy_(st["pristine"])
        V.run_device(case["sigma"], st["noisy"], st["basic"], st["final"], st["p1"], st["p2"], True, case["nb"],
                     fflow_t=st["ff"], bflow_t=st["bf"], stream=torch.cuda.current_stream())
        return [st["noisy"], st["basic"], st["final"]]
    if kind == "host":
        np.copyto(st["noisy"], st["pristine"])
        V.run_vbm3d(case["sigma"], st["noisy"], None, None, st["basic"], st["final"], st["p1"], st["p2"], True, 1)
        return [st["noisy"], st["basic"], st["final"]]
    if kind == "batch":
        for it, z in zip(st["items"], st["pristine"]):
            if it.noisy is not z:
                it.noisy.copy_(z)
        V.run_batch(st["items"], stream=torch.cuda.current_stream())
        return [[it.noisy, it.basic, it.denoised] for it in st["items"]]
    if kind == "flow":
        # the entry runs on its context's own stream and waits for it
        iters = V.tvl1_flow_device(st["I0"], st["I1"], st["u"], st["v"], st["p"])
        return [st["u"], st["v"], iters]
    if kind == "multiscale":
        out, noisy, den = api.multiscale_denoise(st["noisy"], case["sigma"], levels=case["levels"], return_levels=True)
        return [out, noisy, den]
    g = V.step2_adjoint(case["sigma"], st["noisy"], st["basic"], st["grad"], st["p2"], True, 1, final_t=st["final"],
                        stream=torch.cuda.current_stream())
    return [g, st["final"]]


# ---------------------------------------------------------------------
# Work of one pass
# ---------------------------------------------------------------------
def _axis_count(n, k, p):
    return (n - k) // p + 1 + (1 if (n - k) % p else 0)


def _step_flops(w, h, f, c, prm, wiener):
    """Interior count: one search window per predictive frame, folded
    (half-cost) separable transforms, a Haar transform along the group."""
    refs = _axis_count(w, prm.k, prm.p) * _axis_count(h, prm.k, prm.p) * max(f - prm.kt + 1, 1)
    k2 = prm.k * prm.k * prm.kt
    cand = prm.Ns ** 2 + 2 * min(prm.Nf, f - 1) * prm.Npr ** 2
    src = 2 if wiener else 1
    filt = prm.N * c * prm.kt * (src + 1) * 2 * prm.k ** 3 + prm.N * c * k2 * (4 * (src + 1) + 4)
    return refs * (cand * (3.0 * k2 * c + 2) + filt + 4.0 * prm.N * k2 * c)


def _denoise_flops(w, h, f, c, sigma, kt=1):
    p1, p2 = _params(dict(sigma=sigma, kt=kt))
    return _step_flops(w, h, f, c, p1, False) + _step_flops(w, h, f, c, p2, True)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        b = fl = 0.0
        for w, h, f, c, s in _batch_specs(case):
            b += 4.0 * w * h * f * c * (3 if c == 1 else 4)
            fl += _denoise_flops(w, h, f, c, s)
        return {"bytes": b, "flops": fl}
    w, h = case["width"], case["height"]
    if kind == "flow":
        # about 20 iterations per warp on every level, 60 operations each
        return {"bytes": 16.0 * w * h, "flops": 4.0 / 3 * w * h * 5 * (20 * 60 + 300)}
    f, c = case["frames"], case["channels"]
    n = float(w * h * f * c)
    if kind == "multiscale":
        # five full-size transforms' worth of folded matrix products, and the levels' denoising
        dct = f * c * w * h * (w + h) * (2 + 2 * (1 + 0.25 / 2 + 0.0625 / 4))
        fl = sum(_denoise_flops(w >> i, h >> i, f, c, case["sigma"] / 2 ** i) for i in range(case["levels"]))
        return {"bytes": 4 * n * (2 + 2 * (1 + 0.25 + 0.0625)), "flops": dct + fl}
    if kind == "adjoint":
        fl = _step_flops(w, h, f, c, V.initialize_parameters_2(case["sigma"]), True)
        p = V.initialize_parameters_2(case["sigma"])
        refs = _axis_count(w, p.k, p.p) * _axis_count(h, p.k, p.p) * f
        return {"bytes": 4 * n * 5, "flops": fl + refs * p.N * c * (4.0 * p.k ** 3 + 10 * p.k ** 2)}
    return {"bytes": 4 * n * (4 if c == 3 else 3) + (16.0 * w * h * (f - 1) if case.get("flow") else 0),
            "flops": _denoise_flops(w, h, f, c, case["sigma"], case.get("kt", 1))}


# ---------------------------------------------------------------------
# The same computations in 64 bits
# ---------------------------------------------------------------------
def _t64(a):
    return torch.as_tensor(a, dtype=torch.float64, device=DEV)


_YUV = [[0.299, 0.587, 0.114], [-0.14713, -0.28886, 0.436], [0.615, -0.51498, -0.10001]]
_RGB = [[1.0, 0.0, 1.13983], [1.0, -0.39465, -0.5806], [1.0, 2.03211, 0.0]]
_BIOR_ROWS = [
    [0.353553390593274] * 8,
    [0.219417649252501, 0.449283757993216, 0.449283757993216, 0.219417649252501,
     -0.219417649252501, -0.449283757993216, -0.449283757993216, -0.219417649252501],
    [0.569359398342846, 0.402347308162278, -0.402347308162278, -0.569359398342846,
     -0.083506045090284, 0.083506045090284, -0.083506045090284, 0.083506045090284],
    [-0.083506045090284, 0.083506045090284, -0.083506045090284, 0.083506045090284,
     0.569359398342846, 0.402347308162278, -0.402347308162278, -0.569359398342846]]


def _bior():
    m = torch.zeros(8, 8, dtype=torch.float64)
    m[:4] = torch.tensor(_BIOR_ROWS, dtype=torch.float64)
    for i in range(4):
        m[4 + i, 2 * i], m[4 + i, 2 * i + 1] = 2 ** -0.5, -(2 ** -0.5)
    return m.to(DEV), torch.linalg.inv(m).to(DEV)


def _dct(n):
    """Orthonormal DCT-II matrix [frequency][sample]."""
    k = torch.arange(n, dtype=torch.float64)[:, None]
    q = torch.arange(n, dtype=torch.float64)[None, :]
    m = torch.cos(math.pi * k * (2 * q + 1) / (2 * n)) * math.sqrt(2.0 / n)
    m[0] *= 2 ** -0.5
    return m.to(DEV)


def _haar(n):
    """Orthonormal Haar matrix, the mean first."""
    m = torch.ones(1, 1, dtype=torch.float64)
    while m.shape[0] < n:
        s = m.shape[0]
        m = torch.cat([torch.kron(m, torch.tensor([[1.0, 1.0]], dtype=torch.float64)),
                       torch.kron(torch.eye(s, dtype=torch.float64), torch.tensor([[1.0, -1.0]], dtype=torch.float64))])
        m = m * 2 ** -0.5
    return m.to(DEV)


def _kaiser(k):
    if k not in (4, 6, 7, 8, 12):
        return torch.ones(k, k, dtype=torch.float64, device=DEV)
    v = torch.kaiser_window(k, periodic=False, beta=2.0, dtype=torch.float64)
    return (torch.round(torch.outer(v, v) * 1e4) / 1e4).to(DEV)


def _axis(b, e, p):
    v = list(range(b, e + 1, p))
    return v if v[-1] == e else v + [e]


def _grid(w, h, k, p, nb, n=16):
    """Top-left corners of the reference patches of one frame, tile by tile."""
    if nb == 1:
        return [(x, y) for y in _axis(0, h - k, p) for x in _axis(0, w - k, p)]
    b = 2
    while nb % b:
        b += 1
    nw, nh = max(nb // b, b), min(nb // b, b)
    wt, ht, bord = -(-w // nw), -(-h // nh), 2 * n
    out = []
    for ty in range(nh):
        for tx in range(nw):
            ox, oy = max(0, tx * wt - bord), max(0, ty * ht - bord)
            ex, ey = min(w, (tx + 1) * wt + bord), min(h, (ty + 1) * ht + bord)
            ys = _axis(0 if oy == 0 else n, ey - oy - k - (0 if ey == h else n), p)
            xs = _axis(0 if ox == 0 else n, ex - ox - k - (0 if ex == w else n), p)
            out += [(x + ox, y + oy) for y in ys for x in xs]
    return out


class _Step:
    """One step of the filter on a 64-bit video: matching, group filtering
    and weighted aggregation."""

    def __init__(self, shape, prm, sigma, step, nb, ff, bf):
        self.F, self.C, self.H, self.W = shape
        self.p, self.step, self.ff, self.bf = prm, step, ff, bf
        if self.C == 1:
            rows = [1.0]
        else:
            rows = [math.sqrt(a * a + b * b + c * c) for a, b, c in
                    ((0.299, 0.587, 0.114), (0.169, 0.331, 0.5), (0.5, 0.419, 0.081))]
        self.sig = torch.tensor(rows, dtype=torch.float64, device=DEV) * sigma
        self.xy = torch.tensor(_grid(self.W, self.H, prm.k, prm.p, nb), device=DEV)
        k, kt, w, h, c = prm.k, prm.kt, self.W, self.H, self.C
        t, ch, y, x = torch.meshgrid(torch.arange(kt), torch.arange(c), torch.arange(k), torch.arange(k), indexing="ij")
        # offsets of a patch's samples from its corner, [kt][C][k][k]
        self.off = (t * c * h * w + ch * h * w + y * w + x).to(DEV)

    def _window(self, px, py, s):
        """Candidates (x, y, valid) of the s x s windows centred at (px, py)."""
        hs = (s - 1) // 2
        d = torch.arange(-hs, hs + 1, device=DEV)
        x = px[:, None] + d.repeat(len(d))[None]
        y = py[:, None] + d.repeat_interleave(len(d))[None]
        ok = (x >= 0) & (y >= 0) & (x <= self.W - self.p.k) & (y <= self.H - self.p.k)
        return x.clamp(0, self.W - self.p.k), y.clamp(0, self.H - self.p.k), ok

    def _dist(self, vid, ref, rx, ry, x, y, ft, ok):
        whc = self.C * self.H * self.W
        cand = ft[:, None] * whc + y * self.W + x
        acc = torch.zeros(cand.shape, dtype=torch.float64, device=DEV)
        for o in self.off.flatten().tolist():
            acc += (vid[ref + o][:, None] - vid[cand + o]) ** 2
        acc /= self.off.numel()
        acc -= self.p.d * ((x == rx[:, None]) & (y == ry[:, None]))
        return torch.where(ok, acc, math.inf)

    def match(self, vid, t):
        """Groups of the reference patches of frame t: member frame, x, y
        (sorted by distance) and the group size."""
        p, whc = self.p, self.C * self.H * self.W
        rx, ry = self.xy[:, 0], self.xy[:, 1]
        ref = t * whc + ry * self.W + rx
        x, y, ok = self._window(rx, ry, p.Ns)
        ft = torch.full_like(rx, t)
        d, i = torch.topk(self._dist(vid, ref, rx, ry, x, y, ft, ok), p.Nb, dim=1, largest=False)
        best = [(d, torch.full_like(i, t), x.gather(1, i), y.gather(1, i))]
        for sgn in (1, -1):
            cx, cy = best[0][2], best[0][3]
            fl = self.ff if sgn > 0 else self.bf
            for n in range(1, p.Nf + 1):
                tf = t + sgn * n
                if tf < 0 or tf + p.kt > self.F:
                    break
                if fl is not None:
                    fr = fl[tf - 1 if sgn > 0 else tf]
                    hk = p.k // 2
                    dx = fr[0][cy + hk, cx + hk]
                    cx = (cx + torch.sign(dx) * torch.floor(dx.abs() + 0.5)).long().clamp(0, self.W - p.k)
                    dy = fr[1][cy + hk, cx + hk]
                    cy = (cy + torch.sign(dy) * torch.floor(dy.abs() + 0.5)).long().clamp(0, self.H - p.k)
                xs, ys, oks = [], [], []
                hs = (p.Npr - 1) // 2
                for m in range(p.Nb):
                    x, y, ok = self._window(cx[:, m], cy[:, m], p.Npr)
                    for q in range(m):
                        ok = ok & ~(((x - cx[:, q:q + 1]).abs() <= hs) & ((y - cy[:, q:q + 1]).abs() <= hs))
                    xs.append(x), ys.append(y), oks.append(ok)
                x, y, ok = torch.cat(xs, 1), torch.cat(ys, 1), torch.cat(oks, 1)
                ft = torch.full_like(rx, tf)
                d, i = torch.topk(self._dist(vid, ref, rx, ry, x, y, ft, ok), p.Nb, dim=1, largest=False)
                cx, cy = x.gather(1, i), y.gather(1, i)
                best.append((d, torch.full_like(i, tf), cx, cy))
        d, ft, x, y = (torch.cat([b[k] for b in best], 1) for k in range(4))
        nsim = min(p.N, d.shape[1])
        d, i = torch.topk(d, nsim, dim=1, largest=False)
        cnt = (d <= p.tau).sum(1).clamp(min=1)
        size = 2 ** torch.floor(torch.log2(cnt.double()) + 1e-9).long()
        return ft.gather(1, i) * whc + y.gather(1, i) * self.W + x.gather(1, i), size

    def _forward(self, g, ns):
        f2 = _bior()[0] if self.p.T_2D == 1 else _dct(self.p.k)
        g = torch.einsum("ua,rntcab,vb->rntcuv", f2, g, f2)
        if self.p.kt > 1 and self.p.T_2D != 1:
            g = torch.einsum("st,rntcuv->rnscuv", _dct(self.p.kt), g)
        return torch.einsum("mn,rntcuv->rmtcuv", _haar(ns), g)

    def _inverse(self, g, ns):
        i2 = _bior()[1] if self.p.T_2D == 1 else _dct(self.p.k).T
        g = torch.einsum("mn,rmtcuv->rntcuv", _haar(ns), g)
        if self.p.kt > 1 and self.p.T_2D != 1:
            g = torch.einsum("st,rnscuv->rntcuv", _dct(self.p.kt), g)
        return torch.einsum("au,rntcuv,bv->rntcab", i2, g, i2)

    def filter(self, noisy, basic, idx, ns):
        """Filtered members and weights [R][C] of groups of ns members."""
        g = self._forward(noisy[idx[:, :, None, None, None, None] + self.off], ns)
        s = self.sig[None, None, None, :, None, None]
        if self.step == 1:
            keep = g.abs() > self.p.lambda3D * s
            keep[:, 0, 0, :, 0, 0] = True
            w = 1.0 / (self.sig ** 2 * keep.sum((1, 2, 4, 5)))
            g = g * keep
        else:
            e = self._forward(basic[idx[:, :, None, None, None, None] + self.off], ns) ** 2
            v = e / (e + s ** 2)
            w = 1.0 / (self.sig ** 2 * (v ** 2).sum((1, 2, 4, 5)))
            g = g * v
        return self._inverse(g, ns), w

    def __call__(self, noisy, basic=None):
        """Flat numerator and denominator over the whole video."""
        nz, bs = noisy.reshape(-1), None if basic is None else basic.reshape(-1)
        src = nz if self.step == 1 else bs
        num, den = torch.zeros_like(nz), torch.zeros_like(nz)
        kai = _kaiser(self.p.k)
        for t in range(self.F - self.p.kt + 1):
            idx, size = self.match(src, t)
            for ns in torch.unique(size).tolist():
                for i in torch.split(torch.nonzero(size == ns)[:, 0], 40000):
                    gi = idx[i][:, :ns]
                    est, w = self.filter(nz, bs, gi, ns)
                    kw = kai * w[:, None, None, :, None, None].expand(est.shape)
                    at = (gi[:, :, None, None, None, None] + self.off).reshape(-1)
                    num.index_add_(0, at, (kw * est).reshape(-1))
                    den.index_add_(0, at, kw.reshape(-1))
        return num, den


def _denoise64(noisy, sigma, p1, p2, nb=1, ff=None, bf=None):
    """(noisy after the colour round trip, basic, final)."""
    z = _t64(noisy)
    colour = z.shape[1] == 3
    if colour:
        z = torch.einsum("ij,fjhw->fihw", _t64(_YUV), z).contiguous()
    n1, d1 = _Step(z.shape, p1, sigma, 1, nb, ff, bf)(z)
    basic = torch.where(d1 == 0, z.reshape(-1), n1 / d1)
    n2, d2 = _Step(z.shape, p2, sigma, 2, nb, ff, bf)(z, basic)
    final = torch.where(d2 == 0, basic if nb == 1 else z.reshape(-1), n2 / d2)
    out = [z, basic.reshape(z.shape), final.reshape(z.shape)]
    if colour:
        out = [torch.einsum("ij,fjhw->fihw", _t64(_RGB), v) for v in out]
    return out


def _adjoint64(case, seed):
    z, basic, grad = (_t64(v) for v in _adjoint_inputs(case, seed))
    step = _Step(z.shape, V.initialize_parameters_2(case["sigma"]), case["sigma"], 2, 1, None, None)
    # num is linear in the noisy video: its transpose, group by group
    num, den = step(z, basic)
    final = torch.where(den == 0, basic.reshape(-1), num / den)
    u = torch.where(den == 0, torch.zeros_like(den), grad.reshape(-1) / den)
    out = torch.zeros_like(u)
    kai = _kaiser(step.p.k)
    flat, bs = z.reshape(-1), basic.reshape(-1)
    for t in range(step.F):
        idx, size = step.match(bs, t)
        for ns in torch.unique(size).tolist():
            for i in torch.split(torch.nonzero(size == ns)[:, 0], 20000):
                at = idx[i][:, :ns][:, :, None, None, None, None] + step.off
                x = flat[at].requires_grad_(True)
                e = step._forward(bs[at], ns) ** 2
                v = e / (e + step.sig[None, None, None, :, None, None] ** 2)
                w = 1.0 / (step.sig ** 2 * (v ** 2).sum((1, 2, 4, 5)))
                est = step._inverse(step._forward(x, ns) * v, ns)
                (est * kai * w[:, None, None, :, None, None] * u[at]).sum().backward()
                out.index_add_(0, at.reshape(-1), x.grad.reshape(-1))
    return [out.reshape(z.shape), final.reshape(z.shape)]


def _bicubic(img, u, v):
    """Catmull-Rom samples at (u, v); the row above is taken with the sign
    of the x position, as the flow program does.  Also: inside the image."""
    ny, nx = img.shape
    sx, sy = torch.where(u < 0, -1, 1), torch.where(v < 0, -1, 1)
    iu, iv = u.trunc().long(), v.trunc().long()
    xs = [iu - sx, iu, iu + sx, iu + 2 * sx]
    ys = [iv - sx, iv, iv + sy, iv + 2 * sy]
    inside = torch.ones_like(u, dtype=torch.bool)
    for q in xs:
        inside &= (q >= 0) & (q < nx)
    for q in ys:
        inside &= (q >= 0) & (q < ny)
    xs, ys = [q.clamp(0, nx - 1) for q in xs], [q.clamp(0, ny - 1) for q in ys]
    fx, fy = u - xs[1], v - ys[1]

    def cell(a, b, c, d, x):
        return b + 0.5 * x * (c - a + x * (2 * a - 5 * b + 4 * c - d + x * (3 * (b - c) + d - a)))
    cols = [cell(*(img[y, x] for y in ys), fy) for x in xs]
    return cell(*cols, fx), inside


def _gauss(img, sigma):
    size = int(5 * sigma) + 1
    w = [math.exp(-i * i / (2 * sigma * sigma)) for i in range(size)]
    tot = 2 * sum(w) - w[0]
    for dim in (1, 0):
        n = img.shape[dim]
        i = torch.arange(n, device=DEV)
        acc = img * w[0]
        for k in range(1, size):
            lo, hi = (i - k).abs(), i + k
            hi = torch.where(hi >= n, 2 * n - hi - 1, hi)
            acc = acc + w[k] * (img.index_select(dim, lo) + img.index_select(dim, hi))
        img = acc / tot
    return img


def _zoom(img, ny, nx, fy, fx):
    v = (torch.arange(ny, device=DEV, dtype=torch.float64) / fy)[:, None].expand(ny, nx)
    u = (torch.arange(nx, device=DEV, dtype=torch.float64) / fx)[None].expand(ny, nx)
    return _bicubic(img, u, v)[0]


def _flow64(I0, I1, prm):
    """TV-L1 flow (u, v), coarse to fine."""
    a, b = _t64(I0), _t64(I1)
    mn, mx = min(a.min(), b.min()), max(a.max(), b.max())
    lev = [[_gauss(255 * (q - mn) / (mx - mn), 0.8) for q in (a, b)]]
    zf = prm.zfactor
    for _ in range(1, prm.nscales):
        ny, nx = (int(n * zf + 0.5) for n in lev[-1][0].shape)
        zs = 0.6 * math.sqrt(1.0 / (zf * zf) - 1.0)
        lev.append([_zoom(_gauss(q, zs), ny, nx, zf, zf) for q in lev[-1]])
    u = torch.zeros_like(lev[-1][0])
    v = torch.zeros_like(u)
    lt, taut = prm.lambda_ * prm.theta, prm.tau / prm.theta
    for k in range(prm.nscales - 1, -1, -1):
        a, b = lev[k]
        ny, nx = a.shape
        jj = torch.arange(nx, device=DEV, dtype=torch.float64)[None]
        ii = torch.arange(ny, device=DEV, dtype=torch.float64)[:, None]
        pad = torch.nn.functional.pad(b[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]
        bx, by = 0.5 * (pad[1:-1, 2:] - pad[1:-1, :-2]), 0.5 * (pad[2:, 1:-1] - pad[:-2, 1:-1])
        p = torch.zeros(4, ny, nx, dtype=torch.float64, device=DEV)
        for _ in range(prm.nwarps):
            ux, vy = jj + u, ii + v
            smp = [_bicubic(q, ux, vy) for q in (b, bx, by)]
            w, gx, gy = (torch.where(s[1], s[0], 0.0) for s in smp)
            g = gx * gx + gy * gy
            rc = w - gx * u - gy * v - a
            for _it in range(300):
                rho = rc + gx * u + gy * v
                fac = torch.where(rho < -lt * g, lt, torch.where(rho > lt * g, -lt,
                                                                 torch.where(g < 1e-10, 0.0, -rho / g)))
                px, py = p[0::2].clone(), p[1::2].clone()
                px[:, :, -1] = 0
                py[:, -1, :] = 0
                dv = px + py
                dv[:, :, 1:] -= px[:, :, :-1]
                dv[:, 1:, :] -= py[:, :-1, :]
                nu, nv = u + fac * gx + prm.theta * dv[0], v + fac * gy + prm.theta * dv[1]
                err = (((nu - u) ** 2 + (nv - v) ** 2).sum() / (nx * ny))
                u, v = nu, nv
                q = torch.stack([u, v])
                dx, dy = torch.zeros_like(q), torch.zeros_like(q)
                dx[:, :, :-1] = q[:, :, 1:] - q[:, :, :-1]
                dy[:, :-1, :] = q[:, 1:, :] - q[:, :-1, :]
                ng = 1 + taut * torch.sqrt(dx * dx + dy * dy)
                p[0::2], p[1::2] = (p[0::2] + taut * dx) / ng, (p[1::2] + taut * dy) / ng
                if float(err) <= prm.epsilon ** 2:
                    break
        if k:
            fy, fx = (lev[k - 1][0].shape[d] / lev[k][0].shape[d] for d in (0, 1))
            u, v = (_zoom(q, *lev[k - 1][0].shape, fy, fx) / zf for q in (u, v))
    return [u, v, None]


def _multiscale64(case, seed):
    z = _t64(_case_clip(case, seed))
    h, w = z.shape[2:]
    sizes = [(h >> i, w >> i) for i in range(case["levels"])]
    # orthonormal transforms; a level's coefficients carry the size ratio
    coef = _dct(h) @ z @ _dct(w).T
    noisy = []
    for a, b in sizes:
        s = math.sqrt(a * b / (h * w))
        noisy.append(_dct(a).T @ (coef[:, :, :a, :b] * s) @ _dct(b))
    den = []
    for i, v in enumerate(noisy):
        s = math.floor(case["sigma"] / 2 ** i * 100 + 1e-9) / 100
        den.append(_denoise64(v, s, *_params(case, s))[2])
    out = _dct(h) @ den[0] @ _dct(w).T
    for (a, b), v in list(zip(sizes, den))[1:]:
        ba, bb = math.ceil(np.float32(a) * np.float32(0.7)), math.ceil(np.float32(b) * np.float32(0.7))
        s = math.sqrt(h * w / (a * b))
        out[:, :, :ba, :bb] = (_dct(a) @ v @ _dct(b).T)[:, :, :ba, :bb] * s
    out = _dct(h).T @ out @ _dct(w)
    return [out, noisy, den]


def exact(case, seed):
    kind = case["kind"]
    if kind == "flow":
        p = V.tvl1_params()
        p.nscales = V.tvl1_nscales(case["width"], case["height"], p.zfactor, p.nscales)
        return _flow64(*_pair(case, seed), p)
    if kind == "batch":
        if sum(w * h * f * c for w, h, f, c, _ in _batch_specs(case)) > 1.2e8:
            return None
        return [_denoise64(_clip(w, h, f, c, s, 1000 * seed + i), s, *_params(dict(sigma=s)))
                for i, (w, h, f, c, s) in enumerate(_batch_specs(case))]
    if case["width"] * case["height"] * case["frames"] * case["channels"] > 6e7:
        return None  # the 64-bit model takes longer than the case is worth
    if kind == "multiscale":
        return _multiscale64(case, seed)
    if kind == "adjoint":
        return _adjoint64(case, seed)
    ff, bf = (None, None)
    if case.get("flow"):
        ff, bf = _flows(case["width"], case["height"], case["frames"], seed)
    p1, p2 = _params(case)
    return _denoise64(_case_clip(case, seed), case["sigma"], p1, p2, case.get("nb", 1), ff, bf)
