"""The work of a texture compressor's training program, call by call, for timing and for checking results.

A program on this framework fits a latent texture and a small decoder to an image: it initialises a Trainer with the
image and a starting model, then repeats an MLP step (the evolution-strategies population over a minibatch, late in a
run central differences), a latent step over the whole image and, with discrete selectors, a selector search; every so
often it reads the loss and the model, or the decoded error. Each case is one of those calls (or a short stretch of
them) on one model. prepare() gives what the program holds before the call, run() makes the call and reads its result
back, exact() is the same result in 64 bits from plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from neural_block_textures_amd import DctDesc, Layout, PK_UV, Trainer, dct_host, synth

MLP_SIGMA, MLP_LR, LAT_SIGMA, LAT_LR, FD_H = 0.02, 0.005, 0.05, 0.02, 1e-3
NS_LAT, NS_MLP, NS_BATCH = 1, 2, 3
PHI = 0x9E3779B97F4A7C15

# The decoders the draw takes: levels as (divisor of the image, channels, nearest), hidden width, textures, leak, --qat bits.
DECODERS = {
    "default": (((4, 4, False),), 24, 1, 0.01, ()),
    "rgb": (((4, 4, False),), 16, 1, 0.0, ()),
    "two_level": (((4, 8, False), (16, 4, False)), 32, 1, 0.0, ()),
    "plane": (((1, 1, True), (4, 4, False)), 32, 1, 0.01, ()),
    "material": (((1, 2, True), (4, 4, False)), 32, 4, 0.01, (2, 2)),
    "material36": (((1, 2, True), (4, 4, False)), 36, 4, 1.0 / 1024, (2, 2)),
    "maps36": (((4, 4, False), (8, 4, False)), 36, 4, 0.01, ()),
    "plane17": (((1, 1, True), (4, 4, False)), 17, 1, 1.0 / 1024, ()),
    "image27": (((1, 1, True), (8, 4, False)), 27, 1, 1.0 / 1024, (4,)),
    "three24": (((2, 8, False), (4, 4, False)), 24, 3, 0.01, ()),
    "large": (((2, 4, False), (8, 8, False)), 64, 4, 0.0, ()),
}


def listed():
    return [
        # the smallest work of a run: ten iterations between two progress prints of a 256 x 256 RGB image on a 64 x 64 x 4
        # latent, 16,16 decoder, population 64 on 65536 slots; launches and latency count
        {"name": "train_rgb256", "path": "train", "decoder": "rgb", "W": 256, "H": 256, "pairs": 32, "batch": 65536, "lat_pairs": 4, "its": 10},
        # the default decoder (24,24) on an image of odd size with the default population and batch: the smallest single step
        {"name": "step_default", "path": "es", "decoder": "default", "W": 250, "H": 190, "pairs": 64, "batch": 4096},
        # 512 x 512 RGB, 128 x 128 x 8 + 32 x 32 x 4 latents, 32,32, population 1024 on 65536 slots
        {"name": "step_two_level", "path": "es", "decoder": "two_level", "W": 512, "H": 512, "pairs": 512, "batch": 65536},
        # the headline: four 512 x 512 maps with 2-bit selectors, 32,32, population 8192 on 4096 slots
        {"name": "step_material512", "path": "es", "decoder": "material", "W": 512, "H": 512, "pairs": 4096, "batch": 4096},
        # a full-resolution plane beside a block latent, 32,32, population 4096
        {"name": "step_plane512", "path": "es", "decoder": "plane", "W": 512, "H": 512, "pairs": 2048, "batch": 4096},
        # the 36-wide decoder of the published material runs, everything ragged: image, population and batch
        {"name": "step_ragged36", "path": "es", "decoder": "material36", "W": 301, "H": 203, "pairs": 777, "batch": 5001},
        # the largest: four 2048 x 2048 maps, 1024 x 1024 x 4 + 256 x 256 x 8, 64,64, population 16384 on 262144 slots
        {"name": "step_large2048", "path": "es", "decoder": "large", "W": 2048, "H": 2048, "pairs": 8192, "batch": 262144},
        # the end of a run: central differences over all 1740 weights of the material's decoder
        {"name": "fd_material512", "path": "fd", "decoder": "material", "W": 512, "H": 512, "pairs": 64, "batch": 4096},
        # the latent step of two continuous levels over the whole image
        {"name": "latent_two_level", "path": "latent", "decoder": "two_level", "W": 512, "H": 512, "lat_pairs": 16},
        # four iterations of the headline workload: population, latent step, selector search, and the model read back
        {"name": "train_material512", "path": "train", "decoder": "material", "W": 512, "H": 512, "pairs": 4096, "batch": 4096, "lat_pairs": 4, "its": 4},
        # four iterations with a live DCT-coded plane: quantizer, rate proxy, shadow pull
        {"name": "train_dct512", "path": "train", "decoder": "plane", "dct": True, "W": 512, "H": 512, "pairs": 2048, "batch": 4096, "lat_pairs": 4, "its": 4},
        # the decoded error of a progress print over four 2048 x 2048 maps
        {"name": "error_large2048", "path": "error", "decoder": "large", "W": 2048, "H": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A call on a model of random size: any of the decoders, images 96 .. 1024 wide (odd sizes too), populations and
    batches over the range that the listed cases span, the work of a step no more than a sixteenth of the largest's."""
    path = rng.choice(["es", "es", "es", "fd", "latent", "latent", "image", "error"])
    name = rng.choice(sorted(DECODERS))
    c = {"path": path, "decoder": name, "W": _log(rng, 96, 1024), "H": _log(rng, 96, 1024)}
    if path in ("es", "fd"):
        c["pairs"] = _log(rng, 16, 8192) if path == "es" else 64
        most = 2 ** 27 // c["pairs"] if path == "es" else 2 ** 24 // 2048
        c["batch"] = _log(rng, 1000, max(2000, min(262144, most)))
    if path == "latent":
        c["lat_pairs"] = rng.choice([1, 2, 3, 4, 6, 8, 16])
    return c


# ---------------------------------------------------------------- inputs
def _device():
    return torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")


def _layout(case):
    levels, hidden, T, leak, _ = DECODERS[case["decoder"]]
    lv = [((case["W"] + d - 1) // d, (case["H"] + d - 1) // d, c, near) for d, c, near in levels]
    return Layout(case["W"], case["H"], lv, [hidden, hidden], T=T, pos=[PK_UV], leak=leak)


def _texture(gen, W, H, channels):
    """H x W x channels in [0, 1] as bytes / 255: four octaves of smooth noise and a few flat rectangles per channel."""
    dev, img = _device(), None
    for o in range(4):
        n = 4 << o
        grid = torch.rand((1, channels, n + 1, n + 1), generator=gen)
        up = torch.nn.functional.interpolate(grid.to(dev), size=(H, W), mode="bilinear", align_corners=True)[0]
        img = up * 0.5 ** (o + 1) if img is None else img + up * 0.5 ** (o + 1)
    for _ in range(6):
        a = torch.rand(4 + channels, generator=gen).tolist()
        x0, x1, y0, y1 = int(a[0] * W), int(a[1] * W), int(a[2] * H), int(a[3] * H)
        step = torch.tensor(a[4:], device=dev)[:, None, None] * 0.5 - 0.25
        img[:, min(y0, y1):max(y0, y1) + 1, min(x0, x1):max(x0, x1) + 1] += step
    q = torch.round(img.clamp(0, 1) * 255.0).permute(1, 2, 0).contiguous().cpu().numpy()
    return np.ascontiguousarray(q.reshape(-1).astype(np.float32) / np.float32(255.0))


def _inputs(case, seed):
    """(layout, latent, weights, target) of a run in progress: latents of the size training gives them, weights with
    the scale of their layer and small biases, selectors on their grid."""
    lay = _layout(case)
    gen = torch.Generator().manual_seed(seed)
    z = (torch.randn(lay.nz, generator=gen) * 0.4).numpy()
    widths, parts = [lay.nin, *lay.hidden, lay.nout], []
    for l in range(1, len(widths)):
        s = math.sqrt((2.0 if l + 1 < len(widths) else 1.0) / widths[l - 1])
        parts += [torch.randn(widths[l] * widths[l - 1], generator=gen) * s, torch.randn(widths[l], generator=gen) * 0.05]
    p = torch.cat(parts).numpy()
    bits = DECODERS[case["decoder"]][4]
    if bits:
        n0, g = lay.levels[0][0] * lay.levels[0][1] * lay.levels[0][2], synth.qat_grid()
        lv0 = z[:n0].reshape(-1, len(bits))
        for c, b in enumerate(bits):
            lv0[:, c] = synth.qat_snap(lv0[:, c] * np.float32(2.0), b, g)
    return lay, z, p, _texture(gen, lay.W, lay.H, lay.nout)


def prepare(case, seed):
    """An initialised Trainer on the case's model, as a program holds one between calls."""
    lay, z, p, tgt = _inputs(case, seed)
    bits = list(DECODERS[case["decoder"]][4])
    kw = dict(max_pairs=case.get("pairs", 64), max_batch=case.get("batch", 4096), seed=seed)
    if bits:
        kw.update(qat_bits=bits, qat_grid=synth.qat_grid())
    if case.get("dct"):
        kw.update(dct={"C": 1, "q": [50], "dc_step": 4}, dct_basis=dct_host.basis(), dct_zigzag=dct_host.zigzag())
    tr = Trainer()
    tr.init(Trainer.model_desc(lay, **kw), z, p, tgt, lay)
    if case.get("dct"):
        d = DctDesc()
        d.live, d.C, d.BW, d.BH, d.N, d.dc_step = 1, 1, lay.W // 8, lay.H // 8, 8, 4
        t16, d.rate_scale = dct_host.lambda_weights(80.0, lay.W, lay.H, True, True)
        d.rate_es = d.rate_trunc = 1
        for k in range(16):
            d.lam_t16[k] = t16[k]
        d.lo_w16, d.deadzone = 4, 0
        n = d.BW * d.BH
        tr.set_dct(d, np.full(n, 6, np.uint8), np.zeros(n * 64, np.int16), dct_host.steps(50, 4).reshape(-1))
        tr.dct_refit()
    w, h, c, _ = lay.levels[0]
    return {"case": case, "trainer": tr, "it": 0, "qat": bool(bits), "discrete": w * h * c if bits else 0}


# ---------------------------------------------------------------- the calls
def run(state):
    c, tr = state["case"], state["trainer"]
    path = c["path"]
    if path == "es":
        state["it"] += 1
        tr.mlp_step(state["it"], MLP_SIGMA, MLP_LR, c["pairs"], c["batch"])
        loss, spread = tr.mlp_stats()
        return {"grad": tr.debug_last_wgrad(), "loss": loss, "spread": spread}
    if path == "fd":
        state["it"] += 1
        tr.mlp_step_fd(state["it"], FD_H, MLP_LR, c["batch"])
        return {"grad": tr.debug_last_wgrad(), "loss": tr.mlp_stats()[0]}
    if path == "latent":
        state["it"] += 1
        tr.lat_step(state["it"], LAT_SIGMA, LAT_LR, c["lat_pairs"])
        return {"grad": tr.debug_last_zgrad()}
    if path == "train":
        for _ in range(c["its"]):
            state["it"] += 1
            tr.mlp_step(state["it"], MLP_SIGMA, MLP_LR, c["pairs"], c["batch"])
            tr.lat_step(state["it"], LAT_SIGMA, LAT_LR, c["lat_pairs"])
            if c.get("dct"):
                tr.shadow_pull(0, c["W"] * c["H"], 0.01)
            if state["qat"]:
                tr.qat_search()
        loss = tr.mlp_stats()[0]
        z, p = tr.download_model()
        n0 = state["discrete"]   # selectors are values of a small grid: whole values, by their bits
        out = {"selectors": z[:n0].view(np.int32), "latent": z[n0:], "weights": p, "loss": loss}
        if c.get("dct"):
            out["symbols"] = tr.download_dct()[0]
        return out
    if path == "image":
        return {"image": tr.decode_full()}
    tex, weighted = tr.decode_error()
    return {"mse": tex, "weighted": weighted}


def _macs(lay):
    widths = [lay.nin, *lay.hidden, lay.nout]
    return sum(widths[i] * widths[i + 1] for i in range(len(widths) - 1))


def work(case):
    lay = _layout(case)
    npix, path, macs = lay.W * lay.H, case["path"], _macs(lay)
    z, p, tgt = 4 * lay.nz, 4 * lay.nparams, 4 * npix * lay.nout
    bits = DECODERS[case["decoder"]][4]
    moved = sum(w * h * c for l, (w, h, c, _) in enumerate(lay.levels) if not (bits and l == 0)) * 4
    batch = case.get("batch", 0) * 4 * (lay.nin + lay.nout)
    step = {"flops": 2.0 * macs * 2 * case.get("pairs", 0) * case.get("batch", 0), "bytes": batch + 7.0 * p}
    # weights and latents are read, and read and written with their Adam moments
    lat = {"flops": 2.0 * macs * 2 * case.get("lat_pairs", 0) * npix, "bytes": z + tgt + 7.0 * moved}
    qat = {"flops": 2.0 * macs * sum(1 << b for b in bits) * npix, "bytes": z + tgt + 0.0}
    if path == "es":
        return step
    if path == "fd":
        return {"flops": 2.0 * macs * 2 * lay.nparams * case["batch"], "bytes": step["bytes"]}
    if path == "latent":
        return lat
    if path == "train":
        n = case["its"]
        return {k: n * (step[k] + lat[k] + (qat[k] if bits else 0.0)) for k in ("flops", "bytes")}
    return {"flops": 2.0 * macs * npix, "bytes": z + p + tgt + (tgt if path == "error" else 0.0)}


def tolerance(case):
    """About four times what the matrix-core path and the plain vector path (the same sums in another order) differ by on
    an MI355X, over the listed cases and drawn ones, in a first and a second pass."""
    path = case["path"]
    if path == "es":       # 3e-7 from each other, up to 7e-7 from 64 bits
        return {"rel": 5e-6}
    if path == "fd":       # differences of losses one weight apart: 4e-5, 1.7e-4 after an Adam step on them
        return {"rel": 7e-4}
    if path == "latent":   # 1.1e-6 with one pair
        return {"rel": 5e-6, "max": 2e-4}
    if path == "train":    # up to 8e-5 and 2e-2 of a latent after eight Adam steps; a selector or symbol at a tie may differ
        return {"rel": 4e-4, "max": 0.1, "differ": 1e-4}
    return {"rel": 1e-6}   # the decoded values and their 8-bit error are the same to the last bits


# ---------------------------------------------------------------- 64-bit results
def _signed(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _shr(x, n):
    return (x >> n) & ((1 << (64 - n)) - 1)


def _mix(x):
    """splitmix64's output function on int64 tensors (two's complement wraps as unsigned 64-bit does)"""
    x = x + _signed(PHI)
    x = (x ^ _shr(x, 30)) * _signed(0xBF58476D1CE4E5B9)
    x = (x ^ _shr(x, 27)) * _signed(0x94D049BB133111EB)
    return x ^ _shr(x, 31)


def _bits(seed, stream, step, pairs, index):
    """the counter generator's 64 bits for each (pair, index): pairs [n, 1] against index [m]"""
    head = _mix(torch.tensor(_signed(seed ^ (stream << 56) ^ (step << 32)), device=pairs.device) ^ pairs)
    return _mix(head + index * _signed(PHI))


def _gauss(seed, stream, step, pairs, index):
    h = _bits(seed, stream, step, pairs, index)
    u1 = (_shr(h, 40) + 1).double() / 16777216.0
    u2 = (h & 0xFFFFFF).double() / 16777216.0
    return torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(2.0 * math.pi * u2)


def _taps(n_px, n_tex, near, px):
    """the two texels a pixel column reads and the weight of the second, decided in 32 bits as the format does"""
    u = (px.astype(np.float32) + np.float32(0.5)) / np.float32(n_px)
    if near:
        x0 = np.clip(np.floor(u * np.float32(n_tex)).astype(np.int64), 0, n_tex - 1)
        return x0, x0, np.zeros(px.size)
    x = u * np.float32(n_tex) - np.float32(0.5)
    i = np.floor(x).astype(np.int64)
    return np.clip(i, 0, n_tex - 1), np.clip(i + 1, 0, n_tex - 1), (px + 0.5) / n_px * n_tex - 0.5 - i


class _Model:
    """The decoder in 64-bit torch: features of pixels and the MLP over sets of weights."""

    def __init__(self, case, seed):
        self.lay, z, p, tgt = _inputs(case, seed)
        self.dev, lay = _device(), self.lay
        self.z, self.p = (torch.from_numpy(a).to(self.dev).double() for a in (z, p))
        self.p32 = p
        self.tgt = torch.from_numpy(tgt).to(self.dev).view(-1, lay.nout)
        self.cols = [_taps(lay.W, l[0], l[3], np.arange(lay.W)) for l in lay.levels]
        self.rows = [_taps(lay.H, l[1], l[3], np.arange(lay.H)) for l in lay.levels]

    def put(self, a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(self.dev)

    def level_taps(self, l, pix):
        """(texels [4, n], weights [4, n], whether the tap is one of the pixel's distinct texels)"""
        w = self.lay.levels[l][0]
        (x0, x1, fx), (y0, y1, fy) = ([self.put(a) for a in t] for t in (self.cols[l], self.rows[l]))
        x, y = pix % self.lay.W, pix // self.lay.W
        x0, x1, fx, y0, y1, fy = x0[x], x1[x], fx[x], y0[y], y1[y], fy[y]
        texel = torch.stack([y0 * w + x0, y0 * w + x1, y1 * w + x0, y1 * w + x1])
        wt = torch.stack([(1 - fx) * (1 - fy), fx * (1 - fy), (1 - fx) * fy, fx * fy])
        dx, dy = x1 != x0, y1 != y0
        return texel, wt, torch.stack([torch.ones_like(dx), dx, dy, dx & dy])

    def features(self, pix, z):
        """[nin, n] features of the pixels"""
        lay, rows = self.lay, []
        for l, (w, h, c, _) in enumerate(lay.levels):
            texel, wt, _ = self.level_taps(l, pix)
            lv = z[lay.offsets[l]:lay.offsets[l] + w * h * c].view(-1, c)
            rows.append((lv[texel] * wt[..., None]).sum(0).t())
        u, v = (pix % lay.W + 0.5).double() / lay.W, (pix // lay.W + 0.5).double() / lay.H
        return torch.cat([*rows, (2 * u - 1)[None], (2 * v - 1)[None]]).contiguous()

    def outputs(self, sets, f):
        """[members, nout, n] outputs of each weight vector in sets [members, P]"""
        lay, o, cur = self.lay, 0, f
        for l, n in enumerate([*lay.hidden, lay.nout]):
            k = cur.shape[-2]
            w, b = sets[:, o:o + n * k].reshape(-1, n, k).contiguous(), sets[:, o + n * k:o + n * k + n]
            o += n * k + n
            cur = torch.matmul(w, cur) + b[..., None]
            cur = torch.sigmoid(cur) if l == len(lay.hidden) else torch.where(cur > 0, cur, cur * float(np.float32(lay.leak)))
        return cur

    def losses(self, sets, f, t):
        """[members] weighted mean squared errors over the slots"""
        step = max(1, int(2 ** 27 // (max(self.lay.hidden) * f.shape[-1])))
        parts = [((self.outputs(s, f) - t) ** 2).sum((1, 2)) for s in sets.split(step)]
        return torch.cat(parts) / (3.0 * self.lay.T * f.shape[-1])

    def minibatch(self, seed, step, n):
        one = torch.zeros((1, 1), dtype=torch.int64, device=self.dev)
        h = _bits(seed, NS_BATCH, step, one, torch.arange(n, device=self.dev))[0]
        pix = _shr(_shr(h, 32) * (self.lay.W * self.lay.H), 32)
        return self.features(pix, self.z), self.tgt[pix].t().double().contiguous()


def _exact_es(case, seed):
    m, sigma, n = _Model(case, seed), float(np.float32(MLP_SIGMA)), case["pairs"]
    f, t = m.minibatch(seed, 1, case["batch"])
    k = torch.arange(m.p.numel(), device=m.dev)
    lp, lm, grad = [], [], torch.zeros_like(m.p)
    for i in torch.arange(n, device=m.dev).split(512):
        eps = _gauss(seed, NS_MLP, 1, i[:, None], k)
        lp.append(m.losses(m.p + sigma * eps, f, t))
        lm.append(m.losses(m.p - sigma * eps, f, t))
        grad += (lp[-1] - lm[-1]) @ eps / (2.0 * n * sigma)
    lp, lm = torch.cat(lp), torch.cat(lm)
    d = lp - lm
    spread = math.sqrt(max(0.0, float((d * d).mean() - d.mean() ** 2)))
    return {"grad": grad.cpu().numpy(), "loss": float(0.5 * (lp + lm).mean()), "spread": spread}


def _exact_fd(case, seed):
    m = _Model(case, seed)
    f, t = m.minibatch(seed, 1, case["batch"])
    up, down = m.p32 + np.float32(FD_H), m.p32 - np.float32(FD_H)   # the weights a step takes are 32-bit
    wp, wm = (m.put(a).double() for a in (up, down))
    grad = []
    for j in torch.arange(m.p.numel(), device=m.dev).split(128):
        sets = m.p.repeat(2 * j.numel(), 1)
        r = torch.arange(j.numel(), device=m.dev)
        sets[2 * r, j], sets[2 * r + 1, j] = wp[j], wm[j]
        l = m.losses(sets, f, t).view(-1, 2)
        grad.append((l[:, 0] - l[:, 1]) / (wp[j] - wm[j]))
    return {"grad": torch.cat(grad).cpu().numpy(), "loss": float(m.losses(m.p[None], f, t))}


def _exact_latent(case, seed):
    m, sigma, K = _Model(case, seed), float(np.float32(LAT_SIGMA)), case["lat_pairs"]
    lay, searched = m.lay, bool(DECODERS[case["decoder"]][4])
    npix = lay.W * lay.H
    every = torch.arange(npix, device=m.dev)
    moved = torch.ones_like(m.z)
    if searched:
        moved[:lay.levels[0][0] * lay.levels[0][1] * lay.levels[0][2]] = 0.0
    grad = torch.zeros_like(m.z)
    for k in range(K):
        eps = _gauss(seed, NS_LAT, 0, torch.tensor([[k]], device=m.dev), torch.arange(lay.nz, device=m.dev))[0] * moved
        diff = torch.zeros(npix, dtype=torch.float64, device=m.dev)
        for sign in (1.0, -1.0):
            for pix in every.split(1 << 18):
                o = m.outputs(m.p[None], m.features(pix, m.z + sign * sigma * eps))[0]
                diff[pix] += sign * ((o - m.tgt[pix].t().double()) ** 2).sum(0)
        diff /= 3.0 * lay.T * npix
        for l, (w, h, c, _) in enumerate(lay.levels):
            texel, _, distinct = m.level_taps(l, every)
            sums = torch.zeros(w * h, dtype=torch.float64, device=m.dev)
            sums.index_add_(0, texel.reshape(-1), (diff * distinct).reshape(-1))
            part = slice(lay.offsets[l], lay.offsets[l] + w * h * c)
            grad[part] += (sums[:, None] / (2.0 * K * sigma) * eps[part].view(-1, c)).reshape(-1)
    return {"grad": grad.cpu().numpy()}


def _exact_image(case, seed):
    m = _Model(case, seed)
    parts = [m.outputs(m.p[None], m.features(pix, m.z))[0].t() for pix in torch.arange(m.lay.W * m.lay.H, device=m.dev).split(1 << 18)]
    img = torch.cat(parts)
    if case["path"] == "image":
        return {"image": img.reshape(-1).cpu().numpy()}
    a, b = (torch.floor(v.double().clamp(0, 1) * 255.0 + 0.5) for v in (img, m.tgt))
    mse = ((a - b) ** 2).mean(0).view(m.lay.T, 3).mean(1)
    return {"mse": mse.cpu().numpy(), "weighted": float(mse.mean())}


def exact(case, seed):
    """What run() returns on a new state, in 64 bits. A stretch of iterations has no such value: an Adam step's size does
    not shrink with its gradient, so entries whose gradient is nearly zero take their sign from rounding."""
    path = case["path"]
    if path == "train":
        return None
    return {"es": _exact_es, "fd": _exact_fd, "latent": _exact_latent}.get(path, _exact_image)(case, seed)
