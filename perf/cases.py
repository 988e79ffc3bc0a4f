"""Performance cases: the tracking and training work a user of this package runs.

A case is a dict of plain values.  ``prepare`` synthesises a subject on the
GPU (multi-tensor phantom with Rician noise, as ``gpustreamlines_amd.phantom``
does on the host), loads it into a tracker and draws the seeds; ``run`` is one
pass through the public entry points.  Two of them are measured:

* ``api = "tracker"``: ``GPUTracker.generate_streamlines(seeds)``, host seeds
  in, packed host streamlines out: what a Python user calls.
* ``api = "chunk"``: one bounded chunk (``cuslines_chunk_async`` through
  ``ChunkBuffers``) with seeds and results resident on the device: what a
  pipeline that consumes streamlines on the GPU calls.
* ``api = "train"``: loss and gradient of one mini-batch of the learned PTT
  proposal (``learned.Trainer.loss_grad``).

The volume, step size, seed placement, sphere, gradient tables and chunk size
are those of ``bench.py`` (81x106x76, 160 directions + 10 b0, 724 vertices,
half the seeds in white matter and half in border voxels, 25,000-seed chunks),
of the large multi-shell workload (3 x 90 directions + 6 b0, SH order 8) and
of the tests' small phantoms.  Streamlines differ in number and length from
input to input, so ``run`` returns them in arrays of a size that the case
fixes, zero past the last one.
"""

from __future__ import annotations

import functools

import numpy as np
import torch

from gpustreamlines_amd import learned, shm
from gpustreamlines_amd._device import ChunkBuffers, DeviceTracker
from gpustreamlines_amd.direction_getters import BootDirectionGetter, ProbDirectionGetter, PttDirectionGetter
from gpustreamlines_amd.phantom import D_CSF, D_TISSUE, LAMBDA_PAR, LAMBDA_PERP
from gpustreamlines_amd.sphere import multi_shell_gtab, single_shell_gtab, symmetric_sphere
from gpustreamlines_amd.tracker import GPUTracker

STOP_THRESHOLD = 0.1
CHUNK = 25000
FULL = dict(nx=81, ny=106, nz=76)    # the benchmark volume
SMALL = dict(nx=46, ny=55, nz=41)    # a cropped subject, odd sizes
MULTI = dict(nx=61, ny=73, nz=57)    # a downsampled whole brain
# Steps per seed of the 81x106x76 phantom at 0.25 voxel (mixed seeds), from bench.py.
STEPS = dict(prob=510, ptt=433, csa=249, opdt=162)
# Streamlines reserved per seed: peaks are 45 degrees apart, the noisier bootstrap ODFs have more of them.
SLOTS = dict(prob=9, ptt=9, csa=20, opdt=20)


def _track(name, api, getter, vol, seeds, step=0.25, placement="mixed", dirs=160, order=6, verts=724, mfma=True):
    c = dict(api=api, getter=getter, seeds=seeds, step=step, placement=placement, dirs=dirs, order=order,
             verts=verts, mfma=mfma, **vol)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # a look at a handful of seeds in an interactive session: latency
        _track("prob_few", "tracker", "prob", SMALL, 64, step=0.5, placement="mask"),
        # the reference's unit of work: one 25,000-seed chunk
        _track("prob_chunk", "chunk", "prob", FULL, 25000),
        # several chunks in one launch, as whole-brain runs group them
        _track("prob_run", "chunk", "prob", FULL, 100000),
        # PTT, the headline getter: a few seeds, a chunk, a run
        _track("ptt_few", "tracker", "ptt", SMALL, 40, step=0.5, placement="mask"),
        _track("ptt_chunk", "tracker", "ptt", MULTI, 4001, step=0.4),
        _track("ptt_run", "chunk", "ptt", FULL, 25000),
        # residual bootstrap: a few seeds, a chunk, a multi-shell subject with order 8
        _track("csa_few", "tracker", "csa", SMALL, 100, step=0.5, placement="mask"),
        _track("csa_chunk", "chunk", "csa", FULL, 25000),
        _track("csa_multi", "tracker", "csa", MULTI, 6001, step=0.4, dirs=270, order=8),
        _track("opdt_run", "chunk", "opdt", FULL, 40000),
        # the bit-exact bootstrap kernel, the mode results are validated in
        _track("csa_exact", "tracker", "csa", SMALL, 3001, mfma=False),
        # training of the learned proposal: its default mini-batch
        dict(name="train_4096", api="train", pairs=4096),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["prob", "prob", "ptt", "ptt", "csa", "opdt", "exact", "train"])
    if kind == "train":
        return dict(api="train", pairs=logint(33, 60000))
    getter = rng.choice(["csa", "opdt"]) if kind == "exact" else kind
    api = rng.choice(["tracker", "chunk"])
    most = dict(prob=50000, ptt=6000, csa=6000, opdt=20000, exact=2500)[kind]
    vol = dict(nx=rng.randint(37, 80), ny=rng.randint(37, 90), nz=rng.randint(33, 75))
    tables = [(160, 6), (160, 6), (101, 6), (270, 8)]
    dirs, order = rng.choice(tables[:dict(csa=4, opdt=3).get(getter, 1)])
    return _track(None, api, getter, vol, logint(24, most),
                  step=round(rng.uniform(0.2, 0.5), 3), placement=rng.choice(["mask", "mixed"]), dirs=dirs, order=order,
                  verts=rng.choice([724, 724, 362]), mfma=kind != "exact")


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _sphere(n):
    return symmetric_sphere(n)


@functools.lru_cache(maxsize=None)
def _gtab(dirs):
    return multi_shell_gtab(n_per_shell=dirs // 3) if dirs % 3 == 0 else single_shell_gtab(n_dirs=dirs)


@functools.lru_cache(maxsize=None)
def _dti_pinv(dirs):
    g, b = _gtab(dirs).bvecs, _gtab(dirs).bvals
    X = np.stack([np.ones_like(b), -b * g[:, 0] ** 2, -b * g[:, 1] ** 2, -b * g[:, 2] ** 2, -2 * b * g[:, 0] * g[:, 1],
                  -2 * b * g[:, 0] * g[:, 2], -2 * b * g[:, 1] * g[:, 2]], axis=1)
    return np.linalg.pinv(X).astype(np.float32)


@functools.lru_cache(maxsize=None)
def _csa_matrices(dirs, order, verts):
    gt = _gtab(dirs)
    fit = shm.csa_fit_matrix(gt.bvecs[~gt.b0s_mask], order, 0.006)
    _, th, phi = shm.cart2sphere(*_sphere(verts)[0].astype(np.float64).T)
    return fit.astype(np.float32), shm.real_sh_descoteaux(order, th, phi)[0].astype(np.float32)


def _dev(a):
    return torch.as_tensor(np.asarray(a, dtype=np.float32), device="cuda")


def _field(rng, grid, ncomp, nmodes, freq):
    """Smooth random field [n, ncomp]: a sum of low-frequency plane waves."""
    cols = []
    for _ in range(ncomp):
        k = _dev(rng.uniform(-freq, freq, size=(3, nmodes)) * 2 * np.pi)
        ph, a = _dev(rng.uniform(0, 2 * np.pi, nmodes)), _dev(rng.normal(size=nmodes))
        cols.append(torch.sin(grid @ k + ph) @ a)
    return torch.stack(cols, dim=-1)


def _subject(case, seed):
    """(DWI [n, T], FA [n]) on the GPU, voxels in C order: 1-3 fibre
    populations per voxel on smooth direction fields, Rician noise (SNR 20),
    FA of a log-linear tensor fit."""
    rng = np.random.default_rng([seed, 7])
    shape = (case["nx"], case["ny"], case["nz"])
    unit = torch.stack(torch.meshgrid(*[torch.linspace(0, 1, s, device="cuda") for s in shape], indexing="ij"),
                       dim=-1).reshape(-1, 3)
    brain = ((2 * unit - 1) ** 2).sum(1) < 0.92 ** 2
    wm = torch.sigmoid(2.5 * (_field(rng, unit, 1, 5, 4.0)[:, 0] - 0.5)) * brain
    nf = _field(rng, unit, 2, 4, 1.5)
    nfib = 1 + (nf[:, 0] > 0.3).int()
    nfib = nfib + ((nf[:, 1] > 0.9) & (nfib == 2)).int()
    gt = _gtab(case["dirs"])
    bvecs, bvals = _dev(gt.bvecs), _dev(gt.bvals)
    aniso = torch.zeros((len(unit), len(bvals)), device="cuda")
    for k in range(3):
        d = _field(rng, unit, 3, 4, 3.0)
        cosg = (d / d.norm(dim=1, keepdim=True).clamp_min(1e-12)) @ bvecs.T
        att = torch.exp(-bvals * (LAMBDA_PERP + (LAMBDA_PAR - LAMBDA_PERP) * cosg * cosg))
        aniso += torch.where((nfib > k)[:, None], att, torch.zeros_like(att))
    aniso /= nfib[:, None]
    w = wm[:, None]
    tissue = (1 - w) * torch.exp(-bvals * D_TISSUE) + w * aniso
    sig = 1000.0 * torch.where(brain[:, None], tissue, 0.3 * torch.exp(-bvals * D_CSF).expand_as(tissue))
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 1)
    n1 = torch.randn(sig.shape, generator=gen, device="cuda")
    n2 = torch.randn(sig.shape, generator=gen, device="cuda")
    dwi = torch.sqrt((sig + 50.0 * n1) ** 2 + (50.0 * n2) ** 2)
    p = torch.log(dwi.clamp_min(1.0)) @ _dev(_dti_pinv(case["dirs"])).T
    D = torch.stack([p[:, [1, 4, 5]], p[:, [4, 2, 6]], p[:, [5, 6, 3]]], dim=1)
    md = (p[:, 1] + p[:, 2] + p[:, 3]) / 3
    dev = D - md[:, None, None] * torch.eye(3, device="cuda")
    fa = (1.5 * (dev ** 2).sum((1, 2)) / (D ** 2).sum((1, 2)).clamp_min(1e-30)).sqrt().clamp(0, 1)
    return dwi, torch.where(brain, fa, torch.zeros_like(fa))


def _odf(case, dwi, fa):
    """CSA ODF amplitudes, clipped at 0 and zero below the FA threshold."""
    b0 = torch.as_tensor(_gtab(case["dirs"]).b0s_mask, device="cuda")
    fit, smat = _csa_matrices(case["dirs"], case["order"], case["verts"])
    x = (dwi[:, ~b0] / dwi[:, b0].mean(1, keepdim=True)).clamp(0.001, 0.999)
    coef = torch.log(-torch.log(x)) @ _dev(fit).T
    coef[:, 0] = shm.CSA_C0
    odf = (coef @ _dev(smat).T).clamp_min(0)
    odf[fa < STOP_THRESHOLD] = 0
    return odf


def _seeds(case, fa, rng):
    """Uniform over FA > 0.2 voxels ("mask"), or every other seed in a
    0.05 <= FA <= 0.15 border voxel ("mixed"), jittered inside the voxel."""
    shape, n = fa.shape, case["seeds"]
    pools = [np.argwhere(fa > 0.2)]
    if case["placement"] == "mixed":
        pools.append(np.argwhere((fa >= 0.05) & (fa <= 0.15)))
    out = np.empty((n, 3), dtype=np.float32)
    for k, pool in enumerate(pools):
        m = len(out[k::len(pools)])
        out[k::len(pools)] = pool[rng.integers(0, len(pool), m)] + rng.uniform(-0.5, 0.5, (m, 3))
    return out


def _pairs(n, rng):
    """Training pairs as the getter records them: ODF tap sums, direction and
    frame, and the 24 measured supports (between 0 and 9)."""
    p = np.zeros((n, learned.PAIR), dtype=np.float32)
    base = rng.beta(2.0, 1.5, size=(n, 1))
    p[:, :24] = 2 * np.clip(base + 0.25 * rng.standard_normal((n, 24)), 0, 1)
    p[:, 24] = base[:, 0]
    q = rng.standard_normal((n, 2, 3))
    t = q[:, 0] / np.linalg.norm(q[:, 0], axis=1, keepdims=True)
    u = np.cross(t, q[:, 1])
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    p[:, 28:31], p[:, 31:34], p[:, 34:37], p[:, 37:40] = t, t, u, np.cross(t, u)
    p[:, 40:] = np.clip(base + 4 * p[:, :24] + 0.3 * rng.standard_normal((n, 24)), 0, 9)
    return p


# ---------------------------------------------------------------------------
# states
# ---------------------------------------------------------------------------
class _Device:
    """The tracker of one subject and its chunk buffers; their device memory
    goes when the last tensor that views it does."""

    def __init__(self, tracker):
        self.tracker, self.chunk = tracker, None
        tracker.__enter__()

    def __del__(self):
        if self.chunk is not None:
            self.chunk.close()
        self.tracker.__exit__(None, None, None)


class _View:
    """A device buffer as an array (``__cuda_array_interface__``)."""

    def __init__(self, device, buf, shape, typestr):
        self.device = device
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(buf.ptr, False), version=2)


class Tracking:
    """What a tracking program keeps: the subject on the device, the seeds,
    and for resident chunks the chunk's buffers."""

    def __init__(self, case, seed):
        self.case = case
        rng = np.random.default_rng([seed, 11])
        shape = (case["nx"], case["ny"], case["nz"])
        verts, edges = _sphere(case["verts"])
        dwi, fa = _subject(case, seed)
        kind = case["getter"]
        if kind in ("csa", "opdt"):
            make = BootDirectionGetter.from_dipy_csa if kind == "csa" else BootDirectionGetter.from_dipy_opdt
            dg = make(_gtab(case["dirs"]), verts, sh_order_max=case["order"])
            dg.mfma = case["mfma"]
            data = dwi
        else:
            dg = ProbDirectionGetter() if kind == "prob" else PttDirectionGetter(prepare_on_device=True)
            data = _odf(case, dwi, fa)
        host = torch.empty(data.shape, pin_memory=True).copy_(data)
        data = host.reshape(shape + (-1,)).numpy()
        fa = fa.reshape(shape).cpu().numpy()
        self.seeds = _seeds(case, fa, rng)
        self.tracker = GPUTracker(dg, data, fa, STOP_THRESHOLD, verts, edges, step_size=case["step"],
                                  rng_seed=int(seed) & 0xFFFFFFFF, chunk_size=CHUNK)
        self.device = _Device(self.tracker)
        self.tracker.dataf = None  # the volume is on the device
        if case["api"] == "chunk":
            n = len(self.seeds)
            self.chunk = self.device.chunk = cb = ChunkBuffers(self.tracker.device_trackers[0], n, SLOTS[kind] * n)
            cb.sd.upload(self.seeds)
            self.views = [torch.as_tensor(_View(self.device, b, s, t), device="cuda") for b, s, t in (
                (cb.od, (n + 1,), "<i4"), (cb.ssd, (cb.cap,), "<i4"), (cb.sld, (cb.cap,), "<i4"),
                (cb.pod, (cb.cap + 1,), "<i8"), (cb.ptd, (_point_cap(case), 3), "<f4"))]
            for v in self.views:
                v.zero_()


class Training:
    """A trainer of the learned proposal and its pairs on the device."""

    def __init__(self, case, seed):
        self.case = case
        n = case["pairs"]
        self.dt = DeviceTracker(dict(dimx=2, dimy=2, dimz=2, dimt=32, model_type=2, nverts=32, nedges=32,
                                     max_sline_len=501, step_size=0.25, max_angle=1.0472, tc_threshold=STOP_THRESHOLD,
                                     relative_peak_thresh=0.25, min_separation_angle=0.785, min_signal=1.0))
        self.trainer = learned.Trainer(self.dt, learned.init_params(int(seed)), batch=n)
        self.pairs = self.dt.alloc(4 * learned.PAIR * n)
        self.pairs.upload(_pairs(n, np.random.default_rng([seed, 11])))

    def __del__(self):
        self.trainer.free()
        self.pairs.free()
        self.dt.close()


def _point_cap(case):
    """Points kept room for: about 3 times a typical run's, at most what the slots hold."""
    n = case["seeds"]
    typical = n * STEPS[case["getter"]] * 0.25 / case["step"] * (2 if case["placement"] == "mask" else 1)
    typical *= 2 if case["order"] > 6 else 1
    return min(int(3 * typical) + 100000, n * SLOTS[case["getter"]] * 1001)


def _padded(a, n):
    if len(a) > n:
        raise RuntimeError("the streamlines do not fit")
    out = np.zeros((n,) + a.shape[1:], dtype=a.dtype)
    out[:len(a)] = a
    return out


def prepare(case, seed):
    return (Training if case["api"] == "train" else Tracking)(case, seed)


def run(state):
    case = state.case
    if case["api"] == "train":
        loss, grad = state.trainer.loss_grad(state.pairs.ptr, case["pairs"])
        return dict(loss=np.array([loss], dtype=np.float32), grad=grad)
    n = len(state.seeds)
    if case["api"] == "tracker":
        slots = SLOTS[case["getter"]] * n
        s = state.tracker.generate_streamlines(state.seeds)
        return dict(points=_padded(s._data, _point_cap(case)), offsets=_padded(s._offsets, slots),
                    lengths=_padded(s._lengths, slots))
    cb = state.chunk
    cb.enqueue(n, min(n, CHUNK))
    nsl, tracked, npts = cb.totals()
    if tracked < nsl or npts > _point_cap(case):
        raise RuntimeError("the streamlines do not fit")
    off, sseed, slen, poff, pts = state.views
    return dict(streamlines=nsl, offsets=off, seeds=sseed, lengths=slen, point_offsets=poff, points=pts)


def exact(case, seed):
    """Training: loss and gradient in float64.  Tracking draws from random
    streams and each step depends on the last one's rounding: no such value."""
    if case["api"] != "train":
        return None
    rng = np.random.default_rng([seed, 11])
    p = _pairs(case["pairs"], rng).astype(np.float64)
    x, t = (torch.as_tensor(a, device="cuda") for a in (p[:, :learned.N_IN], p[:, learned.N_IN:]))
    w = learned.init_params(int(seed))
    # the forward pass uses the parameters rounded to bf16, as inference does
    par = torch.as_tensor(w).to(torch.bfloat16).to(torch.float64).cuda().requires_grad_(True)
    sizes = [(learned.N_H, learned.N_IN), (learned.N_H, learned.N_H), (learned.N_OUT, learned.N_H)]
    h, at = x, 0
    for k, (no, ni) in enumerate(sizes):
        h = h @ par[at:at + no * ni].reshape(no, ni).T + par[at + no * ni:at + no * ni + no]
        at += no * ni + no
        h = h.relu() if k < 2 else h
    loss = ((h - t) ** 2).mean()
    loss.backward()
    return dict(loss=loss.detach().reshape(1), grad=par.grad)


def work(case):
    if case["api"] == "train":
        n = case["pairs"]
        mac = learned.N_H * learned.N_IN, learned.N_H * learned.N_H, learned.N_OUT * learned.N_H
        return dict(bytes=4 * (learned.PAIR * n + 2 * learned.NPARAM), flops=2 * n * (3 * sum(mac) - mac[0]))
    kind, nv = case["getter"], case["verts"]
    vox = case["nx"] * case["ny"] * case["nz"]
    steps = case["seeds"] * STEPS[kind] * 0.25 / case["step"]
    channels = nv if kind in ("prob", "ptt") else case["dirs"] + 10
    if kind == "prob":  # interpolate every vertex, threshold, cone test, running sum
        flops = steps * nv * (16 + 2 + 6 + 1)
    elif kind == "ptt":  # 24 curves x 8 probes per sub-step: frame and tap
        flops = steps * round(case["step"] / 0.025) * (1 + 24 * 8) * (100 + 30)
    else:  # interpolation, low-rank hat product, fit, ODF projection, peak test
        nc = 28 if case["order"] == 6 else 45
        flops = steps * (16 * channels + 2 * case["dirs"] * nc * 3 + 2 * nv * nc + 16 * nv)
    touched = min(4 * vox * channels, steps * 8 * channels * 4)
    return dict(bytes=touched + 12 * steps + 12 * case["seeds"], flops=flops)
