"""The work whose speed is followed, as this package's users have it done.

Inputs are synthetic and made on the GPU from the seed: a water ellipsoid with
random hot spheres, the matching mu-map, span-11 or span-1 sinograms whose
expected counts follow the chords through that ellipsoid, and list-mode word
streams of the scanner's format. Nothing of the inputs comes out of the
projectors, so both sides of a comparison see the same bytes.

``exact`` repeats a case in float64: the rays are traced from the scanner
tables (crystal positions, ring pairs, sinogram numbers: plain data that a
user's program also holds) with torch sorts, and projections are sums over the
traced pieces.
"""
import math

import numpy as np
import torch

import nipet_amd as nip
from nipet_amd.geom import get_geom
from nipet_amd.lm.mmrhist import Randoms, hist_words
from nipet_amd.mmrnorm import NormSino
from nipet_amd.prj.autograd import Projector, poisson_nll
from nipet_amd.prj.osem import osem_prepare, osem_prepare_batch, osem_run, osem_run_batch

NAW, SUBSET = 68516, 4894
NY, NX, NZ = 320, 320, 127
VOX, VOXZ, AXR, TFOV2 = 0.208626, 0.203125, 0.40625, 890.0
AXES = (9.0, 7.0, 8.0)


def listed():
    return [
        # a profile along a few rays (checks, line integrals of one view): the smallest call
        {'name': 'fp_line', 'kind': 'fp', 'bins': 16, 'span': 11},
        # the emission projection of one of the 14 OSEM subsets
        {'name': 'fp_subset', 'kind': 'fp', 'bins': SUBSET, 'span': 11},
        # attenuation factors of a whole mu-map, once per scan before reconstruction
        {'name': 'att_all', 'kind': 'att', 'bins': NAW, 'span': 11},
        # the back projection of one OSEM subset
        {'name': 'bp_subset', 'kind': 'bp', 'bins': SUBSET, 'span': 11},
        # a clinical reconstruction from corrected inputs: 4 iterations x 14 subsets
        {'name': 'osem_4x14', 'kind': 'osem', 'itr': 4, 'fwhm': 0.0},
        # one iteration with resolution modelling (4.5 mm)
        {'name': 'osem_psf', 'kind': 'osem', 'itr': 1, 'fwhm': 4.5},
        # four bootstrap replicates or frames reconstructed together, one iteration
        {'name': 'batch_4', 'kind': 'batch', 'itr': 1, 'nb': 4},
        # gradients of the Poisson likelihood (image and mu-map) over one subset
        {'name': 'nll_grad', 'kind': 'nll', 'bins': SUBSET},
        # the randoms and the normalisation sinogram of one scan
        {'name': 'corrections', 'kind': 'corr', 'span': 11},
        # a short dynamic frame: 10 s at 1e6 events/s
        {'name': 'hist_frame', 'kind': 'hist', 'seconds': 10, 'per_ms': 1000, 'nrep': 1,
         'span': 11},
        # a whole 10 min acquisition at 1e6 events/s
        {'name': 'hist_600s', 'kind': 'hist', 'seconds': 600, 'per_ms': 1000, 'nrep': 1,
         'span': 11},
        # 16 Poisson bootstrap replicates of a one-minute acquisition
        {'name': 'boot_16', 'kind': 'hist', 'seconds': 60, 'per_ms': 1000, 'nrep': 16,
         'span': 11},
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(['fp', 'fp', 'att', 'bp', 'bp', 'osem', 'batch', 'nll', 'corr', 'hist',
                       'hist', 'boot'])
    if kind in ('fp', 'att', 'bp'):
        return {'kind': kind, 'bins': log(1, SUBSET - 1) | 1, 'span': rng.choice([11, 11, 1])}
    if kind == 'osem':
        return {'kind': kind, 'itr': rng.randint(1, 3),
                'fwhm': rng.choice([0.0, round(rng.uniform(2.5, 6.0), 2)])}
    if kind == 'batch':
        return {'kind': kind, 'itr': 1, 'nb': rng.choice([2, 3, 4, 5, 6])}
    if kind == 'nll':
        return {'kind': kind, 'bins': log(64, SUBSET - 1) | 1}
    if kind == 'corr':
        return {'kind': kind, 'span': rng.choice([11, 1]), 'bias': rng.randint(100, 9000)}
    if kind == 'hist':
        return {'kind': kind, 'seconds': log(2, 300), 'per_ms': log(225, 1000), 'nrep': 1,
                'span': rng.choice([11, 11, 1])}
    return {'kind': 'hist', 'seconds': log(2, 60), 'per_ms': log(225, 1000),
            'nrep': rng.randint(2, 16), 'span': 11}


# --------------------------------------------------------------------- inputs
_PARAMS = {}


def _params(span=11):
    """Scanner parameters, one set per process as in a user's program."""
    if 11 not in _PARAMS:
        _PARAMS[11] = nip.get_mmrparams()
        _PARAMS[11]['Cnt']['SPN'] = 11
        _PARAMS[1] = dict(_PARAMS[11], Cnt=dict(_PARAMS[11]['Cnt'], SPN=1))
    return _PARAMS[span]


def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(1000003 + seed)


def _grid():
    y = (160 - torch.arange(NY, device='cuda') - 0.5) * VOX
    x = (torch.arange(NX, device='cuda') - 160 + 0.5) * VOX
    z = (torch.arange(NZ, device='cuda') - 63) * VOXZ
    return y[:, None, None], x[None, :, None], z[None, None, :]


def _phantom(seed, noise=0.1):
    """Activity 1 in the ellipsoid, 20 spheres of 0.5 .. 4, `noise` per voxel."""
    rng = np.random.default_rng(seed)
    y, x, z = _grid()
    img = ((x / AXES[0])**2 + (y / AXES[1])**2 + (z / AXES[2])**2 <= 1).float()
    for _ in range(20):
        c = rng.uniform(-0.57, 0.57, 3) * AXES
        r, a = rng.uniform(0.5, 2.5), rng.uniform(0.5, 4.0)
        img[(x - c[0])**2 + (y - c[1])**2 + (z - c[2])**2 <= r * r] = a
    return img * (1 + noise * (torch.rand(img.shape, generator=_gen(seed), device='cuda') - 0.5))


def _mumap(seed):
    """Water (0.096 /cm) with a 0.4 cm bone shell, scaled by up to 5 % with the seed."""
    y, x, z = _grid()
    s = 1 + 0.05 * np.random.default_rng(seed + 7).uniform(-1, 1)
    r = lambda k: ((x / (AXES[0] * k))**2 + (y / (AXES[1] * k))**2 +  # noqa: E731
                   (z / (AXES[2] * k))**2 <= 1)
    mu = torch.zeros((NY, NX, NZ), device='cuda')
    mu[r(s)] = 0.15
    mu[r(s * (1 - 0.4 / 7.0))] = 0.096
    return mu


def _tensor(x, dtype):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda().to(dtype)


def _chord(bins=None):
    """Chord of each transaxial bin through the ellipsoid's middle plane [cm]."""
    tx = _params()['txLUT']
    crs, s2c = _tensor(tx['crs'], torch.float64), _tensor(tx['s2c'], torch.int64)
    s2c = s2c if bins is None else s2c[bins]
    mid = 0.5 * (crs[:, :2] + crs[:, 2:]) / torch.tensor(AXES[:2], device='cuda')
    p, q = mid[s2c[:, 0]], mid[s2c[:, 1]]
    n = q - p
    dist2 = (p[:, 0] * n[:, 1] - p[:, 1] * n[:, 0])**2 / (n * n).sum(1)
    return (16.0 * (1 - dist2).clamp(min=0).sqrt()).float()


def _sino(seed, counts=3e8, bins=None):
    """Expected trues, attenuation, norm, randoms, scatter and Poisson prompts (nbins, 837)."""
    ax = _params()['axLUT']
    g = _gen(seed)
    rno, sn = _tensor(ax['li2rno'], torch.float64), _tensor(ax['li2sn'], torch.int64)
    zz = torch.zeros(837, dtype=torch.float64, device='cuda')
    n = torch.zeros_like(zz)
    for k in range(2):
        zz.index_add_(0, sn[:, k], rno.sum(1) - 63.0)
        n.index_add_(0, sn[:, k], torch.ones_like(rno[:, 0]))
    prof = (n * (1 - (zz / n * 0.5 * AXR / 14.0)**2)).float()
    ch = _chord(bins)
    shape = (ch.numel(), 837)
    attn = torch.exp(-0.096 * ch)[:, None].expand(shape).contiguous()
    norm = 0.8 + 0.4 * torch.rand(shape, generator=g, device='cuda')
    lam = ch[:, None] * prof[None, :] * attn * norm
    scale = counts * shape[0] / NAW / (float(lam.sum(dtype=torch.float64)) * 1.37)
    trues = scale * lam
    rnd = torch.full(shape, 0.12 * float(trues.mean(dtype=torch.float64)), device='cuda')
    sct = torch.exp(-((16 - ch) / 12)**2)[:, None] * prof[None, :]
    sct *= 0.25 * float(trues.sum(dtype=torch.float64)) / float(sct.sum(dtype=torch.float64))
    prompts = torch.poisson(trues + rnd + sct, generator=g).clamp_(max=65535)
    return {'trues': trues, 'attn': attn, 'norm': norm, 'randoms': rnd, 'scatter': sct,
            'prompts': prompts.to(torch.int32).to(torch.uint16)}


def _bins(case, seed):
    """Transaxial bins (host int32): a subset's own list, or some of its bins."""
    if case['bins'] == NAW:
        return None
    sub = np.asarray(nip.get_subsets14(seed % 14, _params())[0], np.int32)
    if case['bins'] >= len(sub):
        return sub
    rng = np.random.default_rng(seed)
    return np.sort(rng.choice(sub, case['bins'], replace=False)).astype(np.int32)


def _words(case, seed):
    """List-mode words: per ms a time tag and per_ms events (85 % prompts, more
    of them near the centre; delayeds uniform), 224 singles reports a second."""
    tx = _params()['txLUT']
    g = _gen(seed)
    n, per = case['seconds'] * 1000, case['per_ms']
    ali = _tensor(tx['aw2ali'], torch.int64)
    cdf = torch.cumsum((_chord() + 0.5).double(), 0)
    pick = torch.searchsorted(cdf, (torch.arange(1 << 20, device='cuda') + 0.5) *
                              (cdf[-1] / (1 << 20)))
    pick = ali[pick.clamp_(max=NAW - 1)].to(torch.int32)
    ali = ali.to(torch.int32)
    words = torch.empty((n, per + 1), dtype=torch.int32, device='cuda')
    for m in range(0, n, 50000):
        k = min(50000, n - m)
        shape = (k, per)
        u = torch.randint(0, 1 << 30, shape, generator=g, device='cuda', dtype=torch.int32)
        si = torch.randint(1, 4084, shape, generator=g, device='cuda', dtype=torch.int32)
        prompt = (u >> 20) < 870
        aw = torch.where(prompt, pick[u & 0xfffff], ali[(u & 0xfffff) % NAW])
        words[m:m + k, 1:] = si * 86688 + aw + (prompt.to(torch.int32) << 30)
    ms = torch.arange(n, device='cuda', dtype=torch.int64)
    words[:, 0] = (ms + 1000000 - (1 << 31)).to(torch.int32)
    b = torch.arange(224, device='cuda', dtype=torch.int64)
    val = torch.randint(0, 1 << 19, (case['seconds'], 224), generator=g, device='cuda')
    val[:, ::7] = 0
    words[500::1000, 1:225] = (0xA0000000 - (1 << 32) + (b << 19) + val).to(torch.int32)
    return words.reshape(-1)


def _mask():
    """The 29 cm reconstruction cylinder, one per process as in a user's program."""
    if 'mask' not in _PARAMS:
        cyl = nip.get_cylinder(_params()['Cnt'], rad=29., gpu_dim=True)
        _PARAMS['mask'] = _tensor(cyl > 0.9, torch.uint8)
    return _PARAMS['mask']


def _corr_inputs(case, seed):
    rng = np.random.default_rng(seed)
    live = (_params()['txLUT']['crsri'] >= 0)
    fan = rng.poisson(case.get('bias', 4000) * rng.uniform(0.5, 1.5, (64, 504))) * live
    u = lambda *s: rng.uniform(0.8, 1.2, s).astype(np.float32)  # noqa: E731
    comp = {'geo': u(127, 344), 'cinf': u(344, 9), 'ceff': u(64, 504), 'axe1': u(837),
            'axf1': u(4084), 'dtp': 1e-6 * u(64), 'dtnp': 2e-6 * u(64)}
    return fan.astype(np.int32), comp, rng.integers(2000, 40000, 224).astype(np.int32)


def prepare(case, seed):
    """What a user's program holds on the GPU before the call."""
    k = case['kind']
    s = {'case': case}
    if k in ('fp', 'att', 'bp'):
        s['params'] = _params(case['span'])
        bins = _bins(case, seed)
        s['isub'] = np.array([-1], np.int32) if bins is None else bins
        if k == 'bp':
            # an OSEM ratio: Poisson counts over their mean
            shape = (NAW if bins is None else len(bins), 837 if case['span'] == 11 else 4084)
            lam = 0.5 + 0.3 * _chord(None if bins is None else _tensor(bins, torch.int64))
            s['x'] = torch.poisson(lam[:, None].expand(shape).contiguous(),
                                   generator=_gen(seed)) / lam[:, None]
        else:
            s['x'] = _phantom(seed) if k == 'fp' else _mumap(seed)
        get_geom(s['params'])
    elif k in ('osem', 'batch'):
        s['params'] = _params()
        d = _sino(seed)
        s['d'] = d
        s['subs'] = [nip.get_subsets14(i, s['params'])[0] for i in range(14)]
        if k == 'osem':
            s['mask'] = _mask()
            s['psf'] = nip.psf_config(case['fwhm'], s['params']['Cnt']) if case['fwhm'] else None
        else:
            g = _gen(seed + 1)
            lam = d['prompts'].float()[:, :, None].expand(-1, -1, case['nb'])
            p = torch.poisson(lam.contiguous(), generator=g).clamp_(max=65535)
            s['prompts'] = p.to(torch.int32).to(torch.uint16)
            s['state'] = osem_prepare_batch(s['params'], s['prompts'], d['attn'], d['norm'],
                                            d['randoms'], d['scatter'])
    elif k == 'nll':
        s['params'] = _params()
        bins = _bins(case, seed)
        s['prj'] = Projector(s['params'], bins)
        s['prj'].span1()
        d = _sino(seed, bins=_tensor(bins, torch.int64))
        s['y'], s['norm'] = d['prompts'].to(torch.int32).float(), d['norm']
        s['rs'] = d['randoms'] + d['scatter']
        s['img'] = _phantom(seed) + 0.01
        s['mu'] = _mumap(seed)
    elif k == 'corr':
        s['params'] = _params(case['span'])
        fan, s['comp'], s['buckets'] = _corr_inputs(case, seed)
        s['fan'] = torch.from_numpy(fan).cuda()
        s['rnd'], s['nrm'] = Randoms(s['params']), NormSino(s['params'])
    else:
        s['params'] = _params(case['span'])
        s['words'] = _words(case, seed)
    return s


def run(s):
    case = s['case']
    k = case['kind']
    if k in ('fp', 'att'):
        return nip.frwd_prj(s['x'], s['params'], isub=s['isub'], dev_out=True,
                            attenuation=k == 'att', fullsino_out=False, sync=False)
    if k == 'bp':
        return nip.back_prj(s['x'], s['params'], isub=s['isub'], dev_out=True, sync=False)
    if k == 'osem':
        d = s['d']
        st = osem_prepare(s['params'], d['prompts'], d['attn'], d['norm'], d['randoms'],
                          d['scatter'], subsets=s['subs'], mask=s['mask'], psf=s['psf'])
        return osem_run(st, case['itr'], check_counts=False)
    if k == 'batch':
        return osem_run_batch(s['state'], case['itr'])
    if k == 'nll':
        x, mu = s['img'].detach().requires_grad_(True), s['mu'].detach().requires_grad_(True)
        phi = poisson_nll(x, mu, s['y'], s['norm'], s['rs'], s['prj'])
        return (phi.detach(),) + torch.autograd.grad(phi, (x, mu))
    if k == 'corr':
        rs, cmap = s['rnd'](s['fan'])
        return rs, cmap, s['nrm'](s['comp'], s['buckets'])
    return hist_words(s['words'], s['params'], btp=2 if case['nrep'] > 1 else 0, seed=11,
                      nrep=case['nrep'], span=case['span']).out


# ----------------------------------------------------------------------- work
def _terms(bins):
    """(LOR, voxel) pieces of `bins` rays on average: 272 transaxial segments
    and a z crossing every half ring difference, for 4084 LORs a ray."""
    return bins * 4084 * (272 + 35.0)


def work(case):
    """Inputs read once, outputs written once; two operations per (LOR, voxel)
    piece of a projection, one per PSF tap, ten per list-mode word."""
    k = case['kind']
    img = 4.0 * NY * NX * NZ
    if k in ('fp', 'att', 'bp'):
        nsn = 837 if case['span'] == 11 else 4084
        return {'bytes': img + 4.0 * case['bins'] * nsn, 'flops': 2 * _terms(case['bins'])}
    if k in ('osem', 'batch'):
        nb = case.get('nb', 1)
        sino = 4.0 * NAW * 837
        psf = 14 * case['itr'] * 2 * 3 * 17 * 2 * img / 4 if case.get('fwhm') else 0.0
        # per iteration: prompts (16 bits) and the additive term, the image and
        # 14 sensitivity images; once: attenuation, norm, randoms, scatter
        # (and the sensitivity images of a single reconstruction)
        once = 0.0 if k == 'batch' else 4 * sino
        sens = 14 * img
        pairs = 2 * case['itr'] * nb + (0 if k == 'batch' else 1)
        return {'bytes': once + case['itr'] * ((0.5 * nb + 1) * sino + sens + 28 * nb * img),
                'flops': 2 * pairs * _terms(NAW) + psf}
    if k == 'nll':
        sino = 4.0 * case['bins'] * 837
        return {'bytes': 3 * sino + 4 * img, 'flops': 2 * 5 * _terms(case['bins'])}
    if k == 'corr':
        nsn = 837 if case['span'] == 11 else 4084
        return {'bytes': 2 * 4.0 * NAW * nsn, 'flops': 2 * 2 * NAW * 4084.0}
    words = case['seconds'] * 1000.0 * (case['per_ms'] + 1)
    nsn = 837 if case['span'] == 11 else 4084
    return {'bytes': 4 * words + 2 * 4.0 * nsn * 86688 * case['nrep'],
            'flops': 10 * words * case['nrep']}


# ---------------------------------------------------------------------- exact
F = torch.float64


def _rays(bins):
    """(segment start, length, column, crystal distance) of the bins' rays, padded
    with zero-length segments: every crossing with a grid line inside the field
    of view, in order."""
    tx = _params()['txLUT']
    crs, s2c = _tensor(tx['crs'], F), _tensor(tx['s2c'], torch.int64)[bins]
    mid = 0.5 * (crs[:, :2] + crs[:, 2:])
    p, q = mid[s2c[:, 0]], mid[s2c[:, 1]]
    atn = (q - p).norm(dim=1)
    a = (q - p) / atn[:, None]
    b = (p * a).sum(1)
    sq = (b * b - (p * p).sum(1) + float(np.float32(TFOV2))).clamp(min=0).sqrt()
    vox = float(np.float32(VOX))
    lines = torch.arange(-161, 162, device='cuda', dtype=F) * vox
    t = torch.cat([(lines[None, :] - p[:, k:k + 1]) / a[:, k:k + 1] for k in (0, 1)], 1)
    ok = (t > (-b - sq)[:, None]) & (t < (-b + sq)[:, None]) & (a.abs() > 0).repeat_interleave(
        lines.numel(), 1)
    t = torch.where(ok, t, torch.full_like(t, 1e9)).sort(1).values
    n = max(2, int(ok.sum(1).max()))
    t = t[:, :n]
    live = t[:, 1:] < 1e8
    s = torch.where(live, t[:, :-1], torch.zeros_like(t[:, 1:]))
    ln = torch.where(live, t[:, 1:] - t[:, :-1], torch.zeros_like(s))
    m = s + 0.5 * ln
    u = 160 + torch.floor((p[:, :1] + a[:, :1] * m) / vox).long()
    v = 160 - torch.ceil((p[:, 1:] + a[:, 1:] * m) / vox).long()
    return s, ln, (u + NX * v).clamp_(0, NX * NY - 1), atn


def _pieces(bins):
    """For a block of bins: pieces (weights, column, plane offset) sorted by
    (bin, ring difference d), offsets of those bags, and the obliquity factors.
    A piece of ring difference d on plane offset o of LOR (r0, r0 + d) lies on
    plane o + 2 r0, and on 2 d - o + 2 r0 of its mirror."""
    s, ln, col, atn = _rays(bins)
    d = torch.arange(61, device='cuda', dtype=F)[None, :, None]
    inv = 2 * d / atn[:, None, None]
    w0 = torch.floor(0.5 + inv * s[:, None, :])
    tb = torch.where(d > 0, (w0 + 0.5) / inv.clamp(min=1e-30), torch.full_like(w0, 1e9))
    step = torch.where(d > 0, 1 / inv.clamp(min=1e-30), torch.full_like(inv, 1e9))
    ln = ln[:, None, :].expand_as(w0)
    c1 = torch.minimum((tb - s[:, None, :]).clamp(min=0), ln)
    c2 = torch.minimum((tb + step - s[:, None, :]).clamp(min=0), ln)
    w = torch.stack([c1, c2 - c1, ln - c2], 3).reshape(-1)
    keep = (w > 0).nonzero().squeeze(1)
    nseg = s.shape[1]
    bag = keep // (3 * nseg)
    o = w0.reshape(-1)[keep // 3].long() + keep % 3
    c = col[:, None, :].expand_as(w0).reshape(-1)[keep // 3]
    count = torch.bincount(bag, minlength=len(bins) * 61)
    dd = bag % 61
    sf = torch.sqrt(1 + (2 * d[:, :, 0] * float(np.float32(VOXZ)) / atn[:, None])**2)
    rows = (c * 128 + o, c * 128 + (2 * dd - o).clamp(0, 127))
    return w[keep], rows, torch.cumsum(count, 0) - count, bag, sf


_EXACT_BLOCK = 256


def _unfold(img):
    """U[column * 128 + o][r0] = img[column][o + 2 r0], zero past the image."""
    pad = torch.zeros((NX * NY, 256), dtype=F, device='cuda')
    pad[:, :NZ] = img.reshape(-1, NZ).to(F)
    return pad.as_strided((NX * NY, 128, 64), (256, 1, 2)).reshape(-1, 64)


def _fold(u):
    """The transpose of _unfold."""
    u = u.reshape(NX * NY, 128, 64)
    pad = torch.zeros((NX * NY, 256), dtype=F, device='cuda')
    for r in range(64):
        pad[:, 2 * r:2 * r + 128] += u[:, :, r]
    return pad[:, :NZ].reshape(NY, NX, NZ)


def _lor_maps(span=11):
    """(d, r0) of every ring pair, its and its mirror's output sinogram, number
    of LORs in a sinogram."""
    ax = _params()['axLUT']
    rno = _tensor(ax['li2rno'], torch.int64)
    sn = _tensor(ax['li2sn'] if span == 11 else ax['li2sn1'], torch.int64)
    nos = _tensor(ax['li2nos'], F) if span == 11 else torch.ones(len(rno), dtype=F, device='cuda')
    return rno[:, 1] - rno[:, 0], rno[:, 0], sn, nos


def _fp_lors(u, bins):
    """Line integrals (len(bins), nli, 2) of LORs and mirrors (mirrors of direct planes: 0)."""
    d, r0, _, _ = _lor_maps()
    out = []
    for blk in torch.split(bins, _EXACT_BLOCK):
        w, rows, off, _, sf = _pieces(blk)
        v = [torch.nn.functional.embedding_bag(r, u, off, mode='sum', per_sample_weights=w)
             .reshape(len(blk), 61, 64) * sf[:, :, None] for r in rows]
        out.append(torch.stack([v[0][:, d, r0], v[1][:, d, r0] * (d > 0)], 2))
    return torch.cat(out)


def _bp_lors(vals, bins):
    """Image of LOR values (len(bins), nli, 2): the transpose of _fp_lors."""
    d, r0, _, _ = _lor_maps()
    g = torch.zeros((NX * NY * 128, 64), dtype=F, device='cuda')
    for blk, x in zip(torch.split(bins, _EXACT_BLOCK), torch.split(vals, _EXACT_BLOCK)):
        w, rows, _, bag, sf = _pieces(blk)
        for k in range(2):
            v = torch.zeros((len(blk), 61, 64), dtype=F, device='cuda')
            v[:, d, r0] = x[:, :, k] * ((d > 0) if k else 1)
            v = (v * sf[:, :, None]).reshape(-1, 64)
            g.index_add_(0, rows[k], v[bag] * w[:, None])
    return _fold(g)


def _to_sino(lors, span):
    _, _, sn, _ = _lor_maps(span)
    out = torch.zeros((lors.shape[0], 837 if span == 11 else 4084), dtype=F, device='cuda')
    mir = (_lor_maps()[0] > 0).nonzero().squeeze(1)
    out.index_add_(1, sn[:, 0], lors[:, :, 0])
    out.index_add_(1, sn[mir, 1], lors[:, mir, 1])
    return out


def _to_lors(sino, span):
    _, _, sn, _ = _lor_maps(span)
    return torch.stack([sino[:, sn[:, 0]], sino[:, sn[:, 1]]], 2)


def _blocks(bins, per=4096):
    return torch.split(bins, per)


def _fp(img, bins, span=11, att=False):
    u = _unfold(img)
    out = []
    for b in _blocks(bins):
        lors = _fp_lors(u, b)
        if att:
            lors = torch.exp(-lors) / _lor_maps(span)[3][:, None]
        out.append(_to_sino(lors, span))
    return torch.cat(out)


def _bp(sino, bins, span=11):
    out = 0
    for b, x in zip(_blocks(bins), torch.split(sino, 4096)):
        out = out + _bp_lors(_to_lors(x.to(F), span), b)
    return out


def _psf(img, k):
    """The separable 17-tap kernels along z, x and y, zero outside."""
    for row, axis in ((k[0], 2), (k[1], 1), (k[2], 0)):
        n = img.shape[axis]
        out = torch.zeros_like(img)
        for j in range(-8, 9):
            a, b = max(0, -j), min(n, n - j)
            out.narrow(axis, a, b - a).add_(img.narrow(axis, a + j, b - a), alpha=float(row[8 - j]))
        img = out
    return img


def _exact_osem(case, s):
    eps = 1e-6
    d = s['d']
    an = d['attn'].to(F) * d['norm'].to(F)
    rho = (d['randoms'].to(F) + d['scatter'].to(F)) / an
    p = d['prompts'].to(torch.int32).to(F)
    mask = s['mask'].bool()
    img = torch.ones((NY, NX, NZ), dtype=F, device='cuda')
    conv = (lambda v: _psf(v, s['psf'])) if s['psf'] is not None else (lambda v: v)
    for sub in s['subs']:
        b = _tensor(sub, torch.int64)
        sens = conv(_bp(an[b], b))
        e = _fp(conv(img), b) + rho[b]
        e = torch.where(e.abs() < eps, torch.zeros_like(e), p[b] / e)
        q = conv(_bp(e, b)) / sens
        img = torch.where(mask & (sens.abs() >= eps), img * q, torch.zeros_like(img))
    return img


def _exact_nll(case, seed, s):
    bins = s['prj'].subs.long()
    _, _, _, nos = _lor_maps()
    u = _unfold(s['mu'])
    t = torch.exp(-_fp_lors(u, bins))
    del u
    a = _to_sino(t / nos[:, None], 11)
    ax = _fp(s['img'], bins)
    n, y = s['norm'].to(F), s['y'].to(F)
    yb = a * n * ax + s['rs'].to(F)
    phi = (yb - torch.where(y > 0, y * torch.log(yb), torch.zeros_like(yb))).sum()
    dy = 1 - y / yb
    gx = _bp(dy * a * n, bins)
    gmu = -_bp_lors(t * _to_lors(dy * n * ax, 11) / nos[:, None], bins)
    return phi, gx, gmu


def _members(span):
    """Ring pairs of the span-1 sinograms and their output sinogram."""
    ax = _params()['axLUT']
    out = np.arange(4084) if span == 1 else np.asarray(ax['sn1_sn11'], np.int64)
    return np.asarray(ax['sn1_rno'], np.int64), out


def _pair_products(a, b, span, w=None):
    """sum over the span-1 members (r0, r1) of each sinogram of w a[., r0] b[., r1]."""
    rno, out = _members(span)
    res = torch.zeros((837 if span == 11 else 4084, a.shape[1]), dtype=F, device='cuda')
    for si in range(4084):
        x = a[rno[si, 0]] * b[rno[si, 1]]
        res[out[si]] += x if w is None else x * w[si]
    return res.T.contiguous()


def _exact_corr(case, seed):
    span = case['span']
    tx, ax, Cnt = _params()['txLUT'], _params()['axLUT'], _params()['Cnt']
    fan, comp, bck = _corr_inputs(case, seed)
    live = np.nonzero(np.asarray(tx['crsri']) >= 0)[0]
    f = _tensor(fan[:, live].T, F)                       # (448, 64)
    cij = _tensor(np.asarray(tx['cij']) != 0, F)
    r = torch.arange(64, device='cuda')
    band = ((r[:, None] - r[None, :]).abs() <= Cnt['MRD']).to(F)
    sng = torch.sqrt(f / (cij @ torch.ones_like(f) @ band))
    for _ in range(10):
        sng = 0.5 * sng + 0.5 * f / (cij @ sng @ band)
    c = _tensor(tx['s2cr'], torch.int64)
    rs = _pair_products(sng[c[:, 0]].T.contiguous(), sng[c[:, 1]].T.contiguous(), span)
    cmap = torch.zeros((504, 64), dtype=F, device='cuda')
    cmap[_tensor(live, torch.int64)] = sng
    t = {k: _tensor(v, F) for k, v in comp.items()}
    q = 0.5 * _tensor(bck, F)[(torch.arange(504, device='cuda') // 18)[None, :] + 28 *
                              (r // 8)[:, None]]
    den = 1 + q * t['dtnp'][:, None]
    e = t['ceff'] * torch.exp(q * t['dtp'][:, None] / den) / den
    ali = _tensor(tx['aw2ali'], torch.int64)
    w, a = ali % 344, ali // 344
    c1 = torch.floor((a + 0.5 * (504 - 2 + 172 - w)) % 504).long()
    c2 = torch.floor((a + 0.5 * (1008 - 2 - 172 + w)) % 504).long()
    s11 = _tensor(ax['sn1_sn11'], torch.int64)
    nos = _tensor(ax['sn1_sn11no'], F)
    wt = t['axf1'] / t['axe1'][s11] if span == 1 else 1 / (t['axe1'][s11] * nos)
    ns = _pair_products(e[:, c1], e[:, c2], span, wt)
    return rs, cmap, ns * (t['geo'][0][w] * t['cinf'][w, a % 9])[:, None]


def exact(case, seed):
    """float64 outputs of run(); None where there are only whole numbers, and
    where several iterations or replicates would take too long."""
    k = case['kind']
    if k == 'hist' or k == 'batch' or (k == 'osem' and case['itr'] > 1):
        return None
    if k == 'corr':
        return _exact_corr(case, seed)
    s = prepare(case, seed)
    if k == 'osem':
        return _exact_osem(case, s)
    if k == 'nll':
        return _exact_nll(case, seed, s)
    bins = torch.arange(NAW, device='cuda') if s['isub'][0] < 0 else _tensor(s['isub'],
                                                                              torch.int64)
    if k == 'bp':
        return _bp(s['x'], bins, case['span'])
    return _fp(s['x'], bins, case['span'], att=k == 'att')
