"""Workloads of the scattering transforms, through the public modules.

A case is a dict of plain values; ``prepare`` builds the module and its
inputs on the GPU, ``run`` makes one pass, ``exact`` gives the same outputs
in 64 bits from plain torch (the modules' registered filter buffers are the
weights), ``work`` counts what a pass cannot do without.

kind        transform
scat2d      Scattering2D of a batch of images (inference)
grad2d      Scattering2D forward and the gradient in the images, from a
            cotangent as a linear head or a loss on the coefficients gives it
scat1d      Scattering1D of a batch of signals (inference)
grad1d      Scattering1D forward and the gradient in the signals
jtfs        TimeFrequencyScattering of a batch of signals
harm3d      HarmonicScattering3D of a batch of volumes
"""
import math

import numpy as np
import torch

from kymatio_amd.torch import HarmonicScattering3D, Scattering1D, Scattering2D, TimeFrequencyScattering

DEV = torch.device('cuda')
_POWERS = (1., 2.)  # integrals of the volumes' moduli


def _img(kind, batch, m, n, J, L=8, max_order=2, dtype='float32'):
    return {'kind': kind, 'batch': batch, 'm': m, 'n': n, 'J': J, 'L': L, 'max_order': max_order, 'dtype': dtype}


def _sig(kind, batch, n, J, Q, Q2=1, T='default', max_order=2):
    return {'kind': kind, 'batch': batch, 'n': n, 'J': J, 'Q': Q, 'Q2': Q2, 'T': T, 'max_order': max_order}


def listed():
    return [
        # one thumbnail: an interactive or per-request call, all latency
        dict(_img('scat2d', 1, 32, 32, 2), name='thumb_1x32_j2'),
        # a classifier's mini-batch of 128 colour thumbnails (channels are images)
        dict(_img('scat2d', 384, 32, 32, 2), name='thumbs_384x32_j2'),
        # the benchmark workload: feature extraction over 256 x 256 images
        dict(_img('scat2d', 64, 256, 256, 3), name='images_64x256_j3'),
        # 16 colour photos at the usual network input size
        dict(_img('scat2d', 48, 224, 224, 3), name='photos_48x224_j3'),
        # a few images of an odd, rectangular size
        dict(_img('scat2d', 6, 150, 203, 4), name='ragged_6x150x203_j4'),
        # the largest images of the mixed-size workload, deep averaging
        dict(_img('scat2d', 8, 512, 512, 6), name='large_8x512_j6'),
        # reconstruction / training through the transform
        dict(_img('grad2d', 32, 128, 128, 4), name='grad_32x128_j4'),
        # audio-like signals, many at once
        dict(_sig('scat1d', 256, 4096, 6, 8), name='signals_256x4096_j6q8'),
        # a few short recordings whose length is no power of two
        dict(_sig('scat1d', 3, 1000, 5, 4), name='signals_3x1000_j5q4'),
        # reconstruction of signals from their coefficients, one step
        dict(_sig('grad1d', 64, 4096, 6, 8), name='grad_64x4096_j6q8'),
        # joint time-frequency features of a batch of signals
        {'kind': 'jtfs', 'batch': 64, 'n': 4096, 'J': 6, 'J_fr': 2, 'Q': 8, 'Q2': 1, 'format': 'time',
         'name': 'jtfs_64x4096_j6q8'},
        # electronic densities of small molecules on a grid
        {'kind': 'harm3d', 'batch': 8, 'm': 32, 'n': 32, 'o': 32, 'J': 2, 'L': 3, 'max_order': 2,
         'name': 'volumes_8x32_j2l3'},
    ]


# ------------------------------------------------------------------ ranges
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(v, most=31):
    """Whether v has no prime factor above `most` (the transform's lengths)."""
    for p in (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31):
        while v % p == 0 and p <= most:
            v //= p
    return v == 1


def _ms(case):
    """Rough cost of a case, to keep drawn ones below the largest listed one."""
    w = work(case)
    return w['flops'] + 10 * w['bytes']


def draw(rng):
    """Images of 16 to 512 pixels a side (square or not, mostly no power of
    two), batches of 1 to 256, J from 1 to 6; signals of 200 to 8192 samples;
    volumes of 8 to 64 points a side."""
    cap = {}
    for c in listed():
        cap[c['kind']] = max(cap.get(c['kind'], 0), _ms(c))
    while True:
        c = _draw(rng)
        if c is not None and _ms(c) <= cap[c['kind']]:
            return c


def _draw(rng):
    kind = rng.choices(('scat2d', 'grad2d', 'scat1d', 'grad1d', 'jtfs', 'harm3d'), (9, 4, 4, 2, 1, 1))[0]
    if kind in ('scat2d', 'grad2d'):
        J = rng.randint(1, 6)
        m = _log_int(rng, max(16, 4 * 2 ** J), 512)
        n = m if rng.random() < 0.5 else _log_int(rng, max(16, 4 * 2 ** J), 512)
        if not (_smooth(m // 2 ** J + 2) and _smooth(n // 2 ** J + 2)):
            return None
        dtype = 'float64' if rng.random() < 0.1 and max(m, n) <= 160 else 'float32'
        return _img(kind, _log_int(rng, 1, 256 if kind == 'scat2d' else 64), m, n, J, rng.choice((8, 8, 8, 6, 4)),
                    rng.choice((2, 2, 2, 2, 1)), dtype)
    if kind in ('scat1d', 'grad1d'):
        J = rng.randint(3, 8)
        n = _log_int(rng, max(200, 4 * 2 ** J), 8192)
        T = rng.choice(('default', 'default', 'default', 'global'))
        Q = rng.choice((1, 4, 8, 8, 12, 16))
        c = _sig(kind, _log_int(rng, 1, 256), n, J, Q, rng.choice((1, 1, 2)) if Q > 1 else 1, T,
                 rng.choice((2, 2, 2, 1)))
        return c if _padded1d(c) <= 16384 else None
    if kind == 'jtfs':
        J, J_fr, Q = rng.randint(4, 7), rng.choice((2, 3)), rng.choice((4, 8, 8, 12))
        if not _smooth((J + 1) * Q + 8 * 2 ** J_fr):
            return None
        return {'kind': 'jtfs', 'batch': _log_int(rng, 1, 64), 'n': _log_int(rng, 4 * 2 ** J, 4096), 'J': J,
                'J_fr': J_fr, 'Q': Q, 'Q2': rng.choice((1, 1, 2)), 'format': rng.choice(('time', 'joint'))}
    sides = [rng.choice((8, 12, 16, 20, 24, 32, 40, 48, 64)) for _ in range(3)]
    if rng.random() < 0.5:
        sides = sides[:1] * 3
    return {'kind': 'harm3d', 'batch': _log_int(rng, 1, 16), 'm': sides[0], 'n': sides[1], 'o': sides[2],
            'J': rng.randint(1, 2), 'L': rng.randint(1, 3), 'max_order': rng.choice((2, 2, 1))}


def _padded1d(case):
    """Padded length of a signal: support of the low-pass on both sides."""
    n, width = case['n'], 2 ** case['J']
    return 2 ** min(math.ceil(math.log2(n + 2 * 12 * width)), int(math.floor(math.log2(3 * n - 2))))


# ------------------------------------------------------------------ inputs
def _module(case):
    k = case['kind']
    if k in ('scat2d', 'grad2d'):
        S = Scattering2D(case['J'], (case['m'], case['n']), L=case['L'], max_order=case['max_order'])
        return S.double() if case['dtype'] == 'float64' else S
    if k in ('scat1d', 'grad1d'):
        kw = {'T': 'global'} if case['T'] == 'global' else {}
        return Scattering1D(case['J'], case['n'], (case['Q'], case['Q2']), max_order=case['max_order'], **kw)
    if k == 'jtfs':
        return TimeFrequencyScattering(J=case['J'], J_fr=case['J_fr'], Q=(case['Q'], case['Q2']), shape=case['n'],
                                       format=case['format'])
    return HarmonicScattering3D(J=case['J'], shape=(case['m'], case['n'], case['o']), L=case['L'],
                                max_order=case['max_order'], integral_powers=_POWERS)


def _inputs(case, seed):
    """Images with the 1/f spectrum of photographs, scaled to [0, 1]; chirps
    in noise; sums of Gaussian densities."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    B = case['batch']
    if case['kind'] in ('scat2d', 'grad2d'):
        m, n = case['m'], case['n']
        fy = torch.fft.fftfreq(m, device=DEV, dtype=torch.float64)[:, None]
        fx = torch.fft.fftfreq(n, device=DEV, dtype=torch.float64)[None, :]
        amp = 1 / (fy.square() + fx.square()).sqrt().clamp_min(1 / max(m, n))
        z = torch.randn(B, m, n, device=DEV, generator=g)
        x = torch.fft.ifft2(torch.fft.fft2(z) * amp.float()).real
        lo, hi = x.amin((1, 2), keepdim=True), x.amax((1, 2), keepdim=True)
        x = (x - lo) / (hi - lo)
        return x.to(getattr(torch, case['dtype'])).contiguous()
    if case['kind'] in ('scat1d', 'grad1d', 'jtfs'):
        n = case['n']
        t = torch.arange(n, device=DEV, dtype=torch.float64)
        u = torch.rand(B, 4, 4, device=DEV, dtype=torch.float64, generator=g)[..., None]
        f0, slope = 0.01 + 0.39 * u[:, :, 0], (2 * u[:, :, 1] - 1) * 0.4 / n
        a, ph = torch.exp(math.log(0.1) * u[:, :, 2]), 2 * math.pi * u[:, :, 3]
        x = (a * torch.cos(2 * math.pi * (f0 * t + 0.5 * slope * t * t) + ph)).sum(1)
        return (x + 0.05 * torch.randn(B, n, device=DEV, dtype=torch.float64, generator=g)).float().contiguous()
    dims = [case['m'], case['n'], case['o']]
    axes = [torch.arange(d, device=DEV, dtype=torch.float32) for d in dims]
    x = torch.zeros([B] + dims, device=DEV)
    for _ in range(6):
        c = torch.rand(B, 3, device=DEV, generator=g)
        w = 1 + 5 * torch.rand(B, device=DEV, generator=g)
        e = [torch.exp(-0.5 * ((ax - d * (0.25 + 0.5 * c[:, i:i + 1])) / 1.5) ** 2)
             for i, (ax, d) in enumerate(zip(axes, dims))]
        x += w[:, None, None, None] * e[0][:, :, None, None] * e[1][:, None, :, None] * e[2][:, None, None, :]
    return x.contiguous()


def _out_shape(case, S):
    """Shape of the coefficients a cotangent is drawn for."""
    B, k = case['batch'], case['kind']
    if k == 'grad2d':
        J, L = case['J'], case['L']
        C = 1 + J * L + (L * L * J * (J - 1) // 2 if case['max_order'] == 2 else 0)
        return B, C, case['m'] // 2 ** J, case['n'] // 2 ** J
    C = S.output_size()
    if case['T'] == 'global':
        return B, C, 1
    r = S.log2_stride
    return B, C, S.ind_end[r] - S.ind_start[r]


def _cotangent(case, S, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 7919)
    return torch.randn(_out_shape(case, S), device=DEV, dtype=getattr(torch, case.get('dtype', 'float32')),
                       generator=g)


def prepare(case, seed):
    S = _module(case).to(DEV)
    state = {'S': S, 'x': _inputs(case, seed)}
    if case['kind'].startswith('grad'):
        state['x'].requires_grad_()
        state['w'] = _cotangent(case, S, seed)
    return state


def run(state):
    S, x = state['S'], state['x']
    if 'w' not in state:
        return S(x)
    y = S(x)
    return {'S': y.detach(), 'grad': torch.autograd.grad(y, x, state['w'])[0]}


# ------------------------------------------------------------------ work
def _fft_flops(n):
    return 5 * n * math.log2(max(n, 2))


def work(case):
    """Bytes: inputs, filters and outputs once.  Flops: the filter products
    and FFTs of every node of the scattering tree (a real field's forward
    transform at half a complex one), twice that with a gradient."""
    k, B = case['kind'], case['batch']
    if k in ('scat2d', 'grad2d'):
        J, L, it = case['J'], case['L'], 8 if case['dtype'] == 'float64' else 4
        H, W = (case['m'] // 2 ** J + 2) * 2 ** J, (case['n'] // 2 ** J + 2) * 2 ** J
        n = [H * W // 4 ** r for r in range(J + 1)]
        C = 1 + J * L
        flops, filt = _fft_flops(n[0]) / 2, sum(n[:J])
        for j in range(J):
            kids = case['max_order'] == 2 and j < J - 1
            flops += L * (2 * n[0] + _fft_flops(n[j]) * (1.5 if kids else 1))
            filt += L * sum(n[:min(j + 1, max(J - 1, 1))])
            if kids:
                for j2 in range(j + 1, J):
                    flops += L * L * (2 * n[j] + _fft_flops(n[j2]))
                    C += L * L
        io = B * (case['m'] * case['n'] + C * (H // 2 ** J - 2) * (W // 2 ** J - 2)) * it
        return {'bytes': io * (2 if k == 'grad2d' else 1) + filt * it, 'flops': B * flops * (2 if k == 'grad2d' else 1)}
    if k in ('scat1d', 'grad1d', 'jtfs'):
        n, J, Q, Q2 = _padded1d(case), case['J'], case['Q'], case['Q2']
        flops, C = _fft_flops(n) / 2, 1
        second = case.get('max_order', 2) == 2
        for q in range(J * Q):
            j = q // Q
            flops += 2 * n + _fft_flops(n >> j) * 1.5
            C += 1
            if second:
                for j2 in range(j + 1, J):
                    flops += Q2 * (2 * (n >> j) + _fft_flops(n >> j2) * 1.5)
                    C += Q2
        if k == 'jtfs':
            # every second-order path again along log-frequency, by 2 J_fr + 1 wavelets
            C *= 2 * case['J_fr'] + 1
            flops *= 2 * case['J_fr'] + 2
        io = B * 4 * (case['n'] + C * (1 if case.get('T') == 'global' else max(1, case['n'] >> J)))
        filt = 4 * n * (J * Q + J * Q2 + 1)
        return {'bytes': io * (2 if k == 'grad1d' else 1) + filt, 'flops': B * flops * (2 if k == 'grad1d' else 1)}
    vol = case['m'] * case['n'] * case['o']
    J, L = case['J'], case['L']
    steps = (J + 1) + (J * (J + 1) // 2 if case['max_order'] == 2 else 0)
    per = sum((2 * l + 1) * (8 * vol + _fft_flops(vol)) for l in range(L + 1)) * steps
    per += (L + 1) * (J if case['max_order'] == 2 else 0) * _fft_flops(vol) / 2
    filt = 8 * vol * sum(2 * l + 1 for l in range(L + 1)) * (J + 1)
    return {'bytes': B * 4 * (vol + steps * (L + 1) * len(_POWERS)) + filt, 'flops': B * per}


# ------------------------------------------------------------------ 64 bits
def _levels(f):
    out = []
    for v in f['levels']:
        v = v if torch.is_tensor(v) else torch.from_numpy(np.asarray(v))
        out.append(v.to(device=DEV, dtype=torch.float64).squeeze())
    return dict(f, levels=out)


def _reflect(n, left, total):
    """Source index of each padded sample (the edge sample is not repeated)."""
    i = (torch.arange(total, device=DEV) - left) % (2 * (n - 1))
    return torch.where(i < n, i, 2 * (n - 1) - i)


def _fold2(x, k):
    H, W = x.shape[-2] // k, x.shape[-1] // k
    return x.reshape(x.shape[:-2] + (k, H, k, W)).mean(dim=(-4, -2))


def _exact2d(case, S, x):
    J, M, N = case['J'], case['m'], case['n']
    H, W = (M // 2 ** J + 2) * 2 ** J, (N // 2 ** J + 2) * 2 ** J
    phi, psi = _levels(S.phi), [_levels(p) for p in S.psi]
    x = x.double()
    x = x[:, _reflect(M, (H - M) // 2, H)][:, :, _reflect(N, (W - N) // 2, W)]

    def low(U, r):
        return torch.fft.ifft2(_fold2(U * phi['levels'][r], 2 ** (J - r))).real[:, 1:-1, 1:-1]

    U0 = torch.fft.fft2(x)
    first, second = [low(U0, 0)], []
    for p1 in psi:
        j1 = p1['j']
        U1 = torch.fft.fft2(torch.fft.ifft2(_fold2(U0 * p1['levels'][0], 2 ** j1)).abs())
        first.append(low(U1, j1))
        if case['max_order'] == 2:
            for p2 in psi:
                if p2['j'] > j1:
                    U2 = torch.fft.ifft2(_fold2(U1 * p2['levels'][j1], 2 ** (p2['j'] - j1))).abs()
                    second.append(low(torch.fft.fft2(U2), p2['j']))
    return torch.stack(first + second, 1)


def _fold1(x, k):
    return x.reshape(x.shape[:-1] + (k, x.shape[-1] // k)).mean(dim=-2)


def _exact1d(case, S, x):
    phi, psi1, psi2 = _levels(S.phi_f), [_levels(p) for p in S.psi1_f], [_levels(p) for p in S.psi2_f]
    N, ls = S._N_padded, S.log2_stride
    glob = case['T'] == 'global'
    i0, i1 = S.ind_start[ls], S.ind_end[ls]
    U0 = torch.fft.fft(x.double()[:, _reflect(case['n'], S.pad_left, N)])

    def low(U, r):
        if glob:
            return U[:, :1].real
        return torch.fft.ifft(_fold1(U * phi['levels'][r], 2 ** max(ls - r, 0))).real[:, i0:i1]

    sub = (lambda j: j) if glob else (lambda j: min(j, ls))
    first, second = [low(U0, 0)], []
    for p1 in psi1:
        k1 = sub(p1['j'])
        U1 = torch.fft.fft(torch.fft.ifft(_fold1(U0 * p1['levels'][0], 2 ** k1)).abs())
        first.append(low(U1, k1))
        if case['max_order'] == 2:
            for p2 in psi2:
                if p2['j'] > p1['j']:
                    k2 = max(sub(p2['j']) - k1, 0)
                    U2 = torch.fft.ifft(_fold1(U1 * p2['levels'][k1], 2 ** k2)).abs()
                    second.append(low(torch.fft.fft(U2), k1 + k2))
    return torch.stack(first + second, 1)


def _exact_jtfs(case, S, x):
    phi, psi1, psi2 = _levels(S.phi_f), [_levels(p) for p in S.psi1_f], [_levels(p) for p in S.psi2_f]
    phi_fr, psi_fr = _levels(S.filters_fr[0]), [_levels(p) for p in S.filters_fr[1]]
    N, ls, lf, n_fr = S._N_padded, S.log2_stride, S.log2_stride_fr, S._N_padded_fr
    i0, i1 = S.ind_start[ls], S.ind_end[ls]
    U0 = torch.fft.fft(x.double()[:, _reflect(case['n'], S.pad_left, N)])

    def low(U, r):
        return torch.fft.ifft(_fold1(U * phi['levels'][r], 2 ** (ls - r))).real

    out = [low(U0, 0)[:, None, i0:i1]] if case['format'] == 'time' else []
    bands = [(p, min(p['j'], ls)) for p in psi1]
    U1 = [torch.fft.fft(torch.fft.ifft(_fold1(U0 * p['levels'][0], 2 ** k1)).abs()) for p, k1 in bands]
    rows = [(torch.stack([low(U, k1) for U, (_, k1) in zip(U1, bands)], 1), None)]
    for p2 in psi2:
        y = [torch.fft.ifft(_fold1(U * p2['levels'][k1], 2 ** min(p2['j'] - k1, ls)))
             for U, (p1, k1) in zip(U1, bands) if p2['j'] > p1['j']]
        if y:
            rows.append((torch.stack(y, 1), p2['j']))
    for y, j2 in rows:
        A = y.shape[1]
        Y = torch.fft.fft(torch.nn.functional.pad(y.transpose(1, 2), (0, n_fr - A)))
        for p in psi_fr:
            if j2 is None and p['xi'] < 0:
                continue
            k = min(p['j'], lf)
            u = torch.fft.ifft(_fold1(Y * p['levels'][0], 2 ** k)).abs().transpose(1, 2)
            if j2 is not None:
                u = low(torch.fft.fft(u), j2)
            stride = 2 ** p['j']
            if p['xi'] != 0:
                r = min(p['j'], phi_fr['j'])
                u = torch.fft.ifft(_fold1(torch.fft.fft(u.transpose(1, 2)) * phi_fr['levels'][r],
                                          2 ** (lf - r))).real.transpose(1, 2)
                stride = 2 ** lf
            if case['format'] == 'time':
                out.append(u[:, :len(range(0, A, stride)), i0:i1])
            else:
                out.append(u[:, None, :, i0:i1])
    return torch.cat(out, 1)


def _exact3d(case, S, x):
    J, L = case['J'], case['L']
    bank = [torch.view_as_complex(getattr(S, 'tensor%d' % l).to(DEV).double().contiguous()) for l in range(L + 1)]
    dim = (-3, -2, -1)

    def modulus(U, l, j):
        s = 0
        for m in range(2 * l + 1):
            s = s + torch.fft.ifftn(U * bank[l][j, m], dim=dim).abs().square()
        return s.sqrt()

    def integrals(u):
        return torch.stack([u.pow(p).sum(dim) for p in _POWERS], -1)

    U0 = torch.fft.fftn(x.double(), dim=dim)
    per_l = []
    for l in range(L + 1):
        first, second = [], []
        for j1 in range(J + 1):
            u = modulus(U0, l, j1)
            first.append(integrals(u))
            if case['max_order'] == 2 and j1 < J:
                U1 = torch.fft.fftn(u, dim=dim)
                second += [integrals(modulus(U1, l, j2)) for j2 in range(j1 + 1, J + 1)]
        per_l.append(torch.stack(first + second, 1))
    return torch.stack(per_l, 2)


def exact(case, seed):
    """The same outputs in 64 bits (images and signals a few at a time)."""
    S = _module(case)
    x = _inputs(case, seed)
    f = {'2d': _exact2d, '1d': _exact1d, 'fs': _exact_jtfs, '3d': _exact3d}[case['kind'][-2:]]
    step = max(1, (1 << 19) // x[0].numel()) if case['kind'] == 'grad2d' else max(1, (1 << 22) // x[0].numel())
    if not case['kind'].startswith('grad'):
        return torch.cat([f(case, S, x[i:i + step]) for i in range(0, x.shape[0], step)])
    w = _cotangent(case, S, seed).double()
    ys, gs = [], []
    for i in range(0, x.shape[0], step):
        xi = x[i:i + step].double().requires_grad_()
        y = f(case, S, xi)
        ys.append(y.detach())
        gs.append(torch.autograd.grad(y, xi, w[i:i + step])[0])
        del y
    return {'S': torch.cat(ys), 'grad': torch.cat(gs)}
