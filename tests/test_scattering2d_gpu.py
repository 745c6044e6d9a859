"""Scattering2D on the GPU (through the C ABI) against the reference's
fixture, the golden vectors written from the reference and the oracle.

Parity bar (FP32): per output channel, max |ours - ref| <= 1e-5 * max |ref|
of that channel; the reference fixture is also checked with the reference's
own torch.allclose defaults.  FP64: against the NumPy FP64 oracle, 1e-12."""
import numpy as np
import pytest
import torch

import kymatio_amd
from kymatio_amd import workloads
from kymatio_amd.torch import Scattering2D
from oracle import scat2d
from tests.helpers import RTOL_CHANNEL, channel_rel_err, golden, golden_2d_cases

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def test_fixture_2d():
    """tests/scattering2d/test_torch_scattering2d.py:45-77 on the HIP path."""
    d = golden('test_data_2d.npz')
    x = torch.from_numpy(d['x']).to(DEV)
    S = torch.from_numpy(d['Sx']).to(DEV)
    J = int(d['J'])
    sc = kymatio_amd.Scattering2D(J, shape=(32, 32), pre_pad=bool(d['pre_pad']), frontend='torch').to(DEV)
    Sg = sc(x)
    assert Sg.shape == S.shape
    assert torch.allclose(Sg, S)
    sc1 = Scattering2D(J, shape=(32, 32), max_order=1).to(DEV)
    S1 = sc1(x)
    assert torch.allclose(S1, S[..., :S1.shape[-3], :, :])


@pytest.mark.parametrize('case', golden_2d_cases(), ids=lambda c: c[0])
@pytest.mark.parametrize('lds', [0, 8192], ids=['lds', 'multipass'])
def test_golden(case, lds):
    tag, x, J, shape, kw, ref = case
    print('case', tag, 'lds_limit', lds, flush=True)
    sc = Scattering2D(J, shape, **kw).to(DEV)
    sc.lds_limit = lds
    out = sc(torch.from_numpy(x).to(DEV)).cpu().numpy()
    assert out.shape == ref.shape
    err = channel_rel_err(out, ref)
    print('  per-channel rel err %.3e' % err)
    assert err <= RTOL_CHANNEL


def test_headline_error_by_order_vs_fp64():
    """256x256, J=3: error against the reference (golden) and, per order,
    against the FP64 NumPy restatement."""
    G = golden('golden_scat2d.npz')
    x = G['cfg2_x']
    sc = Scattering2D(3, (256, 256)).to(DEV)
    out = sc(torch.from_numpy(x).to(DEV)).cpu().numpy()
    assert channel_rel_err(out, G['cfg2_Sx']) <= RTOL_CHANNEL
    phi, psi = sc.load_filters()
    fb = {'phi': {'levels': [v.cpu().numpy()[..., 0] for v in phi['levels']]},
          'psi': [{'levels': [v.cpu().numpy()[..., 0] for v in p['levels']], 'j': p['j']} for p in psi]}
    ref64 = scat2d.scattering2d_numpy(x, 3, filters=fb)
    orders = scat2d.channel_orders(3, 8)
    for o in (0, 1, 2):
        e = channel_rel_err(out[:, orders == o], ref64[:, orders == o])
        print('order %d: per-channel rel err vs FP64 %.3e' % (o, e))
        assert e <= RTOL_CHANNEL


def test_headline_more_reference_images():
    """Three more reference-written images of the 256x256 J=3 workload
    (tests/golden/make_headline_golden.py), in one batch with the golden
    cfg2 image: per-channel bar, and the fraction of elements within the
    reference's own torch.allclose(rtol=1e-5, atol=1e-8)."""
    G = golden('golden_headline2d.npz')
    C = golden('golden_scat2d.npz')
    x = np.concatenate([C['cfg2_x'], G['x']])
    ref = np.concatenate([C['cfg2_Sx'], G['Sx']])
    sc = Scattering2D(3, (256, 256)).to(DEV)
    out = sc(torch.from_numpy(x).to(DEV)).cpu().numpy()
    err = channel_rel_err(out, ref)
    close = np.isclose(out, ref, rtol=1e-5, atol=1e-8)
    print('4 reference images: per-channel rel err %.3e, elements within allclose(1e-5, 1e-8): %.6f'
          % (err, close.mean()))
    assert err <= RTOL_CHANNEL
    assert close.mean() >= 0.99


def test_fp64_gpu_vs_numpy():
    G = golden('golden_scat2d.npz')
    x = G['cfg4_x'].astype(np.float64)
    sc = Scattering2D(4, (128, 128)).double().to(DEV)
    out = sc(torch.from_numpy(x).to(DEV)).cpu().numpy()
    phi, psi = sc.load_filters()
    fb = {'phi': {'levels': [v.cpu().numpy()[..., 0] for v in phi['levels']]},
          'psi': [{'levels': [v.cpu().numpy()[..., 0] for v in p['levels']], 'j': p['j']} for p in psi]}
    ref = scat2d.scattering2d_numpy(x, 4, filters=fb)
    assert np.abs(out - ref).max() <= 1e-12 * np.abs(ref).max()


def test_full_batch_properties():
    """Config-2 size (64 x 256 x 256): the batch result equals per-image runs
    bit for bit, is independent of the chunking, deterministic, and finite."""
    x = torch.from_numpy(workloads.grating_images(64, 256, seed=2)).to(DEV)
    sc = Scattering2D(3, (256, 256)).to(DEV)
    a = sc(x)
    b = sc(x)
    assert torch.equal(a, b)
    sc.images_per_chunk = 5
    c = sc(x)
    assert torch.equal(a, c)
    # chunks rotate over the caller's stream and the plan's streams (two by
    # default, up to four) or stay on the caller's stream: the same bits; the
    # plan's streams wait for the caller's pending work (the clone) and the
    # caller's stream for them (the result read right after)
    sc.images_per_chunk = 8
    d2 = sc(x.clone() * 1.0)
    sc.tune = [0, 0, 0, 0, 0, 1]
    d1 = sc(x)
    sc.tune = [0, 0, 0, 0, 0, 4]
    sc._plans.clear()
    d4 = sc(x * 1.0)
    sc.tune = [0, 0, 0, 0, 0, 3]
    sc._plans.clear()
    d3 = sc(x * 1.0)
    assert torch.equal(a, d1) and torch.equal(a, d2) and torch.equal(a, d3) and torch.equal(a, d4)
    sc._plans.clear()
    sc.tune = None
    side = torch.cuda.Stream(device=DEV)
    side.wait_stream(torch.cuda.current_stream(DEV))
    with torch.cuda.stream(side):
        e = sc(x + 0.0)
    torch.cuda.current_stream(DEV).wait_stream(side)
    assert torch.equal(a, e)
    sc.images_per_chunk = None
    for i in (0, 31, 63):
        assert torch.equal(sc(x[i:i + 1].contiguous())[0], a[i])
    assert torch.isfinite(a).all()
    assert a.shape == (64, 217, 32, 32)


def test_batch_shape_agnostic():
    """tests/scattering2d/test_torch_scattering2d.py:91-136."""
    S = Scattering2D(3, (32, 32), 8).to(DEV)
    with pytest.raises(RuntimeError, match='at least two'):
        S(torch.zeros((), device=DEV))
    with pytest.raises(RuntimeError, match='at least two'):
        S(torch.zeros((32,), device=DEV))
    Sx = S(torch.zeros((32, 32), device=DEV))
    assert Sx.shape == (217, 4, 4)
    for shp in ((1, 32, 32), (2, 32, 32), (2, 2, 32, 32), (2, 2, 2, 32, 32)):
        Sx = S(torch.zeros(shp, device=DEV))
        assert Sx.shape == shp[:-2] + (217, 4, 4)


def test_errors():
    """tests/scattering2d/test_torch_scattering2d.py:138-177."""
    S = Scattering2D(3, (32, 32)).to(DEV)
    with pytest.raises(TypeError, match='input should be'):
        S(None)
    x = torch.randn(4, 4, device=DEV)
    with pytest.raises(RuntimeError, match='must be contiguous'):
        S(x[::2, ::2])
    with pytest.raises(RuntimeError, match='Tensor must be of spatial size'):
        S(torch.randn(31, 31, device=DEV))
    S = Scattering2D(3, (32, 32), pre_pad=True).to(DEV)
    with pytest.raises(RuntimeError, match='Padded tensor must be of spatial size'):
        S(torch.randn(31, 31, device=DEV))
    S = Scattering2D(2, (8, 8)).to(DEV)
    y = S(torch.randn(8, 8, device=DEV))
    assert y.device.type == 'cuda'
    with pytest.raises(TypeError, match='same dtype'):
        S(torch.randn(8, 8, device=DEV, dtype=torch.float64))


def test_input_size_agnostic():
    """tests/scattering2d/test_torch_scattering2d.py:179-222 (odd sizes, J up to 5)."""
    for N in (31, 32, 33):
        for J in (1, 2, 4):
            sc = Scattering2D(J, shape=(N, N)).to(DEV)
            sc(torch.zeros(3, 3, N, N, device=DEV))
            sc = Scattering2D(J, shape=(N, N), pre_pad=True).to(DEV)
            sc(torch.zeros(3, 3, sc._M_padded, sc._N_padded, device=DEV))
    sc = Scattering2D(5, shape=(32, 32)).to(DEV)
    assert sc(torch.zeros(3, 3, 32, 32, device=DEV)).shape[-2:] == (1, 1)
    sc = Scattering2D(5, shape=(37, 32)).to(DEV)
    assert sc(torch.zeros(3, 3, 37, 32, device=DEV)).shape[-2:] == (1, 1)


def test_list_output_meta():
    sc = Scattering2D(2, (16, 16), out_type='list').to(DEV)
    x = torch.randn(2, 16, 16, device=DEV)
    out = sc(x)
    arr = Scattering2D(2, (16, 16)).to(DEV)(x)
    assert len(out) == arr.shape[-3]
    ref = scat2d.Scattering2DTorchCPU(2, (16, 16))(x.cpu(), out_type='list')
    for o, r, c in zip(out, ref, range(arr.shape[-3])):
        assert o['j'] == r['j'] and o['n'] == r['n'] and o['theta'] == r['theta']
        assert torch.equal(o['coef'], arr[:, c])


@pytest.mark.parametrize('shape,J,B', [((32, 32), 2, 80), ((28, 34), 2, 70), ((24, 24), 3, 130), ((60, 60), 2, 80)])
def test_many_small_nodes_match_few(shape, J, B):
    """Launches of more than 2048 small nodes run them one wave each, smaller
    launches with 256 threads (nodes of up to 5120 points: 256 and 512): the same coefficients and gradients."""
    sc = Scattering2D(J, shape).to(DEV)
    x = torch.randn((B,) + shape, device=DEV, generator=torch.Generator(DEV).manual_seed(B)).requires_grad_()
    w = torch.randn(sc(x[:1]).shape[1:], device=DEV, generator=torch.Generator(DEV).manual_seed(1))
    many = sc(x)
    gmany, = torch.autograd.grad((many * w).sum(), x)
    few = torch.cat([sc(x[i:i + 4]) for i in range(0, B, 4)])
    gfew, = torch.autograd.grad((few * w).sum(), x)
    # the same butterflies in the same order, only spread over other threads
    assert (many - few).abs().max() <= 1e-6 * few.abs().max()
    assert (gmany - gfew).abs().max() <= 1e-5 * gfew.abs().max()


@pytest.mark.parametrize('lds', [0, 8192], ids=['lds', 'multipass'])
@pytest.mark.parametrize('shape', [(68, 12), (12, 84), (108, 108), (20, 116), (60, 44), (68, 116), (84, 36),
                                   (52, 64), (172, 100), (28, 172)],
                         ids=['19x5', '5x23', '29x29', '7x31', '17x13', '19x31', '23x11',
                              '15x18', '45x27', '9x45'])
def test_prime_lengths(shape, lds):
    """Padded lengths 4 p and 4 q: each family of radices, alone and mixed, and
    products of small primes in one radix (15, 9 from 48 points on): forward
    in both types and the FP64 gradient, against the oracle."""
    sc = Scattering2D(2, shape, L=2).to(DEV)
    sc.lds_limit = lds
    ref = scat2d.Scattering2DTorchCPU(2, shape, L=2, dtype=torch.float64)
    x = torch.randn((2,) + shape, dtype=torch.float64, generator=torch.Generator().manual_seed(shape[0]))
    xr = x.clone().requires_grad_()
    want = ref(xr)
    w = torch.randn(want.shape, dtype=torch.float64, generator=torch.Generator().manual_seed(1))
    gw, = torch.autograd.grad((want * w).sum(), xr)
    out = sc(x.float().to(DEV)).cpu().numpy()
    assert channel_rel_err(out, want.detach().numpy()) <= RTOL_CHANNEL
    sd = Scattering2D(2, shape, L=2).double().to(DEV)
    sd.lds_limit = 3 * lds  # doubles; the backward needs its leaf (45 x 27 at most) in LDS
    xd = x.to(DEV).requires_grad_()
    got = sd(xd)
    gd, = torch.autograd.grad((got * w.to(DEV)).sum(), xd)
    assert (got.detach().cpu() - want.detach()).abs().max() <= 1e-12 * want.abs().max()
    assert torch.allclose(gd.cpu(), gw, rtol=1e-10, atol=1e-12 * gw.abs().max().item())


@pytest.mark.parametrize('B', [1, 2, 39, 40])
def test_streams_either_side_of_the_line(B):
    """Batches of fewer than 9 million node points (227,600 an image here, 39
    images) stay on the caller's stream, larger ones take two: the same
    coefficients and gradients as with one and two streams asked for."""
    x = torch.randn(B, 64, 64, device=DEV, generator=torch.Generator(DEV).manual_seed(B)).requires_grad_()
    res = []
    for streams in (0, 1, 2):
        sc = Scattering2D(3, (64, 64)).to(DEV)
        sc.tune = [0, 0, 0, 0, 0, streams] if streams else None
        out = sc(x * 1.0)
        g, = torch.autograd.grad((out * out).sum(), x)
        with torch.no_grad():
            res.append((out.detach(), g, sc(x * 1.0)))
    for r in res[1:]:
        # the same butterflies, possibly spread over other threads
        for a, b, tol in zip(r, res[0], (1e-6, 1e-5, 1e-6)):
            assert (a - b).abs().max() <= tol * b.abs().max()


@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('shape,J,lds', [((16, 8192), 3, 0), ((144, 488), 3, 0), ((72, 440), 3, 0), ((96, 384), 2, 0),
                                         ((40, 40), 3, 8840), ((40, 40), 3, 7608), ((20, 24), 2, 8696),
                                         ((20, 24), 2, 4952), ((33, 31), 3, 6520), ((45, 30), 1, 9240)])
def test_data_that_fills_the_lds(shape, J, lds, dtype):
    """Lines and nodes that leave no room in LDS for their twiddles (in one
    type or the other), forward and gradient, against the FP64 oracle."""
    L = 2 if shape == (16, 8192) else 8  # nodes stay in one workgroup where there are many
    sc = Scattering2D(J, shape, L=L).to(dtype).to(DEV)
    sc.lds_limit = lds
    ref = scat2d.Scattering2DTorchCPU(J, shape, L=L, dtype=torch.float64)
    x = torch.randn((2,) + shape, generator=torch.Generator().manual_seed(J)).to(dtype)
    xr = x.double().requires_grad_()
    want = ref(xr)
    w = torch.randn(want.shape, dtype=torch.float64, generator=torch.Generator().manual_seed(1)).to(dtype)
    gw, = torch.autograd.grad((want * w.double()).sum(), xr)
    xg = x.to(DEV).requires_grad_()
    got = sc(xg)
    gx, = torch.autograd.grad((got * w.to(DEV)).sum(), xg)
    tol = RTOL_CHANNEL if dtype == torch.float32 else 1e-12
    assert channel_rel_err(got.detach().cpu().numpy(), want.detach().numpy()) <= tol
    if dtype == torch.float32 and shape in ((16, 8192), (144, 488)):
        return  # of so many |u| some are so small that u / |u| is off by 1e-3 and 1.5e-5 in FP32, in plain torch too
    assert (gx.cpu().double() - gw).abs().max() <= (1e-5 if dtype == torch.float32 else 1e-11) * gw.abs().max()


@pytest.mark.parametrize('shape,J,B', [((224, 224), 3, 6), ((58, 58), 1, 70), ((116, 116), 2, 20)])
def test_many_medium_nodes_in_doubles(shape, J, B):
    """FP64 nodes of 2048 to 4095 points and over 64 KB, on 256 threads in
    launches of more than 512, on 512 in smaller ones, with a plan of smaller
    needs of the same kernels made in between: the same outputs and gradients."""
    sc = Scattering2D(J, shape).double().to(DEV)
    x = torch.randn((B,) + shape, device=DEV, dtype=torch.float64,
                    generator=torch.Generator(DEV).manual_seed(B)).requires_grad_()
    few = torch.cat([sc(x[i:i + 1]) for i in range(B)])
    w = torch.randn(few.shape[1:], device=DEV, dtype=torch.float64, generator=torch.Generator(DEV).manual_seed(1))
    gfew, = torch.autograd.grad((few * w).sum(), x)
    Scattering2D(1, (46, 46)).double().to(DEV)(x[:1, :46, :46].detach().contiguous())
    many = sc(x)
    gmany, = torch.autograd.grad((many * w).sum(), x)
    # the same butterflies in the same order, only spread over other threads
    assert (many - few).abs().max() <= 1e-14 * few.abs().max()
    assert (gmany - gfew).abs().max() <= 1e-13 * gfew.abs().max()


@pytest.mark.parametrize('shape,L', [((24, 2280), 3), ((24, 2280), 4), ((20, 4576), 2), ((16, 5600), 2)])
def test_deep_averages_of_long_rows(shape, L):
    """J = 4 with rows of 288, 576 and 704 points at the deepest resolution: forward
    in both types and the FP64 gradient against the FP64 oracle."""
    ref = scat2d.Scattering2DTorchCPU(4, shape, L=L, dtype=torch.float64)
    x = torch.randn((3,) + shape, dtype=torch.float64, generator=torch.Generator().manual_seed(L))
    xr = x.clone().requires_grad_()
    want = ref(xr)
    w = torch.randn(want.shape, dtype=torch.float64, generator=torch.Generator().manual_seed(1))
    gw, = torch.autograd.grad((want * w).sum(), xr)
    out = Scattering2D(4, shape, L=L).to(DEV)(x.float().to(DEV)).cpu().numpy()
    assert channel_rel_err(out, want.detach().numpy()) <= RTOL_CHANNEL
    xd = x.to(DEV).requires_grad_()
    got = Scattering2D(4, shape, L=L).double().to(DEV)(xd)
    gd, = torch.autograd.grad((got * w.to(DEV)).sum(), xd)
    assert (got.detach().cpu() - want.detach()).abs().max() <= 1e-12 * want.abs().max()
    assert (gd.cpu() - gw).abs().max() <= 1e-11 * gw.abs().max()


def test_a_refused_plan_leaves_no_error_behind():
    """A size whose leaf column pass exceeds the LDS (3000 x 40, J = 4) is
    refused as a plan is made, and nothing else fails afterwards."""
    sc = Scattering2D(4, (3000, 40)).to(DEV)
    with pytest.raises(RuntimeError, match='hipFuncSetAttribute'):
        sc(torch.zeros(1, 3000, 40, device=DEV))
    assert torch.ones(8, device=DEV).sum().item() == 8
    assert Scattering2D(2, (32, 32)).to(DEV)(torch.zeros(1, 32, 32, device=DEV)).abs().max().item() == 0
