"""The GPU workgroup bodies, run single-threaded on the CPU by the host-only
harness libkymatio_emu.so, against the golden vectors and the oracle.  This
checks the plan, the digit-reversal maps, the twiddles and every index
formula of the 2D kernels (both the all-in-LDS route and, with a tiny LDS
cap, the column/row multi-pass route) without a GPU."""
import ctypes

import numpy as np
import pytest
import torch

from kymatio_amd.scattering2d.filter_bank import filter_bank
from kymatio_amd.scattering2d.utils import compute_padding
from oracle import scat2d
from tests.helpers import RTOL_CHANNEL, Emu, channel_rel_err, golden, golden_2d_cases, pack_filters_2d


@pytest.fixture(scope='module')
def emu():
    return Emu()


def _filters(shape, J, L, dt=np.float32):
    Mp, Np = compute_padding(shape[0], shape[1], J)
    fb = filter_bank(Mp, Np, J, L)
    return fb, pack_filters_2d(fb, dt)


def test_fixture_2d(emu):
    d = golden('test_data_2d.npz')
    x = d['x'].reshape(-1, 32, 32)
    fb, f = _filters((32, 32), 4, 8)
    for lds in (160 * 1024, 4096):
        out, info = emu.scat2d(x, 4, (32, 32), f, lds_limit=lds, chunk=2)
        assert np.allclose(out, d['Sx'].reshape(out.shape))
        if lds == 4096:
            assert info['big_nodes'] > 0


@pytest.mark.parametrize('case', golden_2d_cases(), ids=lambda c: c[0])
@pytest.mark.parametrize('lds', [160 * 1024, 8192], ids=['lds', 'multipass'])
def test_golden(emu, case, lds):
    tag, x, J, shape, kw, ref = case
    if tag == 'cfg2' and lds == 8192:
        pytest.skip('multi-pass route at 256x256 is covered on the GPU; too slow single-threaded')
    fb, f = _filters(shape, J, kw.get('L', 8))
    out, _ = emu.scat2d(x, J, shape, f, lds_limit=lds, **kw)
    assert out.shape == ref.shape
    assert channel_rel_err(out, ref) <= RTOL_CHANNEL


def test_fp64_matches_numpy_fp64(emu):
    G = golden('golden_scat2d.npz')
    x = G['cfg4_x']
    fb, f = _filters((128, 128), 4, 8, np.float64)
    out, _ = emu.scat2d(x, 4, (128, 128), f)
    ref = scat2d.scattering2d_numpy(x, 4, filters=fb)
    assert np.abs(out - ref).max() < 1e-13


def test_linearity_of_root_and_batch_independence(emu):
    """Images are independent: a batch equals its images run one at a time,
    and chunking does not change results."""
    rng = np.random.default_rng(3)
    x = rng.standard_normal((5, 20, 24)).astype(np.float32)
    fb, f = _filters((20, 24), 2, 8)
    full, _ = emu.scat2d(x, 2, (20, 24), f)
    chunked, _ = emu.scat2d(x, 2, (20, 24), f, chunk=2)
    single = np.concatenate([emu.scat2d(x[i:i + 1], 2, (20, 24), f)[0] for i in range(5)])
    assert np.array_equal(full, chunked)
    assert np.array_equal(full, single)


def test_unsupported_prime_raises(emu):
    # M = 500, J = 2 -> P = 508 = 4 * 127: prime radix 127 is not built
    fb_dummy = np.zeros(1, np.float32)
    with pytest.raises(RuntimeError, match='prime factor'):
        emu.scat2d(np.zeros((1, 500, 500), np.float32), 2, (500, 500), fb_dummy)


def test_small_j_error(emu):
    with pytest.raises(RuntimeError, match='smallest dimension'):
        emu.scat2d(np.zeros((1, 10, 10), np.float32), 4, (10, 10), np.zeros(1, np.float32))


@pytest.mark.parametrize('shape,J,kw,lds', [
    ((20, 24), 2, {}, 160 * 1024),
    ((20, 24), 2, {}, 4096),
    ((16, 16), 2, {'pre_pad': 1}, 160 * 1024),
    ((31, 33), 3, {'max_order': 1}, 160 * 1024),
    ((32, 32), 4, {}, 8192),
    ((32, 32), 5, {}, 160 * 1024),
    ((8, 8), 2, {'L': 4}, 160 * 1024),
], ids=['lds', 'multipass', 'prepad', 'order1', 'J4-multipass', 'J5-fold', 'L4'])
def test_backward_matches_autograd_through_oracle(emu, shape, J, kw, lds):
    """FP64: the hand-written adjoint equals torch autograd through the
    op-for-op restatement of the reference (what the reference's own
    gradients are)."""
    L = kw.get('L', 8)
    fb, f = _filters(shape, J, L, np.float64)
    rng = np.random.default_rng(0)
    from kymatio_amd.scattering2d.utils import compute_padding
    xs = compute_padding(shape[0], shape[1], J) if kw.get('pre_pad') else shape
    x = rng.standard_normal((2,) + tuple(xs))
    sc = scat2d.Scattering2DTorchCPU(J, shape, L=L, max_order=kw.get('max_order', 2),
                                     pre_pad=bool(kw.get('pre_pad')), dtype=torch.float64, filters=fb)
    xt = torch.from_numpy(x).requires_grad_()
    S = sc(xt)
    w = rng.standard_normal(S.shape)
    (S * torch.from_numpy(w)).sum().backward()
    from tests.helpers import emu_train2d
    # three backward passes on one forward: the backward must not consume the saved state
    out, gx = emu_train2d(emu, x, J, shape, f, w, L=L, max_order=kw.get('max_order', 2),
                          pre_pad=kw.get('pre_pad', 0), lds_limit=lds, nbwd=3)
    g = xt.grad.numpy()
    assert np.abs(out - S.detach().numpy()).max() < 1e-13
    assert np.abs(gx - g).max() <= 1e-12 * np.abs(g).max()


@pytest.mark.parametrize('shape,J,tune', [((32, 32), 2, None), ((64, 64), 3, None), ((128, 128), 4, None),
                                          ((128, 128), 4, (16, 0, 16, 8)), ((128, 128), 4, (16, 0, 32, 8))])
def test_backward_fp32_compiled_nodes(emu, shape, J, tune):
    """FP32 backward through the compile-time node kernels (40², 20² and 80²
    nodes with 10² leaves) and, at 128² J=4, the compile-time 160² backward
    passes (the default blocks, and 16 or 32 columns by 8 rows): equals torch
    autograd through the FP64 oracle to FP32 rounding, on two backward passes
    of one forward."""
    fb64, _ = _filters(shape, J, 8, np.float64)
    _, f32 = _filters(shape, J, 8, np.float32)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((2,) + shape)
    _, info = emu.scat2d(x[:1].astype(np.float32), J, shape, f32, tune=list(tune) if tune else None)
    assert info['bwd_spec_launches'] >= (11 if J == 4 else 1)  # at J=4: 6 node launches + 5 of the 160² passes
    sc = scat2d.Scattering2DTorchCPU(J, shape, dtype=torch.float64, filters=fb64)
    xt = torch.from_numpy(x).requires_grad_()
    S = sc(xt)
    w = rng.standard_normal(S.shape)
    (S * torch.from_numpy(w)).sum().backward()
    from tests.helpers import emu_train2d
    out, gx = emu_train2d(emu, x.astype(np.float32), J, shape, f32, w.astype(np.float32), nbwd=2, tune=tune)
    g = xt.grad.numpy()
    assert np.abs(out - S.detach().numpy()).max() <= 1e-5 * np.abs(S.detach().numpy()).max()
    assert np.abs(gx - g).max() <= 1e-5 * np.abs(g).max()


@pytest.mark.parametrize('shape,J,L,dt', [((64, 48), 4, 8, np.float32), ((40, 64), 4, 6, np.float32),
                                          ((32, 90), 5, 5, np.float32), ((64, 64), 4, 3, np.float64),
                                          ((33, 70), 5, 2, np.float64)])
def test_fold_pass_matches_gathers(emu, shape, J, L, dt):
    """Deep periodisations (k >= 8) summed by the fold pass, over tiles of 4,
    3, 2 and 1 parents and wavelets, against the same nodes gathering by
    themselves (the route of a workspace without room for the inputs)."""
    Mp, Np = compute_padding(shape[0], shape[1], J)
    f = pack_filters_2d(filter_bank(Mp, Np, J, L)).astype(dt)
    x = np.random.default_rng(J * L).standard_normal((2,) + shape).astype(dt)
    out, info = emu.scat2d(x, J, shape, f, L=L)
    g = emu.with_taps(f, J, shape, L)
    ref = np.zeros_like(out)
    fn = emu.lib.kym_emu_scat2d_forward_nofold
    fn.argtypes, fn.restype = emu.lib.kym_emu_scat2d_forward.argtypes, ctypes.c_int
    i9 = (ctypes.c_longlong * 9)()
    rc = fn(shape[0], shape[1], J, L, 2, 0, 0 if dt == np.float32 else 1, 160 * 1024, x.ctypes.data, g.ctypes.data,
            ref.ctypes.data, 2, 0, i9)
    assert rc == 0
    # k^2 <= 256 products per point in another order: sqrt(256) eps of the largest term
    assert channel_rel_err(out, ref) < (1e-5 if dt == np.float32 else 1e-13)


def _placement(emu, shape, J, L, dt, lds_limit=160 * 1024, tune=()):
    info = (ctypes.c_longlong * 6)()
    t = (ctypes.c_int * 7)(*tune)
    rc = emu.lib.kym_emu_scat2d_plan(shape[0], shape[1], J, L, 0 if dt == np.float32 else 1,
                                     ctypes.c_longlong(lds_limit), t, len(tune), info)
    assert rc == 0, emu.lib.kym_emu_last_error().decode()
    return dict(zip(('lds', 'big', 'global_tw', 'ws', 'global_tw_nodes', 'gathered'), info))


@pytest.mark.parametrize('shape,J,dt,tune,big', [
    ((16, 8192), 3, np.float32, (), None), ((16, 9000), 3, np.float32, (), None),  # one row and its table: 175, 191 KB
    ((20, 9228), 4, np.float64, (), None),
    ((512, 512), 6, np.float32, (16, 0, 32), None), ((256, 256), 5, np.float32, (16, 0, 64), None),
    ((300, 300), 3, np.float64, (16, 0, 32, 32), None),
    # nodes that fill the LDS by themselves stay in one workgroup, but for those of resolution 0
    ((144, 488), 3, np.float32, (), 9), ((96, 384), 2, np.float64, (), 9),
    ((72, 440), 3, np.float64, (), 9)])
def test_launches_fit_the_workgroup(emu, shape, J, dt, tune, big):
    """Every launch stays within the LDS, twiddles included."""
    p = _placement(emu, shape, J, 8, dt, tune=tune)
    assert p['lds'] <= 160 * 1024
    assert p['global_tw'] > 0
    assert big is None or p['big'] == big


@pytest.mark.parametrize('shape,J,L,dt,limits', [
    ((40, 40), 3, 8, np.float32, (8840, 7608)), ((20, 24), 2, 8, np.float64, (8696, 4952)),
    ((33, 31), 3, 8, np.float32, (6744, 6520)), ((45, 30), 1, 2, np.float64, (9240,))])
def test_twiddles_in_global_memory(emu, shape, J, L, dt, limits):
    """Launches whose LDS has no room for their twiddles, nodes and passes,
    forward and backward, against the default placement."""
    from tests.helpers import emu_train2d
    _, f = _filters(shape, J, L, dt)
    rng = np.random.default_rng(J)
    x = rng.standard_normal((2,) + shape).astype(dt)
    ref, _ = emu.scat2d(x, J, shape, f, L=L)
    w = rng.standard_normal(ref.shape).astype(dt)
    _, gref = emu_train2d(emu, x, J, shape, f, w, L=L)
    eps = 1e-5 if dt == np.float32 else 1e-12
    nodes = passes = 0
    for lim in limits:
        p = _placement(emu, shape, J, L, dt, lim)
        assert p['global_tw'] and p['lds'] <= lim
        nodes += p['global_tw_nodes']
        passes += p['global_tw'] - p['global_tw_nodes']
        out, gx = emu_train2d(emu, x, J, shape, f, w, L=L, lds_limit=lim, nbwd=2)
        assert channel_rel_err(out, ref) <= eps
        assert np.abs(gx - gref).max() <= eps * np.abs(gref).max()
    assert passes and (nodes or J == 1)


def test_gathered_inputs_take_finished_slots(emu):
    """Large images' deep gathers cost no workspace: 480 x 480 J=5 still fits the
    64 MB of a call without allocations, 512 x 512 J=6 takes what its slots take."""
    p = _placement(emu, (480, 480), 5, 8, np.float32)
    assert p['gathered'] > 0 and p['ws'] <= 64 << 20
    p = _placement(emu, (512, 512), 6, 8, np.float32)
    assert p['gathered'] > 0 and p['ws'] <= 113 << 20  # 119 MB with slots of their own


@pytest.mark.parametrize('shape,J,L,dt,lds', [((120, 130), 4, 2, np.float32, 36000), ((100, 96), 5, 1, np.float32, 34000),
                                              ((120, 96), 4, 2, np.float64, 70000)])
def test_fold_into_finished_slots(emu, shape, J, L, dt, lds):
    """Gathered inputs in the slots of finished second-order big nodes, against
    the placement without big nodes, forward and backward."""
    from tests.helpers import emu_train2d
    p = _placement(emu, shape, J, L, dt, lds)
    assert p['gathered'] > 0 and p['big'] > 1 + 2 * L  # second-order ones among the big nodes
    _, f = _filters(shape, J, L, dt)
    rng = np.random.default_rng(J * L)
    x = rng.standard_normal((2,) + shape).astype(dt)
    ref, _ = emu.scat2d(x, J, shape, f, L=L)
    w = rng.standard_normal(ref.shape).astype(dt)
    _, gref = emu_train2d(emu, x, J, shape, f, w, L=L)
    out, _ = emu.scat2d(x, J, shape, f, L=L, lds_limit=lds, chunk=1)
    eps = 1e-5 if dt == np.float32 else 1e-12
    assert channel_rel_err(out, ref) <= eps
    out, gx = emu_train2d(emu, x, J, shape, f, w, L=L, lds_limit=lds, nbwd=2)
    assert channel_rel_err(out, ref) <= eps
    assert np.abs(gx - gref).max() <= eps * np.abs(gref).max()


@pytest.mark.parametrize('shape,J,L,dt', [((24, 2280), 4, 2, np.float32), ((20, 4576), 4, 1, np.float32),
                                          ((24, 2280), 4, 3, np.float64), ((20, 4576), 4, 1, np.float64),
                                          ((16, 5600), 4, 4, np.float64)])
def test_fold_pass_over_long_rows(emu, shape, J, L, dt):
    """Deeply periodised rows of 288, 576 and (in smaller tiles) 704 points, more
    than the fold pass's threads, against the nodes gathering by themselves."""
    assert _placement(emu, shape, J, L, dt)['gathered'] == L + L * L
    Mp, Np = compute_padding(shape[0], shape[1], J)
    f = pack_filters_2d(filter_bank(Mp, Np, J, L)).astype(dt)
    x = np.random.default_rng(L).standard_normal((2,) + shape).astype(dt)
    out, _ = emu.scat2d(x, J, shape, f, L=L)
    g = emu.with_taps(f, J, shape, L)
    ref = np.zeros_like(out)
    fn = emu.lib.kym_emu_scat2d_forward_nofold
    fn.argtypes, fn.restype = emu.lib.kym_emu_scat2d_forward.argtypes, ctypes.c_int
    i9 = (ctypes.c_longlong * 9)()
    assert fn(shape[0], shape[1], J, L, 2, 0, 0 if dt == np.float32 else 1, 160 * 1024, x.ctypes.data, g.ctypes.data,
              ref.ctypes.data, 2, 0, i9) == 0
    assert channel_rel_err(out, ref) < (1e-5 if dt == np.float32 else 1e-13)  # as in test_fold_pass_matches_gathers
