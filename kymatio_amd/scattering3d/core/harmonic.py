"""Solid harmonic scattering as batched HIP launches.

The reference walks l, j1 (and j2 > j1) and, inside, every m of the order-l
wavelets one op at a time: cdgmm3d, ifft, modulus_rotation per m, then one
integral per path (kymatio/scattering3d/core/scattering3d.py:24-75).  Here
each step of one l is two launches over all j, m and images together:

    planes    products U_hat psi_{l, j, m} and their 2D inverse over (N, O)
    lines     inverse along M, then the root of the squares' sum over m (what
              the chained rotation modulus computes, with one rounding)

(kym_op_harmonic_step, for every j of a parent at once) and the moduli of
every (path, l) land in one field array of layout (paths, L + 1, B, n), so
one kym_op_integrals launch computes every output and the result is that
array's integrals moved to (B, paths, L + 1, P).
Path order per l is the reference's: all first-order j1, then the pairs
(j1, j2 > j1) in j1-major order; outputs interleave l inside each path
(scattering3d.py:64-73).
"""
import ctypes

import torch

from ... import _lib


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def harmonic_paths(J, max_order):
    """Paths in output order: (j1,) for j1 <= J, then (j1, j2), j1 < j2 <= J."""
    first = [(j1,) for j1 in range(J + 1)]
    if max_order < 2:
        return first
    return first + [(j1, j2) for j1 in range(J + 1) for j2 in range(j1 + 1, J + 1)]


class _Launcher:
    """The batched ops on one device and stream, for one dtype."""

    def __init__(self, device, dtype):
        self.lib = _lib.lib()
        self.device = device
        self.stream = _lib.stream_of(device)
        self.code = _lib.DTYPE_CODE[dtype]

    def products(self, U_hat, F):
        B, nm = U_hat.shape[0], F.shape[0]
        n = U_hat[0].numel() // 2
        out = torch.empty((B, nm) + tuple(U_hat.shape[1:]), dtype=U_hat.dtype, device=self.device)
        _lib.check(self.lib.kym_op_harmonic_products(_ptr(U_hat), _ptr(F), _ptr(out), B, nm, n, self.code,
                                                       self.stream))
        return out

    def step(self, U_hat, F, nm, dest, vol, dstride):
        """dest[g] (B, n), dstride elements apart = the moduli of scale g of F
        (ng, 2l + 1, ...) over its first nm filters; False where the volume
        does not fit the fused kernels.  Scales are taken together up to 256 MB
        of planes between the two kernels (the MALL)."""
        B, ng, n = U_hat.shape[0], F.shape[0], vol[0] * vol[1] * vol[2]
        fs = F.stride(0) // 2
        each = B * nm * n * 2
        per = max(1, min(ng, (256 << 20) // max(each * U_hat.element_size(), 1)))
        work = torch.empty(per * each, dtype=U_hat.dtype, device=self.device)
        for g in range(0, ng, per):
            rc = self.lib.kym_op_harmonic_step(_ptr(U_hat), _ptr(F[g]), _ptr(work), _ptr(dest[g]), B, min(per, ng - g),
                                               nm, vol[0], vol[1], vol[2], fs, dstride, self.code, self.stream)
            if rc == 5 and g == 0:
                return False
            _lib.check(rc)
        return True

    def rotation_modulus(self, Y, dest):
        """Y: (B, nm, M, N, O, 2) -> dest (B, n) (a contiguous block of the field array)."""
        B, nm = Y.shape[0], Y.shape[1]
        n = dest.shape[1]
        _lib.check(self.lib.kym_op_modulus_rotation_sum(_ptr(Y), _ptr(dest), B, nm, n, n, self.code, self.stream))

    def integrals(self, fields, powers):
        rows, n = fields.shape[0], fields.shape[1]
        P = len(powers)
        pw = (ctypes.c_double * P)(*[float(p) for p in powers])
        out = torch.empty((rows, P), dtype=fields.dtype, device=self.device)
        _lib.check(self.lib.kym_op_integrals(_ptr(fields), _ptr(out), rows, n, pw, P, self.code, self.stream))
        return out


def harmonic_scattering(x, bank, J, L, max_order, rotation_covariant, powers, backend):
    """x: (B, M, N, O, 1) real, contiguous, on the device; bank[l]: the
    (J + 1, 2l + 1, M, N, O, 2) wavelets of order l.  Returns
    (B, paths, L + 1, len(powers)) in float32 (the dtype the reference's
    integrals are allocated in, kymatio/scattering3d/backend/torch_backend.py:145-150)."""
    B = x.shape[0]
    vol = tuple(x.shape[1:4])
    n = vol[0] * vol[1] * vol[2]
    paths = harmonic_paths(J, max_order)
    slot = {p: i for i, p in enumerate(paths)}
    run = _Launcher(x.device, x.dtype)
    fields = torch.empty((len(paths), L + 1, B, n), dtype=x.dtype, device=x.device)

    nm_all = [bank[l].shape[1] for l in range(L + 1)]
    rows = fields.shape[1] * B * n  # field elements between paths

    def moduli(U_hat, l, j0, ng, path0):
        """The moduli of scales j0 .. j0 + ng - 1 of order l into the fields of
        paths path0, path0 + 1, ..."""
        nm = nm_all[l] if rotation_covariant else 1
        if run.step(U_hat, bank[l][j0:j0 + ng], nm, fields[path0:path0 + ng, l], vol, rows):
            return
        for g in range(ng):  # volumes whose planes do not fit a workgroup
            F = bank[l][j0 + g][:nm]
            run.rotation_modulus(backend.ifft(run.products(U_hat, F).reshape((-1,) + vol + (2,))).reshape(
                (B, nm) + vol + (2,)), fields[path0 + g, l])

    U0_hat = backend.rfft(x)
    for l in range(L + 1):
        moduli(U0_hat, l, 0, J + 1, slot[(0,)])
        if max_order > 1:
            for j1 in range(J):
                U1_hat = backend.rfft(fields[slot[(j1,)], l].reshape((B,) + vol + (1,)))
                moduli(U1_hat, l, j1 + 1, J - j1, slot[(j1, j1 + 1)])
    S = run.integrals(fields.reshape(-1, n), powers).reshape(len(paths), L + 1, B, len(powers))
    return S.permute(2, 0, 1, 3).contiguous().to(torch.float32)


__all__ = ['harmonic_paths', 'harmonic_scattering']
