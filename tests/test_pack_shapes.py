"""Packing and unpacking at the edges of their wavefronts' tiles (512 and 256 k, 16 and 64 columns), with rows that are not
16-byte aligned and with column divisors: codes, exponents and held values byte for byte the oracle's."""

import numpy as np
import pytest
import torch

from common.testing import same
from dense_reader import _lib, linear
from oracle import dense_oracle as O

pytestmark = pytest.mark.gpu

FMTS = {"bfp8": linear.bfloat8_b, "bfp4": linear.bfloat4_b, "bf16": linear.bfloat16}


@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("n, k", [(1, 32), (33, 96), (200, 480), (65, 512), (257, 544), (48, 1280)])
def test_pack_unpack(device, fmt, n, k):
    wt = O.matrix(n, k, n + k)
    wt[::7, ::5] *= 60
    wt[0, 3], wt[0, 1] = 0.0, 1e-40
    tw, _ = linear.native_weight(device, wt, FMTS[fmt])
    codes, exps = O.to_layout(wt.T.contiguous(), fmt, n_pad=tw.n_pad)
    same("codes", tw.codes.cpu(), torch.from_numpy(codes))
    if exps is not None:
        same("exponents", tw.exps.cpu(), torch.from_numpy(exps))
    want = torch.from_numpy(O.held(wt.T.contiguous(), fmt))
    same("held", linear.held(tw, n).cpu(), want)
    tc, ts = linear.native_weight(device, wt, FMTS[fmt], col_scale=True)
    c = O.bf16_ceil(wt.abs().amax(dim=1).clamp(min=1e-8))
    same("column divisors", ts.float().cpu().reshape(-1), c)
    same("held of w / c", linear.held(tc, n).cpu(), torch.from_numpy(O.held((wt / c[:, None]).T.contiguous(), fmt)))
    # the same matrix with rows of an odd stride, off 16 bytes: the same bytes
    wide = torch.full((n, k + 3), float("nan"), device=device.torch)
    wide[:, 1:k + 1] = wt.to(device.torch)
    lib, f = _lib.lib(), tw.fmt
    c2, e2 = torch.zeros_like(tw.codes), None if tw.exps is None else torch.zeros_like(tw.exps)
    st = lib.dr_pack(wide[:, 1:].data_ptr(), k + 3, n, k, f, None, c2.data_ptr(), None if e2 is None else e2.data_ptr(),
                     tw.n_pad, tw.k_pad, device.stream())
    _lib.check(st, "dr_pack")
    same("codes of unaligned rows", c2.cpu(), tw.codes.cpu())
    if e2 is not None:
        same("exponents of unaligned rows", e2.cpu(), tw.exps.cpu())
    # a wider output of which only the first columns are written
    out = torch.full((k, n + 5), 7.0, device=device.torch)
    st = lib.dr_unpack(tw.codes.data_ptr(), tw.exps_ptr(), f, n, k, tw.n_pad, tw.k_pad, out.data_ptr(), n + 5, device.stream())
    _lib.check(st, "dr_unpack")
    assert np.array_equal(out[:, :n].cpu().numpy(), want.numpy()) and bool((out[:, n:] == 7.0).all())
