"""The int4 matmul of several rows: 3 to 5 on the GEMV (each row bit for bit the one-token call's), more on the MFMA
kernel (the group sums of an exact 4-bit weight, scaled once each), at the edges of its tiles, against the CPU oracle with
the reference's bars (1 % relative Frobenius error, PCC 0.9999) and, on the MFMA kernel, every value within a bound of its
own (the bf16 rounding, 2^-8 of the value, and float32 sums of exact products in any order, a scale's rounding a group:
at most 2 K 2^-24 of the sum of their magnitudes); what each launch plans, on the host."""

import pytest
import torch

from common.testing import check, same, within
from dense_reader import _lib
from int4 import w4a16
from oracle import dense_oracle as O


def _plan(m, k, n):
    L = _lib.Launch()  # device pointers that are never read: the plan only reads the launch's sizes
    L.x, L.y, L.m, L.k, L.ldx, L.ldy, L.nseg = 16, 16, m, k, k, n, 1
    s = L.seg[0]
    s.fmt, s.n, s.n_pad, s.codes, s.scale = 3, n, -(-n // 32) * 32, 16, 16
    return _lib.launch_info(L), _lib.lib().dr_workspace_bytes(L)


def test_plan_on_the_host():
    """The kernel and rows a pass by rows; never tile pairs (those kernels read block-float weights only); 3 to 5 rows four
    a pass or two by the workgroups and K; and fewer rows a pass where the split-K sums of a long K would not fit
    dr_matmul_noalloc's own workspace."""
    for n in (78, 2048, 14336, 131072):
        few = 4 if n > 8000 else 2
        for m, kernel, rows in ((1, "gemv", 1), (2, "gemv", 2), (3, "gemv", few), (5, "gemv", few), (6, "mfma", 16),
                                (16, "mfma", 16), (17, "mfma", 32), (300, "mfma", 32)):
            p, _ = _plan(m, 4096, n)
            assert (p["kernel"], p["rows_per_pass"], p["tiles_per_workgroup"]) == (kernel, rows, 1), (m, n, p)
    for k, n, rows in ((96, 32, 2), (96, 14336, 4), (96, 65536, 2), (512, 32, 4), (512, 65536, 2), (1024, 32, 4),
                       (1024, 65536, 4), (2048, 4096, 2), (8192, 4096, 2), (14336, 4096, 4), (28672, 2048, 4)):
        assert _plan(4, k, n)[0]["rows_per_pass"] == rows, (k, n)
    cap = _lib.lib().dr_scratch_bytes()
    for n, rows in ((14336, 32), (32768, 16), (65536, 4), (262144, 2)):
        p, need = _plan(32, 14336, n)
        assert p["splits"] == 2 and p["rows_per_pass"] == rows and need <= cap, (n, p, need)


def _case(device, n, k, seed):
    g = torch.Generator().manual_seed(seed)
    codes = torch.randint(-7, 8, (n, k), generator=g).to(torch.int8)
    scales = (torch.rand(n, k // 32, generator=g) * 0.01 + 0.001).to(torch.bfloat16)
    return codes, scales, w4a16.int4_weight(device, codes), w4a16.group_scales(device, scales)


def _products(tx, codes, scales):
    """x @ (q * s) in float64 and the error of its float32 sums."""
    w = (codes.to(tx.device).double() * scales.to(tx.device).double().repeat_interleave(32, dim=1)).t()
    xd = tx.double()
    return xd @ w, (xd.abs() @ w.abs()) * (2 * xd.shape[1] * 2.0**-24)


def _near(name, y, want, err):
    within(name, y, want, want.abs() * 2.0**-8 + err + 1e-30)


@pytest.mark.gpu
@pytest.mark.parametrize("k, n", [(96, 48), (320, 200), (800, 1056), (2080, 8224), (4352, 96), (9216, 320)])
def test_rows(device, k, n):
    codes, scales, wq, ts = _case(device, n, k, k + n)
    x = O.x_input(45, k, 5).to(torch.bfloat16)
    tx = x.to(device.torch)
    want = O.int4_ref(x, codes, scales)
    exact, err = (v.cpu() for v in _products(tx, codes, scales))
    one = [w4a16.w4a16_linear(tx[r].reshape(1, 1, 1, k), wq, ts).float().cpu().reshape(1, n) for r in range(5)]
    for m in (3, 4, 5):
        y = w4a16.rows_matmul(tx[:m], wq, ts).float().cpu()
        for r in range(m):
            same(f"{m} rows: row {r} against the one-token call", y[r:r + 1], one[r])
    for m in (6, 8, 16, 17, 31, 32, 33, 45):
        print(w4a16.launch_plan(tx[:m], wq, ts), flush=True)
        y = w4a16.rows_matmul(tx[:m], wq, ts).float().cpu()
        check(f"{m} rows K {k} N {n}", y, want[:m])
        _near(f"{m} rows, every value", y, exact[:m], err[:m])
        same(f"{m} rows: repeated", w4a16.rows_matmul(tx[:m], wq, ts).float().cpu(), y)
        if m <= 32:
            perm = torch.randperm(m, generator=torch.Generator().manual_seed(m))
            same(f"{m} rows permuted", w4a16.rows_matmul(tx[perm.to(tx.device)], wq, ts).float().cpu(), y[perm])


@pytest.mark.gpu
@pytest.mark.parametrize("m", [6, 20, 40])
@pytest.mark.parametrize("k, n", [(288, 320), (96, 8224), (4128, 64)])
def test_columns_past_k_and_nan(device, m, k, n):
    """A ragged K: the next row's Inf and NaN, which lie past a row's K in memory, enter none of its sums."""
    codes, scales, wq, ts = _case(device, n, k, k)
    x = O.x_input(m, k, 6)
    x[2], x[m - 1] = float("nan"), float("nan")
    x[4, 3] = float("inf")
    tx = x.to(torch.bfloat16).to(device.torch)
    y = w4a16.rows_matmul(tx, wq, ts)
    assert bool(y[2].isnan().all()) and bool(y[m - 1].isnan().all()) and not bool(y[4].isfinite().all())
    keep = torch.tensor([r for r in range(m) if r not in (2, 4, m - 1)], device=device.torch)
    _near(f"{m} rows K {k} N {n}: the other rows", y[keep], *_products(tx[keep], codes, scales))
