"""The matmul of many rows (dense_gemm.hip): every tile of its plan, each format, at the edges of its tiles, against the
CPU oracle; and the order of its staging in the emitted code.

Bars as for the other kernels (the reference's): 1 % relative Frobenius error and PCC 0.9999 for bf16 outputs, 0.1 % for
fp32 outputs; and every value within a bound of its own against the products in float64 (a whole matrix's error hides a
wrong column or store at an edge): the output's rounding, 2^-8 of the value (bf16) or 2^-23, and float32 sums of exact
products in any order, at most K 2^-24 of the sum of their magnitudes (the scales, the GLU and the residual carried
through). Every row is its own MFMA column, summed in an order that depends on K and the tile only, so permuting x's
rows permutes y's bit for bit and repeated calls agree.
"""

import math
import re
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from common.testing import check, same, within
from dense_reader import _lib, linear
from oracle import dense_oracle as O

FMTS = {"bfp8": linear.bfloat8_b, "bfp4": linear.bfloat4_b, "bf16": linear.bfloat16}


def _x(dev, m, k, seed):
    x = O.x_input(m, k, seed)
    return x, x.to(torch.bfloat16).reshape(1, 1, m, k).to(dev.torch)


def _weight(dev, n, k, fmt, seed):
    wt = O.matrix(n, k, seed)
    return linear.native_weight(dev, wt, FMTS[fmt])[0], torch.from_numpy(O.held(wt.T.contiguous(), fmt))


def _host(y, m):
    return y.float().cpu().reshape(m, -1)


def _products(tx, h):
    """x @ h and its terms' magnitudes summed, in float64 on the GPU, and the latter's share of the sums' error."""
    xd, hd = tx.double().reshape(-1, tx.shape[-1]), h.to(tx.device).double()
    return xd @ hd, (xd.abs() @ hd.abs()) * (xd.shape[1] * 2.0**-24)


def _glu(g, ge, u, ue, act):
    """act(g) * u in float64 and its bound for errors of ge and ue (the activations' slopes are below 1.13 and their
    float32 evaluation within 2^-18 of the argument)."""
    z = 2 * (2 / math.pi) ** 0.5 * (g + 0.044715 * g**3) if act == "geglu" else g
    a = g * torch.sigmoid(z)
    ae = 1.13 * ge + g.abs() * 2.0**-18
    return a * u, ae * u.abs() + a.abs() * ue + ae * ue


ROUND = {torch.bfloat16: 2.0**-8, torch.float32: 2.0**-23}


def _near(name, y, want, err):
    within(name, y.reshape(want.shape), want, want.abs() * ROUND[y.dtype] + err + 1e-30)


def test_passes_where_faster():
    """On the host, for 256 CUs: up to K = 14336 (a float32 y: 4096) every call past the row limits is one tiled launch; for
    a longer K the passes of 16 (GLU) and 32 rows stay where few tiles leave most CUs idle, unless their workspace would not fit
    dr_matmul_noalloc's own."""
    def plan(fmt, m, k, n, glu=False, f32=False):
        L = _lib.Launch()  # device pointers that are never read: the plan only reads the launch's sizes
        L.x, L.y, L.m, L.k, L.ldx, L.ldy, L.nseg, L.y_f32 = 16, 16, m, k, k, n, 1, int(f32)
        s = L.seg[0]
        s.fmt, s.n, s.n_pad, s.codes, s.exps = fmt, n, -(-n // 32) * 32, 16, 16
        if glu:
            s.glu, s.codes_up, s.exps_up = 2, 16, 16
        return _lib.launch_info(L), _lib.lib().dr_workspace_bytes(L)

    for fmt in (0, 1, 2):
        for f32 in (False, True):
            for k in (96, 1024, 4096, 14336)[:3 if f32 else 4]:
                for n in (32, 512, 4096):
                    for m, glu in ((33, True), (64, True), (129, False), (256, False)):
                        p, need = plan(fmt, m, k, n, glu, f32)
                        assert p["rows_per_pass"] >= 64 and need == 0, (fmt, m, k, n, glu, f32, p)
            for m, glu, rows in ((33, True, 16), (129, False, 32)):
                for k, n in ((28672, 512), (57344, 32)) if glu or fmt != 2 else ((57344, 32),):
                    p, need = plan(fmt, m, k, n, glu, f32)
                    assert (p["rows_per_pass"], p["splits"]) == (rows, -(-k // 8192)) and need > 0, (fmt, m, k, n, p)
                p, need = plan(fmt, m, 28672, 14336, glu, f32)
                assert p["rows_per_pass"] >= 64 and need == 0, (fmt, m, p)
    cap = _lib.lib().dr_scratch_bytes()
    for n in (32, 256, 512, 1024):
        p, need = plan(0, 129, 1 << 20, n)
        assert need <= cap and (p["rows_per_pass"] == 32) == (need > 0), (n, p, need)


# (rows, K, N, rows a tile, output tiles a workgroup): every tile of the plan; rows past the last tile, K off the
# 256-k group and off the 64-k step, N off the tile, the workgroup's columns and the 4-column store
SHAPES = [
    (129, 96, 40, 64, 2),
    (160, 800, 545, 64, 2),  # the wavefronts split K: groups of 256 k unevenly
    (257, 4352, 96, 64, 2),
    (130, 288, 14340, 64, 8),
    (192, 512, 32768, 128, 8),
    (160, 512, 65537, 192, 8),
    (1023, 256, 16382, 256, 8),
    (1000, 800, 14336, 256, 8),
]


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("m, k, n, rows, tiles", SHAPES)
def test_tiles(device, fmt, m, k, n, rows, tiles):
    tw, h = _weight(device, n, k, fmt, 1)
    x, tx = _x(device, m, k, 2)
    p = linear.launch_plan(tx, tw, None)
    print(p, flush=True)
    assert (p["kernel"], p["rows_per_pass"], p["tiles_per_workgroup"]) == ("mfma", rows, tiles), p
    assert p["passes"] == -(-m // rows) and p["workgroups"] == -(-p["tiles"] // tiles)
    s = torch.rand(n, generator=torch.Generator().manual_seed(3)) + 0.5
    ts = linear.scale_tensor(device, s, dtype=linear.float32)
    yd = linear.matmul(tx, tw, ts)
    y = _host(yd, m)
    check(f"{fmt} rows {m} K {k} N {n} scaled", y, O.ref(x, h, s))
    want, err = _products(tx, h)
    sd = s.to(tx.device).double()
    _near("every value", yd, want * sd, err * sd)
    same("repeated call", _host(linear.matmul(tx, tw, ts), m), y)
    perm = torch.randperm(m, generator=torch.Generator().manual_seed(4))
    yp = _host(linear.matmul(tx[..., perm.to(tx.device), :].contiguous(), tw, ts), m)
    same("rows permuted", yp, y[perm])


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("m, k, n", [(131, 800, 200), (200, 288, 14340)])
def test_epilogue(device, fmt, m, k, n):
    """Residual (both modes, bf16 and fp32 outputs, in place), fp32 output, col0 into a wider output."""
    tw, h = _weight(device, n, k, fmt, 11)
    x, tx = _x(device, m, k, 12)
    want = O.ref(x, h)
    exact, err = _products(tx, h)
    res = torch.randn(m, n, generator=torch.Generator().manual_seed(13)).to(torch.bfloat16)
    tr = res.reshape(1, 1, m, n).to(device.torch)
    plus, err_plus = exact + tr[0, 0].double(), err + tr[0, 0].double().abs() * 2.0**-23
    for mode in ("epilogue", "preload"):
        yd = linear.matmul(tx, tw, None, residual=tr, residual_mode=mode)
        check(f"residual {mode}", _host(yd, m), want + res.float())
        _near(f"residual {mode}, every value", yd, plus, err_plus)
        yd = linear.matmul(tx, tw, None, residual=tr, residual_mode=mode, out32=True)
        check(f"residual {mode} fp32", _host(yd, m), want + res.float(), rel=1e-3, pcc=0.999999)
        _near(f"residual {mode} fp32, every value", yd, plus, err_plus)
    inplace = tr.clone()
    assert linear.matmul(tx, tw, None, residual=inplace, out=inplace) is inplace
    check("residual in place", _host(inplace, m), want + res.float())
    _near("residual in place, every value", inplace, plus, err_plus)
    yd = linear.matmul(tx, tw, None, out32=True)
    check("fp32 output", _host(yd, m), want, rel=1e-3, pcc=0.999999)
    _near("fp32 output, every value", yd, exact, err)
    wide = torch.full((1, 1, m, 32 + n + 32), 7.0, dtype=torch.bfloat16, device=device.torch)
    linear.matmul(tx, tw, None, out=wide, col0=1)
    y = _host(wide, m)
    check("col0", y[:, 32:32 + n], want)
    _near("col0, every value", wide.reshape(m, -1)[:, 32:32 + n], exact, err)
    rest = torch.cat([y[:, :32], y[:, 32 + n:]], 1)
    same("the other columns untouched", rest, torch.full_like(rest, 7.0))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("m, k, n", [(33, 96, 64), (65, 1056, 7200), (129, 800, 96), (150, 256, 7200), (333, 288, 8224), (600, 96, 8192)])
def test_glu(device, fmt, m, k, n):
    """Gate and up apart (with column scales) and interleaved, silu and gelu_tanh."""
    gw, uw = O.matrix(n, k, 21), O.matrix(n, k, 22)
    hg, hu = (torch.from_numpy(O.held(w.T.contiguous(), fmt)).float() for w in (gw, uw))
    tg, tu, ti = (linear.native_weight(device, w, FMTS[fmt])[0] for w in (gw, uw, linear.interleave_glu(gw, uw)))
    x, tx = _x(device, m, k, 23)
    s = torch.rand(2, n, generator=torch.Generator().manual_seed(24)) + 0.5
    tsg, tsu = (linear.scale_tensor(device, v, dtype=linear.float32) for v in s)
    tsi = linear.scale_tensor(device, torch.stack([s[0].reshape(-1, 32), s[1].reshape(-1, 32)], 1).reshape(-1),
                              dtype=linear.float32)
    xd = x.to(torch.bfloat16).double()
    g, u = (xd @ hg.double()) * s[0].double(), (xd @ hu.double()) * s[1].double()
    (gx, ge), (ux, ue) = ([v * sc.to(tx.device).double() for v in _products(tx, h)] for h, sc in ((hg, s[0]), (hu, s[1])))
    for act, code in (("swiglu", 0), ("geglu", 1)):
        yd = linear.matmul(tx, tg, tsg, glu=True, w_up=tu, scale_up=tsu, glu_act=code)
        two = _host(yd, m)
        check(f"{fmt} {act} two weights", two, O.glu_ref(g, u, act))
        _near(f"{act}, every value", yd, *_glu(gx, ge, ux, ue, act))
        same("interleaved against two weights", _host(linear.matmul(tx, ti, tsi, glu=True, glu_act=code), m), two)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("m, k, n", [(132, 512, 96), (160, 4096, 512), (132, 4096, 8192), (131, 2080, 9000), (192, 16896, 64),
                                     (512, 1056, 14336), (999, 4064, 7200), (1000, 2400, 7200), (1000, 8192, 3600)])
def test_float32_error(device, fmt, m, k, n):
    """A float32 y is as exact as that of 32 rows a call, whose kernel sums K over eight wavefronts: its error against
    float64 at most that of the same rows in calls of 32 (and a twentieth: 2 % is what another draw of the inputs moves
    either)."""
    tw, h = _weight(device, n, k, fmt, 41)
    x, tx = _x(device, m, k, 42)
    want = (x.to(torch.bfloat16).to(device.torch).double() @ h.to(device.torch).double()).cpu()
    y = linear.matmul(tx, tw, None, out32=True).cpu().double().reshape(m, n)
    parts = [linear.matmul(tx[..., r:r + 32, :].contiguous(), tw, None, out32=True).reshape(-1, n) for r in range(0, m, 32)]
    one = torch.cat(parts).cpu().double()
    err, ref = ((v - want).norm() / want.norm() for v in (y, one))
    print(f"{fmt} rows {m} K {k} N {n}: {float(err):.3e}, in calls of 32 rows {float(ref):.3e}", flush=True)
    assert err <= 1.05 * ref


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("m, k, n", [(65, 1056, 96), (200, 2336, 14400)])
def test_glu_float32(device, fmt, m, k, n):
    gw, uw = O.matrix(n, k, 51), O.matrix(n, k, 52)
    hg, hu = (torch.from_numpy(O.held(w.T.contiguous(), fmt)).double().to(device.torch) for w in (gw, uw))
    tg, tu = (linear.native_weight(device, w, FMTS[fmt])[0] for w in (gw, uw))
    x, tx = _x(device, m, k, 53)
    xd = x.to(torch.bfloat16).double().to(device.torch)
    yd = linear.matmul(tx, tg, None, glu=True, w_up=tu, out32=True)
    check(f"{fmt} swiglu float32", _host(yd, m), O.glu_ref((xd @ hg).cpu(), (xd @ hu).cpu(), "swiglu"), rel=1e-5, pcc=0.999999)
    _near("every value", yd, *_glu(*_products(tx, hg), *_products(tx, hu), "swiglu"))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("m, k, n, glu", [(140, 288, 64, False), (131, 288, 14340, False), (70, 1056, 7200, True),
                                          (333, 96, 8224, True)])
def test_columns_past_k_and_nan(device, fmt, m, k, n, glu):
    """A ragged K: what lies past K in x's memory (the next row, here Inf and NaN) enters no sum; a NaN row stays its
    own row's. In tiles whose wavefronts split K and in those that share x, each format's order of k, a GLU, and a float32
    y's."""
    tw, h = _weight(device, n, k, fmt, 31)
    tu, hu = _weight(device, n, k, fmt, 33) if glu else (None, None)
    x, _ = _x(device, m, k, 32)
    rows = [5, m - 2]  # (NaN; the row after each has an Inf)
    x[rows] = float("nan")
    x[[r + 1 for r in rows], 3] = float("inf")
    tx = x.to(torch.bfloat16).reshape(1, 1, m, k).to(device.torch)
    keep = torch.tensor([r for r in range(m) if r not in rows and r - 1 not in rows], device=device.torch)
    kept = tx[..., keep, :]
    want = _products(kept, h) if not glu else _glu(*_products(kept, h), *_products(kept, hu), "swiglu")
    for out32 in (False, True):
        y = linear.matmul(tx, tw, None, out32=out32, **({"glu": True, "w_up": tu} if glu else {})).reshape(m, -1)
        for r in rows:
            assert bool(y[r].isnan().all()) and not bool(y[r + 1].isfinite().any())
        _near(f"{fmt} K {k} N {n} {y.dtype}: the other rows", y[keep], *want)


def test_staging_order():
    """In the emitted gfx950 code of dr_gemm every barrier of the K loop follows a wait for the wavefront's LDS reads
    (lgkmcnt(0)) and for all but its newest x loads (vmcnt of at most two stages), and between two such barriers lie one
    stage's loads to LDS, so that a stage is read only after its loads have landed and overwritten only after its reads.
    After the loop's last loads every wavefront waits for all of its own (vmcnt(0)) at a barrier before the first sum is
    written over a stage."""
    import __graft_entry__ as G

    hipcc = G.HIPCC if Path(G.HIPCC).exists() else shutil.which("hipcc")
    if hipcc is None:
        pytest.skip("no hipcc")
    src = next(s for s in G.SOURCES if s.stem == "dense_gemm")
    flags = [f for f in G.FLAGS if f not in ("-shared", "-fPIC")]
    r = subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", str(src), "-o", "-"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    found = 0
    for name, body in re.findall(r"^(_ZN3drk\S*dr_gemmI\S*):(.*?)s_endpgm", r.stdout, re.M | re.S):
        mt, ks = (int(v) for v in re.search(r"dr_gemmILi(\d+)ELi\dELb\dELb(\d)ELb\dE", name).groups())
        stage = 4 * mt if ks else mt  # loads to LDS a stage, of one wavefront
        lines = [s.strip() for s in body.split("\n")]
        lines = [s for s in lines if s and not s.startswith((";", ".")) and not s.endswith(":")]
        dma = [i for i, s in enumerate(lines) if s.startswith("buffer_load") and s.endswith("lds")]
        waits = [(i, int(m.group(1))) for i, s in enumerate(lines)
                 if (m := re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)", s)) and int(m.group(1)) in (stage, 2 * stage)]
        inside = [i for i, v in waits if v == stage]
        # three stages asked for ahead of the loop, then one after each of its waits (four steps a turn)
        assert len(inside) >= 4 and len(inside) % 4 == 0 and len(dma) == (3 + len(inside)) * stage, (name, len(dma))
        assert [v for _, v in waits if v != stage] == [2 * stage] and sum(i < inside[0] for i in dma) == 3 * stage
        for a, b in zip(inside, inside[1:] + [len(lines)]):
            if not ks:
                nxt = next(s for s in lines[a + 1:] if s == "s_barrier" or s.startswith(("ds_", "buffer_", "global_", "flat_")))
                assert nxt == "s_barrier", (name, lines[a], nxt)
            assert sum(a < i < b for i in dma) == stage, (name, a, b)
        # all of the sums' 8 mt LDS writes (others are the ragged K's zeros)
        end = [i for i in range(dma[-1], len(lines) - 1)
               if re.match(r"s_waitcnt vmcnt\(0\) lgkmcnt\(0\)$", lines[i]) and lines[i + 1] == "s_barrier"]
        assert end and sum(s.startswith("ds_write_b128") for s in lines[end[0]:]) >= 8 * mt, (name, end[:1])
        found += 1
    assert found == 46, found
