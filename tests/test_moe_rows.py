"""The MoE over 3 to 32 rows at the edges of its plans. test_down_rows: the two kernels of the down of 17 to 32 rows of
bfloat4_b experts, a tile a workgroup in chunks (one) and dr_mfma_moe_down_pairs (pairs: tiles in pairs, the union's 128-k
steps shared out over the splits' wavefronts), each with one tile and an odd count of tiles (H), an expert's K of a part
of a step, of a step, of a part more than steps and of many (I), unions of one expert (fewer steps than wavefronts) up to
all of them, one split and several. The kernel that 256 CUs run each on stands beside it. Against the float64 sum over h as the
device holds it, so the bound is derived: y is a bf16 rounding (2^-9 of the value) of float32 sums of exact products,
whose order costs at most n 2^-24 of the sum of the products' magnitudes, n their count. test_gate_up_rows: the same
bound carried through the activation."""

import pytest
import torch

from common.testing import same, within
from moe import moe8
from oracle import dense_oracle as O
from oracle import moe_oracle as MO

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


# experts, slots, H, I, rows
@pytest.mark.parametrize("E, k, H, I, R", [
    (2, 1, 32, 32, 17),  # pairs: one tile, a part of a step an expert
    (1, 1, 96, 128, 32),  # pairs: three tiles, one expert of one step
    (4, 2, 64, 160, 24),  # one: a step and a part
    (32, 4, 160, 480, 31),  # one: five tiles
    (8, 8, 1056, 1408, 32),  # pairs: every expert chosen by every row; 33 tiles in 11 splits
    (16, 2, 2080, 256, 18),  # one: 65 tiles in several splits
    (4, 1, 17440, 96, 20),  # pairs: more of them than two a CU, one split
    (16, 4, 4128, 288, 32),  # pairs: 129 tiles, two steps and a part, 6 splits
    (16, 4, 4128, 288, 18),  # pairs: 4 experts chosen of the 16 expected
    (4, 4, 8224, 160, 17),  # pairs: one split
    (8, 4, 1024, 768, 32),  # one: every wavefront two chunks of 256 k
    (256, 8, 64, 1408, 32),  # pairs: the 48 splits' sums of the one-tile kernel would not fit the LDS
])
def test_down_rows(device, E, k, H, I, R):
    print(f"case E {E} k {k} H {H} I {I} rows {R}", flush=True)
    g = torch.Generator().manual_seed(H + I)
    dn = torch.stack([torch.from_numpy(O.held(torch.randn(I, H, generator=g) * 0.05, "bfp4")).float() for _ in range(E)])
    gu = torch.stack([torch.randn(H, 2 * I, generator=g).to(BF) * H ** -0.5 for _ in range(E)])
    P = moe8.pack(device, gu, dn.to(BF))
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(R)])
    if R == 18:
        ids[:] = ids[0]  # (a union of k experts of the 16)
    w = torch.softmax(torch.randn(R, k, generator=g), 1).to(BF)
    tid = ids.to(torch.int16).reshape(1, 1, R, k).to(device.torch)
    x = torch.randn(1, 1, R, H, generator=g).to(BF).to(device.torch)
    h = moe8.gate_up_rows(x, P, tid, w.reshape(1, 1, R, k).to(device.torch), k, R)
    y = moe8.down_rows(h, P, tid, k, R)
    same("y repeated", moe8.down_rows(h, P, tid, k, R).cpu(), y.cpu())
    u = sorted(set(ids.flatten().tolist()))
    hd = h.cpu().double().reshape(-1, h.shape[-1])[:R, :len(u) * I]
    wt = torch.cat([dn[e] for e in u]).double()
    ref, mag = hd @ wt, hd.abs() @ wt.abs()
    yd = y.cpu().double().reshape(-1, y.shape[-1])
    err = (yd[:R, :H] - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + mag * (len(u) * I * 2.0 ** -24) + 1e-30
    assert bool((err <= bound).all()), f"worst {float((err / bound).max()):.3f} of its bound"
    assert not yd[R:].any(), "rows past R"


# What lies past the chosen experts' columns of h (here NaN), or past a row's last ones (the next row, here NaN), enters no
# sum, at an expert's K of a part of a step: both kernels of the down, the one of up to 16 rows, and the K-block one. The
# bound is test_down_rows'.
@pytest.mark.parametrize("E, k, H, I, R, kblock", [
    (16, 4, 4128, 288, 32, False),  # pairs
    (4, 4, 8224, 160, 17, False),  # pairs, one split
    (4, 2, 64, 160, 24, False),  # one
    (16, 2, 2080, 480, 18, False),  # one, several splits
    (16, 4, 1056, 288, 9, False),
    (4, 2, 64, 160, 24, True),
])
@pytest.mark.parametrize("all_chosen", [False, True])
def test_down_nan_beside(device, E, k, H, I, R, kblock, all_chosen):
    print(f"case E {E} k {k} H {H} I {I} rows {R} kblock {kblock} all {all_chosen}", flush=True)
    g = torch.Generator().manual_seed(H + I)

    def grid(w):
        return torch.from_numpy(MO.held_kblock(w.numpy()) if kblock else O.held(w, "bfp4")).float()

    dn = torch.stack([grid(torch.randn(I, H, generator=g) * 0.05) for _ in range(E)])
    P = moe8.pack(device, torch.zeros(E, H, 2 * I, dtype=BF), dn.to(BF), kblock=kblock)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(R)])
    if all_chosen:
        ids = (torch.arange(R * k) % E).reshape(R, k)
    else:
        ids[:] = ids[0]
    tid = ids.to(torch.int16).reshape(1, 1, R, k).to(device.torch)
    u = sorted(set(ids.flatten().tolist()))
    units = min(E, R * k)
    assert (len(u) == units) == all_chosen or k == E
    h = torch.randn(32, units * I, generator=g).to(BF)
    h[:, len(u) * I:] = float("nan")
    h[R - 2] = float("nan")
    y = moe8.down_rows(h.reshape(1, 1, 32, units * I).to(device.torch), P, tid, k, R)
    yd = y.reshape(-1, y.shape[-1])[:R, :H]
    assert bool(yd[R - 2].isnan().all())
    keep = [r for r in range(R) if r != R - 2]
    hd, wt = h[keep, :len(u) * I].double(), torch.cat([dn[e] for e in u]).double()
    ref, mag = hd @ wt, hd.abs() @ wt.abs()
    within("the other rows", yd[keep].cpu(), ref, ref.abs() * 2.0 ** -8 + mag * (len(u) * I * 2.0 ** -24) + 1e-30)


# more workgroups than one round of 8 wavefronts takes: 4 wavefronts of one run of K each (6 and 9 groups of 256 k:
# uneven runs, a wavefront without one), tiles in pairs and an odd one, a row's ids twice the same (the last counts)
@pytest.mark.parametrize("E, k, H, I, R, kblock", [
    (16, 4, 1312, 1056, 32, False),
    (16, 4, 1504, 1056, 17, True),
    (32, 4, 2080, 544, 16, False),
    (32, 8, 1312, 608, 7, True),
])
def test_gate_up_rows(device, E, k, H, I, R, kblock):
    print(f"case E {E} k {k} H {H} I {I} rows {R} kblock {kblock}", flush=True)
    g = torch.Generator().manual_seed(H + I)

    def grid(w):
        return torch.from_numpy(MO.held_kblock(w.numpy()) if kblock else O.held(w, "bfp4")).float()

    gu = torch.stack([grid(torch.randn(H, 2 * I, generator=g) * H ** -0.5) for _ in range(E)])
    gb = torch.randn(E, 2 * I, generator=g).to(BF)
    P = moe8.pack(device, gu.to(BF), torch.zeros(E, I, H, dtype=BF), kblock=kblock, gu_bias=gb)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(R)])
    ids[0, 1] = ids[0, 0]
    w = torch.softmax(torch.randn(R, k, generator=g), 1).to(BF)
    tid = ids.to(torch.int16).reshape(1, 1, R, k).to(device.torch)
    x = torch.randn(R, H, generator=g).to(BF)
    tx, tw = x.reshape(1, 1, R, H).to(device.torch), w.reshape(1, 1, R, k).to(device.torch)
    h = moe8.gate_up_rows(tx, P, tid, tw, k, R, loaders=2)
    same("h repeated", moe8.gate_up_rows(tx, P, tid, tw, k, R, loaders=2).cpu(), h.cpu())
    u = sorted(set(ids.flatten().tolist()))
    ref = torch.zeros(R, len(u) * I, dtype=torch.float64)
    tol = torch.zeros_like(ref)
    for q, e in enumerate(u):
        c = torch.zeros(R, dtype=torch.float64)
        for r in range(R):
            for j in range(k):
                if ids[r, j] == e:
                    c[r] = w[r, j].double()
        z = x.double() @ gu[e].double() + gb[e].double()
        z_err = (x.double().abs() @ gu[e].double().abs() + gb[e].double().abs()) * (H * 2.0 ** -24)
        up, gate, ue, ge = z[:, :I], z[:, I:], z_err[:, :I], z_err[:, I:]  # ([up | gate], as the oracle's layer)
        cols = slice(q * I, (q + 1) * I)
        ref[:, cols] = gate * torch.sigmoid(gate) * up * c[:, None]
        # (silu's slope is at most 1.1; its float32 evaluation within 2^-18 of its argument)
        tol[:, cols] = ((1.1 * ge + gate.abs() * 2.0 ** -18) * up.abs() + gate.abs() * ue) * c[:, None]
    hd = h.cpu().double().reshape(-1, h.shape[-1])[:R, :len(u) * I]
    err, bound = (hd - ref).abs(), ref.abs() * 2.0 ** -8 + 2 * tol + 1e-30
    assert bool((err <= bound).all()), f"worst {float((err / bound).max()):.3f} of its bound"


# The wavefronts of a gate/up workgroup follow the launch's size (four with two chains of chunks each, or eight), its sums
# do not: the first columns of wide experts, whose launch takes four, against the same columns packed alone, bit for bit.
# The two halves of K nearly cancel, so that sums in another order differ in most values.
@pytest.mark.parametrize("H", [1312, 2080, 4160])  # 6, 9 and (512 k each) 9 chunks, the last one a part
@pytest.mark.parametrize("R, kblock", [(6, False), (16, True), (17, False), (32, False), (32, True)])
def test_gate_up_bits(device, H, R, kblock):
    print(f"case H {H} rows {R} kblock {kblock}", flush=True)
    E, k, I, few = 32, 4, 1056, 64
    g = torch.Generator().manual_seed(H + R)
    half = torch.randn(E, H // 2, 2 * I, generator=g) * H ** -0.5
    gu = torch.cat([half, -half + 2.0 ** -7 * torch.randn(E, H // 2, 2 * I, generator=g) * H ** -0.5], 1).to(BF)
    first = torch.cat([gu[:, :, :few], gu[:, :, I:I + few]], 2)
    x = torch.randn(R, H // 2, generator=g)
    tx = torch.cat([x, x], 1).to(BF).reshape(1, 1, R, H).to(device.torch)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(R)]).to(torch.int16)
    tid = ids.reshape(1, 1, R, k).to(device.torch)
    tw = torch.softmax(torch.randn(1, 1, R, k, generator=g), -1).to(BF).to(device.torch)
    u = len(set(ids.flatten().tolist()))

    def h(w, n):
        P = moe8.pack(device, w, torch.zeros(E, n, H, dtype=BF), kblock=kblock)
        return moe8.gate_up_rows(tx, P, tid, tw, k, R, loaders=2).cpu().reshape(-1, min(E, R * k), n)[:R, :u]

    same("the first columns", h(gu, I)[:, :, :few], h(first, few))
