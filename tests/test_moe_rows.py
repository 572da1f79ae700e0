"""The MoE down over 17 to 32 rows of bfloat4_b experts (dr_mfma_moe_down_pairs: tiles in pairs, the union's 128-k
steps shared out over the splits' wavefronts), at the shapes where its plan has an edge: one tile and an odd count of
tiles (H), an expert's K of a part of a step, of a step, of one more than a step and of many (I), unions of one expert
(fewer steps than wavefronts) up to all of them, one split and several. Against the oracle's float64 sum over h as the
device holds it, so the bound is derived: y is a bf16 rounding (2^-9 of the value) of float32 sums of exact products,
whose order costs at most n 2^-24 of the sum of the products' magnitudes, n their count."""

import pytest
import torch

from common.testing import same
from moe import moe8
from oracle import dense_oracle as O

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


# experts, slots, H, I, rows
@pytest.mark.parametrize("E, k, H, I, R", [
    (2, 1, 32, 32, 17),  # one tile, a part of a step an expert
    (1, 1, 96, 128, 32),  # three tiles, one expert of one step
    (4, 2, 64, 160, 24),  # a step and a part
    (32, 4, 160, 480, 31),
    (8, 8, 1056, 1408, 32),  # every expert chosen by every row; 33 tiles
    (16, 2, 2080, 256, 18),  # 65 tiles in several splits
    (4, 1, 17440, 96, 20),  # more tile pairs than two a CU: one split
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
