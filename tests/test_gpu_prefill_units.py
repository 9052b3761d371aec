"""The grouped MXFP4 GEMMs over every unit shape: plan blocks of 1..4 M-tiles with full and ragged
last tiles, K that runs on from unit to unit (a multiple of 2048) and K that starts afresh."""
import numpy as np
import pytest
import torch

from conftest import bf16_bits, bits_to_f32, f16_bits, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter", [(1024, 256), (1024, 768), (2048, 512), (3072, 2048), (6144, 256)])
def test_unit_shapes_match_oracle(cuda, orc, hidden, inter):
    from mlxlr8_amd import synth
    from mlxlr8_amd.joined_mxfp4 import JoinedMXFP4
    lens = [1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 130]  # rows of expert 1, 2, ..; expert 0 takes the rest
    L = synth.mxfp4_layer(cuda, 5, hidden=hidden, intermediate=inter, experts=len(lens) + 2)  # the last has no rows
    side = L["side"]
    joined = JoinedMXFP4(L["weights"], L["unit"], {"gate": (None, side["out_gate"]), "up": (None, side["out_up"]),
                                                   "down": (side["in_down"], side["out_down"])}, hidden, inter)
    rows = (sum(lens) + 3) // 9 + 1
    flat = np.concatenate([np.full(n, e + 1) for e, n in enumerate(lens)])
    flat = np.concatenate([flat, np.zeros(9 * rows - flat.size, np.int64)]).astype(np.int32)
    np.random.default_rng(hidden + inter).shuffle(flat)
    ids = flat.reshape(rows, 9)
    x, _ = synth.activations(cuda, 6, rows, hidden)
    print(f"case: unit shapes h={hidden} m={inter} rows={rows}", flush=True)
    values = joined.slots(x, torch.from_numpy(ids).to(cuda))
    again = joined.slots(x, torch.from_numpy(ids).to(cuda))
    assert torch.equal(values.view(torch.int16), again.view(torch.int16))  # whatever block took a unit
    (gc, gs), (dc, ds) = L["weights"]["gate_up"], L["weights"]["down"]
    _, want = orc.mxfp4_moe(bf16_bits(x), ids.astype(np.uint32), np.zeros((rows, 8), np.float32),
                            np.zeros((rows, hidden), np.uint16), hidden, inter, gc.cpu().numpy(), gs.cpu().numpy(),
                            dc.cpu().numpy(), ds.cpu().numpy(), f16_bits(L["unit"]), f16_bits(side["out_gate"]),
                            f16_bits(side["out_up"]), f16_bits(side["in_down"]), f16_bits(side["out_down"]),
                            want_values=True)
    got = bits_to_f32(bf16_bits(values.reshape(rows * 9, hidden)))
    want = bits_to_f32(want).reshape(rows * 9, hidden)
    for e in range(len(lens) + 1):  # expert by expert: a lost tile must not hide in the whole
        at = flat == e
        assert rel_l2(got[at], want[at]) <= 1e-3, f"expert {e} with {at.sum()} rows"  # bf16 casts: 3.6e-4 typical
