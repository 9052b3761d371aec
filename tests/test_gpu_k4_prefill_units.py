"""The grouped K4 and K3 GEMMs' items of 33..64 rows (each piece decoded once for all rows): full and ragged
M-tiles, and an output width whose last item has one 128-column block."""
import numpy as np
import pytest
import torch

from conftest import bf16_bits, bits_to_f32, f16_bits, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [4, 3])
@pytest.mark.parametrize("h,m", [(256, 128), (384, 256), (1024, 384)])
def test_wide_items_match_oracle(cuda, orc, h, m, k):
    from mlxlr8_amd import synth
    from mlxlr8_amd.fast_prefill import grouped_expert_mlp
    lens = [33, 40, 41, 63, 64, 65, 97, 128, 32]
    layer = synth.k4_layer(cuda, 77, hidden=h, intermediate=m, experts=len(lens) + 1, k=k)
    rows = sum(lens) // 9 + 1
    flat = np.concatenate([np.full(n, e) for e, n in enumerate(lens)])
    flat = np.concatenate([flat, np.full(9 * rows - flat.size, len(lens))]).astype(np.int32)
    rng = np.random.default_rng(h + m)
    rng.shuffle(flat)
    ids = flat.reshape(rows, 9)
    x = torch.from_numpy(rng.normal(size=(rows, h)).astype(np.float32)).to(cuda).to(torch.bfloat16)
    print(f"case: K{k} wide items h={h} m={m} rows={rows}", flush=True)
    values = grouped_expert_mlp(x, torch.from_numpy(ids).to(cuda), layer["packed"], layer["scales"], k, h, m)
    host = {p: layer["packed"][p].cpu().numpy() for p in ("gate", "up", "down")}
    sc = {p: tuple(f16_bits(v) for v in layer["scales"][p]) for p in ("gate", "up", "down")}
    _, want = orc.k4_moe(bf16_bits(x), ids.astype(np.uint32), np.zeros((rows, 8), np.float32),
                         np.zeros((rows, h), np.uint16), h, m, host["gate"], host["up"], host["down"], sc["gate"][0],
                         sc["gate"][1], sc["up"][0], sc["up"][1], sc["down"][0], sc["down"][1], want_values=True, k=k)
    got = bits_to_f32(bf16_bits(values.reshape(rows * 9, h)))
    want = bits_to_f32(want).reshape(rows * 9, h)
    for e in range(len(lens)):  # expert by expert: a lost tile must not hide in the whole
        at = flat == e
        assert rel_l2(got[at], want[at]) <= 1e-3, f"expert {e} with {at.sum()} rows"
