"""Router logits of every tile shape (single, 2 x 2, 4 x 2 tiles of 16 rows x 16 experts) are the same
bits: rows just around each change of shape and ragged ones, against batches of 100 rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [9, 512, 513, 529, 1024, 1025, 1087, 2049])
def test_logits_do_not_depend_on_the_tile(cuda, rows):
    from mlxlr8_amd.fast_router import router_logits
    g = torch.Generator(device=cuda)
    g.manual_seed(rows)
    x = torch.randn((rows, 2048), generator=g, device=cuda).bfloat16()
    w = torch.randn((256, 2048), generator=g, device=cuda) * 0.02
    print(f"case: router tiles rows={rows}", flush=True)
    got = router_logits(x, w)
    for r0 in range(0, rows, 100):
        part = x[r0:r0 + 100]
        pad = torch.cat([part, part[:1].expand(max(0, 9 - part.shape[0]), -1)])  # at least 9 rows: the same kernel
        want = router_logits(pad.contiguous(), w)[:part.shape[0]]
        assert torch.equal(got[r0:r0 + 100], want)
    ref = x.double() @ w.double().T  # 2048 fp32 sums of terms ~0.02: 2048^0.5 * 2^-24 * |partial sum| ~ 5e-6
    assert (got.double() - ref).abs().max().item() <= 2e-5
