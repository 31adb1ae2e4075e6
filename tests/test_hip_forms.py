"""Kernels that come in several forms, at the sizes where the choice falls and at the forms' edges."""
import pytest
import torch

from oracle import zipage_oracle as O

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _rand(*shape, seed, std=1.0, dtype=BF16):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std).to(dtype)


# ------------------------------------------------------------------ compaction
# pairs of (row, tensor): up to 512 take workgroups of sixteen waves, up to 256 workgroups are cut by columns of at
# least 128 bytes; 513 and more take the general form
@pytest.mark.parametrize("dtype,L,B,Hkv,D", [(torch.float32, 1, 1, 1, 256), (torch.float32, 1, 1, 8, 128), (BF16, 1, 1, 2, 128),
                                             (BF16, 2, 8, 8, 128), (torch.float16, 1, 32, 8, 64), (BF16, 1, 33, 8, 64),
                                             (BF16, 1, 2, 3, 48), (torch.float32, 1, 16, 8, 64)])
@pytest.mark.parametrize("style", ["aliased", "cow"])
def test_compaction_of_few_rows(dev, dtype, L, B, Hkv, D, style):
    from zipage_amd.kernel import compress_kv
    BS, budget, NB = 32, 3, 5
    g = torch.Generator().manual_seed(B * 7 + D)
    pages = torch.randperm(B * (NB + 2), generator=g).tolist()
    tables = [[pages.pop() for _ in range(NB - b % 2)] for b in range(B)]
    enc = O.encode_block_table(tables)
    head = [t[:budget + 1] for t in tables]
    if style == "cow":
        head = [[pages.pop(), pages.pop()] + t[2:] for t in head]
    target = torch.tensor(head, dtype=torch.int32)
    k, v = (_rand(L, B * (NB + 2), BS, Hkv, D, seed=s, dtype=dtype) for s in (1, 2))
    scores = O.pad_mask(torch.rand((L, B, Hkv, NB, BS), generator=g), enc).view(L, B, Hkv, NB * BS)
    flag = O.topk_mask(scores, budget * BS).view(L, B, Hkv, NB, BS)
    wk, wv = k.clone(), v.clone()
    O.compress_kv_loop(wk, wv, flag, enc, target)
    gk, gv = k.to(dev), v.to(dev)
    compress_kv(gk, gv, flag.to(dev), enc.to(dev), target.to(dev))
    assert torch.equal(gk.cpu().view(torch.uint8), wk.view(torch.uint8))
    assert torch.equal(gv.cpu().view(torch.uint8), wv.view(torch.uint8))
