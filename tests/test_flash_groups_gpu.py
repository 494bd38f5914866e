"""dK / dV of few (key tile, kv head) items: two groups of waves share an item's (head, query tile) steps."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def gradients(qkv, do, lens, nh, nkv, causal):
    from lumen.ops.attention import flash_attention_qkv

    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    x = qkv.clone().requires_grad_(True)
    o = flash_attention_qkv(x, tuple(cu), nh, nkv, D, causal)
    return torch.autograd.grad(o, x, do.view_as(o))[0]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("hand_over", [True, False])
@pytest.mark.parametrize("nh,nkv,lens", [(1, 1, [1]), (2, 2, [64, 65, 1]), (3, 1, [129, 63]), (3, 3, [300, 192]), (8, 2, [511, 130]),
                                         (32, 8, [520, 448, 512, 66])])
def test_two_groups(nh, nkv, lens, causal, hand_over, dtype, monkeypatch):
    """Against one group, which the same sequences take among so many others that the items fill the chip: the steps' sums
    in another order, fp32 sums of at most 36 x 64 products, so 2^-13 of the largest gradient at most, and a result that may
    round the other way."""
    import lumen.ops.attention as att

    if not hand_over:
        monkeypatch.setattr(att, "FA_DS_MB", 0)
    g = torch.Generator().manual_seed(sum(lens) + nh)
    T = sum(lens)
    qkv = (torch.randn(T, (nh + 2 * nkv) * D, generator=g) * 0.5).to(dtype).cuda()
    do = torch.randn(T, nh * D, generator=g).to(dtype).cuda()
    items = sum(-(-n // 64) for n in lens) * nkv
    assert items <= 256
    times = 512 // items + 1
    got = gradients(qkv, do, lens, nh, nkv, causal)
    one = gradients(qkv.repeat(times, 1), do.repeat(times, 1), lens * times, nh, nkv, causal)
    assert torch.equal(one[:T], one[T:2 * T])
    a, b = got.float(), one[:T].float()
    ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    assert torch.equal(a[:, :nh * D], b[:, :nh * D]) or (a - b)[:, :nh * D].abs().max() <= 2 * ulp * b[:, :nh * D].abs().max()
    for part in (slice(nh * D, (nh + nkv) * D), slice((nh + nkv) * D, None)):
        d = (a[:, part] - b[:, part]).abs()
        assert (d <= ulp * b[:, part].abs() + 2.0 ** -13 * b[:, part].abs().max()).all()
