"""dK / dV of few (key tile, kv head) items: two groups of waves share an item's (head, query tile) steps."""
import os
import subprocess
import sys

import pytest
import torch

from launches import launches

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
                                         (32, 8, [520, 448, 512, 66]), (1, 1, [512]), (2, 2, [450, 65, 1]), (3, 3, [700, 192])])
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


def against_float64(dx, qkv, do, lens, nh, nkv, causal):
    """The largest errors of dq, dk and dv over the largest entry of each."""
    x, r0 = qkv.double().cpu().requires_grad_(True), 0
    out = []
    for n in lens:
        q, k, v = x[r0:r0 + n].split([nh * D, nkv * D, nkv * D], 1)
        q, k, v = (t.view(n, -1, D).transpose(0, 1) for t in (q, k, v))
        k, v = (t.repeat_interleave(nh // nkv, 0) for t in (k, v))
        s = q @ k.transpose(1, 2) / D ** 0.5
        if causal:
            s = s.masked_fill(~torch.ones(n, n, dtype=torch.bool).tril(), -float("inf"))
        out.append((s.softmax(-1) @ v).transpose(0, 1).reshape(n, nh * D))
        r0 += n
    want = torch.autograd.grad(torch.cat(out), x, do.double().cpu())[0]
    cut = (nh * D, nkv * D, nkv * D)
    return [((a.double().cpu() - b).abs().max() / b.abs().max()).item() for a, b in zip(dx.split(cut, 1), want.split(cut, 1))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("nh,nkv,lens", [(1, 1, [513]), (2, 2, [450, 65, 1]), (8, 2, [130, 64])])
def test_two_groups_against_float64(nh, nkv, lens, causal, dtype):
    """P and dS are rounded to 16 bits once (half an ulp of entries up to the largest), their sums over at most 513 x 4 rows average out:
    one ulp of the largest gradient holds four times what is seen."""
    g = torch.Generator().manual_seed(sum(lens))
    T = sum(lens)
    qkv = (torch.randn(T, (nh + 2 * nkv) * D, generator=g) * 0.5).to(dtype).cuda()
    do = torch.randn(T, nh * D, generator=g).to(dtype).cuda()
    names = [n for n, _, _ in launches(lambda: gradients(qkv, do, lens, nh, nkv, causal))]
    assert [grouped(n) for n in names if "dkdv" in n] == [True]
    assert max(against_float64(gradients(qkv, do, lens, nh, nkv, causal), qkv, do, lens, nh, nkv, causal)) < 2.0 ** (-7 if dtype == torch.bfloat16 else -10)


def grouped(name):
    """Is the kernel the one with two groups of waves (its last template argument)?"""
    return name.split("bwd_dkdv_kernel<")[1].split(">(")[0].rstrip().endswith("2")


@pytest.mark.parametrize("hand_over", [True, False])
@pytest.mark.parametrize("nh,nkv,lens,two", [
    (8, 8, [30], False), (16, 16, [64] * 4, False), (32, 32, [128] * 2, False), (8, 8, [256] * 4, False), (8, 8, [512], True), (8, 8, [64, 449], True),
    (16, 4, [64] * 30, False), (32, 8, [128], True), (16, 2, [1], True), (32, 16, [64] * 30, False), (32, 16, [512] * 4, False), (32, 16, [1024] * 2, True),
    (16, 4, [512] * 9, True), (16, 4, [100] * 40, False), (32, 32, [512] * 2, False)])
def test_short_chains_keep_one_group(nh, nkv, lens, two, hand_over, monkeypatch):
    """Two groups' sums cost more to add than a chain of few (head, query tile) steps saves."""
    import lumen.ops.attention as att

    if not hand_over:
        monkeypatch.setattr(att, "FA_DS_MB", 0)
    qkv = torch.randn(sum(lens), (nh + 2 * nkv) * D, device="cuda", dtype=torch.bfloat16)
    do = torch.randn(sum(lens), nh * D, device="cuda", dtype=torch.bfloat16)
    names = [n for n, _, _ in launches(lambda: gradients(qkv, do, lens, nh, nkv, True)) if "dkdv" in n]
    assert [grouped(n) for n in names] == [two]


@pytest.mark.parametrize("hand_over", [2048, 0])
@pytest.mark.parametrize("switch,grid", [("15", (256, 1, 1)), ("14", (72, 4, 1))])
def test_the_switch_of_persistent_launches(switch, grid, hand_over):
    """288 items: persistent workgroups are one a CU, else there is one an item.  (The switch is read once a process.)"""
    run = """
import torch, test_flash_groups_gpu as t
qkv, do = (torch.randn(9 * 512, n * 128, device="cuda", dtype=torch.bfloat16) for n in (24, 16))
print(*[g for n, g, _ in t.launches(lambda: t.gradients(qkv, do, [512] * 9, 16, 4, True)) if "dkdv" in n])
"""
    tests = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, LUMEN_FA_PERSIST=switch, LUMEN_FA_DS_MB=str(hand_over), PYTHONPATH=os.pathsep.join([os.path.dirname(tests), tests]))
    out = subprocess.run([sys.executable, "-c", run], env=env, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    assert out.stdout.strip().splitlines()[-1] == str(grid)
