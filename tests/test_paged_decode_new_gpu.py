"""A decode step's rotary turn and cache write inside its paged attention, against the two-launch form."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(D, nh, nkv, lens, dt, fp8, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    bs, N = 2048 // D, len(lens)
    need = [(n + bs - 1) // bs for n in lens]
    nb = sum(need) + 2
    free = torch.randperm(nb - 1, generator=torch.Generator().manual_seed(seed)).tolist()
    bt = torch.zeros(N, max(need) + 1, dtype=torch.int32)
    for i, n in enumerate(need):
        bt[i, :n] = torch.tensor([1 + free.pop() for _ in range(n)], dtype=torch.int32)
    bt, cl = bt.cuda(), torch.tensor(lens, dtype=torch.int32, device="cuda")
    pos = cl - 1
    slots = bt[torch.arange(N, device="cuda"), (pos // bs).long()].long() * bs + pos.long() % bs
    kc = torch.randn(nb, nkv, bs, D, device="cuda", generator=g).to(dt)
    vc = torch.randn(nb, nkv, bs, D, device="cuda", generator=g).to(dt)
    if fp8:
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    qkv = torch.randn(N, (nh + 2 * nkv) * D, device="cuda", generator=g).to(dt)
    from lumen.ops.rope import rope_tables

    cos, sin = rope_tables(D, max(lens) + 1, 10000.0, torch.device("cuda"))
    return qkv, kc, vc, bt, cl, pos, slots, cos, sin


@pytest.mark.parametrize("D,nh,nkv,dt,fp8", [
    (128, 8, 8, torch.bfloat16, False), (128, 8, 1, torch.float16, False), (64, 4, 2, torch.bfloat16, False),
    (64, 2, 2, torch.bfloat16, True), (32, 4, 1, torch.float16, False), (256, 2, 2, torch.bfloat16, False),
    (256, 4, 1, torch.bfloat16, False), (128, 8, 2, torch.bfloat16, True)])
def test_new_tokens(D, nh, nkv, dt, fp8):
    """Contexts of one token, at the edges of blocks, steps and partitions; a row whose slot is -1."""
    from lumen.ops.attention import paged_decode, paged_decode_new, paged_decode_new_ok, rope_write_kv

    bs = 2048 // D
    lens = [1, 2, bs, bs + 1, 4 * bs, 4 * bs + 1, 64, 65, 128, 129, 300, 513]
    args = _case(D, nh, nkv, lens, dt, fp8)
    qkv, kc, vc, bt, cl, pos, slots, cos, sin = args
    slots[3] = -1                                       # not written: its output is compared all the same
    for part in (64, 512):
        k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
        assert paged_decode_new_ok(qkv, k1, nh, part)
        keep = qkv.clone()
        got = paged_decode_new(qkv, k1, v1, pos, cos, sin, slots, bt, cl, max(lens) + 700, nh, 1 / math.sqrt(D), part)
        assert torch.equal(qkv, keep)
        x = qkv.clone()
        rope_write_kv(x, pos, nh, nkv, D, cos, sin, k2, v2, slots)
        assert torch.equal(k1.view(torch.uint8), k2.view(torch.uint8))
        assert torch.equal(v1.view(torch.uint8), v2.view(torch.uint8))
        ref = paged_decode(x[:, :nh * D].view(len(lens), nh, D), k2, v2, bt, cl, max(lens) + 700,
                           1 / math.sqrt(D), part)
        on = torch.arange(len(lens), device="cuda") != 3
        # the same rows and rounding, summed in another order: fp32 sums, results rounded to 16 bits once
        err = (got.float() - ref.float())[on].norm() / ref.float()[on].norm()
        assert err < (4e-3 if dt == torch.bfloat16 else 5e-4)
        # one token: its value row itself
        v = qkv[0, (nh + nkv) * D:].view(nkv, 1, D).expand(nkv, nh // nkv, D).reshape(nh, D)
        v = v.to(torch.float8_e4m3fn).to(dt) if fp8 else v
        assert torch.equal(got[0], v)


@pytest.mark.parametrize("D,nh,nkv,dt,fp8", [
    (128, 8, 8, torch.bfloat16, False), (128, 32, 8, torch.bfloat16, True), (64, 16, 8, torch.float16, False),
    (128, 8, 8, torch.float16, False), (32, 8, 8, torch.float16, False), (256, 8, 8, torch.float16, False)])
@pytest.mark.parametrize("part", [128, 512])
def test_large_batches_walk_the_heads_first(D, nh, nkv, dt, fp8, part):
    """From 512 (sequence, key head) pairs on the grid's axes change places: ragged contexts over several partitions, with
    and without the step's own tokens; a few of the sequences alone, which keep the other grid, give the same bits."""
    from lumen.ops.attention import paged_decode, paged_decode_new, paged_decode_ref, rope_write_kv

    lens = [1 + (i * 97) % 701 for i in range(64)]                   # 64 x 8 pairs; a few x 8
    qkv, kc, vc, bt, cl, pos, slots, cos, sin = _case(D, nh, nkv, lens, dt, fp8, 3)
    scale, few = 1 / math.sqrt(D), 9
    x, k2, v2 = qkv.clone(), kc.clone(), vc.clone()
    rope_write_kv(x, pos, nh, nkv, D, cos, sin, k2, v2, slots)
    q = x[:, :nh * D].view(len(lens), nh, D)
    ref = paged_decode_ref(q.float(), k2.float(), v2.float(), bt, cl, scale)
    for n in (len(lens), few):
        k1, v1 = kc.clone(), vc.clone()
        got = paged_decode_new(qkv[:n], k1, v1, pos[:n], cos, sin, slots[:n], bt[:n], cl[:n], 701, nh, scale, part)
        old = paged_decode(q[:n], k2, v2, bt[:n], cl[:n], 701, scale, part)
        if n > few:
            assert torch.equal(k1.view(torch.uint8), k2.view(torch.uint8))
            assert torch.equal(v1.view(torch.uint8), v2.view(torch.uint8))
            all_new, all_old = got, old
        for y in (got, old):
            # the result's rounding and the weights' and sums' in fp32, relative to the largest entry
            err = (y.float() - ref[:n]).abs().max() / ref.abs().max()
            assert err < (2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11) * 1.1
    assert torch.equal(got, all_new[:few]) and torch.equal(old, all_old[:few])


def test_refused():
    """Rows the kernel cannot take stay with the two-launch form; what does not fit is an error."""
    from lumen.ops.attention import paged_decode_new_ok
    from lumen.ops._native import native

    qkv, kc, vc, bt, cl, pos, slots, cos, sin = _case(128, 4, 4, [5, 9], torch.bfloat16, False)
    assert paged_decode_new_ok(qkv, kc, 4, 64)
    assert not paged_decode_new_ok(qkv, kc[:, :, :8].contiguous(), 4, 64)
    assert not paged_decode_new_ok(qkv, kc, 4, 24)
    assert not paged_decode_new_ok(qkv[:, 8:], kc, 4, 64)
    assert not paged_decode_new_ok(torch.cat([qkv, qkv], 1)[:, 4:], kc, 4, 64)
    q = qkv[:, :512].reshape(2, 4, 128).contiguous()                 # no key and value behind the query
    one = torch.empty(1, 1, 1, device="cuda")
    with pytest.raises(ValueError):
        native().paged_attention_decode(torch.empty_like(q), q, kc, vc, bt, cl, 4, 16, bt.shape[1], 0.1, one, one,
                                        one, 64, None, 3, pos, cos, sin, slots)


@pytest.mark.parametrize("D,nh,nkv,dt", [(128, 5, 5, torch.bfloat16), (64, 6, 3, torch.float16), (32, 4, 1, torch.bfloat16), (256, 2, 2, torch.float16)])
def test_merge_of_partitions(D, nh, nkv, dt):
    """Up to 130 partitions, at the edges of the merge's 4 and 16 rows and 64 lanes, over parts that hold NaN where no partition
    lies; against the context in one partition, whose fp32 sums have another order, so a result may round the other way."""
    from lumen.ops._native import native
    from lumen.ops.attention import PA_ONE_PASS, paged_decode

    lens = [64, 65, 128, 129, 4 * 64, 4 * 64 + 1, 16 * 64, 16 * 64 + 1, 32 * 64 + 7, 64 * 64 - 1, 64 * 64 + 1, 80 * 64 + 1, 130 * 64 - 5]
    qkv, kc, vc, bt, cl, *_ = _case(D, nh, nkv, lens, dt, False)
    q = qkv[:, :nh * D].view(len(lens), nh, D)
    m, l = (torch.full((len(lens), nh, 140), math.nan, device="cuda") for _ in range(2))
    o = torch.full((len(lens), nh, 140, D), math.nan, device="cuda")
    got = torch.full((len(lens), nh, D), math.nan, device="cuda", dtype=dt)
    native().paged_attention_decode(got, q, kc, vc, bt, cl, nkv, kc.shape[2], bt.shape[1], 1 / math.sqrt(D), m, l, o, 64, None, PA_ONE_PASS)
    for i, n in enumerate(lens):
        parts = -(-n // 64) if n > 64 else 0                 # (one partition writes its result at once)
        assert m[i, :, parts:].isnan().all() and l[i, :, parts:].isnan().all() and o[i, :, parts:].isnan().all()
        assert parts == 0 or m[i, :, :parts].isfinite().all()
    got = got.float()
    one = paged_decode(q, kc, vc, bt, cl, 140 * 64, 1 / math.sqrt(D), 140 * 64).float()
    ulp = 2.0 ** (-7 if dt == torch.bfloat16 else -10)
    assert ((got - one).abs() <= ulp * one.abs() + 2.0 ** -16 * one.abs().max()).all()
