"""Decode attention at head dim 64: the MFMA kernel (GQA 4 and 8, and one-split
rows of MHA and GQA 2) and the VALU kernel beside it, at the edges of their
splits, steps and pages, against 64-bit attention.  Tolerance: both hold the
weights in fp32 (the MFMA form as two fp16 parts), so outputs, weighted means
of N(0, 1) values, are off by their fp16 rounding (2^-11 of at most 5) and
fp32 sums."""
import math

import pytest

pytestmark = pytest.mark.gpu

TOL = 5 * 2 ** -11 + 2 ** -12


def _ref(torch, q, k, v):
    """q [heads, d], k / v [positions, kv_heads, d]."""
    group = q.shape[0] // k.shape[1]
    out = []
    for h in range(q.shape[0]):
        kh, vh = k[:, h // group].double().contiguous(), v[:, h // group].double().contiguous()
        out.append(torch.softmax(kh @ q[h].double() / math.sqrt(q.shape[1]), 0) @ vh)
    return torch.stack(out)


@pytest.mark.parametrize("qh,kvh,p,lengths,capacity,sharp", [
    (8, 2, 16, [1, 15, 16, 17, 31, 33, 127, 129], 256, 1),
    (16, 2, 16, [1, 255, 256, 257, 600, 1000], 1024, 1), (32, 8, 16, [2047, 5, 1300] * 8, 2048, 30),
    (8, 1, 48, [700, 47, 49, 95], 960, 30), (4, 4, 16, [1, 32, 511, 512, 513, 1023], 1024, 1),
    (8, 4, 32, [900, 3, 33], 1024, 30), (32, 32, 16, [300] * 9 + [1], 512, 1),
    (8, 2, 12, [500, 11, 12, 13], 504, 1), (4, 4, 16, [1500, 20], 2048, 1),
    # one VALU split; the first row lengths past it
    (4, 4, 16, [1, 15, 127, 128], 128, 1), (8, 4, 16, [255, 256, 33], 256, 30),
    (4, 4, 16, [256, 257, 272], 272, 1)])
def test_paged_d64_matches_fp64(tmc, qh, kvh, p, lengths, capacity, sharp):
    import torch
    torch.manual_seed(qh * 100 + p)
    d, b, max_pages = 64, len(lengths), capacity // p
    need = [-(-n // p) for n in lengths]
    pages = sum(need) + 2
    order = torch.randperm(pages)
    table = torch.full((b, max_pages), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n].int()
        at += n
    k, v = (torch.randn((pages, kvh, p, d), device="cuda").half() for _ in range(2))
    k *= sharp ** 0.5
    q = torch.randn((b, qh * d), device="cuda").half() * sharp ** 0.5
    out = torch.full_like(q, float("nan"))
    ws = torch.zeros(max(tmc.attention_workspace_bytes(b, qh, kvh, d, capacity) // 4, 1),
                     dtype=torch.float32, device="cuda")
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).cuda()  # noqa: E731
    args = (q, k, v, i32(lengths), i32(table), i32([b]))
    tmc.paged_decode_attention(*args, out, b, qh, kvh, d, p, max_pages, kvh * p * d, p * d, ws)
    for i, n in enumerate(lengths):
        rows = table[i, :need[i]].long().cuda()
        flat = [t[rows].permute(0, 2, 1, 3).reshape(-1, kvh, d)[:n] for t in (k, v)]
        err = (out[i].view(qh, d).double() - _ref(torch, q[i].view(qh, d), *flat)).abs().max().item()
        assert err <= TOL, (i, n, err)
    # a missing page leaves its row's output untouched, the others as they were
    hit = max(range(b), key=lambda i: need[i])
    table[hit, need[hit] // 2] = -1
    again = torch.full_like(q, float("nan"))
    tmc.paged_decode_attention(*args[:4], i32(table), args[5], again, b, qh, kvh, d, p, max_pages,
                               kvh * p * d, p * d, ws)
    assert bool(torch.isnan(again[hit]).all())
    keep = [i for i in range(b) if i != hit]
    assert torch.equal(again[keep], out[keep])


@pytest.mark.parametrize("b,qh,kvh,capacity,length", [
    (1, 8, 2, 2048, 2047), (1, 32, 8, 4096, 1025), (2, 8, 1, 512, 31), (1, 8, 8, 1024, 900),
    (1, 4, 4, 2000, 1999), (1, 8, 8, 512, 511), (2, 8, 4, 257, 257), (1, 4, 4, 256, 256),
    (2, 48, 24, 1024, 1023), (1, 47, 47, 1024, 513),  # 48 and 47 rows past 512 positions
    (64, 32, 32, 16384, 300)])  # 4 GiB a cache: past the buffer loads' range
def test_contiguous_d64_matches_fp64(tmc, b, qh, kvh, capacity, length):
    import torch
    torch.manual_seed(capacity + length)
    d = 64
    k = torch.zeros((b, kvh, capacity, d), dtype=torch.float16, device="cuda")
    v = torch.zeros_like(k)
    for t in (k, v):
        t[:, :, :length] = torch.randn((b, kvh, length, d), device="cuda").half()
    q = torch.randn((b, qh * d), device="cuda").half()
    out = torch.full_like(q, float("nan"))
    ws = torch.zeros(max(tmc.attention_workspace_bytes(b, qh, kvh, d, capacity) // 4, 1),
                     dtype=torch.float32, device="cuda")
    tmc.decode_attention(q, k, v, torch.tensor([length], dtype=torch.int32, device="cuda"), out, b,
                         qh, kvh, d, capacity, ws)
    for i in sorted({0, b - 1}):
        ref = _ref(torch, q[i].view(qh, d), k[i, :, :length].transpose(0, 1),
                   v[i, :, :length].transpose(0, 1))
        err = (out[i].view(qh, d).double() - ref).abs().max().item()
        assert err <= TOL, (i, err)


@pytest.mark.parametrize("qh,kvh,gap,length", [(8, 2, 12.5, 500), (8, 1, 16.4, 2000),
                                               (32, 8, 20.6, 1000), (8, 2, 22.4, 4000)])
def test_small_weights_keep_their_bits(tmc, qh, kvh, gap, length):
    """One position holds the greatest weight and a value of zero, all others
    weigh 2^-gap of it: the output is theirs alone.  fp32 weights (or two fp16
    parts of 22 bits in all down to 2^-18, and 2^-37 absolute below) leave its
    own fp16 rounding, 2^-11, and up to 2^-37 / 2^-gap of it."""
    import torch
    torch.manual_seed(gap)
    d, p = 64, 16
    capacity = -(-length // p) * p
    pages = capacity // p
    k = torch.zeros((pages, kvh, p, d), dtype=torch.float16, device="cuda")
    v = (torch.rand((pages, kvh, p, d), device="cuda") + 1).half() * 2 ** int(gap - 10)
    v[length // 3 // p, :, length // 3 % p] = 0
    k[length // 3 // p, :, length // 3 % p, 0] = gap * math.log(2)
    q = torch.zeros((1, qh, d), dtype=torch.float16, device="cuda")
    q[..., 0] = 8
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).cuda()  # noqa: E731
    out = torch.full((1, qh * d), float("nan"), dtype=torch.float16, device="cuda")
    ws = torch.zeros(max(tmc.attention_workspace_bytes(1, qh, kvh, d, capacity) // 4, 1),
                     dtype=torch.float32, device="cuda")
    tmc.paged_decode_attention(q.view(1, -1), k, v, i32([length]), i32(list(range(pages))), i32([1]),
                               out, 1, qh, kvh, d, p, pages, kvh * p * d, p * d, ws)
    flat = [t.permute(0, 2, 1, 3).reshape(-1, kvh, d)[:length] for t in (k, v)]
    ref = _ref(torch, q[0], *flat)
    err = ((out[0].view(qh, d).double() - ref).abs() / ref.abs()).max().item()
    assert err <= 2 ** -11 + 2 ** -20 + 2.0 ** (gap - 38), err


@pytest.mark.parametrize("qh,kvh,p,length,capacity", [(8, 2, 16, 300, 512), (8, 1, 16, 700, 4096),
                                                      (8, 2, 12, 300, 516), (8, 8, 16, 300, 512)])
def test_infinite_values_stay_infinite(tmc, qh, kvh, p, length, capacity):
    """A V element of +-inf makes its column +-inf, two of opposite sign NaN,
    and reaches nothing else: GQA on the MFMA kernel as on the VALU one (page
    size 12) and in the one-block rows."""
    import torch
    torch.manual_seed(p + length)
    d, pages = 64, -(-capacity // p)
    k, v = (torch.randn((pages, kvh, p, d), device="cuda").half() for _ in range(2))
    q = torch.randn((1, qh * d), device="cuda").half()
    flat = v.permute(0, 2, 1, 3).reshape(-1, kvh, d).clone()
    inf = float("inf")
    put = lambda at, head, col, x: v[at // p, head, at % p].__setitem__(col, x)  # noqa: E731
    for at in range(0, length, 7):
        put(at, 0, 3, inf)
    put(length - 1, 0, 10, inf)
    put(31, kvh - 1, 20, -inf)
    put(5, 0, 40, inf)
    put(length // 2, 0, 40, -inf)
    put(length, 0, 50, inf)  # past the row's length
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).cuda()  # noqa: E731
    out = torch.zeros((1, qh * d), dtype=torch.float16, device="cuda")
    ws = torch.zeros(max(tmc.attention_workspace_bytes(1, qh, kvh, d, pages * p) // 4, 1),
                     dtype=torch.float32, device="cuda")
    tmc.paged_decode_attention(q, k, v, i32([length]), i32(list(range(pages))), i32([1]), out, 1,
                               qh, kvh, d, p, pages, kvh * p * d, p * d, ws)
    kf = k.permute(0, 2, 1, 3).reshape(-1, kvh, d)[:length]
    want = _ref(torch, q.view(qh, d), kf, flat[:length])
    g = qh // kvh
    want[:g, 3] = want[:g, 10] = inf
    want[qh - g:, 20] = -inf
    want[:g, 40] = float("nan")
    got = out.view(qh, d).double()
    assert bool((torch.isnan(got) == torch.isnan(want)).all())
    for sign in (inf, -inf):
        assert bool(((got == sign) == (want == sign)).all())
    fin = torch.isfinite(want)
    assert (got - want)[fin].abs().max().item() <= TOL
