"""Causal chunk attention staged by LDS loads: both position-group forms
(at most 256 tiles over more than 1024 positions take four), lengths around
the 32-, 64- and 128-position edges, page sizes that are and are not powers
of two, GQA groups up to 64, strides that fall back to the staged-register
kernel, and scores that keep raising the running maximum."""
import math

import pytest

pytestmark = pytest.mark.gpu


def _attend64(torch, q, k, v, start):
    rows, heads, d = q.shape
    group = heads // k.shape[1]
    mask = (torch.arange(k.shape[0], device="cuda")[None]
            > start + torch.arange(rows, device="cuda")[:, None])
    out = torch.empty((rows, heads, d), dtype=torch.float64, device="cuda")
    for h in range(heads):
        s = q[:, h].double() @ k[:, h // group].double().t().contiguous() / math.sqrt(d)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[:, h // group].double()
    return out


@pytest.mark.parametrize("rows,qh,kvh,d,p,start,capacity,pad,sharp", [
    (1, 4, 4, 128, 16, 0, 64, 0, 1), (33, 8, 8, 64, 16, 0, 4096, 0, 1),
    (64, 8, 2, 128, 16, 64, 2048, 0, 1), (65, 8, 1, 128, 12, 127, 1200, 0, 1),
    (31, 64, 1, 64, 64, 1000, 2048, 0, 1), (130, 32, 32, 128, 16, 31, 200, 0, 1),
    (257, 64, 64, 64, 4, 95, 400, 0, 1), (520, 32, 32, 128, 16, 600, 1200, 0, 30),
    (40, 16, 4, 128, 16, 1500, 2048, 0, 30), (50, 8, 4, 128, 16, 70, 128, 3, 1),
    (40, 8, 2, 64, 4, 100, 32000, 0, 1), (33, 8, 2, 64, 2, 75, 16000, 0, 30),
    (50, 8, 4, 64, 16, 70, 128, 5, 30), (50, 8, 4, 128, 12, 70, 132, 3, 1),
    (20, 4, 4, 128, 1, 30, 64, 1, 1), (600, 32, 32, 128, 1, 0, 4096, 0, 1),
    (600, 32, 32, 128, 1, 40, 5000, 0, 1),
    # one to four position groups with attended positions, of two and of four
    (1, 8, 8, 128, 16, 0, 2048, 0, 1), (32, 8, 8, 128, 16, 0, 2048, 0, 30),
    (64, 8, 2, 128, 16, 0, 2048, 0, 1), (65, 4, 4, 128, 16, 0, 2048, 0, 30),
    (97, 8, 8, 64, 16, 0, 4096, 0, 1), (16, 64, 8, 64, 16, 0, 2048, 0, 1),
    (31, 8, 1, 128, 16, 33, 2048, 0, 1), (33, 8, 2, 128, 16, 0, 512, 0, 1),
    (64, 64, 8, 64, 16, 0, 512, 0, 30)])
def test_prefill_tiles_match_fp64(tmc, rows, qh, kvh, d, p, start, capacity, pad, sharp):
    """pad > 0 moves the heads of a page apart by an odd element count; these,
    and tables past 28 KiB, run the staged-register kernel with the table in
    LDS (as byte offsets where the page size is a power of two from 4 on)."""
    import torch
    torch.manual_seed(rows + start)
    end = start + rows
    pages, max_pages = -(-end // p) + 2, -(-capacity // p)
    table = torch.full((max_pages,), -1, dtype=torch.int32, device="cuda")
    table[:-(-end // p)] = torch.randperm(pages, device="cuda")[:-(-end // p)].int()
    head = p * d + pad
    k, v = (torch.randn((pages, kvh, head), device="cuda").half() for _ in range(2))
    k *= sharp ** 0.5
    q = torch.randn((rows, qh * d), device="cuda").half() * sharp ** 0.5
    valid = torch.arange(start + 1, end + 1, dtype=torch.int32, device="cuda")
    out = torch.full_like(q, float("nan"))
    tmc.prefill_attention(q, k, v, valid, table,
                          torch.tensor([rows], dtype=torch.int32, device="cuda"), out, rows, qh,
                          kvh, d, p, max_pages, kvh * head, head)
    flat = [t[table[:-(-end // p)].long(), :, :p * d].view(-1, kvh, p, d).permute(0, 2, 1, 3)
            .reshape(-1, kvh, d)[:end] for t in (k, v)]
    ref = _attend64(torch, q.view(rows, qh, d), *flat, start).view(rows, -1)
    err = (out.double() - ref).abs().max().item()
    # outputs are weighted means of N(0, 1) values: fp16 weights and results
    # (2^-11 each) of magnitude up to 5
    assert err <= 5 * 2 ** -10 + 2 ** -12, err
