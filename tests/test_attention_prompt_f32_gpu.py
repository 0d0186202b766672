"""Float32 prompts through the matrix-instruction kernel against the general kernel, which takes
queries that are not 16-byte aligned, against attention in float64, and a row alone against the same
row among others."""
import pytest
import torch
from helpers import paged_attention

pytestmark = pytest.mark.gpu
DEV = "cuda"
OPTIONS = {
    "plain": {}, "window": dict(window=50), "kept": dict(window=40, keep_first=70),
    "chunk": dict(chunk=48), "slopes": dict(slopes=True), "sinks": dict(sinks=True),
    "cap": dict(softcap=3.0), "gate": dict(gate=True),
}


@pytest.mark.parametrize("option", OPTIONS)
@pytest.mark.parametrize("D,heads,kv_heads", [(64, 3, 3), (128, 4, 2), (64, 6, 2), (128, 16, 1), (128, 20, 1),
                                              (64, 17, 1)])
def test_prompts(option, D, heads, kv_heads):
    """Prompts of one row, of an item's and a page's edges and of several pages, one that goes on
    behind 130 cached tokens; a padding item; pages in any order, stale bytes (NaN) behind the last
    key, a page released behind the window.  Both kernels do float32 arithmetic in another order:
    results of order one within 2e-6 (as for the decode kernel)."""
    from edge_infer_amd.csrc import lib
    how = OPTIONS[option]
    g = torch.Generator().manual_seed(D + heads)
    starts, counts = [0, 0, 0, 130, 0, 63], [1, 16, 65, 70, 260, 2]
    n_seqs, width = len(counts), 6
    order = torch.randperm(n_seqs * width, generator=g).view(n_seqs, width)
    k = torch.randn(n_seqs * width, kv_heads, 64, D, generator=g)
    v = torch.randn(n_seqs * width, kv_heads, 64, D, generator=g)
    for s in range(n_seqs):
        end = starts[s] + counts[s]
        k[order[s, (end - 1) // 64], :, (end - 1) % 64 + 1:] = float("nan")
        v[order[s, (end - 1) // 64], :, (end - 1) % 64 + 1:] = float("nan")
    table = order.clone()
    if option == "window":
        table[3, 0] = -1
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    size = lib.attention_positions_per_item(heads // kv_heads)
    items, row_pos, row_seq, row0 = [], [], [], 0
    for s in range(n_seqs):
        items += [(s, row0 + p, min(size, counts[s] - p)) for p in range(0, counts[s], size)]
        row_pos += range(starts[s], starts[s] + counts[s])
        row_seq += [s] * counts[s]
        row0 += counts[s]
    items.append((-1, row0, 0))
    rows = row0 + 1                                             # (the last one is padding)
    row_pos, row_seq = row_pos + [0], row_seq + [-1]
    q = torch.randn(rows, heads * D, generator=g).to(DEV)
    shifted = torch.empty(q.numel() + 1, device=DEV)[1:].view(q.shape)
    shifted.copy_(q)
    more = dict(window=how.get("window"), chunk=how.get("chunk"), keep_first=how.get("keep_first", 0),
                softcap=how.get("softcap"))
    if how.get("slopes"):
        more["slopes"] = torch.rand(heads, generator=g).to(DEV) * 0.1
    if how.get("sinks"):
        more["sinks"] = torch.randn(heads, generator=g).to(DEV)
    if how.get("gate"):
        more["gate"] = torch.randn(rows, heads, generator=g).to(DEV)

    def run(queries, work):
        out = torch.full((rows, heads * D), 7.0, device=DEV)
        seq, first, npos = (i32([w[i] for w in work]) for i in range(3))
        lib.attention(queries, k.to(DEV), v.to(DEV), seq, first, npos, len(work), i32(row_pos), i32(row_seq),
                      i32(table), out, heads, kv_heads, D, scale=D ** -0.5, **more)
        return out.cpu()

    general, fast = run(shifted, items), run(q, items)
    assert not bool(torch.isnan(fast).any())
    assert (general - fast).abs().max().item() <= 2e-6 * general.abs().max().clamp(min=1.0).item()
    assert torch.equal(general[-1], fast[-1])                   # padding is not written
    # against float64 (see the decode kernel's test for the bound): every seventh row, and the last
    some = sorted({*range(0, rows - 1, 7), rows - 2})
    host = {n: x.cpu() if isinstance(x, torch.Tensor) else x for n, x in more.items()}
    if "gate" in host:
        host["gate"] = host["gate"][some]
    want, _ = paged_attention(q[some].cpu(), k, v, table, [row_seq[r] for r in some], [row_pos[r] for r in some],
                              heads, kv_heads, D ** -0.5, **host)
    got = fast[some].double().view(len(some), heads, D)
    assert (got - want).abs().max().item() <= 4e-6 * want.abs().max().clamp(min=1.0).item()
    alone = run(q, [(s, first + i, 1) for s, first, npos in items for i in range(npos)])
    assert torch.equal(alone, fast)
