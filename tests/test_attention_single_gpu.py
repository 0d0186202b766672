"""Decoding through the generic kernels: one position an item against the kernel of many rows, and
against attention in float64."""
import pytest
import torch
from helpers import paged_attention

pytestmark = pytest.mark.gpu
DEV = "cuda"
OPTIONS = {
    "plain": {}, "window": dict(window=50), "kept": dict(window=40, keep_first=70),
    "chunk": dict(chunk=48), "slopes": dict(slopes=True), "sinks": dict(sinks=True),
    "cap": dict(softcap=3.0), "gate": dict(gate=True), "pool": dict(window=40, pool=3),
    "pool_only": dict(window=40, pool=3, pool_only=True),
}


@pytest.mark.parametrize("option", OPTIONS)
@pytest.mark.parametrize("D,heads,kv_heads", [(64, 3, 3), (128, 4, 2), (64, 6, 2), (128, 8, 1), (128, 10, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("splits", [1, 3])
def test_one_position_an_item(option, D, heads, kv_heads, dtype, splits):
    """Contexts of one token, of a page's edges and of several pages; a padding item; pages in any
    order with stale bytes (NaN) behind the last key and one page released behind the window.  Both
    kernels do the same float32 arithmetic in another order: results of order one within 2e-6, and
    within a step of the storage type."""
    from edge_infer_amd.csrc import lib
    how = dict(OPTIONS[option])
    if how.get("pool_only") and splits > 1:
        splits = 1
    g = torch.Generator().manual_seed(D + heads + splits)
    contexts = [1, 64, 65, 130, 401]
    width = 8
    order = torch.randperm(len(contexts) * width, generator=g).view(len(contexts), width)
    k = torch.randn(len(contexts) * width, kv_heads, 64, D, generator=g).to(dtype)
    v = torch.randn(len(contexts) * width, kv_heads, 64, D, generator=g).to(dtype)
    for s, n in enumerate(contexts):
        last = order[s, (n - 1) // 64]
        k[last, :, (n - 1) % 64 + 1:] = float("nan")
        v[last, :, (n - 1) % 64 + 1:] = float("nan")
    table = order.clone()
    if "window" in how and "keep_first" not in how:
        table[4, 0] = -1
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    rows = len(contexts) + 1                                    # (the last one is padding)
    q = torch.randn(rows, heads * D, generator=g).to(dtype).to(DEV)
    more = dict(window=how.get("window"), chunk=how.get("chunk"), keep_first=how.get("keep_first", 0),
                softcap=how.get("softcap"))
    if how.get("slopes"):
        more["slopes"] = torch.rand(heads, generator=g).to(DEV) * 0.1
    if how.get("sinks"):
        more["sinks"] = torch.randn(heads, generator=g).to(DEV)
    if how.get("gate"):
        more["gate"] = torch.randn(rows, heads, generator=g).to(DEV)
    if how.get("pool"):
        more.update(pool=how["pool"], pool_only=bool(how.get("pool_only")),
                    pool_k=torch.randn(k.shape, generator=g).to(dtype).to(DEV),
                    pool_v=torch.randn(k.shape, generator=g).to(dtype).to(DEV),
                    pool_table=i32(order.flip(0)))
    results = []
    for single in (False, True):
        out = torch.full((rows, heads * D), 7.0, device=DEV, dtype=dtype)
        part_o = torch.full((rows * heads * splits * D,), 7.0, device=DEV)
        part_ml = torch.full((rows * heads * splits * 2,), 7.0, device=DEV)
        lib.attention(q, k.to(DEV), v.to(DEV), i32([0, 1, 2, 3, 4, -1]), i32(range(rows)), i32([1] * 5 + [0]),
                      rows, i32([n - 1 for n in contexts] + [0]), i32([0, 1, 2, 3, 4, -1]), i32(table), out,
                      heads, kv_heads, D, scale=D ** -0.5, n_splits=splits, part_o=part_o, part_ml=part_ml,
                      single=single, **more)
        if how.get("pool_only"):       # the sums over their own maximum, as the next kernel reads them
            ml = part_ml.view(rows, heads, 2)
            out = torch.cat([part_o.view(rows, heads, D), ml], dim=2)
        results.append(out.float().cpu())
    slow, fast = results
    assert not bool(torch.isnan(fast).any())
    bound = 2e-6 * slow.abs().max().clamp(min=1.0) + (2.0 ** -7 * slow.abs() if dtype == torch.bfloat16 else 0.0)
    assert bool(((slow - fast).abs() <= bound).all())
    assert torch.equal(slow[-1], fast[-1])                      # padding is not written
    # Against float64: scores of a few units are sums of D products (some 1e-6 off), and a weight is
    # off by what its score is; the sums over keys and their join add a few roundings
    host = {n: x.cpu() if isinstance(x, torch.Tensor) else x for n, x in more.items()}
    want, logs = paged_attention(q.cpu(), k, v, table, [0, 1, 2, 3, 4, -1], [n - 1 for n in contexts] + [0], heads,
                                 kv_heads, D ** -0.5, **host)
    if how.get("pool_only"):
        sums, top, total = fast[:, :, :D], fast[:, :, D], fast[:, :, D + 1]
        live = logs[:-1].isfinite()
        assert torch.equal(total[:-1] > 0, live)
        assert ((top + total.log())[:-1][live] - logs[:-1][live]).abs().max().item() <= 4e-6
        got, want = (sums / total[:, :, None])[:-1][live].double(), want[:-1][live]
        assert ((got - want).abs() <= 4e-6 * want.abs().max().clamp(min=1.0)).all()
        return
    got, want = fast.double().view(rows, heads, D)[:-1], want[:-1]
    bound = 4e-6 * want.abs().max().clamp(min=1.0) + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0)
    assert ((got - want).abs() <= bound).all()
