"""The experts' products over groups of row tiles (csrc/moe.hip, many rows per expert and K in whole steps of 64): one step of K, two,
an odd number of them, columns that are no multiple of a tile or of four, groups with one row and with 128, experts with more groups
than a band, experts without rows, every form of the product; and the same rows a tile of 16 at a time; against float64."""
import pytest
import torch

from tests.gpu_util import close, require_gpu

pytestmark = pytest.mark.gpu


def rows_for(kind, E, top, g):
    """ids [T, top]: how many rows the experts get."""
    if kind in ("even", "few"):                  # few: eight to fifteen rows an expert on average
        return torch.stack([torch.randperm(E, generator=g)[:top] for _ in range((40 if kind == "even" else 9) * E // top)]).int()
    # the first expert gets every token (more groups than a band), the last none, the others a few
    T = {"one": 700, "edges": 128}[kind]
    ids = torch.zeros((T, top), dtype=torch.int32)
    for t in range(T):
        ids[t, 1:] = torch.randperm(E - 2, generator=g)[:top - 1].int() + 1
    return ids


@pytest.mark.parametrize("by_groups", [True, False])
@pytest.mark.parametrize("form", ["silu", "clamped", "weighted", "gelu"])
@pytest.mark.parametrize("kind,E,top,K,F", [("even", 6, 2, 64, 64), ("one", 5, 2, 128, 192), ("edges", 9, 3, 192, 320), ("one", 4, 2, 320, 130), ("even", 7, 3, 256, 67 * 4),
                                             ("few", 8, 2, 128, 192), ("few", 16, 4, 64, 320)])
def test_products_over_groups(kind, E, top, K, F, form, by_groups, monkeypatch):
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "experts_by_groups", lambda *sizes: by_groups)         # (few and small experts would not go by groups)
    dev = require_gpu()
    g = torch.Generator().manual_seed(E + K)
    ids = rows_for(kind, E, top, g)
    T, gated = ids.shape[0], form != "gelu"
    bf = lambda *s, std=1.0: (torch.randn(s, generator=g) * std).bfloat16()
    x, wgu, wd = bf(T, K), bf(E, (2 if gated else 1) * F, K, std=K ** -0.5), bf(E, K, F, std=F ** -0.5)
    w = torch.rand((T, top), generator=g)
    kw = dict(silu={}, clamped=dict(activation="clamped", limit=0.8), weighted=dict(activation="clamped", limit=0.8, weight_input=True), gelu=dict(activation="gelu"))[form]
    out = ops.moe_experts(x.to(dev), ids.to(dev), w.to(dev), wgu.to(dev), wd.to(dev), **kw)
    ref = torch.zeros((T, K), dtype=torch.float64)
    xd, wgud, wdd = x.double(), wgu.double(), wd.double()
    for e in range(E):
        for j in range(top):
            at = (ids[:, j] == e).nonzero()[:, 0]
            scale = w[at, j].double()[:, None]
            h = xd[at] @ wgud[e].T * (scale if form == "weighted" else 1.0)
            if form == "gelu":
                a = torch.nn.functional.gelu(h)
            elif form == "silu":
                a = torch.nn.functional.silu(h[:, :F]) * h[:, F:]
            else:
                gate, up = h[:, :F].clamp(max=0.8), h[:, F:].clamp(-0.8, 0.8)
                a = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
            ref[at] += (a @ wdd[e].T) * (1.0 if form == "weighted" else scale)
    close(out, ref, torch.bfloat16, scale=2.0, what="experts over groups")


def test_groups_of_an_alignment():
    """Every sorted row of an expert lies in one group, groups begin every eight tiles of an expert, bands hold up to four of them."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(5)
    for T, E, top in ((1, 1, 1), (3, 7, 2), (900, 3, 1), (700, 40, 3)):
        routes = ops.ExpertTables()
        table = torch.rand((11, E), generator=g).argsort(dim=1)[:, :top].to(torch.int32).contiguous()
        routes.add(table.to(dev), E)
        al = routes.align(torch.randint(0, 11, (T,), generator=g, dtype=torch.int32).to(dev))[0]
        te, gr = al.tile_expert.cpu().tolist(), al.groups.cpu().tolist()
        seen, n = [], gr[0]
        assert 1 + 2 * n <= len(gr)
        for i in range(n):
            tile, tiles, first, in_band = gr[1 + 2 * i] >> 4, gr[1 + 2 * i] & 15, gr[2 + 2 * i] >> 3, gr[2 + 2 * i] & 7
            assert 1 <= tiles <= 8 and len({te[t] for t in range(tile, tile + tiles)}) == 1 and te[tile] >= 0
            assert first <= i < first + in_band and 1 <= in_band <= 4
            assert all(te[gr[1 + 2 * j] >> 4] == te[tile] for j in range(first, first + in_band))
            seen += list(range(tile, tile + tiles))
        assert seen == [t for t, e in enumerate(te) if e >= 0]


@pytest.mark.parametrize("by_groups", [True, False])
@pytest.mark.parametrize("form", ["silu", "weighted", "gelu"])
@pytest.mark.parametrize("kind,E,top,K,F", [("even", 6, 2, 128, 128), ("one", 5, 2, 384, 128), ("edges", 9, 3, 256, 640), ("few", 16, 4, 128, 384), ("one", 40, 3, 640, 1024), ("few", 3, 1, 128, 384)])
def test_experts_in_operand_order(kind, E, top, K, F, form, by_groups, monkeypatch):
    """Matrices in operand order: one turn of 128 of K, an odd number of them, groups in halves and whole, as many blocks as the grid can have at most, against the rows' kernels."""
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "experts_by_groups", lambda *sizes: by_groups)
    dev = require_gpu()
    g = torch.Generator().manual_seed(E + K)
    ids = rows_for(kind, E, top, g)
    T, gated = ids.shape[0], form != "gelu"
    bf = lambda *s, std=1.0: (torch.randn(s, generator=g) * std).bfloat16().to(dev)
    x, wgu, wd, w = bf(T, K), bf(E, (2 if gated else 1) * F, K, std=K ** -0.5), bf(E, K, F, std=F ** -0.5), torch.rand((T, top), generator=g).to(dev)
    kw = dict(silu={}, weighted=dict(activation="clamped", limit=0.8, weight_input=True), gelu=dict(activation="gelu"))[form]
    tiled = [ops.expert_forms([m.tensor_split(2) if gated and mats is wgu else [m] for m in mats]) for mats in (wgu, wd)]
    assert all(isinstance(m, ops.TiledExperts) for m in tiled) and torch.equal(tiled[0].rows(), wgu)
    out = ops.moe_experts(x, ids.to(dev), w, *tiled, **kw)
    ref = ops.moe_experts(x.float(), ids.to(dev), w, wgu.float(), wd.float(), **kw)          # (float32 kernels, no rounding in between)
    close(out, ref, torch.bfloat16, scale=2.0, what="experts in operand order")
    if kind == "even":
        close(ops.moe_experts(x.float(), ids.to(dev), w, *tiled, **kw), ref, torch.float32, what="float32 rows of the same matrices")


@pytest.mark.parametrize("dtype,form", [("float32", "silu"), ("float32", "gelu"), ("bfloat16", "silu"), ("bfloat16", "gelu")])
def test_plain_kernel_reads_operand_order(dtype, form, monkeypatch):
    """The plain kernel (float32 rows; bfloat16 ones with MOE_MFMA off) reads matrices in operand order as they lie, and sums the same values
    in the same order as from rows; no copy of the matrices is made."""
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "MOE_MFMA", False)
    dev = require_gpu()
    g = torch.Generator().manual_seed(11)
    E, top, K, F, T, gated = 5, 2, 256, 384, 37, form != "gelu"
    bf = lambda *s, std=1.0: (torch.randn(s, generator=g) * std).bfloat16().to(dev)
    x, wgu, wd = bf(T, K).to(getattr(torch, dtype)), bf(E, (2 if gated else 1) * F, K, std=K ** -0.5), bf(E, K, F, std=F ** -0.5)
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).int().to(dev)
    w = torch.rand((T, top), generator=g).to(dev)
    tiled = [ops.expert_forms([[m] for m in mats]) for mats in (wgu, wd)]
    assert all(isinstance(m, ops.TiledExperts) for m in tiled)
    ref = ops.moe_experts(x, ids, w, wgu, wd, activation=form)
    monkeypatch.setattr(ops.TiledExperts, "rows", lambda self: pytest.fail("the matrices were copied"))
    assert torch.equal(ops.moe_experts(x, ids, w, *tiled, activation=form), ref)


def test_more_rows_than_offsets_of_31_bits_reach():
    """Experts in operand order where the activations pass 2^31 bytes and the sorted rows 2^20."""
    from spyinfer_amd.kernels import ops
    dev = require_gpu()
    g = torch.Generator().manual_seed(12)
    E, K, F, T = 8, 128, 1024, 131200
    bf = lambda *s, std=1.0: (torch.randn(s, generator=g) * std).bfloat16()
    x, wgu, wd, w = bf(T, K), bf(E, 2 * F, K, std=K ** -0.5), bf(E, K, F, std=F ** -0.5), torch.rand((T, E), generator=g)
    ids = torch.arange(E, dtype=torch.int32).expand(T, E).contiguous()
    assert 2 * T * E * F >= 1 << 31 and T * E > 1 << 20 and ops.experts_by_groups(T * E, E, K, F, True, True)
    mats = [ops.expert_forms([[m] for m in mats.to(dev)]) for mats in (wgu, wd)]
    assert all(isinstance(m, ops.TiledExperts) for m in mats)
    out = ops.moe_experts(x.to(dev), ids.to(dev), w.to(dev), *mats)
    at = torch.tensor([0, 1, 16, 77777, T // 2, T - 17, T - 1])
    h = torch.einsum("tk,enk->ten", x[at].double(), wgu.double())
    ref = torch.einsum("tef,ekf,te->tk", torch.nn.functional.silu(h[..., :F]) * h[..., F:], wd.double(), w[at].double())
    close(out[at.to(dev)], ref, torch.bfloat16, scale=2.0, what="experts of many rows")


@pytest.mark.parametrize("by_groups", [True, False])
def test_nan_stays_with_its_token(by_groups, monkeypatch):
    """Rows that do not exist are read as row 0: what it holds stays with its own token."""
    from spyinfer_amd.kernels import ops
    monkeypatch.setattr(ops, "experts_by_groups", lambda *sizes: by_groups)
    dev = require_gpu()
    g = torch.Generator().manual_seed(13)
    E, top, K, F = 6, 2, 256, 384
    ids = rows_for("even", E, top, g).to(dev)
    T = ids.shape[0]
    bf = lambda *s, std=1.0: (torch.randn(s, generator=g) * std).bfloat16().to(dev)
    x, w = bf(T, K), torch.rand((T, top), generator=g).to(dev)
    mats = [ops.expert_forms([[m] for m in t]) for t in (bf(E, 2 * F, K, std=K ** -0.5), bf(E, K, F, std=F ** -0.5))]
    ref = ops.moe_experts(x, ids, w, *mats)
    x[0, 5], x[T - 1, 7] = float("nan"), float("inf")
    out = ops.moe_experts(x, ids, w, *mats)
    assert not ref.isnan().any() and out[0].isnan().all() and torch.equal(out[1:-1], ref[1:-1])
