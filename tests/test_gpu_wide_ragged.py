"""Rows of 64 lane vectors (streamed) and rows of any other width (the ragged kernel) at the edges of their
inputs, on the GPU: Inf, NaN, overflow and subnormals among the rows, with row 0 not finite (the rows that a
lane reads past its bag must leave no trace); malformed offsets (decreasing, negative, past nnz); tables beside
and beyond the 4 GiB that 32-bit row offsets reach.

Bar: the oracle's result bit for bit (NaN where it has NaN); with the LayerNorm, the tolerance of
test_gpu_fused_norm.py, or the two launches' result.
"""
import numpy as np
import pytest
import torch

from _cases import random_case
from oracle import ebag_oracle as orc
from test_gpu_fused_norm import check, expected, run_fused
from test_gpu_parity import TORCH_DT, _special_rows, to_np
from test_gpu_stream import _malformed

pytestmark = pytest.mark.gpu

WIDE = {"f32": 256, "bf16": 512, "f16": 512, "i8": 512}


def _to_dev(arr, tdt, dev, layout):
    """A table on the device: rows next to one another, 16 bytes further apart, or from the second element on."""
    t = torch.from_numpy(np.ascontiguousarray(arr))
    if tdt in ("bf16", "f16"):
        t = t.view(torch.int16).view(TORCH_DT[tdt])
    V, D = t.shape
    pitch, first = {"packed": (D, 0), "padded": (D + 16 // t.element_size(), 0), "odd base": (D, 1)}[layout]
    view = torch.as_strided(torch.zeros(V * pitch + first, dtype=t.dtype, device=dev), (V, D), (pitch, 1), first)
    view.copy_(t)
    return view


def _tables(host, tdt, dev, layout):
    if tdt == "i8":
        return [(_to_dev(q, tdt, dev, layout), torch.from_numpy(s).to(dev)) for q, s in host]
    return [_to_dev(t, tdt, dev, layout) for t in host]


def _int8(case, seed):
    """int8 tables of a case's shapes."""
    rng = np.random.default_rng(seed)
    return [(rng.integers(-128, 128, t.shape).astype(np.int8), (rng.random(len(t)) * 0.02 + 1e-4).astype(np.float32))
            for t in case.tables]


def _pool(pkg, dev, values, offsets, tables, pooling, odt):
    out = pkg.embedding_bag_pooled(torch.from_numpy(values).to(dev), torch.from_numpy(offsets).to(dev), tables,
                                   pooling=pooling, out_dtype=TORCH_DT[odt])
    return to_np(out, odt)


def _same(got, want, odt):
    g, w = orc.decode(got, odt), orc.decode(want, odt)
    assert np.array_equal(np.isnan(g), np.isnan(w))
    finite = ~np.isnan(w)
    assert np.array_equal(got[finite], want[finite])


@pytest.mark.parametrize("tdt,D", [(t, d) for t in ("f32", "bf16", "f16", "i8") for d in (3, 9, 50, 100, 300, WIDE[t])])
@pytest.mark.parametrize("layout", ["packed", "padded", "odd base"])
@pytest.mark.parametrize("pooling", ["sum", "mean"])
def test_special_values(pkg, dev, tdt, D, layout, pooling):
    print(f"special values {tdt} D={D} {layout} {pooling}", flush=True)
    rows = _special_rows(D)
    n = len(rows)
    if tdt == "i8":  # the special values as the rows' scales
        rng = np.random.default_rng(D)
        host = [(rng.integers(-3, 4, (n, D)).astype(np.int8), rows[:, 0].copy())]
    else:
        host = [orc.encode(rows, tdt)]
    bags = [[]] * 9 + [[i] for i in range(n)] + [[i, j] for i in range(n) for j in range(n)] + \
           [[i, j, k] for i in range(0, n, 3) for j in range(1, n, 4) for k in range(2, n, 5)] + \
           [[9] * m + [17] for m in (7, 63, 64, 65, 130)]
    np.random.default_rng(6).shuffle(bags)
    values = np.concatenate([np.array(b, np.int64) for b in bags])
    offsets = np.concatenate([[0], np.cumsum([len(b) for b in bags])]).astype(np.int64)
    tables = _tables(host, tdt, dev, layout)
    for odt in ("f32", "bf16"):
        _same(_pool(pkg, dev, values, offsets, tables, pooling, odt),
              orc.pool_c(values, offsets, host, tdt, pooling, odt), odt)


@pytest.mark.parametrize("tdt,dims", [("bf16", (512,)), ("f32", (256,)), ("f16", (512,)), ("i8", (512,)),
                                      ("bf16", (9, 100, 300, 1030)), ("f32", (3, 50, 260)), ("i8", (7, 50, 513))])
@pytest.mark.parametrize("layout", ["packed", "padded", "odd base"])
def test_malformed_global_offsets(pkg, dev, tdt, dims, layout):
    print(f"malformed global {tdt} {dims} {layout}", flush=True)
    rng = np.random.default_rng(sum(dims))
    for B in (45, 1200):  # few bags: tiles of two; many: of four
        case = random_case(dims[0] + B, F=8, B=B, dims=dims, V=(300,), max_len=12, tdt="f32" if tdt == "i8" else tdt)
        host = _int8(case, B) if tdt == "i8" else case.tables
        bad = _malformed(case.offsets, case.values.size, rng)
        tables = _tables(host, tdt, dev, layout)
        for pooling in ("sum", "mean"):
            want = orc.pool_c(case.values, bad, host, tdt, pooling, "f32")
            assert np.array_equal(_pool(pkg, dev, case.values, bad, tables, pooling, "f32"), want), (B, pooling)


def _reference_batch(seed, S, B, V, max_len):
    """(values, malformed row offsets, slot starts) of the reference layout."""
    case = random_case(seed, F=S, B=B, dims=(8,), V=(V,), max_len=max_len, tdt="f32")
    ro, vo = case.reference_layout()
    return case.values, _malformed(ro, case.values.size, np.random.default_rng(seed)), vo


@pytest.mark.parametrize("tdt,D", [("bf16", 512), ("f32", 256)])
@pytest.mark.parametrize("max_len", [4, 20])  # rounds of bags, and walks over them
def test_malformed_offsets_with_the_layer_norm(pkg, dev, tdt, D, max_len):
    print(f"malformed fused norm {tdt} D={D} max_len={max_len}", flush=True)
    S, B, V = 12, 41, 500
    v, ro, vo = _reference_batch(max_len, S, B, V, max_len)
    rng = np.random.default_rng(D)
    w = torch.from_numpy(rng.integers(-8, 9, (V, D)).astype(np.float32)).to(TORCH_DT[tdt]).to(dev)
    g = torch.from_numpy((1 + 0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(dev)
    b = torch.from_numpy((0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(dev)
    for pooling in ("sum", "mean"):
        check(run_fused(pkg, dev, v, ro, vo, w, g, b, B, pooling), expected(v, ro, vo, w, g, b, B, pooling, tdt), tdt)


@pytest.mark.parametrize("max_len", [4, 20])
def test_malformed_offsets_with_the_int8_layer_norm(pkg, dev, max_len):
    print(f"malformed int8 fused norm max_len={max_len}", flush=True)
    S, B, V, D = 12, 41, 500, 512
    v, ro, vo = (torch.from_numpy(a).to(dev) for a in _reference_batch(max_len, S, B, V, max_len))
    gen = torch.Generator(device="cpu").manual_seed(max_len)
    q = torch.randint(-128, 128, (V, D), generator=gen, dtype=torch.int8).to(dev)
    scale = (torch.rand(V, generator=gen) * 0.01 + 1e-4).to(dev)
    gamma = (1 + 0.1 * torch.randn(S * D, generator=gen)).to(dev)
    beta = (0.1 * torch.randn(S * D, generator=gen)).to(dev)
    pooled = torch.empty(B, S * D, dtype=torch.bfloat16, device=dev)
    pkg.fused_all_slots_embedding_int8(v, vo, ro, q, scale, pooled, B, D, V - 1)
    host = [(q.cpu().numpy(), scale.cpu().numpy())] * S
    oracle = orc.pool_c(v.cpu().numpy(), ro.cpu().numpy(), host, "i8", "sum", "bf16", batch=B, val_base=vo.cpu().numpy())
    assert np.array_equal(to_np(pooled, "bf16"), oracle)
    got = torch.full_like(pooled, float("nan"))
    pkg.fused_all_slots_embedding_int8_layernorm(v, vo, ro, q, scale, got, B, D, V - 1, gamma, beta, 1e-5)
    want = pkg.layer_norm(pooled, gamma, beta, 1e-5).double()
    # as test_fused_int8_layernorm_equals_two_launches
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -7 * (1 + 2.0 ** -7) + 2e-5).all()


@pytest.mark.parametrize("tdt,D", [("bf16", 512), ("f32", 256)])
def test_walks_and_rounds_pool_alike(pkg, dev, tdt, D):
    """A sample's normalised row is the same bits in a batch whose mean bag length takes the walk and in one
    whose empty samples take the rounds; and pooled, in tiles of two bags and of four."""
    print(f"walk and rounds {tdt} D={D}", flush=True)
    S, B, V, more = 28, 67, 900, 1300
    rng = np.random.default_rng(D)
    L = rng.integers(0, 17, (S, B))
    L[::5, ::7] = 90
    wide = np.concatenate([L, np.zeros((S, more), np.int64)], axis=1)
    assert L.sum() > 4 * L.size and wide.sum() < 4 * wide.size
    ids = torch.from_numpy(rng.integers(0, V, int(L.sum()))).to(dev)
    w = torch.from_numpy(rng.standard_normal((V, D)).astype(np.float32)).to(TORCH_DT[tdt]).to(dev)
    g = torch.from_numpy((1 + 0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(dev)
    b = torch.from_numpy((0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(dev)
    rows = []
    for lens in (L, wide):
        n = lens.shape[1]
        ro = np.zeros((S, n + 1), np.int64)
        np.cumsum(lens, axis=1, out=ro[:, 1:])
        vo = torch.from_numpy(np.concatenate([[0], np.cumsum(lens.sum(axis=1))[:-1]]).astype(np.int64)).to(dev)
        ro = torch.from_numpy(ro.reshape(-1)).to(dev)
        normed, pooled = (torch.empty((n, S * D), dtype=w.dtype, device=dev) for _ in range(2))
        pkg.fused_all_slots_embedding_layernorm(ids, vo, ro, w, normed, n, D, V - 1, g, b, 1e-5)
        pkg.fused_all_slots_embedding(ids, vo, ro, w, pooled, n, D, V - 1)
        rows.append((normed[:B], pooled[:B]))
    for x, y in zip(*rows):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("tdt,D,over", [("bf16", 100, 0), ("bf16", 100, 1), ("f32", 50, 0), ("f32", 50, 300_000),
                                        ("bf16", 301, 0), ("i8", 50, 5_000_000)])
def test_ragged_table_beside_and_beyond_4_gib(pkg, dev, tdt, D, over):
    """The largest table that 32-bit offsets reach (over = 0), one row more, and far more: bags of its first and
    last rows, of every length beside empty ones, give what the oracle gives for those rows alone."""
    elem = {"bf16": 2, "f32": 4, "i8": 1}[tdt]
    V = (2 ** 32 - D * elem - 1) // (D * elem) + over
    print(f"ragged {tdt} D={D} rows={V}", flush=True)
    rng = np.random.default_rng(D + over)
    dt = torch.int8 if tdt == "i8" else TORCH_DT[tdt]
    table = torch.zeros(V, D, dtype=dt, device=dev)
    used = np.unique(np.concatenate([np.arange(40), V - 1 - np.arange(90), rng.integers(0, V, 60)]))
    small = rng.integers(-128, 128, (len(used), D))
    at = torch.from_numpy(used).to(dev)
    if tdt == "i8":
        host = (small.astype(np.int8), (rng.random(len(used)) * 0.02 + 1e-4).astype(np.float32))
        table[at] = torch.from_numpy(host[0]).to(dev)
        scale = torch.zeros(V, device=dev)
        scale[at] = torch.from_numpy(host[1]).to(dev)
        arg = (table, scale)
    else:
        host = orc.encode(small.astype(np.float32) * np.float32(0.37), tdt)
        t = torch.from_numpy(host)
        table[at] = (t if tdt == "f32" else t.view(torch.int16).view(dt)).to(dev)
        arg = table
    L = np.concatenate([rng.integers(0, 9, 150), [70, 0, 0, 1, 200], np.zeros(40, np.int64)])
    rng.shuffle(L)
    pick = rng.integers(0, len(used), int(L.sum()))
    offsets = np.concatenate([[0], np.cumsum(L)]).astype(np.int64)
    ids = used[pick].astype(np.int64)
    past = pick == len(used) - 1
    ids[past] += rng.integers(0, 3, int(past.sum()))  # the last row's ids, also past the table (clamped to it)
    for pooling in ("sum", "mean"):
        got = _pool(pkg, dev, ids, offsets, [arg], pooling, "f32")
        want = orc.pool_c(pick.astype(np.int64), offsets, [host], tdt, pooling, "f32")
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), pooling
