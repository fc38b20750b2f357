"""Pooling with the input LayerNorm fused into the writer, on the GPU.

Bar: the fused kernel's output equals LayerNorm(pooled row) where the pooled row is the oracle's
(bit-exact for bags pooled by one lane group, rounded to the table dtype) and the LayerNorm is
the oracle's fp32 restatement (online_best/infer.py:829-858): within 2e-5 absolute before the
final rounding (fp32 output) or half an output ulp plus 2e-5 (bf16 output). It also agrees with
running the pooling kernel and the LayerNorm kernel one after the other, and is deterministic.
"""
import numpy as np
import pytest
import torch

from oracle import ebag_oracle as orc

pytestmark = pytest.mark.gpu

TORCH_DT = {"f32": torch.float32, "bf16": torch.bfloat16}


def ref_layout(rng, S, B, V, max_len, long_every=0, long_len=0):
    L = rng.integers(0, max_len + 1, (S, B))
    L[:, rng.random(B) < 0.1] = 0
    if long_every:
        L[:, ::long_every] = long_len
    ro = np.zeros((S, B + 1), np.int64)
    np.cumsum(L, axis=1, out=ro[:, 1:])
    vo = np.concatenate([[0], np.cumsum(L.sum(axis=1))[:-1]]).astype(np.int64)
    v = rng.integers(-3, V + 3, int(L.sum())).astype(np.int64)
    return v, ro.reshape(-1), vo


def run_fused(pkg, dev, v, ro, vo, w, g, bb, B, pooling="sum", eps=1e-5):
    S = vo.size
    D = w.shape[1]
    out = torch.empty((B, S * D), dtype=w.dtype, device=dev)
    pkg.fused_all_slots_embedding_layernorm(torch.from_numpy(v).to(dev), torch.from_numpy(vo).to(dev),
                                            torch.from_numpy(ro).to(dev), w, out, B, D, w.shape[0] - 1, g, bb, eps,
                                            pooling=pooling)
    torch.cuda.synchronize()
    return out


def expected(v, ro, vo, w, g, bb, B, pooling, dt, eps=1e-5):
    """Oracle pooling (rounded to the table dtype) then the oracle LayerNorm, fp32."""
    S = vo.size
    wn = w.cpu()
    tab = wn.numpy() if dt == "f32" else wn.view(torch.int16).numpy().view(np.uint16)
    pooled = orc.pool_c(v, ro, [tab] * S, dt, pooling, dt, batch=B, val_base=vo)
    x = orc.decode(pooled, dt)
    y, _, _ = orc.layer_norm_np(x, g.float().cpu().numpy(), bb.float().cpu().numpy(), eps)
    return y


def check(out, y, dt):
    got = out.float().cpu().numpy()
    if dt == "f32":
        tol = 2e-5 + 1e-5 * np.abs(y)
    else:
        tol = 2e-5 + np.abs(y) * 2.0 ** -8
    assert (np.abs(got - y) <= tol).all(), np.abs(got - y).max()


@pytest.mark.parametrize("dt", ["bf16", "f32"])
@pytest.mark.parametrize("pdt", ["f32", "bf16"])
@pytest.mark.parametrize("D", [32, 64, 128, 256, 512])
@pytest.mark.parametrize("pooling", ["sum", "mean"])
def test_fused_matches_oracle(pkg, dev, dt, pdt, D, pooling):
    print(f"fused dt={dt} pdt={pdt} D={D} pooling={pooling}", flush=True)
    rng = np.random.default_rng(D + len(dt) * 7 + len(pdt) + len(pooling))
    S, B, V = 28 if D <= 128 else 12, 37, 700
    v, ro, vo = ref_layout(rng, S, B, V, 20)
    w = torch.from_numpy(rng.standard_normal((V, D)).astype(np.float32)).to(TORCH_DT[dt]).to(dev)
    g = torch.from_numpy((1 + 0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(TORCH_DT[pdt]).to(dev)
    bb = torch.from_numpy((0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(TORCH_DT[pdt]).to(dev)
    if dt == "f32" and D == 512 and pooling == "mean":
        # 2 KiB rows are outside the fused kernel and the unfused fallback pools by sum only
        with pytest.raises(pkg.EbagError, match="fused LayerNorm"):
            run_fused(pkg, dev, v, ro, vo, w, g, bb, B, pooling)
        return
    out = run_fused(pkg, dev, v, ro, vo, w, g, bb, B, pooling)
    check(out, expected(v, ro, vo, w, g, bb, B, pooling, dt), dt)


@pytest.mark.parametrize("S", [1, 5, 64])
@pytest.mark.parametrize("B", [1, 2, 3])
def test_fused_slot_counts_and_small_batches(pkg, dev, S, B):
    """Workgroups pool two samples when the slots allow it; odd batches leave the last one half
    full, and 64 slots (16 bags per wavefront per sample) is the largest fused shape."""
    print(f"fused S={S} B={B}", flush=True)
    rng = np.random.default_rng(S * 10 + B)
    V, D = 400, 32
    v, ro, vo = ref_layout(rng, S, B, V, 24, long_every=2, long_len=70)
    # integer rows: the split sums of the 70-id bags are exact, so the pooled rows equal the oracle's
    w = torch.from_numpy(rng.integers(-8, 9, (V, D)).astype(np.float32)).to(torch.bfloat16).to(dev)
    g = torch.from_numpy((1 + 0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(dev)
    bb = torch.from_numpy((0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(dev)
    for pooling in ("sum", "mean"):
        out = run_fused(pkg, dev, v, ro, vo, w, g, bb, B, pooling)
        check(out, expected(v, ro, vo, w, g, bb, B, pooling, "bf16"), "bf16")


def test_fused_long_bags_and_int32_inputs(pkg, dev):
    """Bags longer than the short-bag limit are pooled by the whole wavefront (split sums: the
    pooled row is within the reassociation bound, the LayerNorm tolerance covers it)."""
    rng = np.random.default_rng(5)
    S, B, V, D = 28, 20, 900, 128
    v, ro, vo = ref_layout(rng, S, B, V, 30, long_every=3, long_len=300)
    w = torch.from_numpy((rng.integers(-8, 9, (V, D))).astype(np.float32)).to(torch.bfloat16).to(dev)  # exact sums
    g = torch.ones(S * D, dtype=torch.float32, device=dev)
    bb = torch.zeros(S * D, dtype=torch.float32, device=dev)
    a = run_fused(pkg, dev, v, ro, vo, w, g, bb, B)
    check(a, expected(v, ro, vo, w, g, bb, B, "sum", "bf16"), "bf16")
    b = run_fused(pkg, dev, v.astype(np.int32), ro.astype(np.int32), vo.astype(np.int32), w, g, bb, B)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_fused_agrees_with_separate_kernels_and_is_deterministic(pkg, dev):
    rng = np.random.default_rng(9)
    S, B, V, D = 28, 300, 5000, 128
    v, ro, vo = ref_layout(rng, S, B, V, 16)
    w = torch.from_numpy((0.01 * rng.standard_normal((V, D))).astype(np.float32)).to(torch.bfloat16).to(dev)
    g = torch.from_numpy((1 + 0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(torch.bfloat16).to(dev)
    bb = torch.from_numpy((0.1 * rng.standard_normal(S * D)).astype(np.float32)).to(torch.bfloat16).to(dev)
    fused = run_fused(pkg, dev, v, ro, vo, w, g, bb, B)
    again = run_fused(pkg, dev, v, ro, vo, w, g, bb, B)
    assert torch.equal(fused.view(torch.int16), again.view(torch.int16))
    pooled = torch.empty((B, S * D), dtype=torch.bfloat16, device=dev)
    pkg.fused_all_slots_embedding(torch.from_numpy(v).to(dev), torch.from_numpy(vo).to(dev),
                                  torch.from_numpy(ro).to(dev), w, pooled, B, D, V - 1)
    sep = pkg.layer_norm(pooled, g, bb, 1e-5)
    torch.cuda.synchronize()
    # the pooled rows are the same bits; the two LayerNorms reduce in different orders, so their
    # fp32 results differ in the last bits and a bf16 rounding may land one ulp apart
    # (one ulp <= 2^-7 of the value)
    diff = (fused.float() - sep.float()).abs()
    big = torch.maximum(fused.float().abs(), sep.float().abs())
    assert (diff <= big * 2.0 ** -7 + 1e-5).all(), (diff - big * 2.0 ** -7).max().item()
    assert (diff == 0).float().mean().item() > 0.95


def test_unfused_shapes_fall_back(pkg, dev):
    """16-byte rows (bf16 D=8) are outside the fused kernel: the wrapper runs the pooling and
    LayerNorm kernels instead and the result is the same within the LayerNorm tolerance."""
    rng = np.random.default_rng(3)
    S, B, V, D = 28, 25, 300, 8
    v, ro, vo = ref_layout(rng, S, B, V, 10)
    w = torch.from_numpy(rng.standard_normal((V, D)).astype(np.float32)).to(torch.bfloat16).to(dev)
    g = torch.ones(S * D, device=dev)
    bb = torch.zeros(S * D, device=dev)
    out = run_fused(pkg, dev, v, ro, vo, w, g, bb, B)
    check(out, expected(v, ro, vo, w, g, bb, B, "sum", "bf16"), "bf16")
    with pytest.raises(pkg.EbagError, match="fused LayerNorm"):
        run_fused(pkg, dev, v, ro, vo, w, g, bb, B, pooling="mean")


def test_encoder_normalized_uses_fused_path(pkg, dev):
    torch.manual_seed(0)
    S, D = 28, 128
    enc = pkg.RepEncoder(vocab_size=4000, emb_dim=D, padding_idx=0, slot_num=S, d_model=32).to(dev).to(torch.bfloat16)
    with torch.no_grad():
        enc.input_norm.weight.copy_(1 + 0.1 * torch.randn(S * D))
        enc.input_norm.bias.copy_(0.1 * torch.randn(S * D))
    rng = np.random.default_rng(1)
    B = 64
    v, ro, vo = ref_layout(rng, S, B, 4000, 12)
    batch = {"_flat_values": torch.from_numpy(v).to(dev), "_flat_row_offsets": torch.from_numpy(ro).to(dev),
             "_val_offsets": torch.from_numpy(vo).to(dev)}
    y = enc.normalized(batch)
    torch.cuda.synchronize()
    check(y, expected(v, ro, vo, enc.emb.weight.detach(), enc.input_norm.weight.detach(),
                      enc.input_norm.bias.detach(), B, "sum", "bf16"), "bf16")


# rows of 64 lane vectors are streamed: tiles of 4 bags (2 of few long ones or with a dispatch order), tables read through
# buffers below 4 GiB and with power-of-two rows, else at 64-bit addresses
@pytest.mark.parametrize("tdt", ["bf16", "f32", "f16", "i8"])
@pytest.mark.parametrize("B", [1, 4, 5, 67])
@pytest.mark.parametrize("padded", [False, True])
def test_wide_rows_match_oracle(pkg, dev, tdt, B, padded):
    print(f"wide rows {tdt} B={B} padded={padded}", flush=True)
    D = 256 if tdt == "f32" else 512
    rng = np.random.default_rng(B)
    F, V = 3, 200
    L = rng.integers(0, 12, (F, B))
    L[:, ::4] = rng.choice([0, 63, 64, 65, 130], L[:, ::4].shape)
    off = np.concatenate([[0], np.cumsum(L.reshape(-1))]).astype(np.int64)
    ids = rng.integers(-3, V + 3, int(off[-1])).astype(np.int64)
    host, tables = [], []
    for f in range(F):
        if tdt == "i8":
            q = rng.integers(-128, 128, (V, D)).astype(np.int8)
            scale = (rng.random(V) * 0.02 + 1e-4).astype(np.float32)
            host.append((q, scale))
            t = torch.from_numpy(q).to(dev)
        else:
            host.append(orc.encode(rng.standard_normal((V, D)).astype(np.float32), tdt))
            t = torch.from_numpy(host[-1].view(np.int16) if tdt != "f32" else host[-1]).to(dev)
            t = t if tdt == "f32" else t.view(torch.bfloat16 if tdt == "bf16" else torch.float16)
        if padded:  # rows 16 bytes apart more than their width
            wide = torch.zeros(V, D + 16 // t.element_size(), dtype=t.dtype, device=dev)
            wide[:, :D] = t
            t = wide[:, :D]
        tables.append((t, torch.from_numpy(scale).to(dev)) if tdt == "i8" else t)
    for idt in (torch.int64, torch.int32):
        for pooling in ("sum", "mean"):
            got = pkg.embedding_bag_pooled(torch.from_numpy(ids).to(dev).to(idt), torch.from_numpy(off).to(dev), tables,
                                           pooling=pooling, out_dtype=torch.float32).cpu().numpy()
            want = orc.pool_c(ids, off, host, tdt, pooling, "f32")
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (idt, pooling)


@pytest.mark.parametrize("int8", [False, True])
def test_wide_table_beyond_4_gib(pkg, dev, int8):
    """A table of 4.4 GB (rows at 64-bit addresses) gives what a small table of the same rows gives
    (rows through buffers), pooled and pooled with the LayerNorm, bit for bit."""
    S, B, D = 28, 37, 512
    V = 8_600_000 if int8 else 4_300_000
    g = torch.Generator(device="cpu").manual_seed(5)
    lens = torch.randint(0, 15, (S, B), generator=g)
    rows = torch.zeros(S, B + 1, dtype=torch.int64)
    rows[:, 1:] = torch.cumsum(lens, 1)
    starts = torch.cumsum(rows[:, -1], 0) - rows[:, -1]
    n = int(lens.sum())
    ids = torch.randint(0, V, (n,), generator=g)
    ids[::7] = V - 1 - ids[::7] % 100
    uniq, small_ids = torch.unique(ids, return_inverse=True)
    out = {}
    with torch.device("meta"):
        encs = {"big": pkg.RepEncoder(V, D, slot_num=S, d_model=8), "small": pkg.RepEncoder(len(uniq), D, slot_num=S, d_model=8)}
    gamma = (1 + 0.1 * torch.randn(S * D, generator=g)).to(dev).to(torch.bfloat16)
    beta = (0.1 * torch.randn(S * D, generator=g)).to(dev).to(torch.bfloat16)
    if int8:
        big = torch.randint(-128, 128, (V, D), dtype=torch.int8, device=dev)
        scale = torch.rand(V, device=dev) * 0.01 + 1e-4
    else:
        big = torch.empty(V, D, dtype=torch.bfloat16, device=dev).normal_()
    for name, enc in encs.items():
        sel = slice(None) if name == "big" else uniq.to(dev)
        enc.input_norm.weight = torch.nn.Parameter(gamma, requires_grad=False)
        enc.input_norm.bias = torch.nn.Parameter(beta, requires_grad=False)
        if int8:
            weight = torch.empty(1, D, dtype=torch.bfloat16, device=dev).expand(enc.emb.num_embeddings, D)
            enc._int8_weight, enc._int8_scale = big[sel].contiguous(), scale[sel].contiguous()
        else:
            weight = big[sel]
        enc.emb.weight = torch.nn.Parameter(weight, requires_grad=False)
        batch = {"_flat_values": (ids if name == "big" else small_ids).to(dev),
                 "_flat_row_offsets": rows.reshape(-1).to(dev), "_val_offsets": starts.to(dev)}
        out[name] = (enc.pooled(batch), enc.normalized(batch))
    for a, b in zip(out["big"], out["small"]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("B", [1, 9, 131])
@pytest.mark.parametrize("S", [1, 5, 28, 64])
@pytest.mark.parametrize("pdt", [torch.bfloat16, torch.float32])
def test_fused_int8_layernorm_equals_two_launches(pkg, dev, B, S, pdt):
    """Rows pooled and normalised in one launch: the pooled rows are the int8 pooling's (rounded to
    bf16), so the result is the LayerNorm kernel's up to its fp32 rounding and one bf16 ulp."""
    print(f"int8 fused norm B={B} S={S} params={pdt}", flush=True)
    D, V = 512, 300
    g = torch.Generator(device="cpu").manual_seed(B * 100 + S)
    lens = torch.randint(0, 9, (S, B), generator=g)
    lens[::3, ::5] = 70
    rows = torch.zeros(S, B + 1, dtype=torch.int64)
    rows[:, 1:] = torch.cumsum(lens, 1)
    starts = (torch.cumsum(rows[:, -1], 0) - rows[:, -1]).to(dev)
    ids = torch.randint(-2, V + 2, (int(lens.sum()),), generator=g).to(dev)
    rows = rows.reshape(-1).to(dev)
    q = torch.randint(-128, 128, (V, D), generator=g, dtype=torch.int8).to(dev)
    scale = (torch.rand(V, generator=g) * 0.01 + 1e-4).to(dev)
    gamma = (1 + 0.1 * torch.randn(S * D, generator=g)).to(dev).to(pdt)
    beta = (0.1 * torch.randn(S * D, generator=g)).to(dev).to(pdt)
    want = torch.empty(B, S * D, dtype=torch.bfloat16, device=dev)
    pkg.fused_all_slots_embedding_int8(ids, starts, rows, q, scale, want, B, D, V - 1)
    want = pkg.layer_norm(want, gamma, beta, 1e-5).double()
    for idt in (torch.int64, torch.int32):
        got = torch.full((B, S * D), float("nan"), dtype=torch.bfloat16, device=dev)
        pkg.fused_all_slots_embedding_int8_layernorm(ids.to(idt), starts.to(idt), rows.to(idt), q, scale, got, B, D, V - 1,
                                                     gamma, beta, 1e-5)
        # the same pooled rows and formula, the sums in another order of fp32 additions (2e-5): values that
        # close round to the same bf16 or to neighbours, which are at most 2^-7 of the larger apart
        assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -7 * (1 + 2.0 ** -7) + 2e-5).all()
        assert (got.double() != want).double().mean() < 0.01
