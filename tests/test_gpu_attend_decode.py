"""Decode attention (attend_decode.hip) at the sizes where it can go wrong:
counts around a wave's 32-key run, a block's 128-key step and past 64 steps (a
share of two), every group size and both head widths over both cache forms, a
context far longer than the position (shares without keys), and a workspace
that held NaN before (those shares' values are never written).  Gate: 1e-5 of
the peak against the oracle, as tests/test_gpu_kernels.py test_attention.
"""

import numpy as np
import pytest
import torch

import oracle
from molla_amd import synth

pytestmark = pytest.mark.gpu


def caches(form, count, kvw, seed):
    from tests.test_gpu_kernels import q8_decode, q8_rows
    dev, host = [], []
    for i in (0, 1):
        raw = synth.normal(count * kvw, seed + i).numpy()
        h = q8_rows(raw, kvw) if form == "q8" else raw.astype(np.float16).view(np.uint16)
        dev.append(torch.from_numpy(h.view(np.int16).copy()).view(torch.float16).cuda())
        host.append(q8_decode(h, kvw, count).reshape(-1) if form == "q8" else h.view(np.float16).astype(np.float32))
    return dev, host


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("heads,kv,hd", [(2, 2, 128), (4, 2, 64), (8, 2, 128), (8, 1, 64), (16, 2, 128)])
@pytest.mark.parametrize("count", [1, 31, 32, 33, 128, 129, 8193])
def test_decode_attention_edges(form, heads, kv, hd, count):
    from molla_amd import gpu
    ctx = gpu.DeviceContext(0)
    (kd, vd), (kh, vh) = caches(form, count, kv * hd, 40)
    q = synth.normal(heads * hd, 42).numpy()
    scale = float(np.float32(1 / np.sqrt(hd)))
    out = torch.zeros(heads * hd, device="cuda")
    f = gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16
    gpu.device_attend(ctx, torch.from_numpy(q).cuda(), kd, vd, heads, kv, hd, scale, count, out, f)
    want = oracle.attend(heads, kv, hd, scale, q, kh, vh, count)
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("heads,kv,hd", [(2, 2, 128), (16, 2, 64)])
def test_several_steps_a_share(form, heads, kv, hd):
    """20000 keys are 157 steps of a block's 128: three a share, the last of
    them short."""
    test_decode_attention_edges(form, heads, kv, hd, 20000)


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("heads,kv,hd", [(16, 8, 64), (8, 8, 128)])
@pytest.mark.parametrize("tokens", [3, 8])
def test_paged_steps(form, heads, kv, hd, tokens):
    """Sequences of unequal length, many steps a share: rows in the cells of a
    pool, in no order, give the contiguous caches' result to the bit; with some
    positions not held, the oracle's over the rows that are (the gate of
    tests/test_gpu_layer.py)."""
    from molla_amd import block, gpu
    from tests.test_gpu_kernels import q8_decode
    from tests.test_gpu_layer import assert_layer_close, device_layer_from, layer_gate, make_layer_weights, spec_of
    ctx = gpu.DeviceContext(0)
    f = gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16
    spec = spec_of(256, 256, heads, kv, hd)
    host = make_layer_weights(spec, 35)
    host["attn_norm"] = (host["attn_norm"] * 0.05).astype(np.float32)  # scores of a model's size
    kind, r, c, blob = host["down"]
    host["down"] = (kind, r, c, np.zeros_like(blob))  # (no MLP, which magnifies a last bit)
    bs, layer = device_layer_from(host, spec)
    kvw, length = bs.kv_width(), 2600
    row = gpu.cache_row(f, kvw)
    (k, v), _ = caches(form, tokens * length, kvw, 64)
    pos = [length - 1 - 290 * t for t in range(tokens)]
    posd = torch.tensor(pos, dtype=torch.int32, device="cuda")
    x = synth.normal(tokens * bs.width, 66).cuda()

    def contiguous(ks, vs, at):
        xd, kd, vd = x.clone(), ks.clone(), vs.clone()
        block.device_layer(ctx, layer, xd, kd, vd, length * row, at, length, tokens, form=f)
        return xd.cpu()

    def paged(held):
        order = torch.randperm(tokens * length, generator=torch.Generator().manual_seed(6))
        pools = []
        for c in (k, v):
            pool = torch.zeros(tokens * length, row, dtype=torch.float16, device="cuda")
            pool[order.cuda()] = c.reshape(-1, row)
            pools.append(pool.reshape(-1))
        index = torch.where(held, order.reshape(tokens, length), -1).to(torch.int32).cuda()
        xd = x.clone()
        block.device_layer_paged(ctx, layer, xd, *pools, index, length, posd, length, tokens, form=f)
        return xd.cpu()

    held = torch.ones(tokens, length, dtype=torch.bool)
    assert torch.equal(paged(held), contiguous(k, v, posd))

    held[:, 5::9] = False
    for t in range(tokens):
        held[t, pos[t]] = True
    got = paged(held)
    keep = []
    L = oracle.make_layer(spec, host, keep)

    def floats(c):
        a = c.cpu().view(torch.int16).numpy().view(np.uint16)
        n = a.size // row
        if form == "q8":
            return q8_decode(a, kvw, n).reshape(n, kvw)
        return a.view(np.float16).astype(np.float32).reshape(n, kvw)

    for t in (0, tokens - 1):
        rows = [j for j in range(pos[t]) if held[t, j]]
        kr, vr = (np.concatenate([floats(c.reshape(tokens, length, row)[t])[rows], np.zeros((1, kvw), np.float32)])
                  .astype(np.float32).reshape(-1) for c in (k, v))
        xr = x.cpu().numpy().reshape(tokens, -1)[t].copy()
        bound = layer_gate(spec, host, xr, kr, vr, len(rows))
        oracle.layer_step(L, xr, kr, vr, len(rows), pos[t], f16_store=form != "q8", q8_store=form == "q8", threads=8)
        assert_layer_close(got.numpy().reshape(tokens, -1)[t], xr, bound, f"sequence {t}:")


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("hd", [64, 128])
def test_weights_to_the_last_bits(form, hd):
    """Two keys with scores 0 and -a and values 0 and 1: the result is the second
    one's weight, e^-a / (1 + e^-a).  At a up to 1.4 the score's factor and its
    product with a (2^-24 of at most 2 in base 2), the exponential (an ulp), the
    sum and the quotient (2^-24) round it: together within 1.1e-7 in the root
    mean square (6e-8 to 7e-8 is seen).  With P's lift by 2^14 in the exponential's
    argument, which that rounds to 2^-21, it is 1.4e-7 to 1.5e-7."""
    from molla_amd import gpu
    from tests.test_gpu_kernels import q8_rows
    ctx = gpu.DeviceContext(0)
    heads, kv = 64, 8
    kvw = kv * hd
    k, v = np.zeros((2, kvw), np.float32), np.zeros((2, kvw), np.float32)
    k[1, ::hd] = -1.0
    v[1] = 1.0
    # (a q8_0 factor that is a power of two: 1 / 127 would not be exact)
    unit = np.float32(127 / 128 if form == "q8" else 1.0)
    rows = [q8_rows(c * unit, kvw) if form == "q8" else c.astype(np.float16).view(np.uint16).reshape(-1) for c in (k, v)]
    kd, vd = (torch.from_numpy(r.view(np.int16).copy()).view(torch.float16).cuda() for r in rows)
    errs = []
    for seed in range(8):
        a = np.random.default_rng(seed).uniform(0.05, 1.4, heads).astype(np.float32)
        q = np.zeros((heads, hd), np.float32)
        q[:, 0] = a
        out = torch.zeros(heads * hd, device="cuda")
        gpu.device_attend(ctx, torch.from_numpy(q.reshape(-1)).cuda(), kd, vd, heads, kv, hd, 1.0, 2, out,
                          gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16)
        x = a.astype(np.float64) * unit
        want = np.exp(-x) / (1 + np.exp(-x)) * unit
        errs.append(out.cpu().numpy().reshape(heads, hd).astype(np.float64) / want[:, None] - 1)
    assert np.sqrt(np.mean(np.square(errs))) <= 1.1e-7


@pytest.mark.parametrize("form", ["f16", "q8"])
def test_scores_of_1e8(form):
    """Scores whose rounding is worth several powers of two of a weight: the
    largest weight stays 1.  Neighbouring scores lie 1e5 apart and more, so the
    gate above holds (one key has all the weight)."""
    from molla_amd import gpu
    ctx = gpu.DeviceContext(0)
    heads, kv, hd, count = 8, 2, 128, 300
    (kd, vd), (kh, vh) = caches(form, count, kv * hd, 60)
    q = synth.normal(heads * hd, 62).numpy()
    q *= np.float32(3e4 / np.abs(q).max())
    scale = np.float32(1e3)
    out = torch.zeros(heads * hd, device="cuda")
    f = gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16
    gpu.device_attend(ctx, torch.from_numpy(q).cuda(), kd, vd, heads, kv, hd, float(scale), count, out, f)
    want = oracle.attend(heads, kv, hd, float(scale), q, kh, vh, count)
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("tokens", [1, 3])
def test_context_longer_than_the_position(form, tokens):
    """The shares are cut by the context and filled by the position: the layer
    over a context of 5000 gives the layer over one of pos + 1 within the
    rounding of differently grouped sums (1e-6 of each element's own bound
    would be tests/layer64.py's gate a hundred times over)."""
    from molla_amd import block, gpu
    from tests.test_gpu_layer import device_layer_from, make_layer_weights, spec_of
    ctx = gpu.DeviceContext(0)
    f = gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16
    bs, layer = device_layer_from(make_layer_weights(spec_of(512, 512, 8, 2, 64), 31), spec_of(512, 512, 8, 2, 64))
    kvw, pos, ctx_len = bs.kv_width(), 140, 5000
    row = gpu.cache_row(f, kvw)
    (k, v), _ = caches(form, tokens * ctx_len, kvw, 50)
    x = synth.normal(tokens * bs.width, 52).cuda()
    posd = torch.tensor([pos - 60 * t for t in range(tokens)], dtype=torch.int32, device="cuda")
    outs = []
    for max_count in (pos + 1, ctx_len):
        work = torch.empty(block.layer_workspace(layer, max_count, tokens), dtype=torch.uint8, device="cuda")
        work.fill_(255)  # NaN as floats
        xd, kd, vd = x.clone(), k.clone(), v.clone()
        block.device_layer(ctx, layer, xd, kd, vd, ctx_len * row, posd, max_count, tokens, work=work, form=f)
        outs.append(xd.cpu().double())
    assert torch.isfinite(outs[1]).all()
    assert (outs[0] - outs[1]).norm() <= 1e-5 * outs[0].norm()


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("dims", [(256, 256, 8, 2, 64), (256, 256, 16, 2, 128), (256, 256, 4, 4, 128)])
def test_block_sizes(form, dims):
    """Eight sequences that end at the edges of a run and of a step, in a context
    that gives every 64 keys a compute unit (blocks of two waves) and in one
    that does not (four): the same within the rounding of sums in another
    order."""
    from molla_amd import block, gpu
    from tests.test_gpu_layer import device_layer_from, make_layer_weights, spec_of
    ctx = gpu.DeviceContext(0)
    f = gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16
    bs, layer = device_layer_from(make_layer_weights(spec_of(*dims), 37), spec_of(*dims))
    pos = [0, 30, 31, 32, 63, 127, 128, 299]
    kvw, length, tokens = bs.kv_width(), 300, len(pos)
    row = gpu.cache_row(f, kvw)
    (k, v), _ = caches(form, tokens * length, kvw, 68)
    x = synth.normal(tokens * bs.width, 69).cuda()
    posd = torch.tensor(pos, dtype=torch.int32, device="cuda")
    outs = []
    for context in (length, 20000):
        # (the same rows, the longer cache's padded with ones that no position reaches)
        kd, vd = (torch.cat([c.reshape(tokens, length * row), torch.zeros(tokens, (context - length) * row,
                                                                         dtype=c.dtype, device="cuda")], 1).reshape(-1)
                  for c in (k, v))
        xd = x.clone()
        block.device_layer(ctx, layer, xd, kd, vd, context * row, posd, context, tokens, form=f)
        outs.append(xd.cpu().double().reshape(tokens, -1))
    assert ((outs[0] - outs[1]).norm(dim=1) <= 1e-5 * outs[0].norm(dim=1)).all()


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("heads,kv,hd", [(8, 2, 128), (8, 1, 64)])
@pytest.mark.parametrize("power", [-90, -40, -12, 4, 20, 100])
def test_query_of_any_size(form, heads, kv, hd, power):
    """A query times 2^power and the scale times 2^-power are the same scores:
    the result is the same to the bit, whatever the query's size (a half alone
    would overflow from 2^16 on, and lose its low bits below 1/2)."""
    from molla_amd import gpu
    ctx = gpu.DeviceContext(0)
    count = 300
    (kd, vd), _ = caches(form, count, kv * hd, 70)
    q = synth.normal(heads * hd, 72).cuda()
    f = gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16
    outs = []
    for p in (0, power):
        out = torch.zeros(heads * hd, device="cuda")
        # (no query value and neither scale leaves the normal floats)
        gpu.device_attend(ctx, q * 2.0 ** p, kd, vd, heads, kv, hd, 2.0 ** (-3 - p), count, out, f)
        outs.append(out.cpu())
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("size,keys", [(1e6, 1.0), (1e-6, 1e4)])
def test_large_and_small_queries(form, size, keys):
    """The same against the oracle, with the keys as they are in a cache of
    large ones: scores of a few units."""
    from molla_amd import gpu
    from tests.test_gpu_kernels import q8_decode, q8_rows
    ctx = gpu.DeviceContext(0)
    heads, kv, hd, count = 16, 2, 128, 400
    dev, host = [], []
    for i, m in enumerate((keys, 1.0)):
        raw = synth.normal(count * kv * hd, 80 + i).numpy() * np.float32(m)
        h = q8_rows(raw, kv * hd) if form == "q8" else raw.astype(np.float16).view(np.uint16)
        dev.append(torch.from_numpy(h.view(np.int16).copy()).view(torch.float16).cuda())
        host.append(q8_decode(h, kv * hd, count).reshape(-1) if form == "q8" else h.view(np.float16).astype(np.float32))
    q = synth.normal(heads * hd, 82).numpy() * np.float32(size)
    scale = float(np.float32(1 / np.sqrt(hd) / size / keys))
    out = torch.zeros(heads * hd, device="cuda")
    gpu.device_attend(ctx, torch.from_numpy(q).cuda(), dev[0], dev[1], heads, kv, hd, scale, count, out,
                      gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16)
    want = oracle.attend(heads, kv, hd, scale, q, host[0], host[1], count)
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("heads,kv,hd", [(8, 2, 128), (8, 1, 64)])
def test_q8_value_factors_of_any_range(heads, kv, hd):
    """Values 2^28 apart in the same block of 32: keys of large ones with
    weights of e^-40 leave the others their bits."""
    from molla_amd import gpu
    from tests.test_gpu_kernels import q8_decode, q8_rows
    ctx = gpu.DeviceContext(0)
    count, kvw, scale = 700, kv * hd, np.float32(1 / np.sqrt(hd))
    q = synth.normal(heads * hd, 84).numpy()
    k = synth.normal(count * kvw, 85).numpy().reshape(count, kvw)
    v = synth.normal(count * kvw, 86).numpy().reshape(count, kvw) * np.float32(2.0 ** -8)
    big = np.arange(count) % 9 == 4
    away = q.reshape(kv, -1, hd).sum(1).reshape(-1)  # every head of a group scores about -40 along it
    k[big] = -away * np.float32(40 / (hd * scale))
    v[big] *= np.float32(2.0 ** 28)
    rows = [q8_rows(c, kvw) for c in (k, v)]
    kd, vd = (torch.from_numpy(r.view(np.int16).copy()).view(torch.float16).cuda() for r in rows)
    kh, vh = (q8_decode(r, kvw, count).reshape(-1) for r in rows)
    out = torch.zeros(heads * hd, device="cuda")
    gpu.device_attend(ctx, torch.from_numpy(q).cuda(), kd, vd, heads, kv, hd, float(scale), count, out, gpu.CACHE_Q8)
    want = oracle.attend(heads, kv, hd, float(scale), q, kh, vh, count)
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("tokens", [1, 3])
@pytest.mark.parametrize("factor", [0x7c00, 0x7bff])
def test_q8_cells_not_held_leave_no_trace(tokens, factor):
    """Positions that are not held read cell 0, which is another sequence's: an
    infinite or the largest factor there changes no bit."""
    from molla_amd import block, gpu
    from tests.test_gpu_layer import device_layer_from, make_layer_weights, spec_of
    ctx = gpu.DeviceContext(0)
    spec = spec_of(512, 512, 8, 2, 64)
    bs, layer = device_layer_from(make_layer_weights(spec, 33), spec)
    kvw, pos = bs.kv_width(), 300
    row = gpu.cache_row(gpu.CACHE_Q8, kvw)
    (k, v), _ = caches("q8", 1 + tokens * (pos + 1), kvw, 54)
    index = 1 + torch.randperm(tokens * (pos + 1), generator=torch.Generator().manual_seed(5)).reshape(tokens, pos + 1)
    index[:, 3:pos:5] = -1
    index = index.to(torch.int32).cuda()
    x = synth.normal(tokens * bs.width, 56).cuda()
    posd = torch.full((tokens,), pos, dtype=torch.int32, device="cuda")
    outs = []
    for poison in (False, True):
        xd, kd, vd = x.clone(), k.clone(), v.clone()
        if poison:
            for c in (kd, vd):
                c[kvw // 2:row] = torch.tensor([factor] * (row - kvw // 2), dtype=torch.int16).view(torch.float16).cuda()
        block.device_layer_paged(ctx, layer, xd, kd, vd, index, pos + 1, posd, pos + 1, tokens, form=gpu.CACHE_Q8)
        outs.append(xd.cpu())
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])
