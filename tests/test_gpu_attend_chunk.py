"""A prompt chunk's attention (attend_flash.hip) at the sizes where it can go
wrong: a chunk that starts at 0 and one that starts inside a 64-key slice, one
slice (no split of the keys) and several, fewer tokens than a block's rows
and more, every group size, both head widths, both cache forms, contiguous and
paged, positions that are not held, a negative attention scale.

The layer over the chunk is checked at its first tokens, its last and some
between, against the oracle run on that token alone over the rows the device
stored for the chunk's earlier tokens (the gate of tests/test_gpu_layer.py).
"""

import numpy as np
import pytest
import torch

import oracle
from molla_amd import synth
from tests.test_gpu_layer import assert_layer_close, device_layer_from, layer_gate, make_layer_weights, spec_of

pytestmark = pytest.mark.gpu

CASES = [
    # (width, hidden, heads, kv_heads, head_dim), first position, tokens
    ((256, 256, 4, 4, 64), 0, 9),       # one slice: the finished row, no second launch
    ((256, 256, 4, 4, 64), 55, 130),    # group 1: two blocks of rows, a slice's edge inside the chunk
    ((256, 256, 2, 1, 128), 64, 64),    # group 2, whole slices
    ((512, 256, 8, 2, 64), 190, 33),    # group 4, a block's rows one token past full
    ((512, 256, 8, 1, 64), 1, 63),      # group 8
    ((1024, 256, 8, 1, 128), 300, 17),  # group 8, one token past a block
]


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("dims,first,tokens", CASES)
@pytest.mark.parametrize("paged", [False, True])
def test_chunk_attention_edges(form, dims, first, tokens, paged):
    against_oracle(form, dims, first, tokens, paged)


# (the same), several slices a block
LONG_CASES = [
    ((512, 256, 8, 2, 64), 2500, 130),    # 16 shares of 3 slices, the last ones short
    ((512, 256, 4, 4, 128), 2500, 40),
    ((512, 256, 8, 1, 128), 3000, 17),
    ((256, 256, 4, 4, 64), 40, 1000),     # waves of a block end in different slices
    ((256, 256, 128, 16, 64), 100, 512),  # one share of up to 10 slices: the finished row
    ((256, 256, 128, 16, 128), 250, 500),
]


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("dims,first,tokens", LONG_CASES)
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("growing", [False, True])
def test_chunk_attention_over_several_slices(form, dims, first, tokens, paged, growing):
    """A block that walks several slices: the buffers' hand-over, the running
    maximum, and, where the values of every slice are 2^0, 2^7 or 2^-7 of the
    others' size, the change of the factors' exponent X in a block."""
    against_oracle(form, dims, first, tokens, paged, growing)


def against_oracle(form, dims, first, tokens, paged, growing=False):
    from molla_amd import block, gpu
    from tests.test_gpu_kernels import q8_decode, q8_rows
    ctx = gpu.DeviceContext(0)
    q8 = form == "q8"
    f = gpu.CACHE_Q8 if q8 else gpu.CACHE_F16
    spec = spec_of(*dims)
    if first == 190:
        spec["attn_scale"] = -spec["attn_scale"]
    host = make_layer_weights(spec, 23)
    host["attn_norm"] = (host["attn_norm"] * 0.05).astype(np.float32)  # scores of a model's size
    # no MLP: behind random weights it magnifies a last bit of the attention
    # (the oracle's own rounding of the token's key is 30 times the gate there)
    kind, r, c, blob = host["down"]
    host["down"] = (kind, r, c, np.zeros_like(blob))
    bs, layer = device_layer_from(host, spec)
    layer.desc.attn_scale = spec["attn_scale"]
    kvw, count = bs.kv_width(), first + tokens
    row = gpu.cache_row(f, kvw)
    raw = [synth.normal(count * kvw, 90 + i).numpy().reshape(count, kvw) for i in (0, 1)]
    if growing:
        raw[1] *= (2.0 ** (7 * ((np.arange(count) // 64 * 5 + np.arange(count) // 192) % 3 - 1))).astype(np.float32)[:, None]
    rows = [q8_rows(r, kvw).reshape(count, row) if q8 else r.astype(np.float16).view(np.uint16) for r in raw]
    x = synth.normal(tokens * bs.width, 92).numpy()
    xd = torch.from_numpy(x.copy()).cuda()
    posd = torch.arange(first, count, dtype=torch.int32, device="cuda")

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).view(torch.float16).cuda()

    held = np.ones(count, bool)
    if paged:
        held[1:first:7] = False  # positions trimmed out of the window
        order = np.random.default_rng(3).permutation(count + 5)[:count].astype(np.int32)
        pools = [np.zeros((count + 5, row), np.uint16) for _ in rows]
        for p, r in zip(pools, rows):
            p[order] = r
        kd, vd = (dev(p.reshape(-1)) for p in pools)
        idx = torch.from_numpy(np.where(held, order, -1).astype(np.int32)).cuda()
        block.device_layer_paged(ctx, layer, xd, kd, vd, idx, 0, posd, count, tokens, form=f)
    else:
        order = np.arange(count)
        kd, vd = (dev(r.reshape(-1)) for r in rows)
        block.device_layer(ctx, layer, xd, kd, vd, 0, posd, count, tokens, form=f)
    ctx.synchronize()
    got = [c.cpu().view(torch.int16).numpy().view(np.uint16).reshape(-1, row)[order] for c in (kd, vd)]
    got = [q8_decode(g.reshape(-1), kvw, count) if q8 else g.view(np.float16).astype(np.float32) for g in got]
    keep = []
    L = oracle.make_layer(spec, host, keep)
    for i in sorted({0, 1, 8, tokens // 2, tokens - 2, tokens - 1}):
        p = first + i
        kept = [j for j in range(p) if held[j]]
        slot = len(kept)
        kr, vr = (np.concatenate([g[kept], np.zeros((1, kvw), np.float32)]).astype(np.float32).reshape(-1) for g in got)
        xr = x.reshape(tokens, -1)[i].copy()
        # the oracle's own position is the slot count: give the float64 layer
        # the kept rows, the rope the true position
        bound = layer_gate(spec, host, xr, kr, vr, slot)
        oracle.layer_step(L, xr, kr, vr, slot, p, f16_store=not q8, q8_store=q8, threads=8)
        assert_layer_close(xd.cpu().numpy().reshape(tokens, -1)[i], xr, bound, f"token {i}:")


@pytest.mark.parametrize("form", ["f16", "q8"])
@pytest.mark.parametrize("dims", [(512, 256, 8, 2, 64), (1024, 256, 8, 1, 128)])
@pytest.mark.parametrize("power", [-40, -12, 20, 60])
def test_chunk_query_of_any_size(form, dims, power):
    """Queries times 2^power (the gain of the per-head query norm) and the
    attention scale times 2^-power are the same scores: the layer is the same
    to the bit (a half alone would overflow from 2^16 on, and lose its low bits
    below 1/2)."""
    from molla_amd import block, gpu
    ctx = gpu.DeviceContext(0)
    f = gpu.CACHE_Q8 if form == "q8" else gpu.CACHE_F16
    spec = spec_of(*dims)
    first, tokens = 70, 40
    bs, layer = device_layer_from(make_layer_weights(spec, 27), spec)
    kvw, hd, count = bs.kv_width(), dims[4], first + tokens
    k, v = (synth.normal(count * kvw, 94 + i) for i in (0, 1))
    if form == "q8":
        from tests.test_gpu_kernels import q8_rows
        k, v = (torch.from_numpy(q8_rows(c.numpy(), kvw).view(np.int16).copy()).view(torch.float16) for c in (k, v))
    x = synth.normal(tokens * bs.width, 96).cuda()
    posd = torch.arange(first, count, dtype=torch.int32, device="cuda")
    ones = torch.ones(hd, device="cuda")
    outs = []
    for p in (0, power):
        l = block.DeviceLayer(bs, layer.attn_norm, layer.ffn_norm, layer.weights, layer.rope_steps,
                              extras={"q_norm": ones * 2.0 ** p, "k_norm": ones})
        l.desc.attn_scale = 2.0 ** (-3 - p)
        xd, kd, vd = x.clone(), k.half().cuda(), v.half().cuda()
        block.device_layer(ctx, l, xd, kd, vd, 0, posd, count, tokens, form=f)
        outs.append(xd.cpu())
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dims", [(512, 256, 8, 2, 64), (1024, 256, 8, 1, 128), (256, 256, 4, 4, 64)])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("infinite", [False, True])
def test_q8_value_factors_of_any_range(dims, paged, infinite):
    """Value factors 2^28 apart, or infinite, at positions that only the chunk's
    last token reaches (and in cell 0 of the pool, where positions that are not
    held look): the earlier tokens keep every bit, and the last one, which sums
    both sizes, is right too.  The gate is the layer's own."""
    from molla_amd import block, gpu
    from tests.test_gpu_kernels import q8_decode, q8_rows
    ctx = gpu.DeviceContext(0)
    spec = spec_of(*dims)
    host = make_layer_weights(spec, 29)
    host["attn_norm"] = (host["attn_norm"] * 0.05).astype(np.float32)
    kind, r, c, blob = host["down"]
    host["down"] = (kind, r, c, np.zeros_like(blob))
    bs, layer = device_layer_from(host, spec)
    kvw, count = bs.kv_width(), 200
    row = gpu.cache_row(gpu.CACHE_Q8, kvw)
    pos = np.array(list(range(60, 71)) + [count - 1])  # 11 tokens, and one past rows that lie there
    k, v = (synth.normal(count * kvw, 98 + i).numpy().reshape(count, kvw) for i in (0, 1))
    v *= np.float32(2.0 ** -8)
    big = np.arange(count) % 7 == 3
    big[:71] = False
    v[big] *= np.float32(2.0 ** 28)
    rows = [q8_rows(a, kvw).reshape(count, row) for a in (k, v)]
    if infinite:
        rows[1][big, kvw // 2:] = 0x7c00
    held = np.ones(count, bool)
    held[5:60:6] = False
    if not paged:
        held[:] = True
    order = 1 + np.random.default_rng(4).permutation(count + 3)[:count].astype(np.int32)
    x = synth.normal(pos.size * bs.width, 101).numpy()
    xd = torch.from_numpy(x.copy()).cuda()
    posd = torch.from_numpy(pos.astype(np.int32)).cuda()

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).view(torch.float16).cuda()

    if paged:
        pools = [np.zeros((count + 4, row), np.uint16) for _ in rows]
        for p, a in zip(pools, rows):
            p[order] = a
            p[0, :kvw // 2] = 0x0101
            p[0, kvw // 2:] = 0x7c00
        kd, vd = (dev(p.reshape(-1)) for p in pools)
        idx = torch.from_numpy(np.where(held, order, -1).astype(np.int32)).cuda()
        block.device_layer_paged(ctx, layer, xd, kd, vd, idx, 0, posd, count, pos.size, form=gpu.CACHE_Q8)
    else:
        order = np.arange(count)
        kd, vd = (dev(a.reshape(-1)) for a in rows)
        block.device_layer(ctx, layer, xd, kd, vd, 0, posd, count, pos.size, form=gpu.CACHE_Q8)
    ctx.synchronize()
    got = [c.cpu().view(torch.int16).numpy().view(np.uint16).reshape(-1, row)[order] for c in (kd, vd)]
    with np.errstate(invalid="ignore"):  # 0 x infinity, in rows that are not looked at
        got = [q8_decode(g.reshape(-1), kvw, count) for g in got]
    keep = []
    L = oracle.make_layer(spec, host, keep)
    for i in (0, 1, 10) + (() if infinite else (11,)):
        kept = [j for j in range(pos[i]) if held[j]]
        slot = len(kept)
        kr, vr = (np.concatenate([g[kept], np.zeros((1, kvw), np.float32)]).astype(np.float32).reshape(-1) for g in got)
        xr = x.reshape(pos.size, -1)[i].copy()
        bound = layer_gate(spec, host, xr, kr, vr, slot)
        oracle.layer_step(L, xr, kr, vr, slot, int(pos[i]), f16_store=False, q8_store=True, threads=8)
        assert_layer_close(xd.cpu().numpy().reshape(pos.size, -1)[i], xr, bound, f"token {i}:")
