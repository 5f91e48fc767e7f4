"""Each kernel alone against a plain torch statement of the same operation, at sizes other than
the engine's test models: primes, sizes that are no multiple of a tile, single rows."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def ops():
    from geneinfer_amd.kernels import ops as o
    return o


def rel(got, want):
    got, want = got.double().cpu(), want.double().cpu()
    return float((got - want).abs().max() / want.abs().max().clamp_min(1e-30))


def randn(*shape, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (scale * torch.randn(*shape, generator=g)).to(dtype).to(DEV)


# ------------------------------------------------------------------------------------------ gemm
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 7, 13), (5, 64, 64), (64, 65, 17), (130, 257, 96), (3, 1000, 515)])
@pytest.mark.parametrize("dtypes", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16)])
def test_gemm_exact(m, n, k, dtypes):
    a, w = randn(m, k, dtype=dtypes[0], seed=1), randn(n, k, dtype=dtypes[1], seed=2)
    out = torch.full((m, n + 3), -777.25, device=DEV)                 # a wider output keeps its rim
    ops().gemm_exact(a, w, out[:, :n])
    want = a.double() @ w.double().T
    assert rel(out[:, :n], want) < 2e-6
    assert torch.all(out[:, n:] == -777.25)
    before = out[:, :n].clone()
    ops().gemm_exact(a, w, out[:, :n], accumulate=True)
    assert rel(out[:, :n], 2 * want) < 2e-6 and not torch.equal(before, out[:, :n])


@pytest.mark.parametrize("w_dtype,k", [(torch.float32, 200), (torch.float32, 203), (torch.bfloat16, 264), (torch.bfloat16, 520)])
def test_gemm_exact_rows_alone_have_the_same_bits(w_dtype, k):
    """Few rows take the kernel without tiles where their rows lie aligned, more rows (and k = 203, which no 16-byte load may step through)
    one with tiles; k = 200, 264 and 520 end within a range of k, or within a block of it."""
    a, w = randn(37, k, seed=3), randn(90, -(-k // 8) * 8, dtype=w_dtype, seed=4)[:, :k]      # the row stride stays a multiple of the 16-byte piece
    full = torch.empty(37, 90, device=DEV)
    ops().gemm_exact(a, w, full)
    for first, rows in ((0, 1), (17, 1), (36, 1), (5, 2), (9, 3), (30, 4)):
        few = torch.empty(rows, 90, device=DEV)
        ops().gemm_exact(a[first:first + rows], w, few)
        assert torch.equal(few, full[first:first + rows])
        ops().gemm_exact(a[first:first + rows], w, few, accumulate=True)
        both = full[first:first + rows].clone()
        ops().gemm_exact(a[first:first + rows].repeat(17, 1)[:rows + 13], w, (wide := torch.cat([both, torch.zeros(13, 90, device=DEV)])), accumulate=True)
        assert torch.equal(few, wide[:rows])                                # adding onto what is there, the same in both kernels


@pytest.mark.parametrize("k", [4, 36, 260, 1056, 2052, 2820, 4100])            # a range of k in 32-bit: none to sixteen whole lines of 32 k, four in flight, and what is left
@pytest.mark.parametrize("m,n", [(1, 5), (8, 520), (9, 130), (3, 8200)])       # strips of 8 and of 16 weight rows, the last ones partly beyond the output
def test_gemm_exact_few_rows_line_by_line(m, n, k):
    """In the bits of the kernel with tiles, which serves more rows, stored and added, and near the 64-bit product (the bound of the tests above)."""
    a, w, x0 = randn(40, k, seed=5), randn(n, k + 4, seed=6)[:, :k], randn(m, n + 2, seed=7)
    tiles, few, x = torch.empty(40, n, device=DEV), torch.empty(m, n, device=DEV), x0.clone()
    ops().gemm_exact(a, w, tiles)
    ops().gemm_exact(a[:m], w, few)
    ops().gemm_exact(a[:m], w, x[:, :n], accumulate=True)
    assert torch.equal(few, tiles[:m]) and rel(few, a[:m].double() @ w.double().T) < 2e-6
    assert torch.equal(x[:, :n], x0[:, :n] + few) and torch.equal(x[:, n:], x0[:, n:])


@pytest.mark.parametrize("m,n,k", [(64, 256, 8192), (33, 130, 2080), (300, 160, 64), (129, 65, 4128), (16, 2048, 8192), (17, 90, 32), (70, 100, 1000), (40, 70, 203),
                                   # three, five, six and seven ranges of k that are not empty, the last ones whole or not
                                   (40, 70, 96), (300, 160, 160), (33, 90, 192), (70, 100, 224), (40, 70, 75), (70, 90, 141), (40, 70, 201)])
def test_gemm_exact_kernels_agree_in_bits(m, n, k):
    """Whole blocks of 32 k go through LDS in a ring (tiles of 32 and 64 rows, k shared out over 1 to 8 workgroups where the tiles are few),
    other aligned rows are staged through registers, unaligned ones element by element, a few rows need no tiles: one order of every sum."""
    a, w = randn(m, k, seed=31), randn(n, k, seed=32)
    full = torch.empty(m, n, device=DEV)
    ops().gemm_exact(a, w, full)
    assert rel(full, a.double() @ w.double().T) < 2e-6
    shifted = torch.zeros(n, -(-k // 4) * 4 + 4, device=DEV)[:, 1:1 + k].copy_(w)              # the same weights where no 16-byte load may touch them
    out = torch.empty_like(full)
    ops().gemm_exact(a, shifted, out)
    assert torch.equal(out, full)
    for rows in {1, min(8, m), min(16, m), min(32, m)}:
        few = torch.ones(rows, n, device=DEV)
        ops().gemm_exact(a[m - rows:], w, few, accumulate=True)
        assert torch.equal(few, 1.0 + full[m - rows:])
    wide = torch.empty(m + 200, n, device=DEV)
    ops().gemm_exact(torch.cat([a, a.new_ones(200, k)]), w, wide)
    assert torch.equal(wide[:m], full)


@pytest.mark.parametrize("m,hidden,n_heads,n_kv,hd,page_size,rotate", [(3, 2048, 32, 8, 64, 16, True), (8, 264, 6, 3, 8, 4, True), (1, 1000, 5, 1, 128, 12, True), (5, 36, 2, 2, 24, 7, False)])
def test_gemm_exact_qkv_has_the_bits_of_two_kernels(m, hidden, n_heads, n_kv, hd, page_size, rotate):
    """A few rows' q/k/v product in 32-bit that rotates and fills the pages itself: queries and pages in the bits of product and `rope_store`, and nothing else touched."""
    o = ops()
    n, a_dim, kv_dim = (n_heads + 2 * n_kv) * hd, n_heads * hd, n_kv * hd
    a, w = randn(m, hidden, seed=1), randn(n, hidden, seed=2, scale=0.05)
    cos, sin = (torch.cos(randn(m, hd // 2, seed=3)), torch.sin(randn(m, hd // 2, seed=3))) if rotate else (None, None)
    table = torch.randperm(12, generator=torch.Generator().manual_seed(4)).view(4, 3).to(torch.int32).to(DEV)
    slots = torch.tensor([i % 4 for i in range(m)], dtype=torch.int32, device=DEV)
    positions = torch.tensor([(page_size - 1 + (i // 4) * page_size + i % 4) % (3 * page_size) for i in range(m)], dtype=torch.int32, device=DEV)
    caches = [torch.full((12, 2, n_kv, page_size, hd), 7.0, device=DEV) for _ in range(2)]
    qkv, want, got = torch.empty(m, n, device=DEV), torch.empty(m, a_dim, device=DEV), torch.empty(m, a_dim, device=DEV)
    o.gemm_exact(a, w, qkv)
    o.rope_store(qkv[:, :a_dim], qkv[:, a_dim:a_dim + kv_dim], qkv[:, a_dim + kv_dim:], cos, sin, positions, slots, table, want, caches[0], n_heads, n_kv, hd)
    o.gemm_exact_qkv_rope_store(a, w, cos, sin, positions, slots, table, got, caches[1], n_heads, n_kv, hd)
    assert torch.equal(got, want) and torch.equal(caches[0], caches[1]) and bool((caches[1] != 7).any())


@pytest.mark.parametrize("m,n,k,gated", [(3, 16384, 2048, "silu"), (1, 1000, 4096, "gelu_tanh"), (8, 34, 36, "swish_clamped"), (16, 1004, 264, "gelu_tanh"), (9, 2, 4, "silu")])
def test_gemm_exact_gated_has_the_bits_of_two_kernels(m, n, k, gated):
    o = ops()
    a, w = randn(m, k + 4, seed=5)[:, :k], randn(n, k, seed=6, scale=2.0 / k ** 0.5)
    product = o.gemm_exact(a, w, torch.empty(m, n, device=DEV))
    want = torch.empty(m, n // 2, device=DEV)
    o.act_mul(product, want, gated, 1.5)
    got = torch.full((m, n // 2 + 3), 7.0, device=DEV)
    o.gemm_exact_gated(a, w, got[:, :n // 2], gated, 1.5)
    assert torch.equal(got[:, :n // 2], want) and bool((got[:, n // 2:] == 7).all())


@pytest.mark.parametrize("m,n,k", [(1, 16, 8), (1, 2048, 2048), (3, 100, 136), (8, 130, 264), (16, 64, 128), (17, 1000, 520),
                                   (33, 48, 72), (64, 515, 1032), (65, 128, 64), (100, 300, 200), (128, 128, 128), (200, 257, 96),
                                   (513, 384, 1024), (2048, 96, 160),
                                   # the kernels for more than 128 rows: one block of k, edge tiles (which kernel is whose: the next test)
                                   (256, 160, 64), (130, 129, 192), (2100, 2200, 192), (4000, 8200, 128),
                                   # the ping-pong kernel (256 x 256 tiles for every compute unit or more): one block of k, an odd number of them, edges
                                   (4100, 4104, 64), (4096, 4100, 320),
                                   # ... with tiles for three quarters of the compute units only (3 x 64, and 3 x 65 with an edge on both sides)
                                   (768, 16384, 64), (520, 16400, 192),
                                   # ... and with k shared out over workgroups because the tiles are few
                                   (200, 256, 1024), (300, 2048, 2048), (129, 130, 512),
                                   # 65 to 128 rows: the skinny kernel with six or eight tiles of rows, narrow outputs (k shared out) and wide ones
                                   (72, 256, 1024), (65, 130, 512), (72, 2048, 2048), (96, 3072, 2048), (128, 2048, 8192), (80, 12300, 264), (113, 12288, 520),
                                   # wide outputs finished by the skinny kernel itself, from 12 rows and from 5
                                   (12, 12300, 520), (40, 12300, 264), (5, 65600, 72), (16, 12288, 256),
                                   # 17 to 32 rows, narrow outputs, short k: the slim kernel with two tiles of rows
                                   (32, 2048, 2048), (20, 3072, 2048), (31, 130, 136), (17, 16, 8),
                                   # up to 8 rows and a narrow output: 8 weight rows at two places in k to a matrix instruction (steps of 64, cut anywhere)
                                   (8, 2048, 8192), (4, 3072, 2048), (2, 3072, 264), (6, 1000, 1000), (7, 60, 8200), (8, 8, 32), (5, 24, 40),
                                   # ... and 9 to 16 rows, in two groups of 8 that share the weights
                                   (12, 2048, 8192), (9, 100, 136), (16, 3072, 2048), (13, 1000, 1000), (16, 8, 32),
                                   # 12 or 8 weight rows a workgroup, which fill the compute units evenly, the last one's fewer (up to 16 rows, and 17 to 32)
                                   (13, 3000, 264), (8, 3071, 264), (3, 3072, 2048), (20, 2000, 264), (32, 2920, 2048)])
@pytest.mark.parametrize("out_dtype,accumulate", [(torch.float32, False), (torch.float32, True), (torch.bfloat16, False)])
def test_gemm_bf16(m, n, k, out_dtype, accumulate):
    a, w = randn(m, k, dtype=torch.bfloat16, seed=5), randn(n, k, dtype=torch.bfloat16, seed=6)
    base = randn(m, n + 5, seed=7).to(out_dtype)
    out = base.clone()
    ops().gemm_bf16(a, w, out[:, :n], accumulate=accumulate)
    want = a.double() @ w.double().T + (base[:, :n].double() if accumulate else 0)
    tol = 1e-5 if out_dtype == torch.float32 else 5e-3
    assert rel(out[:, :n], want) < tol, (m, n, k)
    assert torch.equal(out[:, n:], base[:, n:])


@pytest.mark.parametrize("kernel,kind,m,n,k", [
    # two workgroups of four waves a unit; one of eight
    ("128x128", "stored", 2600, 3072, 2048), ("128x128", "added", 2600, 3072, 2048), ("128x128", "added handing a norm on", 2600, 3072, 1024), ("128x128", "gated", 2600, 3072, 192),
    ("128x128", "xielu", 2600, 3072, 192), ("128x128", "stored", 2590, 3070, 64), ("128x128", "added", 2590, 3070, 128), ("128x128", "gated", 2590, 3040, 64),
    ("128x128", "stored", 300, 3000, 320), ("128x128", "added", 300, 3000, 64), ("128x128", "added handing a norm on", 1300, 1024, 256), ("128x128", "gated", 300, 3040, 128), ("128x128", "xielu", 300, 3000, 320),
    # one block of k, two (where the loop's first and last waits meet), more; edge tiles
    ("256x128", "added", 2048, 3072, 64), ("256x128", "added", 2048, 3072, 128), ("256x128", "added", 2047, 3050, 192), ("256x128", "stored", 2030, 3050, 1536), ("256x128", "stored", 2048, 3072, 2048),
    ("256x128", "added handing a norm on", 2048, 3072, 1024), ("256x128", "added handing a norm on", 1700, 3072, 2048), ("256x128", "gated", 300, 16384, 512), ("256x128", "gated", 390, 16352, 384),
    ("256x128", "xielu", 2048, 3072, 64), ("256x128", "xielu", 2030, 3050, 128),
    ("256x256", "stored", 4100, 4104, 64), ("256x256", "added", 4100, 4104, 128), ("256x256", "gated", 2048, 16384, 192), ("256x256", "xielu", 2048, 8192, 64)])
def test_products_of_prompts_in_each_kernel(kernel, kind, m, n, k):
    """Every kernel for more than 128 rows with every end of a product it may be given, at sizes the library's rule sends to it, against 64 bits.
    (Rotated into the pages: `test_qkv_product_that_rotates_and_fills_the_pages`.)"""
    o = ops()
    assert o.gemm_bf16_large_kernel(m, n, k, kind) == kernel
    a, w = randn(m, k, dtype=torch.bfloat16, seed=11), randn(n, k, dtype=torch.bfloat16, seed=12, scale=1.5 / k ** 0.5)
    want = a.double() @ w.double().T
    if kind == "stored":
        out, half = torch.full((m, n + 3), 7.0, device=DEV), torch.full((m, n + 4), 7.0, dtype=torch.bfloat16, device=DEV)
        o.gemm_bf16(a, w, out[:, :n])
        o.gemm_bf16(a, w, half[:, :n])
        assert rel(out[:, :n], want) < 1e-5 and torch.equal(half[:, :n], out[:, :n].to(torch.bfloat16))
        assert bool((out[:, n:] == 7).all()) and bool((half[:, n:] == 7).all())
    elif kind == "added":
        base = randn(m, n + 1, seed=13)
        out = base.clone()
        o.gemm_bf16(a, w, out[:, :n], accumulate=True)
        assert rel(out[:, :n], want + base[:, :n].double()) < 1e-5 and torch.equal(out[:, n:], base[:, n:])
    elif kind == "added handing a norm on":
        parts = o.gemm_bf16_norm_parts(m, n, k)
        assert parts == n // 128
        base, g = randn(m, n, seed=13), (1 + 0.1 * randn(n, seed=14)).float()
        plain, x = base.clone(), base.clone()
        o.gemm_bf16(a, w, plain, accumulate=True)
        scaled, squares = torch.empty(m, n, dtype=torch.bfloat16, device=DEV), torch.empty(m, parts, device=DEV)
        o.gemm_bf16(a, w, x, accumulate=True, norm_out=(g, scaled, squares))
        assert rel(x, want + base.double()) < 1e-5 and torch.equal(x, plain) and torch.equal(scaled, (g * x).to(torch.bfloat16))
        assert rel(squares.double(), (x.double() ** 2).view(m, parts, 128).sum(2)) < 1e-6
    elif kind == "gated":
        v = want.view(m, n // 32, 2, 16)
        gate, up = v[:, :, 0].reshape(m, -1), v[:, :, 1].reshape(m, -1)
        ends = dict(silu=torch.nn.functional.silu(gate) * up, gelu_tanh=torch.nn.functional.gelu(gate, approximate="tanh") * up)
        low = gate.clamp(max=1.5)
        ends["swish_clamped"] = low * torch.sigmoid(1.702 * low) * (up.clamp(-1.5, 1.5) + 1)
        for name, right in ends.items():
            out = torch.full((m, n // 2 + 1), 7.0, dtype=torch.bfloat16, device=DEV)
            o.gemm_bf16(a, w, out[:, :n // 2], gated=name, gate_limit=1.5)
            assert rel(out[:, :n // 2], right) < 4e-3 and bool((out[:, n // 2:] == 7).all()), name        # (one rounding to bfloat16: 2^-8 of the largest at most)
    else:
        params = torch.tensor([0.3, -0.7], device=DEV)
        pa, pb = torch.nn.functional.softplus(params.double())
        right = torch.where(want > 0, pa * want * want + 0.5 * want, (0.5 + pb) * (torch.expm1(want) - want) + 0.5 * want)
        out = torch.full((m, n + 5), 7.0, dtype=torch.bfloat16, device=DEV)
        o.gemm_bf16_xielu(a, w, params, out[:, :n])
        assert rel(out[:, :n], right) < 4e-3 and bool((out[:, n:] == 7).all())


@pytest.mark.parametrize("kind,m,n,k,shares", [
    # no whole round: two shares of equal and of unequal parts of k, ragged tiles; one whole round and a few tiles in four, three and two shares
    ("added", 2048, 2048, 8192, 2), ("added", 1777, 2050, 8256, 2), ("handing", 2048, 2048, 8192, 2), ("stored", 1777, 2050, 8256, 2), ("bfloat16", 1777, 2050, 8256, 2),
    ("rotated", 2048, 5120, 3072, 4), ("added", 2047, 5130, 3072, 3), ("gated", 2600, 4064, 4160, 2)])
def test_products_whose_last_tiles_share_k_out(kind, m, n, k, shares):
    """The tiles of 256 x 128 of an incomplete round, each made by several workgroups: against 64 bits, and every time the same bits, whoever came last; counters that are
    given come back as they were."""
    o = ops()
    asked = {"handing": "added handing a norm on", "bfloat16": "stored"}.get(kind, kind)
    assert o.gemm_bf16_large_kernel(m, n, k, asked) == "256x128" and o.lib().gi_gemm_bf16_tall_shares(m, n, k) == shares
    a, w = randn(m, k, dtype=torch.bfloat16, seed=11), randn(n, k, dtype=torch.bfloat16, seed=12, scale=1.5 / k ** 0.5)
    want = a.double() @ w.double().T
    seen, counters = [], torch.zeros(o.lib().gi_gemm_bf16_counters(), dtype=torch.int32, device=DEV)
    for given in (None, counters, counters, None):
        if kind == "rotated":
            heads, hd, page = n // 128 - 16, 128, 16
            q, cache = torch.zeros(m, heads * hd, dtype=torch.bfloat16, device=DEV), torch.zeros(m // page, 2, 8, page, hd, dtype=torch.bfloat16, device=DEV)
            positions, slots = torch.arange(m, dtype=torch.int32, device=DEV), torch.zeros(m, dtype=torch.int32, device=DEV)
            o.gemm_bf16_qkv_rope_store(a, w, None, None, positions, slots, torch.arange(m // page, dtype=torch.int32, device=DEV).view(1, -1), q, cache, heads, 8, hd,
                                       counters=given)
            keys, values = cache[:, 0].permute(0, 2, 1, 3).reshape(m, -1), cache[:, 1].reshape(-1, 8, hd, page).permute(0, 3, 1, 2).reshape(m, -1)
            got, right, tol = torch.cat([q, keys, values], dim=1), want, 4e-3
        elif kind == "gated":
            got = torch.empty(m, n // 2, dtype=torch.bfloat16, device=DEV)
            o.gemm_bf16(a, w, got, gated=True, counters=given)
            v = want.view(m, n // 32, 2, 16)
            right, tol = torch.nn.functional.silu(v[:, :, 0].reshape(m, -1)) * v[:, :, 1].reshape(m, -1), 4e-3
        else:
            got = torch.full((m, n), 0.5, dtype=torch.bfloat16 if kind == "bfloat16" else torch.float32, device=DEV)
            norm_out = None
            if kind == "handing":
                norm_out = (torch.ones(n, device=DEV), torch.empty(m, n, dtype=torch.bfloat16, device=DEV), torch.empty(m, o.gemm_bf16_norm_parts(m, n, k), device=DEV))
            o.gemm_bf16(a, w, got, accumulate=kind in ("added", "handing"), norm_out=norm_out, counters=given)
            right, tol = want + (0.5 if kind in ("added", "handing") else 0.0), 4e-3 if kind == "bfloat16" else 1e-5
            if kind == "handing":
                assert torch.equal(norm_out[1], got.to(torch.bfloat16))
        assert rel(got, right) < tol
        seen.append(got)
    assert all(torch.equal(seen[0], s) for s in seen[1:]) and not bool(counters.any())


@pytest.mark.parametrize("m,inter,k", [(1, 16, 8), (5, 48, 136), (16, 160, 96), (17, 176, 64), (64, 32, 264), (70, 192, 128), (300, 8192 // 16, 2048 // 8),
                                       (72, 8192, 2048), (128, 6144, 264), (100, 288, 136),
                                       (40, 6144, 264), (13, 6160, 72), (64, 8192, 512), (2048, 1024, 192), (600, 288, 64), (200, 512, 1024),
                                       (4100, 2064, 128), (640, 8192, 128), (530, 8208, 192)])
def test_gemm_bf16_gated(m, inter, k):
    a = randn(m, k, dtype=torch.bfloat16, seed=15)
    gate, up = randn(inter, k, dtype=torch.bfloat16, seed=16, scale=0.3), randn(inter, k, dtype=torch.bfloat16, seed=17, scale=0.3)
    w = ops().interleave_gate_up(gate, up)
    out = torch.full((m, inter + 2), 3.0, dtype=torch.bfloat16, device=DEV)
    ops().gemm_bf16(a, w, out[:, :inter], gated=True)
    want = torch.nn.functional.silu(a.double() @ gate.double().T) * (a.double() @ up.double().T)
    assert rel(out[:, :inter], want) < 6e-3
    assert torch.all(out[:, inter:] == 3.0)
    # the same product gated by the tanh form of GELU, stated here as 0.5 z (1 + tanh(sqrt(2 / pi) (z + 0.044715 z^3)))
    ops().gemm_bf16(a, w, out[:, :inter], gated="gelu_tanh")
    z = a.double() @ gate.double().T
    want = 0.5 * z * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (z + 0.044715 * z ** 3))) * (a.double() @ up.double().T)
    assert rel(out[:, :inter], want) < 6e-3
    assert torch.all(out[:, inter:] == 3.0)


@pytest.mark.parametrize("gated,limit", [(True, 0.0), ("gelu_tanh", 0.0), ("swish_clamped", 1.5)])
@pytest.mark.parametrize("m,inter,k,few,columns,stride", [(300, 8192, 2048, 256, 8192, 8192), (500, 8192, 512, 131, 8192, 8195), (200, 14336, 512, 200, 8192, 14336), (257, 8176, 512, 256, 8176, 8178)])
def test_gated_products_have_one_gate(m, inter, k, few, columns, stride, gated, limit):
    """The tiles of 256 x 128 gate as those of 128 x 128 do, which fewer rows or fewer columns take: the same sums, the same results in bits."""
    a = randn(m, k, dtype=torch.bfloat16, seed=15)
    w = randn(2 * inter, k, dtype=torch.bfloat16, seed=16, scale=2.0 / k ** 0.5)
    out = torch.full((m, stride), 3.0, dtype=torch.bfloat16, device=DEV)
    assert ops().gemm_bf16_large_kernel(m, 2 * inter, k, "gated") == "256x128" and ops().gemm_bf16_large_kernel(few, 2 * columns, k, "gated") == "128x128"
    ops().gemm_bf16(a, w, out[:, :inter], gated=gated, gate_limit=limit)
    alone = torch.empty(few, columns, dtype=torch.bfloat16, device=DEV)
    ops().gemm_bf16(a[:few], w[:2 * columns], alone, gated=gated, gate_limit=limit)
    assert torch.equal(out[:few, :columns], alone) and bool((out[:, inter:] == 3.0).all())


@pytest.mark.parametrize("m", [1, 17, 33, 64, 65, 97, 128, 129, 160, 161, 192, 193, 225, 256])
@pytest.mark.parametrize("n,k", [(12320, 64), (12288 + 48, 192), (16384, 576), (200, 1088), (3072, 1536), (2048, 2112)])
def test_gemm_bf16_strips(m, n, k):
    """64 columns by all rows, 17 to 128 of them (one row: the kernel for few rows): on both sides of every height, one to more blocks of k than the ring has stages, a last strip of 8, 32 and 48 columns, k whole and in two to seven shares
    (uneven ones too), stored, added, in bfloat16 and gated.  With more rows strips make some of these products: two tiles of rows in two shares (3,072 x 1,536), gated ones with all of k."""
    a, w = randn(m, k, dtype=torch.bfloat16, seed=1), randn(n, k, dtype=torch.bfloat16, seed=2, scale=0.1)
    want = a.double() @ w.double().T
    out = torch.full((m, n + 4), 3.0, device=DEV)
    ops().gemm_bf16(a, w, out[:, :n])
    assert rel(out[:, :n], want) < 2e-6 and bool((out[:, n:] == 3.0).all())
    ops().gemm_bf16(a, w, out[:, :n], accumulate=True)
    assert rel(out[:, :n], 2 * want) < 2e-6 and bool((out[:, n:] == 3.0).all())
    rounded = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    ops().gemm_bf16(a, w, rounded)
    assert torch.equal(rounded, (out[:, :n] / 2).bfloat16()) or rel(rounded, want) < 4.1e-3          # half of bfloat16's last place
    if n % 32 == 0:
        gate, up = want.view(m, n // 32, 2, 16).unbind(2)
        gated = torch.full((m + 1, n // 2), 3.0, dtype=torch.bfloat16, device=DEV)
        ops().gemm_bf16(a, w, gated[:m], gated=True)
        assert rel(gated[:m], (torch.nn.functional.silu(gate) * up).reshape(m, n // 2)) < 4.1e-3 and bool((gated[m:] == 3.0).all())


# m, n, k -> tiles of rows, rows of the last one, shares of k, blocks of 64 of a share and of the last one
@pytest.mark.parametrize("m,n,k,tiles,last,shares,blocks,last_blocks",
                         [(m, 3072, 8192, 1, m, 5, 26, 24) for m in (17, 33, 65, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256)] +
                         [(33, 200, 1088, 1, 33, 5, 4, 1), (129, 200, 4096, 3, 43, 13, 5, 4), (193, 2048, 2048, 4, 46, 2, 16, 16), (257, 2048, 8192, 2, 128, 4, 32, 32), (301, 2048, 2048, 4, 73, 2, 16, 16),
                          (400, 500, 4096, 7, 52, 4, 16, 16), (897, 2048, 8192, 4, 222, 2, 64, 64), (897, 2048, 2048, 8, 106, 1, 32, 32), (1536, 1920, 640, 8, 192, 1, 10, 10), (225, 3072, 1536, 4, 54, 1, 24, 24)])
def test_gemm_bf16_strips_of_shared_k(m, n, k, tiles, last, shares, blocks, last_blocks):
    """k in even and uneven shares, one tile of every height (both ends of the rows that each has) or several of equal height, the last of them a few rows lower: stored, added and in bfloat16, whole
    matrices and columns of wider ones; the cut is the one named."""
    assert ops().gemm_bf16_strip_cut(m, n, k) == (tiles, shares)
    tile_rows, per = -(-m // tiles), -(-(k // 64) // shares)
    assert (m - (tiles - 1) * tile_rows, per, k // 64 - (shares - 1) * per) == (last, blocks, last_blocks)
    wide_a, wide_w = randn(m, k + 24, dtype=torch.bfloat16, seed=1), randn(n, k + 40, dtype=torch.bfloat16, seed=2, scale=0.1)
    a, w = wide_a[:, 8:8 + k], wide_w[:, 16:16 + k]
    want = a.double() @ w.double().T
    seen = []
    for left, right in ((a, w), (a.contiguous(), w.contiguous())):
        out = torch.full((m + 1, n + 4), 3.0, device=DEV)
        ops().gemm_bf16(left, right, out[:m, :n])
        assert rel(out[:m, :n], want) < 2e-6 and bool((out[:, n:] == 3.0).all()) and bool((out[m:] == 3.0).all())
        rounded = torch.full((m + 1, n), 3.0, dtype=torch.bfloat16, device=DEV)
        ops().gemm_bf16(left, right, rounded[:m])
        assert torch.equal(rounded[:m], out[:m, :n].bfloat16()) and bool((rounded[m:] == 3.0).all())
        ops().gemm_bf16(left, right, out[:m, :n], accumulate=True)
        assert rel(out[:m, :n], 2 * want) < 2e-6 and bool((out[m:] == 3.0).all())
        seen.append(out)
    assert torch.equal(*seen)


@pytest.mark.parametrize("gated,limit", [(True, 0.0), ("gelu_tanh", 0.0), ("swish_clamped", 1.5)])
@pytest.mark.parametrize("m", [129, 160, 161, 192])
def test_gemm_bf16_strips_gate_up_to_192_rows(m, gated, limit):
    """Every gate at both heights of strips above 128 rows, the last strip of 32 columns; whole matrices and columns of wider ones in bits."""
    inter, k = 6160, 1088
    assert ops().gemm_bf16_large_kernel(m, 2 * inter, k, "gated") == "strips"
    wide_a, wide_w = randn(m, k + 24, dtype=torch.bfloat16, seed=1), randn(2 * inter, k + 40, dtype=torch.bfloat16, seed=2, scale=0.05)
    a, w = wide_a[:, 8:8 + k], wide_w[:, 16:16 + k]
    gate, up = (a.double() @ w.double().T).view(m, inter // 16, 2, 16).unbind(2)
    if gated == "swish_clamped":
        gate, up = gate.clamp(max=limit), up.clamp(-limit, limit) + 1
        want = gate * torch.sigmoid(1.702 * gate) * up
    else:
        want = (torch.nn.functional.silu(gate) if gated is True else 0.5 * gate * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (gate + 0.044715 * gate ** 3)))) * up
    seen = []
    for left, right in ((a, w), (a.contiguous(), w.contiguous())):
        out = torch.full((m + 1, inter + 2), 3.0, dtype=torch.bfloat16, device=DEV)
        ops().gemm_bf16(left, right, out[:m, :inter], gated=gated, gate_limit=limit)
        assert rel(out[:m, :inter], want.reshape(m, inter)) < 4.1e-3 and bool((out[m:] == 3.0).all()) and bool((out[:, inter:] == 3.0).all())
        seen.append(out)
    assert torch.equal(*seen)


@pytest.mark.parametrize("m,n,k", [(1, 17608, 64), (12, 28680, 384), (20, 16384, 576), (64, 12320, 192), (97, 12320, 576), (128, 16384, 1088)])
def test_gemm_bf16_strips_of_columns_of_wider_matrices(m, n, k):
    """All of k in a workgroup: rows of A and W further apart than k, in bits as whole matrices."""
    assert ops().gemm_bf16_small_kernel(m, n, k) == "strips"
    wide_a, wide_w = randn(m, k + 24, dtype=torch.bfloat16, seed=1), randn(n, k + 40, dtype=torch.bfloat16, seed=2, scale=0.1)
    a, w = wide_a[:, 8:8 + k], wide_w[:, 16:16 + k]
    out, whole = torch.full((m + 1, n + 4), 3.0, device=DEV), torch.empty(m, n, device=DEV)
    ops().gemm_bf16(a, w, out[:m, :n])
    ops().gemm_bf16(a.contiguous(), w.contiguous(), whole)
    assert torch.equal(out[:m, :n], whole) and rel(whole, a.double() @ w.double().T) < 2e-6 and bool((out[:, n:] == 3.0).all()) and bool((out[m:] == 3.0).all())


@pytest.mark.parametrize("m,n,k", [(33, 3072, 8192), (131, 3072, 8192)])
@pytest.mark.parametrize("short_of", ["scratch", "strides"])
def test_products_that_strips_do_not_make_go_the_way_before(m, n, k, short_of, monkeypatch):
    """With the scratch of the kernels before strips, fewer shares of k than strips make, and with rows of A further apart than a strip's 32-bit offsets are asked to reach."""
    o = ops()
    before = o.lib().gi_gemm_bf16_skinny_splits(n, k) if m <= 128 else o.lib().gi_gemm_bf16_piped_splits(m, n, k)
    assert 0 < before < o.gemm_bf16_strip_cut(m, n, k)[1]
    a, w = randn(m, k, dtype=torch.bfloat16, seed=1), randn(n, k, dtype=torch.bfloat16, seed=2, scale=0.1)
    strips, out = torch.empty(m, n, device=DEV), torch.full((m + 1, n + 4), 3.0, device=DEV)
    o.gemm_bf16(a, w, strips)
    if short_of == "scratch":
        monkeypatch.setattr(o, "_scratch_floats", lambda *_: before * m * n)
    else:
        far = torch.empty(m, 1 << 22, dtype=torch.bfloat16, device=DEV)[:, :k]
        far.copy_(a)
        a = far
    o.gemm_bf16(a, w, out[:m, :n])
    want = a.double() @ w.double().T
    assert rel(out[:m, :n], want) < 2e-6 and rel(strips, want) < 2e-6 and bool((out[:, n:] == 3.0).all()) and bool((out[m:] == 3.0).all())
    assert not torch.equal(out[:m, :n], strips)                            # (the sums of other shares)


@pytest.mark.parametrize("n", [5, 2300, 4600, 7000])                      # weight rows a workgroup: 8, 9, 18 and 28 (15 where added, or of the longest k), the last workgroup's fewer
@pytest.mark.parametrize("m,k", [(1, 8), (8, 72), (9, 520), (16, 1032), (3, 1536), (8, 2056), (16, 2560), (7, 3080), (12, 4160), (1, 5120)])
def test_gemm_bf16_few_rows_at_every_height(m, n, k):
    """Workgroups of 8 to 32 weight rows with partly full groups, waves of none to ten steps of 64 k, the last one ragged; operands and outputs within wider ones.  The 32-bit sums' bound: 2e-6."""
    wide_a, wide_w = randn(m, k + 24, dtype=torch.bfloat16, seed=1), randn(n, k + 8, dtype=torch.bfloat16, seed=2, scale=0.1)
    a, w, x0 = wide_a[:, 8:8 + k], wide_w[:, :k], randn(m, n, seed=3)
    want = a.double() @ w.double().T
    out, x, low = torch.full((m + 1, n + 3), 3.0, device=DEV), x0.clone(), torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    ops().gemm_bf16(a, w, out[:m, :n])
    ops().gemm_bf16(a, w, x, accumulate=True)
    ops().gemm_bf16(a, w, low)
    assert rel(out[:m, :n], want) < 2e-6 and rel(x, x0.double() + want) < 2e-6 and rel(low, want) < 4.1e-3
    assert bool((out[m:] == 3.0).all()) and bool((out[:, n:] == 3.0).all())
    cols = n // 32 * 16                                                    # gated: pairs of 16 weight rows, by halves of them or whole ones
    if cols:
        gate, up = want[:, :2 * cols].reshape(m, cols // 16, 2, 16).unbind(2)
        gated = torch.full((m + 1, cols + 2), 3.0, dtype=torch.bfloat16, device=DEV)
        ops().gemm_bf16(a, w[:2 * cols], gated[:m, :cols], gated=True)
        assert rel(gated[:m, :cols], (torch.nn.functional.silu(gate) * up).reshape(m, cols)) < 4.1e-3
        assert bool((gated[m:] == 3.0).all()) and bool((gated[:, cols:] == 3.0).all())


@pytest.mark.parametrize("m,n,k,lda8,reach", [(16, 8192, 256, ((1 << 28) - 32) // 15, (32, False)), (16, 8192, 256, ((1 << 28) - 32) // 15 + 1, (24, False)), (16, 8192, 264, ((1 << 32) - 33) // 15, (24, False)),
                                              (16, 6144, 264, ((1 << 32) - 33) // 15 + 1, (24, True)), (16, 300, 56, ((1 << 32) - 7) // 15 + 1, (8, True))])
def test_gemm_bf16_few_rows_far_apart(m, n, k, lda8, reach):
    """Rows of A that the ends of 32 bits lie in, 4.3 and 68.7 GB behind the first: stored, added with a norm taken and handed on, gated, through xielu, and weight rows so far apart.
    (Weights of a multiple of 64 of k beyond 12,288 columns go another way, which takes no such rows.)"""
    o = ops()
    assert o.gemm_bf16_slim_reach(m, n, k, 8 * lda8, k) == reach
    torch.cuda.empty_cache()
    far = torch.as_strided(torch.empty(8 * lda8 * (m - 1) + k, dtype=torch.bfloat16, device=DEV), (m, k), (8 * lda8, 1))
    far.copy_(randn(m, k, dtype=torch.bfloat16, seed=1))
    a, w, x0 = far.contiguous(), randn(n, k, dtype=torch.bfloat16, seed=2, scale=0.1), randn(m, n, seed=3)
    want = a.double() @ w.double().T
    out, x, low = torch.full((m + 1, n + 3), 3.0, device=DEV), x0.clone(), torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    o.gemm_bf16(far, w, out[:m, :n])
    o.gemm_bf16(far, w, x, accumulate=True)
    o.gemm_bf16(far, w, low)
    assert rel(out[:m, :n], want) < 2e-6 and rel(x, x0.double() + want) < 2e-6 and rel(low, want) < 4.1e-3
    assert bool((out[m:] == 3.0).all()) and bool((out[:, n:] == 3.0).all())
    cols = n // 32 * 16
    gate, up = want[:, :2 * cols].reshape(m, cols // 16, 2, 16).unbind(2)
    gated = torch.full((m + 1, cols + 2), 3.0, dtype=torch.bfloat16, device=DEV)
    o.gemm_bf16(far, w[:2 * cols], gated[:m, :cols], gated=True)
    assert rel(gated[:m, :cols], (torch.nn.functional.silu(gate) * up).reshape(m, cols)) < 4.1e-3 and bool((gated[m:] == 3.0).all()) and bool((gated[:, cols:] == 3.0).all())
    if reach[1]:
        weights = far[::m - 1]                                             # (the first row and the last as weight rows)
        assert o.gemm_bf16_slim_reach(1, 2, k, k, weights.stride(0)) == (8, True)
        o.gemm_bf16(a[:1], weights, out[:1, :2])
        assert rel(out[:1, :2], a[:1].double() @ a[::m - 1].double().T) < 2e-6
        mid, mid_near, params = torch.empty(m, n, dtype=torch.bfloat16, device=DEV), torch.empty(m, n, dtype=torch.bfloat16, device=DEV), torch.tensor([0.3, -0.2], device=DEV)
        o.gemm_bf16_xielu(far, w, params, mid)
        o.gemm_bf16_xielu(a, w, params, mid_near)
        assert torch.equal(mid, mid_near)                                  # (as many weight rows a workgroup: the same sums)
        squares, g = torch.rand(m, 3, device=DEV) * k, torch.rand(n, device=DEV)
        results = []
        for rows in (far, a):
            y, scaled, pieces = x0.clone(), torch.empty(m, n, dtype=torch.bfloat16, device=DEV), torch.zeros(m, o.gemm_bf16_norm_parts(m, n, k), device=DEV)
            o.gemm_bf16(rows, w, y, accumulate=True, norm_in=(squares, 1e-5), norm_out=(g, scaled, pieces))
            results.append((y, scaled, pieces))
        assert all(torch.equal(got, beside) for got, beside in zip(*results))
    del far
    torch.cuda.empty_cache()


@pytest.mark.parametrize("m,parts", [(1, 512), (8, 300), (9, 256), (16, 3), (17, 256), (32, 2), (33, 8), (64, 1), (128, 5)])
def test_gemm_bf16_strips_finish_a_norm(m, parts):
    n, k = 28672, 3072 if m > 10 else 192
    assert ops().gemm_bf16_small_kernel(m, n, k, True) == "strips"
    a, w, squares = randn(m, k, dtype=torch.bfloat16, seed=1), randn(n, k, dtype=torch.bfloat16, seed=2, scale=0.1), randn(m, parts, seed=3).abs() * k / parts
    product = (a.double() @ w.double().T) * torch.rsqrt(squares.double().sum(1, keepdim=True) / k + 1e-5)
    gate, up = product.view(m, n // 32, 2, 16).unbind(2)
    out = torch.empty(m, n // 2, dtype=torch.bfloat16, device=DEV)
    ops().gemm_bf16(a, w, out, gated=True, norm_in=(squares, 1e-5))
    assert rel(out, (torch.nn.functional.silu(gate) * up).reshape(m, n // 2)) < 4.1e-3


@pytest.mark.parametrize("m,n,k", [(4109, 4120, 192), (4096, 4096, 448)])
def test_gemm_bf16_ping_pong_with_whole_lines(m, n, k):
    """Outputs whose rows are 16-byte aligned leave the ping-pong kernel in whole cache lines: every epilogue, with edge tiles."""
    a, w = randn(m, k, dtype=torch.bfloat16, seed=25), randn(n, k, dtype=torch.bfloat16, seed=26, scale=0.3)
    want = a.double() @ w.double().T
    for out_dtype, accumulate in ((torch.float32, False), (torch.float32, True), (torch.bfloat16, False)):
        base = randn(m, n, seed=27).to(out_dtype)
        out = base.clone()
        ops().gemm_bf16(a, w, out, accumulate=accumulate)
        assert rel(out, want + (base.double() if accumulate else 0)) < (1e-5 if out_dtype == torch.float32 else 5e-3), (out_dtype, accumulate)
    gate, up = w[:n // 2 // 16 * 16], w[n // 2:n // 2 + n // 2 // 16 * 16]
    out = torch.full((m, gate.shape[0]), 3.0, dtype=torch.bfloat16, device=DEV)
    ops().gemm_bf16(a, ops().interleave_gate_up(gate.contiguous(), up.contiguous()), out, gated=True)
    assert rel(out, torch.nn.functional.silu(a.double() @ gate.double().T) * (a.double() @ up.double().T)) < 6e-3


def test_gemm_bf16_refuses_what_it_cannot_do():
    o = ops()
    a, w = randn(4, 12, dtype=torch.bfloat16), randn(6, 12, dtype=torch.bfloat16)
    out = torch.empty(4, 6, device=DEV)
    assert not o.gemm_bf16_supports(a, w, out)                       # K = 12 is no multiple of 8
    with pytest.raises(o.KernelError):
        o.gemm_bf16(a, w, out)


# ------------------------------------------------------------------------------- row-wise kernels
@pytest.mark.parametrize("n,dim", [(1, 1), (3, 17), (5, 256), (2, 1000), (7, 4099)])
@pytest.mark.parametrize("w_dtype,out_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16)])
def test_rmsnorm(n, dim, w_dtype, out_dtype):
    x, w = randn(n, dim, seed=8, scale=3.0), (1 + 0.1 * randn(dim, seed=9)).to(w_dtype)
    for eps in (1e-6, 0.05):                                         # a large eps shows an eps in the wrong place
        out = torch.empty(n, dim, dtype=out_dtype, device=DEV)
        ops().rmsnorm(x, w, eps, out)
        xd = x.double()
        want = w.double() * (xd / torch.sqrt((xd * xd).mean(-1, keepdim=True) + eps))
        assert rel(out, want) < (2e-6 if out_dtype == torch.float32 else 5e-3)
    zero = torch.zeros(1, dim, device=DEV)
    out = torch.empty(1, dim, device=DEV)
    ops().rmsnorm(zero, w.float(), 1e-6, out)
    assert torch.isfinite(out).all() and float(out.abs().max()) == 0.0


def test_embed_and_gather():
    table = randn(50, 24, dtype=torch.bfloat16, seed=10)
    toks = torch.tensor([3, 49, 0, 3], dtype=torch.int32, device=DEV)
    out = torch.empty(4, 24, device=DEV)
    ops().embed(table, toks, out)
    assert torch.equal(out, table[toks.long()].float())
    picked = torch.empty(2, 24, device=DEV)
    ops().gather_rows(out, torch.tensor([2, 1], dtype=torch.int32, device=DEV), picked)
    assert torch.equal(picked, out[[2, 1]])


@pytest.mark.parametrize("dim,dtype", [(2048, torch.bfloat16), (24, torch.bfloat16), (37, torch.bfloat16), (100, torch.float32)])
def test_embed_with_the_first_half_of_a_norm(dim, dtype):
    """The fetch of token rows that also writes them times a norm's weights in bfloat16 and their sums of squares (widths with and
    without the four-channel path), against the plain statement; with the product's share (times rsqrt(mean square + eps)) the
    rows are the norm's."""
    table = randn(50, dim, dtype=dtype, seed=10)
    toks = torch.tensor([3, 49, 0, 3, 17], dtype=torch.int32, device=DEV)
    g = (1 + 0.1 * randn(dim, seed=12)).contiguous()
    out, scaled, squares = torch.empty(5, dim, device=DEV), torch.empty(5, dim, dtype=torch.bfloat16, device=DEV), torch.empty(5, 1, device=DEV)
    ops().embed_handing(table, toks, out, g, scaled, squares)
    rows = table[toks.long()].double()
    assert torch.equal(out, rows.float())
    assert torch.equal(scaled, (g * out).to(torch.bfloat16))
    assert rel(squares[:, 0], (rows ** 2).sum(1)) < 1e-6
    normed = scaled.double() * torch.rsqrt(squares.double() / dim + 1e-5)
    assert rel(normed, g.double() * rows * torch.rsqrt((rows ** 2).mean(1, keepdim=True) + 1e-5)) < 5e-3


@pytest.mark.parametrize("dim,dtype", [(2048, torch.bfloat16), (24, torch.bfloat16), (37, torch.bfloat16), (100, torch.float32), (1028, torch.float32)])
def test_embed_with_a_factor(dim, dtype):
    """A scale behind the token table is a factor of the fetch: the bits of the two, with and without the four-channel path."""
    table, toks, factor = randn(50, dim, dtype=dtype, seed=10), torch.tensor([3, 49, 0, 3, 17], dtype=torch.int32, device=DEV), 45.25
    want = ops().scale_rows(table[toks.long()].float(), factor)
    assert torch.equal(ops().embed(table, toks, torch.empty(5, dim, device=DEV), factor), want)


def test_silu_mul():
    gu = randn(5, 2 * 37, seed=11, scale=4.0)
    gu[0, 0], gu[0, 1] = 100.0, -100.0                               # extremes stay finite
    out = torch.empty(5, 37, device=DEV)
    ops().silu_mul(gu, out)
    want = torch.nn.functional.silu(gu[:, :37].double()) * gu[:, 37:].double()
    assert rel(out, want) < 2e-6 and torch.isfinite(out).all()


def test_rope_cos_sin_uses_64_bit_angles():
    pos = torch.tensor([0, 1, 4095, 131071, 2 ** 24 + 1], dtype=torch.int32, device=DEV)
    inv = torch.tensor([1.0, 0.3, 1e-3], dtype=torch.float64, device=DEV)
    cos, sin = torch.empty(5, 3, device=DEV), torch.empty(5, 3, device=DEV)
    ops().rope_cos_sin(pos, inv, cos, sin)
    ang = pos.double()[:, None] * inv[None, :]
    assert (cos.double() - torch.cos(ang)).abs().max() < 1e-7 and (sin.double() - torch.sin(ang)).abs().max() < 1e-7


@pytest.mark.parametrize("m,d,k1,n2,gated", [(1, 2048, 2048, 3072, False), (8, 2048, 8192, 16384, True), (8, 2048, 2048, 16384, True), (9, 2048, 2048, 3072, False),
                                            (16, 136, 264, 96, False), (5, 3072, 3072, 5120, False), (3, 4096, 4096, 6144, False), (7, 264, 136, 64, True),
                                            (64, 2048, 8192, 16384, True), (64, 2048, 2048, 3072, False), (40, 2048, 8192, 3072, False), (17, 2048, 8192, 16384, True),
                                            (100, 4096, 14336, 6144, False), (128, 3072, 8192, 16384, True), (33, 1024, 512, 12288, False),
                                            (24, 2048, 2048, 16384, True), (24, 2048, 8192, 3072, False), (14, 2048, 2048, 16384, True), (32, 2048, 2048, 2048, False),
                                            (17, 264, 136, 12288, False), (13, 4096, 4096, 28672, True),
                                            # 12 and 16 weight rows a workgroup, with as many pieces of a row's sum of squares as a reader takes at 9 to 16 rows, and at
                                            # up to 8
                                            (12, 3072, 8192, 5120, False), (16, 3072, 3072, 16384, True), (8, 4096, 14336, 6144, False), (4, 4096, 4096, 28672, True),
                                            # the rows of prompts: from the tiles of 128 x 128 (or the kernel that adds the shares of k) to the gated
                                            # product on the kernel with tiles of 256 x 256
                                            (2048, 2048, 2048, 16384, True), (2048, 2048, 8192, 16384, True), (1024, 2048, 2048, 16384, True),
                                            (1500, 3072, 1024, 16384, True),
                                            # ... with tiles of 256 x 256 for three quarters of the compute units
                                            (640, 2048, 2048, 16384, True), (530, 2048, 8192, 16384, True)])
def test_norm_handed_from_one_product_to_the_next(m, d, k1, n2, gated):
    """A product that adds onto rows x also writes g * x and the pieces of the rows' sums of squares; the next product reads
    g * x and multiplies its results by rsqrt(mean(x^2) + eps).  The rows x are what the plain product leaves, bit for bit; the
    second product's results are as near the 64-bit norm and product as those of the norm's own kernel followed by the product."""
    o = ops()
    eps = 1e-5
    a = randn(m, k1, dtype=torch.bfloat16, seed=1)
    w1 = randn(d, k1, dtype=torch.bfloat16, seed=2, scale=0.05)
    w2 = randn(n2, d, dtype=torch.bfloat16, seed=3, scale=0.05)
    g = (1 + 0.1 * randn(d, seed=4)).float()
    x0 = randn(m, d, seed=5)
    parts = o.gemm_bf16_norm_parts(m, d, k1)
    assert parts and o.gemm_bf16_takes_norm(m, n2, d, gated), "every case here is one the kernels take"
    plain_x = x0.clone()
    o.gemm_bf16(a, w1, plain_x, accumulate=True)
    x, scaled, squares = x0.clone(), torch.full((m, d), float("nan"), dtype=torch.bfloat16, device=DEV), torch.full((m, parts), float("nan"), device=DEV)
    o.gemm_bf16(a, w1, x, accumulate=True, norm_out=(g, scaled, squares))
    assert torch.equal(x, plain_x)
    assert torch.equal(scaled, (g * x).to(torch.bfloat16))
    assert rel(squares.double().sum(1), (x.double() ** 2).sum(1)) < 1e-6
    out_shape = (m, n2 // 2) if gated else (m, n2)
    out_dtype = torch.bfloat16 if gated else torch.float32
    w2k = o.interleave_gate_up(w2[:n2 // 2], w2[n2 // 2:]) if gated else w2
    handed = torch.empty(out_shape, dtype=out_dtype, device=DEV)
    o.gemm_bf16(scaled, w2k, handed, gated=gated, norm_in=(squares, eps))
    normed = torch.empty((m, d), dtype=torch.bfloat16, device=DEV)
    o.rmsnorm(x, g, eps, normed)
    usual = torch.empty(out_shape, dtype=out_dtype, device=DEV)
    o.gemm_bf16(normed, w2k, usual, gated=gated)
    xd = x.double()
    exact = (g.double() * xd * torch.rsqrt((xd ** 2).mean(1, keepdim=True) + eps)) @ w2.double().T
    if gated:
        exact = torch.nn.functional.silu(exact[:, :n2 // 2]) * exact[:, n2 // 2:]
    err_handed, err_usual = rel(handed, exact), rel(usual, exact)
    assert err_handed < 1.5 * err_usual + 1e-6, (err_handed, err_usual)


@pytest.mark.parametrize("m,d,k1", [(2048, 2048, 8192), (1100, 2048, 2048), (300, 2048, 2048), (2048, 3072, 8192), (700, 1024, 512), (130, 256, 192),
                                    (3000, 3072, 256), (4100, 2048, 256)])
def test_norm_handed_on_by_a_product_of_many_rows(m, d, k1):
    """The rows of prompts: the product that adds onto the residual writes g * x and the pieces of the rows' sums of squares from
    its tiles' epilogues (one piece per 128 columns), or from the kernel that adds the shares of k (one per 1024).  The rows are
    what the plain product leaves, bit for bit; sizes at which the kernels do not do it are refused."""
    o = ops()
    a = randn(m, k1, dtype=torch.bfloat16, seed=1)
    w1 = randn(d, k1, dtype=torch.bfloat16, seed=2, scale=0.05)
    g = (1 + 0.1 * randn(d, seed=4)).float()
    x0 = randn(m, d, seed=5)
    parts = o.gemm_bf16_norm_parts(m, d, k1)
    assert parts in (d // 128, d // 1024), parts
    plain_x = x0.clone()
    o.gemm_bf16(a, w1, plain_x, accumulate=True)
    x, scaled, squares = x0.clone(), torch.full((m, d), float("nan"), dtype=torch.bfloat16, device=DEV), torch.full((m, parts), float("nan"), device=DEV)
    o.gemm_bf16(a, w1, x, accumulate=True, norm_out=(g, scaled, squares))
    assert torch.equal(x, plain_x)
    assert torch.equal(scaled, (g * x).to(torch.bfloat16))
    assert rel(squares.double().sum(1), (x.double() ** 2).sum(1)) < 1e-6
    width = d // parts
    assert rel(squares.double(), (x.double() ** 2).view(m, parts, width).sum(2)) < 1e-6            # every piece is its columns' sum
    assert o.gemm_bf16_norm_parts(8192, 8192, 512) == 0 and o.gemm_bf16_norm_parts(300, 200, 512) == 0        # the ping-pong kernel; a ragged width
    with pytest.raises(o.KernelError):
        o.gemm_bf16(randn(8192, 512, dtype=torch.bfloat16, seed=1), randn(8192, 512, dtype=torch.bfloat16, seed=2), torch.zeros(8192, 8192, device=DEV),
                    accumulate=True, norm_out=((1 + 0 * randn(8192, seed=4)).float(), torch.empty(8192, 8192, dtype=torch.bfloat16, device=DEV), torch.empty(8192, 64, device=DEV)))


@pytest.mark.parametrize("m,hidden,n_heads,n_kv,hd,page_size,rotate,handed", [(64, 2048, 32, 8, 64, 16, True, True), (40, 2048, 32, 8, 64, 16, True, False),
                                                                              (128, 3072, 24, 8, 128, 16, True, True), (33, 512, 6, 1, 32, 8, False, False),
                                                                              (17, 4096, 32, 8, 128, 32, True, False), (100, 1024, 2, 1, 256, 16, True, True),
                                                                              # rows of prompts: tiles of 256 x 128 and of 128 x 128 whose epilogue rotates and stores (the
                                                                              # smaller ones with two workgroups of four waves a unit, and with one of eight), and shapes
                                                                              # whose k is shared out over workgroups
                                                                              (2048, 2048, 32, 8, 64, 16, True, False), (2048, 2048, 32, 8, 64, 16, True, True), (777, 2048, 24, 8, 128, 12, False, True),
                                                                              (2600, 2048, 32, 8, 64, 16, True, False), (2600, 1024, 32, 8, 64, 16, True, True), (1100, 256, 20, 2, 128, 16, True, True),
                                                                              (1100, 256, 80, 8, 32, 8, False, True), (300, 3072, 24, 8, 128, 16, True, True),
                                                                              (520, 512, 28, 2, 64, 16, True, False), (129, 2048, 32, 8, 64, 16, True, True)])
def test_qkv_product_that_rotates_and_fills_the_pages(m, hidden, n_heads, n_kv, hd, page_size, rotate, handed):
    """The q/k/v product whose last step rotates and writes the pages itself (the kernel that adds up the shares of k, or the
    epilogue over a tile of a prompt's rows) against the product followed by the kernel that does that, which
    `test_rope_store_writes_the_right_places` holds against the plain statement: the same queries and the same pages, also with
    a norm handed on."""
    o = ops()
    n = (n_heads + 2 * n_kv) * hd
    assert o.gemm_bf16_qkv_rope_store_takes(m, n, hidden, hd)
    if m in (777, 2048, 2600):
        assert o.gemm_bf16_large_kernel(m, n, hidden, "rotated") == ("128x128" if m == 2600 else "256x128")
    a = randn(m, hidden, dtype=torch.bfloat16, seed=1)
    w = randn(n, hidden, dtype=torch.bfloat16, seed=2, scale=0.05)
    g = torch.Generator().manual_seed(9)
    ang = torch.rand(m, hd // 2, generator=g) * 6.28
    cos, sin = (torch.cos(ang).to(DEV), torch.sin(ang).to(DEV)) if rotate else (None, None)
    n_slots = 5
    pages_per = max(4, -(-2 * m // (n_slots * page_size)))
    n_pages = n_slots * pages_per + 2
    table = torch.randperm(n_pages, generator=g)[:n_slots * pages_per].view(n_slots, pages_per).to(torch.int32).to(DEV)
    slots = torch.randint(0, n_slots, (m,), generator=g).to(torch.int32)
    positions = torch.empty(m, dtype=torch.int32)
    seen = {}
    for i in range(m):                                                # distinct (slot, position) per row
        while True:
            p = int(torch.randint(0, pages_per * page_size, (1,), generator=g))
            if (int(slots[i]), p) not in seen:
                seen[(int(slots[i]), p)] = True
                positions[i] = p
                break
    slots, positions = slots.to(DEV), positions.to(DEV)
    norm_in = None
    fill = lambda: torch.full((n_pages, 2, n_kv, page_size, hd), 7.0, dtype=torch.bfloat16, device=DEV)
    want_cache, got_cache = fill(), fill()
    qkv = torch.empty(m, n, device=DEV)
    o.gemm_bf16(a, w, qkv)
    if handed:
        parts = min(16, o.gemm_bf16_qkv_rope_store_max_parts(m, n, hidden))
        squares = (torch.rand(m, parts, generator=g) * hidden / parts).to(DEV)
        norm_in = (squares, 1e-5)
        qkv *= torch.rsqrt(squares.sum(1, keepdim=True) / hidden + 1e-5)
    a_dim, kv_dim = n_heads * hd, n_kv * hd
    want_q = torch.empty(m, a_dim, dtype=torch.bfloat16, device=DEV)
    o.rope_store(qkv[:, :a_dim], qkv[:, a_dim:a_dim + kv_dim], qkv[:, a_dim + kv_dim:], cos, sin, positions, slots, table, want_q, want_cache, n_heads, n_kv, hd)
    got_q = torch.full((m, a_dim), float("nan"), dtype=torch.bfloat16, device=DEV)
    o.gemm_bf16_qkv_rope_store(a, w, cos, sin, positions, slots, table, got_q, got_cache, n_heads, n_kv, hd, norm_in)
    step = lambda t: t.float().abs().clamp_min(1e-3) * 2.0 ** -7          # a rounding step of bfloat16 at most: the two kernels may fuse a * cos - b * sin differently
    assert ((got_q.float() - want_q.float()).abs() <= step(want_q)).all()
    assert ((got_cache.float() - want_cache.float()).abs() <= step(want_cache)).all()
    assert float((got_q.float() != want_q.float()).float().mean()) < 0.01 and float((got_cache.float() != want_cache.float()).float().mean()) < 0.01


@pytest.mark.parametrize("m,hidden,n_heads,n_kv,hd,page_size,rotate", [(2500, 3072, 24, 8, 128, 16, True), (2390, 3072, 23, 8, 128, 12, True), (4000, 2048, 32, 8, 64, 16, True), (2330, 4096, 40, 4, 128, 24, False),
                                                                       (2305, 3072, 128, 16, 32, 8, True)])
def test_qkv_product_of_many_tiles_rotates_and_fills_the_pages(m, hidden, n_heads, n_kv, hd, page_size, rotate):
    """Tiles of 256 x 256 whose halves of rows and of columns end anywhere: a last tile of one row, without a second half of rows or of columns; portions that begin anywhere, and single rows."""
    o = ops()
    n = (n_heads + 2 * n_kv) * hd
    assert o.gemm_bf16_qkv_rope_store_takes(m, n, hidden, hd) and o.gemm_bf16_large_kernel(m, n, hidden, "rotated") == "256x256"
    a, w = randn(m, hidden, dtype=torch.bfloat16, seed=1), randn(n, hidden, dtype=torch.bfloat16, seed=2, scale=hidden ** -0.5)
    ang = 6.28 * torch.rand(m, hd // 2, generator=torch.Generator().manual_seed(9))
    cos, sin = (torch.cos(ang).to(DEV), torch.sin(ang).to(DEV)) if rotate else (None, None)
    starts, pos0 = [0, 1, 2, 3, 24, 1000, m], [5, 16, 7, 0, 701, 3]
    positions = torch.cat([p + torch.arange(e - b, dtype=torch.int32) for b, e, p in zip(starts, starts[1:], pos0)]).to(DEV)
    slots = torch.cat([torch.full((e - b,), i, dtype=torch.int32) for i, (b, e) in enumerate(zip(starts, starts[1:]))]).to(DEV)
    pages = -(-(m + 800) // page_size)
    table = torch.randperm(6 * pages, generator=torch.Generator().manual_seed(3)).view(6, pages).to(torch.int32).to(DEV)
    want_cache, got_cache = (torch.full((6 * pages, 2, n_kv, page_size, hd), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    want_q, got_q = (torch.full((m + 1, n_heads * hd), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    qkv = (a.double() @ w.double().T).float()
    a_dim, kv_dim = n_heads * hd, n_kv * hd
    o.rope_store(qkv[:, :a_dim], qkv[:, a_dim:a_dim + kv_dim], qkv[:, a_dim + kv_dim:], cos, sin, positions, slots, table, want_q[:m], want_cache, n_heads, n_kv, hd)
    o.gemm_bf16_qkv_rope_store(a, w, cos, sin, positions, slots, table, got_q[:m], got_cache, n_heads, n_kv, hd)
    step = lambda t: t.float().abs() * 2.0 ** -7 + 2.0 ** -16             # a rounding step of bfloat16 at most, and what 32-bit sums of numbers about 1 may be off
    for got, want in ((got_q, want_q), (got_cache, want_cache)):
        assert ((got.float() - want.float()).abs() <= step(want)).all() and float((got.float() != want.float()).float().mean()) < 0.01


@pytest.mark.parametrize("m,page_size,portions", [(2048, 16, [(0, 24, 0), (24, 1300, 701), (1324, 724, 3)]),      # single rows, then portions that begin anywhere
                                                  (1500, 16, [(0, 3, 0), (3, 9, 5), (12, 8, 16), (20, 1, 7), (21, 1479, 1000)]),
                                                  (2048, 12, [(0, 1000, 5), (1000, 1048, 0)]), (1410, 24, [(0, 1410, 23)])])
def test_qkv_product_fills_the_pages_of_portions(m, page_size, portions):
    """The epilogue of tiles of a prompt's rows: values of eight consecutive positions leave their pages' way as one piece wherever in the
    tile their rows lie, those around them one by one: what the kernel that rotates and stores writes, at every place."""
    o = ops()
    hidden, n_heads, n_kv, hd = 192, 24, 8, 128
    n = (n_heads + 2 * n_kv) * hd
    assert o.gemm_bf16_qkv_rope_store_takes(m, n, hidden, hd)
    a, w = randn(m, hidden, dtype=torch.bfloat16, seed=41), randn(n, hidden, dtype=torch.bfloat16, seed=42, scale=0.05)
    slots, positions = torch.empty(m, dtype=torch.int32), torch.empty(m, dtype=torch.int32)
    for slot, (first, rows, pos0) in enumerate(portions):
        slots[first:first + rows] = slot
        positions[first:first + rows] = pos0 + torch.arange(rows, dtype=torch.int32)
    slots[:portions[0][1]] = torch.where(torch.tensor(portions[0][1] <= 24), len(portions) + torch.arange(portions[0][1]), torch.zeros(portions[0][1])).int()      # (few rows: a request each)
    n_slots, pages = len(portions) + 25, -(-2600 // page_size)
    table = torch.randperm(n_slots * pages, generator=torch.Generator().manual_seed(3)).view(n_slots, pages).to(torch.int32).to(DEV)
    slots, positions = slots.to(DEV), positions.to(DEV)
    want_cache, got_cache = (torch.full((n_slots * pages, 2, n_kv, page_size, hd), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    want_q, got_q = (torch.full((m, n_heads * hd), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    qkv = torch.empty(m, n, device=DEV)
    o.gemm_bf16(a, w, qkv)
    a_dim, kv_dim = n_heads * hd, n_kv * hd
    o.rope_store(qkv[:, :a_dim], qkv[:, a_dim:a_dim + kv_dim], qkv[:, a_dim + kv_dim:], None, None, positions, slots, table, want_q, want_cache, n_heads, n_kv, hd)
    o.gemm_bf16_qkv_rope_store(a, w, None, None, positions, slots, table, got_q, got_cache, n_heads, n_kv, hd)
    assert torch.equal(got_q, want_q) and torch.equal(got_cache, want_cache)             # (nothing is rotated: the same sums, rounded once)


# -------------------------------------------------------------------------------------- sampling
def test_argmax_lowest_index_on_ties():
    rows = [[1, 5, 5, 2], [3, 3, 3, 3], [-7, -8, -9, -10], [0, -1, 9, 9]]          # tests/verify_sampler.py:173-178
    logits = torch.tensor(rows, dtype=torch.float32, device=DEV)
    out = torch.empty(4, dtype=torch.int32, device=DEV)
    ops().argmax(logits, out)
    assert out.tolist() == [1, 0, 0, 2]
    big = randn(3, 128256, seed=12)
    big[1, 70000] = big[1, 5] = 50.0
    out = torch.empty(3, dtype=torch.int32, device=DEV)
    ops().argmax(big, out)
    assert out.tolist() == [int(torch.argmax(big[0])), 5, int(torch.argmax(big[2]))]


def test_sample_temperature_matches_the_inverse_distribution():
    import numpy as np
    from plain_sampler import sample
    g = torch.Generator().manual_seed(0)
    for vocab in (2, 5, 100, 3001, 128256):
        logits = (2 * torch.randn(8, vocab, generator=g)).float()
        temps = torch.tensor([0.3, 1.0, 2.0, 0.8, 1.0, 0.01, 1.5, 0.7])
        us = torch.cat([torch.rand(5, generator=g), torch.tensor([0.0, 0.5, 1.0 - 2.0 ** -24])]).float()
        out = torch.empty(8, dtype=torch.int32, device=DEV)
        ops().sample_temperature(logits.to(DEV), temps.to(DEV), us.to(DEV), out)
        for i, got in enumerate(out.tolist()):
            want = sample(logits[i].numpy(), float(temps[i]), 0, 1.0, float(us[i]))
            if got != want:                                          # only a draw on the edge between two tokens may differ
                p = torch.softmax(logits[i].double() / float(temps[i]), 0)
                cum = torch.cumsum(p, 0)
                assert abs(got - want) == 1 and float((cum - float(us[i])).abs().min()) < 1e-6, (vocab, i, got, want)


@pytest.mark.parametrize("vocab,light,heavy", [(100, 5, 40), (3000, 100, 1000), (3000, 17, 2999), (9000, 4000, 4095), (9000, 70, 5000)])
def test_a_draw_of_zero_takes_the_first_token_that_has_any_probability(vocab, light, heavy):
    """u = 0 stops at the first token whose probability is not zero (src/sampler/sampler.cpp:119-128), however little it weighs
    beside a later one: 1e-35 before a token of probability 1 is below the last bit of the running sum in 64-bit, so a thread that
    found where its tokens start by taking its own sum off the running one would start at 0 too and claim the draw."""
    from plain_sampler import sample
    logits = torch.full((3, vocab), -30.0)
    logits[:, heavy] = 0.0
    logits[0, light], logits[1, light], logits[2, light] = -0.8, -1.0, -1.04          # p = 1.8e-35, 3.8e-44 (subnormal), 0 at T = 0.01
    out = torch.empty(3, dtype=torch.int32, device=DEV)
    ops().sample_temperature(logits.to(DEV), torch.full((3,), 0.01, device=DEV), torch.zeros(3, device=DEV), out)
    assert [sample(row.numpy(), 0.01, 0, 1.0, 0.0) for row in logits] == [light, light, heavy]
    assert out.tolist() == [light, light, heavy]


def on_an_edge(logits, temperature, top_k, top_p, u, got, want):
    """Whether the plain sampler could give `got` for `want` by rounding alone: two tokens whose probabilities differ in the
    last bits change places in the order, or u, or top_p times the kept mass, falls within 2e-6 of a boundary."""
    from plain_sampler import sample
    p = torch.softmax(torch.from_numpy(logits).double() / temperature, 0)
    if abs(float(p[got]) - float(p[want])) <= 1e-6 * float(p[want]):
        return True
    near = set()
    for dp in (-2e-6, 0.0, 2e-6):
        for du in (-2e-6, 0.0, 2e-6):
            near.add(sample(logits, temperature, top_k, top_p if top_p >= 1.0 else min(max(top_p + dp, 1e-6), 1.0 - 1e-7),
                            min(max(u + du, 0.0), 1.0 - 2.0 ** -24)))
    return got in near


def filtered_on_device(logits, temps, ks, ps, us):
    n = logits.shape[0]
    out = torch.empty(n, dtype=torch.int32, device=DEV)
    ops().sample_filtered(logits.to(DEV), torch.tensor(temps, dtype=torch.float32, device=DEV), torch.tensor(ks, dtype=torch.int32, device=DEV),
                          torch.tensor(ps, dtype=torch.float32, device=DEV), torch.tensor(us, dtype=torch.float32, device=DEV), out)
    return out.tolist()


def test_filters_on_the_device_keep_what_they_should():
    """The sets that the filters leave, as the reference's test states them (tests/verify_sampler.py:161-166): among equal
    probabilities the lowest indices stay."""
    g = torch.Generator().manual_seed(3)
    us = torch.rand(300, generator=g).tolist()
    flat = torch.zeros(300, 10)
    assert set(filtered_on_device(flat, [1.0] * 300, [3] * 300, [1.0] * 300, us)) == {0, 1, 2}
    assert set(filtered_on_device(flat, [1.0] * 300, [0] * 300, [0.35] * 300, us)) == {0, 1, 2, 3}
    assert set(filtered_on_device(flat, [1.0] * 300, [7] * 300, [0.35] * 300, us)) == {0, 1, 2}          # 0.35 of the mass of seven
    peaked = torch.zeros(300, 20)
    peaked[:, 13] = 30.0
    assert set(filtered_on_device(peaked, [1.0] * 300, [0] * 300, [0.9] * 300, us)) == {13}
    assert set(filtered_on_device(peaked, [1.0] * 300, [1] * 300, [1.0] * 300, us)) == {13}
    wide = torch.zeros(300, 5000)                                   # equal probabilities far beyond one wave's reach
    wide[:, 4000:] = 1.0
    got = filtered_on_device(wide, [1.0] * 300, [600] * 300, [1.0] * 300, us)
    assert min(got) >= 4000 and max(got) < 4600 and len(set(got)) > 150
    got = filtered_on_device(wide, [1.0] * 300, [1300] * 300, [1.0] * 300, us)                            # all of the likely ones and 300 of the rest
    assert set(t for t in got if t < 4000) <= set(range(300)) and any(t < 4000 for t in got) and max(got) < 5000


def test_sample_filtered_matches_the_plain_sampler():
    """Top-k and top-p on the device against the plain sampler, row by row: random logits, logits on a coarse grid (many
    tokens of exactly equal probability, so that the filters cut through groups of equals), and the real vocabulary."""
    from plain_sampler import sample
    g = torch.Generator().manual_seed(1)
    settings = [(1.0, 0, 0.9), (0.8, 0, 0.5), (1.0, 0, 0.05), (1.0, 3, 1.0), (1.5, 50, 1.0), (1.0, 5, 0.9), (0.7, 1, 1.0), (1.0, 4, 0.3),
                (0.3, 0, 0.999), (2.0, 40, 0.95), (1.0, 10 ** 6, 0.7), (1.0, 0, 2.0 ** -20)]
    exact = total = 0
    for vocab, coarse in ((2, False), (5, False), (100, False), (100, True), (3001, False), (3001, True), (128256, False), (128256, True)):
        rows = []
        for t, k, p in settings:
            if not (0 < k < vocab or p < 1.0):
                continue
            for u in torch.rand(2 if vocab > 100000 else 6, generator=g).tolist() + [0.0, 1.0 - 2.0 ** -24]:
                rows.append((t, k, p, u))
        logits = 2 * torch.randn(len(rows), vocab, generator=g)
        if coarse:
            logits = torch.round(logits * 2) / 2
        got = filtered_on_device(logits, *zip(*rows))
        for i, (t, k, p, u) in enumerate(rows):
            row = logits[i].numpy()
            want = sample(row, t, k, p, np.float32(u))
            total += 1
            exact += got[i] == want
            assert got[i] == want or on_an_edge(row, t, k, p, u, got[i], want), (vocab, coarse, i, (t, k, p, u), got[i], want)
    assert exact >= 0.98 * total, (exact, total)


def test_rows_of_every_kind_of_sampler_in_one_call():
    """Greedy, plain and filtered samplers side by side get what each gets alone, and every one draws from its own stream."""
    from geneinfer_amd.sampling import Sampler, SamplerConfig, sample_rows
    g = torch.Generator().manual_seed(5)
    vocab = 777
    configs = [SamplerConfig(0.0), SamplerConfig(0.9, seed=4), SamplerConfig(1.0, top_k=7, seed=5), SamplerConfig(0.0), SamplerConfig(0.7, top_p=0.8, seed=6),
               SamplerConfig(1.2, seed=7), SamplerConfig(1.0, top_k=20, top_p=0.5, seed=8)]
    together = [Sampler(c, vocab) for c in configs]
    alone = [Sampler(c, vocab) for c in configs]
    for step in range(5):
        logits = (2 * torch.randn(len(configs), vocab, generator=g)).to(DEV)
        got = sample_rows(logits, together)
        want = [sample_rows(logits[i:i + 1], [alone[i]])[0] for i in range(len(configs))]
        assert got == want, (step, got, want)
        assert [s.stream.state for s in together] == [s.stream.state for s in alone]
    some = [together[i] for i in (2, 4, 6)]                           # only filtered ones: no gathering
    logits = (2 * torch.randn(3, vocab, generator=g)).to(DEV)
    assert sample_rows(logits, some) == [sample_rows(logits[i:i + 1], [alone[j]])[0] for i, j in enumerate((2, 4, 6))]


# ------------------------------------------------------------------------------------- attention
def build_paged(requests, n_kv, hd, page_size, dtype, seed, scale_one=None, gone_before=None, shape_keys=None):
    """Dense keys/values per request, written into a paged cache with scrambled pages and a rim of
    NaN pages that nothing may touch.  requests: list of context lengths.  gone_before: per request index, a position;
    pages that lie wholly before it have been given back (a window has passed them): their table entries are -1 and
    nothing of them is in the cache.  Returns cache, table, dense."""
    g = torch.Generator().manual_seed(seed)
    n_pages_needed = sum(-(-n // page_size) for n in requests)
    n_pages = n_pages_needed + 3
    perm = torch.randperm(n_pages, generator=g).tolist()
    cache = torch.full((n_pages, 2, n_kv, page_size, hd), float("nan"), dtype=dtype)
    width = max(-(-n // page_size) for n in requests) + 2
    table = torch.full((len(requests) + 1, width), -1, dtype=torch.int32)
    dense, nxt = [], 0
    for slot, n in enumerate(requests):
        k = torch.randn(n, n_kv, hd, generator=g).to(dtype)
        v = torch.randn(n, n_kv, hd, generator=g).to(dtype)
        if scale_one is not None and n > scale_one[0]:
            k[scale_one[0]] *= scale_one[1]                    # one far key that must stand out
        if shape_keys is not None:
            k = shape_keys(slot, k.float()).to(dtype)
        dense.append((k, v))
        for i in range(-(-n // page_size)):
            if gone_before is not None and (i + 1) * page_size <= gone_before.get(slot, 0):
                continue
            page = perm[nxt]; nxt += 1
            table[slot + 1, i] = page                          # slot 0 of the table stays unused (-1)
            cache[page] = 0
            m = min(page_size, n - i * page_size)
            cache[page, 0, :, :m, :] = k[i * page_size:i * page_size + m].permute(1, 0, 2)
            cache[page, 1].view(n_kv, hd, page_size)[:, :, :m] = v[i * page_size:i * page_size + m].permute(1, 2, 0)
    return cache.to(DEV), table.to(DEV), dense


def plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, window):
    """rows: (slot, pos) per row of q [n, heads*hd]; float64 softmax(q k / sqrt(hd)) v over keys <= pos."""
    out = torch.zeros(q.shape[0], n_heads, hd, dtype=torch.float64)
    qd = q.double().cpu().view(-1, n_heads, hd)
    for i, (slot, pos) in enumerate(rows):
        k, v = dense[slot]
        lo = max(0, pos - window + 1) if window else 0
        for h in range(n_heads):
            kv = h // (n_heads // n_kv)
            s = (k[lo:pos + 1, kv].double() @ qd[i, h]) / math.sqrt(hd)
            out[i, h] = torch.softmax(s, 0) @ v[lo:pos + 1, kv].double()
    return out.view(q.shape[0], n_heads * hd)


ATT_CASES = [  # n_heads, n_kv, hd, page_size, window
    (4, 2, 64, 16, None), (3, 1, 32, 16, None), (8, 8, 128, 32, None), (6, 2, 96, 16, None), (4, 4, 64, 16, 40), (32, 8, 64, 16, None),
    (5, 5, 48, 16, None), (2, 1, 16, 4, 9), (4, 2, 256, 16, None), (8, 2, 128, 16, 50), (6, 3, 128, 48, None),
]


SEGMENTS = {
    # request 0: rows at positions 150..299 (a portion on top of 150 cached positions); request 1: its last row;
    # request 2: its only row; request 3: rows 0..76 (a whole prompt); request 4: its last row
    "long portions": [(0, 150, 150), (1, 130, 1), (2, 0, 1), (3, 0, 77), (4, 529, 1)],
    # short portions, 60 rows in all: the matrix-core path takes them row by row through the decode kernel
    "short portions": [(0, 250, 50), (1, 130, 1), (2, 0, 1), (3, 70, 7), (4, 527, 3)],
    # short portions that sum to more than 64 rows stay tiles
    "many short portions": [(0, 240, 60), (1, 130, 1), (3, 47, 30), (4, 490, 40)],
    # portions of several tiles: a late tile shares its workgroup with an early one (3 tiles: the middle one alone; 4: two pairs)
    "several tiles": [(0, 0, 300), (1, 130, 1), (4, 100, 430)],
}


@pytest.mark.parametrize("n_heads,n_kv,hd,ps,window", ATT_CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("portions,tile", [(name, 0) for name in SEGMENTS] + [("long portions", 128), ("several tiles", 128)])
def test_attention_over_pages(n_heads, n_kv, hd, ps, window, dtype, portions, tile, monkeypatch):
    """Portions of prompts on top of an existing cache, beside single decoded rows, on scrambled pages.
    tile: rows of a prompt tile (0: as the step's size decides, which is 64 for steps as small as these)."""
    from geneinfer_amd.parts import StepContext
    monkeypatch.setattr(ops().AttentionPlan, "TILE", tile)
    contexts = [300, 131, 1, 77, 530]
    segs = SEGMENTS[portions]
    # with a window, the pages that no row of the step can see have been given back
    gone = {slot: max(0, pos0 - window + 1) for slot, pos0, _ in segs} if window else None
    cache, table, dense = build_paged(contexts, n_kv, hd, ps, dtype, seed=hd + n_heads, gone_before=gone)
    if window:
        assert int((table[1:] == -1).sum()) > int((build_paged(contexts, n_kv, hd, ps, dtype, seed=hd + n_heads)[1][1:] == -1).sum())
    rows, seg_start, seg_len, seg_pos0, seg_slot = [], [], [], [], []
    for slot, pos0, n in segs:
        seg_start.append(len(rows)); seg_len.append(n); seg_pos0.append(pos0); seg_slot.append(slot + 1)
        rows += [(slot, pos0 + i) for i in range(n)]
    T = len(rows)
    q = randn(T, n_heads * hd, dtype=dtype, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s + 1 for s, _ in rows], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=dtype, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=seg_slot,
                      seg_start=seg_start, seg_len=seg_len, seg_pos0=seg_pos0)
    out = torch.full((T, n_heads * hd), float("nan"), dtype=dtype, device=DEV)
    before = cache.clone()
    ops().attention(q, cache, out, ctx, table, n_heads, n_kv, hd, window)
    want = plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, window)
    err = rel(out, want)
    assert err < (2e-6 if dtype == torch.float32 else 8e-3), err
    assert torch.equal(torch.nan_to_num(cache, nan=-1.0), torch.nan_to_num(before, nan=-1.0)), "attention wrote into the cache"


@pytest.mark.parametrize("n_heads,n_kv,hd,ps,window", [(4, 2, 64, 16, None), (3, 1, 32, 16, None), (8, 8, 128, 32, None), (6, 2, 96, 16, 700), (4, 4, 64, 16, 450),
                                                       (4, 1, 128, 16, 600)])
def test_few_prompt_tiles_over_a_long_context_share_their_keys_out(n_heads, n_kv, hd, ps, window):
    """Two portions on top of long cached contexts: few tiles, so each tile's keys go to several workgroups and a combine
    kernel; among the keys one far one is scaled so that a lost share would show."""
    from geneinfer_amd.parts import StepContext
    o = ops()
    contexts = [1500, 730, 40]
    segs = [(0, 1400, 100), (1, 600, 130), (2, 39, 1)]
    gone = {slot: max(0, pos0 - window + 1) for slot, pos0, _ in segs} if window else None          # what a window has given back
    cache, table, dense = build_paged(contexts, n_kv, hd, ps, torch.bfloat16, seed=hd + n_heads + 7, scale_one=(333, 3.0), gone_before=gone)
    rows, seg_start, seg_len, seg_pos0, seg_slot = [], [], [], [], []
    for slot, pos0, n in segs:
        seg_start.append(len(rows)); seg_len.append(n); seg_pos0.append(pos0); seg_slot.append(slot + 1)
        rows += [(slot, pos0 + i) for i in range(n)]
    T = len(rows)
    q = randn(T, n_heads * hd, dtype=torch.bfloat16, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s_ + 1 for s_, _ in rows], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=seg_slot,
                      seg_start=seg_start, seg_len=seg_len, seg_pos0=seg_pos0)
    assert o.prompt_attention_splits(3, n_heads, 1500 if not window else window + 128) > 1
    out = torch.full((T, n_heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    o.attention(q, cache, out, ctx, table, n_heads, n_kv, hd, window)
    want = plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, window)
    assert rel(out, want) < 8e-3, rel(out, want)


@pytest.mark.parametrize("n_single, portion, n_heads, n_kv, hd, window", [(40, 0, 16, 8, 64, None), (65, 0, 8, 4, 128, 100), (33, 90, 32, 8, 128, None), (200, 80, 4, 2, 64, None), (17, 0, 64, 16, 64, None)])
def test_decoded_rows_of_unequal_contexts_dealt_out_over_the_chip(n_single, portion, n_heads, n_kv, hd, window):
    """More workgroups than compute units: the single rows are taken longest context first, there and back.  Each row's result is what it is in the step's own
    order (where neither cuts a context), and the right one; a prompt's portion in the middle makes the single rows a list."""
    from geneinfer_amd.parts import StepContext
    g = torch.Generator().manual_seed(n_single)
    contexts = [int(c) for c in torch.randint(1, 700, (n_single,), generator=g)]
    contexts[3] = contexts[7] = 700
    if portion:
        contexts.insert(n_single // 2, 200 + portion)
    cache, table, dense = build_paged(contexts, n_kv, hd, 16, torch.bfloat16, seed=5)
    rows, seg_start, seg_len, seg_pos0, seg_slot = [], [], [], [], []
    for slot, c in enumerate(contexts):
        n = portion if portion and slot == n_single // 2 else 1
        seg_start.append(len(rows)); seg_len.append(n); seg_pos0.append(c - n); seg_slot.append(slot + 1)
        rows += [(slot, c - n + i) for i in range(n)]
    T = len(rows)
    q = randn(T, n_heads * hd, dtype=torch.bfloat16, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s_ + 1 for s_, _ in rows], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=seg_slot,
                      seg_start=seg_start, seg_len=seg_len, seg_pos0=seg_pos0)
    out = torch.full((T, n_heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops().attention(q, cache, out, ctx, table, n_heads, n_kv, hd, window)
    want = plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, window)
    assert rel(out, want) < 8e-3, rel(out, want)
    order = ctx.memo["decode_order"].tolist()
    single = [i for i, (slot, _) in enumerate(rows) if not (portion and slot == n_single // 2)]
    assert order == sorted(single, key=lambda i: (-rows[i][1], i))
    plan = ops().AttentionPlan(seg_start, seg_len, seg_pos0, seg_slot, DEV)
    assert plan.decode_positions == sum(rows[i][1] + 1 for i in single)
    plan.decode_positions = None
    both = []
    for memo in ({}, None):
        both.append(torch.full_like(out, float("nan")))
        ops().attention_bf16(q, cache, both[-1], plan, pos, slots, table, n_heads, n_kv, hd, window, memo=memo)
    assert torch.equal(*both)


@pytest.mark.parametrize("n_single, n_heads, n_kv, hd, splits", [(24, 24, 8, 128, 3), (38, 32, 4, 64, 4)])
def test_ordered_rows_whose_contexts_are_cut(n_single, n_heads, n_kv, hd, splits):
    """Single rows at 500 to 3,000 positions beside a prompt's portion: taken longest context first, and each context cut.  The pieces are kept by the place in that
    order and come back to their rows."""
    from geneinfer_amd.parts import StepContext
    o = ops()
    g = torch.Generator().manual_seed(n_single)
    contexts = [int(c) for c in torch.randint(500, 1700, (n_single,), generator=g)]
    contexts[5], contexts[n_single - 2] = 3000, 2900
    contexts.insert(n_single // 2, 300)                        # a portion of 100 rows in the middle
    cache, table, dense = build_paged(contexts, n_kv, hd, 16, torch.bfloat16, seed=5, scale_one=(2000, 3.0))
    rows, seg_start, seg_len, seg_pos0, seg_slot = [], [], [], [], []
    for slot, c in enumerate(contexts):
        n = 100 if slot == n_single // 2 else 1
        seg_start.append(len(rows)); seg_len.append(n); seg_pos0.append(c - n); seg_slot.append(slot + 1)
        rows += [(slot, c - n + i) for i in range(n)]
    T = len(rows)
    q = randn(T, n_heads * hd, dtype=torch.bfloat16, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s_ + 1 for s_, _ in rows], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=seg_slot,
                      seg_start=seg_start, seg_len=seg_len, seg_pos0=seg_pos0)
    plan = o._plan_of(ctx)
    assert o.decode_attention_shape(n_single, n_heads, n_kv, hd, 3000)[0] == 1
    assert o._decode_ragged_split(n_single * n_kv, 3000, plan.decode_positions / n_single, hd, 8)[0] == splits
    out = torch.full((T, n_heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    o.attention(q, cache, out, ctx, table, n_heads, n_kv, hd)
    assert "decode_order" in ctx.memo
    want = plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, None)
    worst = float(((out.double().cpu() - want).norm(dim=1) / want.norm(dim=1)).max())
    assert rel(out, want) < 8e-3 and worst < 3e-2, (rel(out, want), worst)


@pytest.mark.parametrize("n_heads", [32, 24])
def test_ordered_rows_in_the_kernel_that_rotates_and_stores(n_heads):
    """The rows of a decode step whose contexts are cut and whose workgroups are more than the compute units: each still writes its own key and value, once."""
    from geneinfer_amd.parts import StepContext
    o = ops()
    n, longest, n_kv, hd = 17, 4096, 8, 64
    g = torch.Generator().manual_seed(n_heads)
    contexts = [int(c) for c in torch.randint(2, longest, (n,), generator=g)]
    contexts[3] = longest
    cache, table, dense = build_paged(contexts, n_kv, hd, 16, torch.bfloat16, seed=5)
    a, kv = n_heads * hd, n_kv * hd
    pos = torch.tensor([c - 1 for c in contexts], dtype=torch.int32, device=DEV)
    slots = torch.arange(1, n + 1, dtype=torch.int32, device=DEV)
    qkv = randn(n, a + 2 * kv, seed=31)
    inv = torch.tensor([1.0 / (10000.0 ** (2 * k / hd)) for k in range(hd // 2)], dtype=torch.float64, device=DEV)
    cos, sin = torch.empty(n, hd // 2, device=DEV), torch.empty(n, hd // 2, device=DEV)
    o.rope_cos_sin(pos, inv, cos, sin)
    want_cache, q_rot = cache.clone(), torch.empty(n, a, dtype=torch.bfloat16, device=DEV)
    o.rope_store(qkv[:, :a], qkv[:, a:a + kv], qkv[:, a + kv:], cos, sin, pos, slots, table, q_rot, want_cache, n_heads, n_kv, hd)
    for i, c in enumerate(contexts):
        page, place = int(table[i + 1, (c - 1) // 16]), (c - 1) % 16
        dense[i][0][c - 1], dense[i][1][c - 1] = want_cache[page, 0, :, place].cpu(), want_cache[page, 1].view(n_kv, hd, 16)[:, :, place].cpu()
    ctx = StepContext(n_rows=n, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=list(range(1, n + 1)), seg_start=list(range(n)),
                      seg_len=[1] * n, seg_pos0=[c - 1 for c in contexts])
    splits = o.decode_attention_shape(n, n_heads, n_kv, hd, longest, fused=True)[0]
    assert splits > 1 and n * n_kv * splits > o.lib().gi_compute_units()
    out = torch.full((n, a), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert o.attention_from_products(qkv[:, :a], qkv[:, a:a + kv], qkv[:, a + kv:], cos, sin, cache, out, ctx, table, n_heads, n_kv, hd) and "decode_order" in ctx.memo
    got, kept = torch.nan_to_num(cache.float(), nan=-1.0), torch.nan_to_num(want_cache.float(), nan=-1.0)
    assert rel(got, kept) < 1e-3 and float(((got - kept).abs() > 0.02 * kept.abs() + 1e-6).sum()) == 0           # (a rotated key may round the other way in 32-bit)
    want = plain_attention_rows(q_rot, dense, [(i, c - 1) for i, c in enumerate(contexts)], n_heads, n_kv, hd, None)
    assert rel(out, want) < 8e-3


@pytest.mark.parametrize("window", [None, 200])
def test_many_prompt_tiles_of_many_heads(window):
    """More workgroups than compute units at head size 64 (5 pairs of tiles x 64 heads): the step takes the kernel with a
    workgroup per tile, several to a compute unit, which head size 128 always takes.  A whole prompt of 900 rows, a portion of
    130 rows on 300 cached positions and a single row; with a window the pages behind it are gone."""
    from geneinfer_amd.parts import StepContext
    n_heads, n_kv, hd, ps = 64, 16, 64, 16
    contexts = [900, 430, 50]
    segs = [(0, 0, 900), (1, 300, 130), (2, 49, 1)]
    gone = {slot: max(0, pos0 - window + 1) for slot, pos0, _ in segs} if window else None
    cache, table, dense = build_paged(contexts, n_kv, hd, ps, torch.bfloat16, seed=5, scale_one=(77, 3.0), gone_before=gone)
    rows, seg_start, seg_len, seg_pos0, seg_slot = [], [], [], [], []
    for slot, pos0, n in segs:
        seg_start.append(len(rows)); seg_len.append(n); seg_pos0.append(pos0); seg_slot.append(slot + 1)
        rows += [(slot, pos0 + i) for i in range(n)]
    T = len(rows)
    q = randn(T, n_heads * hd, dtype=torch.bfloat16, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s_ + 1 for s_, _ in rows], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=seg_slot,
                      seg_start=seg_start, seg_len=seg_len, seg_pos0=seg_pos0)
    plan = ops().AttentionPlan(seg_start, seg_len, seg_pos0, seg_slot, DEV)
    assert plan.paired and plan.tile == 128 and plan.n_tiles // 2 * n_heads > 256
    out = torch.full((T, n_heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops().attention(q, cache, out, ctx, table, n_heads, n_kv, hd, window)
    want = plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, window)
    assert rel(out, want) < 8e-3, rel(out, want)


@pytest.mark.parametrize("n_heads,n_kv,hd,segs,window,known", [
    (24, 8, 128, [(0, 1020, 1350), (1, 0, 674), (2, 49, 1)], None, "3"), (32, 8, 128, [(0, 0, 1000)], None, "2"), (16, 8, 128, [(0, 4000, 260), (1, 0, 1900)], None, "4"), (24, 8, 128, [(0, 1020, 1350), (1, 0, 674)], None, "sinks"),
    (24, 8, 128, [(0, 1020, 1350), (1, 0, 674)], None, "cap"), (64, 16, 64, [(0, 3000, 900), (1, 0, 401)], None, "3"), (64, 16, 64, [(0, 3000, 130), (1, 0, 960)], 2000, "2"),
    (32, 8, 64, [(0, 0, 1500)], None, "3"), (32, 8, 64, [(0, 0, 1777)], 1024, "3"), (32, 8, 64, [(0, 1300, 300), (1, 0, 200)], None, "3")])
def test_long_walks_of_prompt_tiles_share_their_keys_out(n_heads, n_kv, hd, segs, window, known):
    """Portions far behind others whose tiles fill the chip all the same: the tiles with long walks are made by several workgroups that meet in the kernel.
    Against 64 bits where that is stated plainly, against one workgroup a tile, and in bits against themselves, whoever came last."""
    o = ops()
    contexts = [pos0 + n for _, pos0, n in segs]
    cache, table, dense = build_paged(contexts, n_kv, hd, 16, torch.bfloat16, seed=5, scale_one=(77, 3.0))
    rows = [(slot, pos0 + i) for slot, pos0, n in segs for i in range(n)]
    starts = [sum(n for _, _, n in segs[:i]) for i in range(len(segs))]
    plan = o.AttentionPlan(starts, [n for _, _, n in segs], [p for _, p, _ in segs], [s_ + 1 for s_, _, _ in segs], DEV)
    most, keys = o.prompt_attention_shares([min(c, (window or c) + plan.tile) for c in plan.tile_contexts], n_heads, hd, plan.tile,
                                           plan.n_tiles // 2 * n_heads <= o.lib().gi_compute_units())
    assert plan.n_tiles and most > 1 and (known not in "234" or most == int(known)), (most, keys)
    q = randn(len(rows), n_heads * hd, dtype=torch.bfloat16, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s_ + 1 for s_, _ in rows], dtype=torch.int32, device=DEV)
    extras = dict(sinks=randn(n_heads, seed=9)) if known == "sinks" else dict(cap=20.0) if known == "cap" else {}
    seen, memo = [], {}
    for m in (memo, memo, {}, None):
        seen.append(torch.full((len(rows), n_heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV))
        o.attention_bf16(q, cache, seen[-1], plan, pos, slots, table, n_heads, n_kv, hd, window, memo=m, **extras)
    assert torch.equal(seen[0], seen[1]) and torch.equal(seen[0], seen[2]) and not bool(memo["attention_counters"].any())
    # (the probabilities are rounded to bfloat16 about another maximum, 2^-9 of each at most on either side, and the results, 2^-8 between the two)
    assert rel(seen[0], seen[3]) < 2 * 2.0 ** -9 + 2.0 ** -8, rel(seen[0], seen[3])
    if not extras:
        assert rel(seen[0], plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, window)) < 8e-3


@pytest.mark.parametrize("n_heads,n_kv,hd,ps,portions,singles,splits,window,extra", [
    # walks in shares; one more single row than a workgroup of eight fills, contexts of 1 and 33; pages of 16, 32 and 48; several splits; a window and chunks; more workgroups of either kind
    (24, 8, 128, 16, [(1020, 1350), (0, 674)], [1, 33, 700, 2990] * 6, 1, None, None), (24, 8, 128, 32, [(500, 600)], [900, 64, 31], 2, None, None),
    (32, 8, 64, 16, [(0, 1500)], [1, 1200, 16, 17, 500], 1, None, None), (64, 16, 64, 48, [(3000, 900), (0, 401)], [2000] * 9, 3, None, None), (64, 16, 64, 16, [(300, 1200)], [900, 30, 1700], 2, 200, None),
    (20, 1, 128, 16, [(0, 300)], [40, 999, 1], 1, None, None), (40, 2, 128, 16, [(100, 800)], [640, 65], 3, None, None), (4, 4, 128, 48, [(1400, 100), (600, 130)], [300, 800], 1, 450, None),
    (4, 1, 128, 16, [(0, 200)], [500] * 70, 4, None, None), (16, 8, 128, 16, [(640, 900)], [300, 129, 128, 1], 1, None, "chunk"), (16, 8, 128, 16, [(0, 900)], [300, 129], 2, None, "sinks"),
    (24, 8, 128, 16, [(0, 700)], [800, 2], 2, None, "gate"), (32, 8, 64, 16, [(0, 1500)], [600, 3], 2, None, "channels"),
    # short portions, which go row by row among the single rows: several rows of one request in the list
    (24, 8, 128, 16, [(1020, 900), (700, 30)], [1, 2990, 64], 1, None, None), (32, 8, 64, 16, [(0, 1500), (33, 2), (900, 17)], [600] * 5, 2, None, None), (40, 2, 128, 32, [(100, 800), (0, 40)], [640], 1, 300, None)])
def test_single_rows_and_tiles_in_one_launch(n_heads, n_kv, hd, ps, portions, singles, splits, window, extra, monkeypatch):
    """A step's single rows beside portions of prompts: the tiles' rows are in bits those of a launch of their own, the single rows those of another cut of their contexts; every time the
    same bits; and without room for shares."""
    o = ops()
    segs = [(c - 1, 1) for c in singles[:len(singles) // 2]] + portions + [(c - 1, 1) for c in singles[len(singles) // 2:]]
    contexts = [p + n for p, n in segs]
    gone = {s: max(0, p - window + 1) for s, (p, _) in enumerate(segs)} if window else None
    cache, table, dense = build_paged(contexts, n_kv, hd, ps, torch.bfloat16, seed=5, scale_one=(0, 2.0), gone_before=gone)
    rows = [(s, p + i) for s, (p, n) in enumerate(segs) for i in range(n)]
    starts = [sum(n for _, n in segs[:i]) for i in range(len(segs))]
    q = randn(len(rows), n_heads * hd, dtype=torch.bfloat16, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s + 1 for s, _ in rows], dtype=torch.int32, device=DEV)
    extras = {None: {}, "chunk": dict(chunk=128), "sinks": dict(sinks=randn(n_heads, seed=9)), "gate": dict(gate=randn(len(rows), n_heads, seed=9)),
              "channels": dict(channel_gate=randn(len(rows), n_heads * hd, seed=9))}[extra]
    asked, call = [], o._call
    monkeypatch.setattr(o, "_call", lambda name, *a: (asked.append(name), call(name, *a))[1])
    monkeypatch.setattr(o, "_both_splits", lambda *a: splits)

    def made(together, memo):
        plan = o.AttentionPlan(starts, [n for _, n in segs], [p for p, _ in segs], [s + 1 for s in range(len(segs))], DEV)
        out = torch.full((len(rows), n_heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        return o.attention_bf16(q, cache, out, plan, pos, slots, table, n_heads, n_kv, hd, window, memo=memo, together=together, **extras)

    before, memo = cache.clone(), {}
    apart, got, again = made(False, {}), made(True, memo), made(True, memo)
    assert asked.count("gi_attention_both_bf16") == 2 and asked.count("gi_attention_prompt_bf16") == 1
    single = torch.tensor([s + i for s, (_, n) in zip(starts, segs) if n <= 64 for i in range(n)], device=DEV)
    tiles = torch.ones(len(rows), dtype=torch.bool, device=DEV).index_fill_(0, single, False)
    assert torch.equal(got, again) and torch.equal(got[tiles], apart[tiles])
    # (probabilities are rounded to bfloat16 about other maxima, 2^-9 of each at most on either side, and the results, 2^-8 between the two)
    assert rel(got[single], apart[single]) < 2 * 2.0 ** -9 + 2.0 ** -8
    if extra is None:
        assert rel(got, plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, window)) < 8e-3
    assert torch.equal(torch.nan_to_num(cache, nan=-1.0), torch.nan_to_num(before, nan=-1.0)) and ("attention_counters" not in memo or not bool(memo["attention_counters"].any()))
    monkeypatch.setattr(o, "_room", lambda *_: None)
    asked.clear()
    without = made(True, {})
    assert rel(without, got) < 2 * 2.0 ** -9 + 2.0 ** -8 and len(asked) <= 3


def test_workgroups_that_meet_in_a_kernel_under_capture():
    """A product with shared tiles and an attention with shared walks in one captured pass, whose counters are filled in the pass: every replay gives the bits of
    the same calls made one by one, with other work and a synchronization between."""
    from types import SimpleNamespace
    o = ops()
    m, n_heads, n_kv, hd = 1000, 32, 8, 128
    width = n_heads * hd
    cache, table, _ = build_paged([m], n_kv, hd, 16, torch.bfloat16, seed=5)
    plan = o.AttentionPlan([0], [m], [0], [1], DEV)
    assert o.prompt_attention_shares(plan.tile_contexts, n_heads, hd)[0] > 1 and o.gemm_bf16_tall_shares(2 * m, width // 2, 2 * width) == 2
    pos, slots = torch.arange(m, dtype=torch.int32, device=DEV), torch.ones(m, dtype=torch.int32, device=DEV)
    q, a, w = randn(m, width, dtype=torch.bfloat16, seed=3), randn(2 * m, 2 * width, dtype=torch.bfloat16, seed=4), randn(width // 2, 2 * width, dtype=torch.bfloat16, seed=6)
    att, out = torch.empty(m, width, dtype=torch.bfloat16, device=DEV), torch.empty(2 * m, width // 2, device=DEV)

    def step():
        ctx = SimpleNamespace(memo={}, device=torch.device(DEV))
        for _ in range(2):
            o.attention_bf16(q, cache, att, plan, pos, slots, table, n_heads, n_kv, hd, memo=ctx.memo)
            o.gemm_bf16(a, w, out, counters=o.step_counters(ctx, 2 * m, *w.shape))

    step()
    want = att.clone(), out.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(4):
        att.fill_(7), out.fill_(7)
        graph.replay()
        assert torch.equal(att, want[0]) and torch.equal(out, want[1])
        torch.cuda.synchronize()
        o.gemm_bf16(a, w, torch.empty_like(out))


def test_workgroups_that_meet_on_two_streams_at_once():
    """Two steps side by side, each with counters of its own, and products that clear their own: every result has the bits it has alone."""
    from types import SimpleNamespace
    o = ops()
    m, n_heads, n_kv, hd, rows, n, k = 1000, 32, 8, 128, 2048, 2048, 8192
    cache, table, _ = build_paged([m], n_kv, hd, 16, torch.bfloat16, seed=5)
    plan = o.AttentionPlan([0], [m], [0], [1], DEV)
    pos, slots = torch.arange(m, dtype=torch.int32, device=DEV), torch.ones(m, dtype=torch.int32, device=DEV)
    q, a, w = randn(m, n_heads * hd, dtype=torch.bfloat16, seed=3), randn(rows, k, dtype=torch.bfloat16, seed=4), randn(n, k, dtype=torch.bfloat16, seed=6)
    assert o._shares(rows, n, k, 0, False) == o._shares(rows, n, k, 0, True) == 2

    def step(times):
        ctx, got = SimpleNamespace(memo={}, device=torch.device(DEV)), []
        for _ in range(times):
            got.append(o.attention_bf16(q, cache, torch.empty_like(q), plan, pos, slots, table, n_heads, n_kv, hd, memo=ctx.memo))
            got.append(o.gemm_bf16(a, w, torch.empty(rows, n, device=DEV), counters=o.step_counters(ctx, rows, n, k)))
            got.append(o.gemm_bf16(a, w, torch.empty(rows, n, device=DEV)))
        return got

    want = step(1)
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream(), torch.cuda.Stream()], []
    for stream in streams:
        with torch.cuda.stream(stream):
            got.append(step(6))
    torch.cuda.synchronize()
    for results in got:
        assert all(torch.equal(x, want[i % 3]) for i, x in enumerate(results))


@pytest.mark.parametrize("m", [33, 131])
def test_a_product_without_room_for_strips_is_made_beside_them(m, monkeypatch):
    """A device that has no room for the sums of strips' shares of k (five here): those of the kernels before them (four) are enough."""
    o, n, k = ops(), 3072, 8192
    a, w = randn(m, k, dtype=torch.bfloat16, seed=1), randn(n, k, dtype=torch.bfloat16, seed=2, scale=0.1)
    strips, out, asked = o.gemm_bf16(a, w, torch.empty(m, n, device=DEV)), torch.full((m + 1, n), 3.0, device=DEV), []
    monkeypatch.setattr(o, "_room", lambda floats, device: asked.append(floats))
    o.gemm_bf16(a, w, out[:m])
    want = a.double() @ w.double().T
    assert asked == [5 * m * n] and o.lib().gi_gemm_bf16_least_scratch_floats(m, n, k) == 4 * m * n
    assert rel(out[:m], want) < 2e-6 and rel(strips, want) < 2e-6 and not torch.equal(out[:m], strips) and bool((out[m:] == 3.0).all())


@pytest.mark.parametrize("hd, m", [(128, 1000), (64, 1500)])
def test_without_room_for_scratch_nothing_is_shared_out(hd, m, monkeypatch):
    """A device that has no room for the sums of shared tiles and walks: the kernels that share nothing out serve, as without a step's memory of its own."""
    o = ops()
    n_heads, n_kv, rows, n, k = 32, 8, 2048, 2048, 8192
    cache, table, _ = build_paged([m], n_kv, hd, 16, torch.bfloat16, seed=5)
    plan = o.AttentionPlan([0], [m], [0], [1], DEV)
    pos, slots = torch.arange(m, dtype=torch.int32, device=DEV), torch.ones(m, dtype=torch.int32, device=DEV)
    q, a, w = randn(m, n_heads * hd, dtype=torch.bfloat16, seed=3), randn(rows, k, dtype=torch.bfloat16, seed=4), randn(n, k, dtype=torch.bfloat16, seed=6)

    def attend(memo):
        return o.attention_bf16(q, cache, torch.empty_like(q), plan, pos, slots, table, n_heads, n_kv, hd, memo=memo)

    alone, memo = attend(None), {}
    shared, product = attend(memo), o.gemm_bf16(a, w, torch.empty(rows, n, device=DEV))
    assert "attention_counters" in memo and o._shares(rows, n, k, 0, False) == 2
    asked = []
    monkeypatch.setattr(o, "_room", lambda floats, device: asked.append(4 * floats))
    memo = {}
    assert torch.equal(attend(memo), alone) and not torch.equal(shared, alone) and "attention_counters" not in memo
    whole = o.gemm_bf16(a, w, torch.empty(rows, n, device=DEV))
    assert rel(whole, a.double() @ w.double().T) < 1e-5 and not torch.equal(whole, product)
    # 68 KB (heads of 128 channels; 36) for every share of every tile and head, 128 KB for every share of a product's tile
    assert asked == [plan.n_tiles * n_heads * {128: 2 * 69632, 64: 3 * 36864}[hd], 4 * (512 + 128 * 2 * 32768)]


def test_a_meeting_of_workgroups_ends_whatever_its_counters_held():
    """Counters that were not 0 (a workgroup has been counted that never comes): the launch ends, the results that are not whole are no numbers, all others are right,
    and the counters are 0 again."""
    o = ops()
    m, n, k = 2048, 2048, 8192                                # 128 tiles of 256 x 128, each in two shares; a tile's counters: {drawn, raised} of its upper half, of its lower half
    a, w = randn(m, k, dtype=torch.bfloat16, seed=4), randn(n, k, dtype=torch.bfloat16, seed=6)
    counters = torch.zeros(o.lib().gi_gemm_bf16_counters(), dtype=torch.int32, device=DEV)
    right = o.gemm_bf16(a, w, torch.empty(m, n, device=DEV), counters=counters)
    assert o.gemm_bf16_tall_shares(m, n, k) == 2 and bool(torch.isfinite(right).all())
    counters[4 * 5 + 2] = 1                                   # the sixth tile's lower half
    hurt = o.gemm_bf16(a, w, torch.empty(m, n, device=DEV), counters=counters)
    bad = torch.isnan(hurt)
    rows, columns = bad.any(1).nonzero().flatten(), bad.any(0).nonzero().flatten()
    assert rows.numel() == columns.numel() == 128 and int(rows[0]) % 256 == 128 and int(columns[0]) % 128 == 0 and int(bad.sum()) == 128 * 128
    assert torch.equal(hurt[~bad], right[~bad]) and not bool(counters.any())
    m, n_heads, n_kv, hd = 1000, 32, 8, 128
    cache, table, _ = build_paged([m], n_kv, hd, 16, torch.bfloat16, seed=5)
    plan = o.AttentionPlan([0], [m], [0], [1], DEV)
    pos, slots = torch.arange(m, dtype=torch.int32, device=DEV), torch.ones(m, dtype=torch.int32, device=DEV)
    q, memo = randn(m, n_heads * hd, dtype=torch.bfloat16, seed=3), {}

    def attend():
        return o.attention_bf16(q, cache, torch.empty_like(q), plan, pos, slots, table, n_heads, n_kv, hd, memo=memo)

    right = attend()
    late = plan.tiles.view(-1, 4)[:, 0].argmax().item()       # the tile of the last rows: two shares
    memo["attention_counters"][2 * (late * n_heads + 7)] = 1
    hurt = attend()
    bad = torch.isnan(hurt).view(m, n_heads, hd)
    assert bool(bad[896:, 7].all()) and int(bad.sum()) == (m - 896) * hd and torch.equal(hurt[~bad.view(m, -1)], right[~bad.view(m, -1)])
    assert not bool(memo["attention_counters"].any()) and torch.equal(attend(), right)


@pytest.mark.parametrize("n_heads,n_kv,hd", [(4, 2, 64), (4, 2, 128), (64, 16, 64)])
def test_prompt_attention_with_scores_that_climb_along_the_context(n_heads, n_kv, hd):
    """Every query points along one direction and the keys' share of that direction climbs with their position, by 2 to 12
    units of log2 e from one tile of 64 keys to the next, and falls again behind position 800: the running maximum of a
    row moves in every tile, by less and by more than what the kernels let it lag behind.  Scores reach 60 and more, so a
    maximum applied wrongly once is a factor and not a rounding error.  A whole prompt of several tiles, a portion on a
    cached context and a single row (in the last case: more workgroups than compute units, the other prompt kernel)."""
    from geneinfer_amd.parts import StepContext
    ps = 16
    contexts = [1200, 900, 50]
    segs = [(0, 0, 1200), (1, 700, 200), (2, 49, 1)]
    g = torch.Generator().manual_seed(11)
    direction = torch.nn.functional.normalize(torch.randn(n_kv, hd, generator=g), dim=-1)
    pos_all = torch.arange(1200, dtype=torch.float32)
    # slope per position in nats of the final score: gentle, then steep, then falling
    slope = torch.where(pos_all < 300, 0.02, torch.where(pos_all < 800, 0.13, -0.09))
    height = torch.cumsum(slope, 0)                                        # the score a unit query gives the key at a position
    q_gain = 3.0

    def shape_keys(slot, k):
        n = k.shape[0]
        return 0.3 * k + (height[:n] * math.sqrt(hd) / q_gain)[:, None, None] * direction[None]

    cache, table, dense = build_paged(contexts, n_kv, hd, ps, torch.bfloat16, seed=hd + 2, shape_keys=shape_keys)
    rows, seg_start, seg_len, seg_pos0, seg_slot = [], [], [], [], []
    for slot, pos0, n in segs:
        seg_start.append(len(rows)); seg_len.append(n); seg_pos0.append(pos0); seg_slot.append(slot + 1)
        rows += [(slot, pos0 + i) for i in range(n)]
    T = len(rows)
    q = (q_gain * direction.repeat_interleave(n_heads // n_kv, 0).reshape(1, n_heads * hd) + 0.3 * torch.randn(T, n_heads * hd, generator=g)).to(torch.bfloat16).to(DEV)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s_ + 1 for s_, _ in rows], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=seg_slot,
                      seg_start=seg_start, seg_len=seg_len, seg_pos0=seg_pos0)
    out = torch.full((T, n_heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops().attention(q, cache, out, ctx, table, n_heads, n_kv, hd, None)
    k0 = dense[0][0]
    top = float((k0[:, 0].double() @ q[0].double().cpu().view(n_heads, hd)[0]).max() / math.sqrt(hd))
    assert top > 40, top                                                   # the scores do climb as meant
    want = plain_attention_rows(q, dense, rows, n_heads, n_kv, hd, None)
    assert rel(out, want) < 8e-3, rel(out, want)
    worst_row = float(((out.double().cpu() - want).norm(dim=1) / want.norm(dim=1)).max())
    assert worst_row < 3e-2, worst_row                                     # no row is off by a factor


@pytest.mark.parametrize("n_heads,n_kv,hd,ps,window,chunk", [(4, 2, 64, 16, None, None), (6, 2, 128, 12, None, None), (40, 2, 32, 4, None, None), (3, 3, 96, 16, 300, None),
                                                             (8, 1, 16, 20, None, 320), (32, 8, 64, 16, 256, None)])
def test_attention_exact_has_one_order_of_sums(n_heads, n_kv, hd, ps, window, chunk):
    """32-bit: tiles of several rows, of one row, contexts shared out over workgroups or not, rows alone: equal in bits; at contexts around
    the blocks of 64 keys and spans of 256.  A value that is no number is met only by the rows that see its position."""
    contexts = [1025, 256, 64, 513]
    cache, table, dense = build_paged(contexts, n_kv, hd, ps, torch.float32, seed=hd + n_heads)
    segs = [(0, 1018, 7), (1, 255, 1), (2, 0, 64), (3, 510, 3), (0, 766, 3)]
    rows = [(slot, pos0 + i) for slot, pos0, n in segs for i in range(n)]
    T = len(rows)
    q = randn(T, n_heads * hd, seed=3)
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s_ + 1 for s_, _ in rows], dtype=torch.int32, device=DEV)

    def attend(pick=slice(None), **known):
        out = torch.full((T, n_heads * hd), float("nan"), device=DEV)[pick]
        return ops().attention_exact(q[pick].contiguous(), cache, out, pos[pick].contiguous(), slots[pick].contiguous(), table, n_heads, n_kv, hd, window, chunk=chunk, **known)

    whole = attend()
    lows = [max(0, p - window + 1) if window else p - p % chunk if chunk else 0 for _, p in rows]
    want = torch.cat([plain_attention_rows(q[i:i + 1], {s_: (dense[s_][0][lo:], dense[s_][1][lo:])}, [(s_, p - lo)], n_heads, n_kv, hd, None)
                      for i, ((s_, p), lo) in enumerate(zip(rows, lows))])
    assert rel(whole, want) < 2e-6
    assert torch.equal(attend(max_context=1025), whole) and torch.equal(attend(max_context=4096), whole)
    assert torch.equal(attend(single_rows=True), whole) and torch.equal(attend(single_rows=True, max_context=1025), whole)
    for known in (dict(single_rows=5), dict(single_rows=8, n_requests=1), dict(single_rows=T - 1, n_requests=1, max_context=1025), dict(n_requests=2), dict(n_requests=5, max_context=1025)):
        assert torch.equal(attend(**known), whole), known
    for i in (0, 6, 7, 40, T - 4, T - 1):
        assert torch.equal(attend(slice(i, i + 1)), whole[i:i + 1]) and torch.equal(attend(slice(i, i + 1), max_context=2048), whole[i:i + 1])
    place = 1022                                             # of request 0, whose rows 1018 .. 1024 share tiles
    cache[int(table[1, place // ps]), 1].view(n_kv, hd, ps)[:, :, place % ps] = float("inf")
    for known in (dict(), dict(max_context=1025), dict(single_rows=True)):
        hurt = attend(**known)
        sees = torch.tensor([s_ == 0 and p >= place and lo <= place for (s_, p), lo in zip(rows, lows)], device=DEV)
        assert torch.equal(hurt[~sees], whole[~sees]) and not bool(torch.isfinite(hurt[sees]).any())


@pytest.mark.parametrize("window,chunk", [(1, None), (16, None), (17, None), (40, None), (None, 1), (None, 16), (None, 17), (None, 48)])
@pytest.mark.parametrize("n_heads,n_kv,hd,ps", [(4, 2, 64, 16), (3, 1, 128, 12)])
def test_attention_exact_with_few_keys(n_heads, n_kv, hd, ps, window, chunk):
    """32-bit: short contexts, and windows and chunks on both sides of the line between the two kernels: groups of 16 keys that no row of a tile sees, at
    all ends of blocks of 64 and spans of 256; the same bits whatever is known of the step, and alone."""
    contexts = [600, 70, 18, 1]
    cache, table, dense = build_paged(contexts, n_kv, hd, ps, torch.float32, seed=hd + n_heads)
    rows = [(3, 0)] + [(0, p) for p in (0, 14, 15, 16, 17, 47, 48, 63, 64, 65, 79, 255, 256, 257, 271, 272, 300, 511, 512, 599)] + [(1, p) for p in range(50, 70)] + [(2, p) for p in range(18)]
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s_ + 1 for s_, _ in rows], dtype=torch.int32, device=DEV)
    q = randn(len(rows), n_heads * hd, seed=3)

    def attend(pick=slice(None), **known):
        out = torch.full_like(q, float("nan"))[pick]
        return ops().attention_exact(q[pick].contiguous(), cache, out, pos[pick].contiguous(), slots[pick].contiguous(), table, n_heads, n_kv, hd, window, chunk=chunk, **known)

    lows = [max(0, p - window + 1) if window else p - p % chunk for _, p in rows]
    want = torch.cat([plain_attention_rows(q[i:i + 1], {s_: (dense[s_][0][lo:], dense[s_][1][lo:])}, [(s_, p - lo)], n_heads, n_kv, hd, None)
                      for i, ((s_, p), lo) in enumerate(zip(rows, lows))])
    whole = attend()
    assert rel(whole, want) < 2e-6
    for known in (dict(single_rows=21), dict(single_rows=True, max_context=600), dict(n_requests=4, max_context=600)):
        assert torch.equal(attend(**known), whole), known
    for i in (0, 4, 12, 20, 25, len(rows) - 1):
        assert torch.equal(attend(slice(i, i + 1)), whole[i:i + 1])


@pytest.mark.parametrize("sinks", [False, True])
@pytest.mark.parametrize("n_heads,n_kv,hd,ps,window", [(4, 2, 64, 16, None), (6, 1, 128, 4, None), (2, 2, 32, 16, 400)])
@pytest.mark.parametrize("known", [dict(), dict(max_context=770), dict(single_rows=True), dict(single_rows=True, max_context=770)], ids=["whole", "shared", "single", "single-shared"])
def test_attention_exact_hands_on_what_is_no_number(n_heads, n_kv, hd, ps, window, sinks, known):
    """32-bit: a query, a key or a value that is no number shows in every row that sees it and in no other, also where it is all that a row
    sees of a span of 256 keys (positions 256, 512, 768), with sinks that keep the denominator finite, and where its block's factor is zero."""
    contexts = [770, 300]
    cache, table, _ = build_paged(contexts, n_kv, hd, ps, torch.float32, seed=5)
    rows = [(0, p) for p in (0, 2, 3, 255, 256, 257, 300, 511, 512, 513, 767, 768, 769)] + [(1, p) for p in (256, 299)]
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    slots = torch.tensor([r + 1 for r, _ in rows], dtype=torch.int32, device=DEV)
    one = randn(hd, seed=7)
    q = one.repeat(len(rows), n_heads).contiguous()
    s = randn(n_heads, seed=8) if sinks else None

    def attend():
        out = torch.full_like(q, 7.0)
        return ops().attention_exact(q, cache, out, pos, slots, table, n_heads, n_kv, hd, window, sinks=s, **known)

    def sees(request, place):
        return torch.tensor([r == request and p >= place and (window is None or p - window < place) for r, p in rows], device=DEV)

    def keys(place):
        return cache[int(table[1, place // ps]), 0][:, place % ps]

    clean = attend()
    assert bool(torch.isfinite(clean).all())
    for place in (256, 512, 768, 300):
        kept = keys(place).clone()
        for bad in (float("nan"), float("inf")):                              # (infinite keys: scores of +inf, -inf or none, by the query's signs)
            keys(place)[:] = bad
            hurt, hit = attend(), sees(0, place)
            assert torch.equal(hurt[~hit], clean[~hit]) and (bad == float("inf") or bool(torch.isnan(hurt[hit]).all()))
        keys(place)[:] = kept
    kept, q[4] = q[4].clone(), float("nan")                                    # position 256
    hurt = attend()
    assert bool(torch.isnan(hurt[4]).all()) and torch.equal(hurt[:4], clean[:4]) and torch.equal(hurt[5:], clean[5:])
    q[4] = kept
    keys(300)[:] = 30 * one                                                   # all others' shares are zero in 32 bits wherever this key is seen
    cache[int(table[1, 3 // ps]), 1].view(n_kv, hd, ps)[:, :, 3 % ps] = float("inf")
    hurt, hit, moved = attend(), sees(0, 3), sees(0, 300)
    assert not bool(torch.isfinite(hurt[hit]).any())
    assert torch.equal(hurt[~hit & ~moved], clean[~hit & ~moved]) and bool(torch.isfinite(hurt[~hit]).all())


@pytest.mark.parametrize("n_heads,n_kv,hd,vd,cap,sinks,gate,chunk", [(6, 2, 64, 128, None, True, None, None), (4, 1, 128, 48, 5.0, False, "head", None), (8, 8, 32, 16, None, True, "channel", None),
                                                                    (20, 1, 64, 64, 3.0, True, "head", 600), (3, 3, 16, 96, None, False, "channel", 320)])
def test_attention_exact_shares_contexts_out_with_all_it_takes(n_heads, n_kv, hd, vd, cap, sinks, gate, chunk):
    """32-bit: value heads of another size, capped scores, sinks, gates: a context shared out over workgroups gives the bits of one that is not,
    and both are the plain statement's in 64 bits."""
    ps, contexts = 8, [1030, 257]
    g = torch.Generator().manual_seed(hd + vd)
    pages = [-(-n // ps) for n in contexts]
    order = torch.randperm(sum(pages), generator=g)
    table = torch.full((2, max(pages)), -1, dtype=torch.int32)
    cache = torch.full((sum(pages), n_kv * ps * (hd + vd)), float("nan"))
    dense, at = [], 0
    for r, n in enumerate(contexts):
        k, v = torch.randn(pages[r] * ps, n_kv, hd, generator=g), torch.randn(pages[r] * ps, n_kv, vd, generator=g)
        dense.append((k[:n].double(), v[:n].double()))
        for i in range(pages[r]):
            page = int(order[at])
            table[r, i], at = page, at + 1
            cache[page, :n_kv * ps * hd] = k[i * ps:(i + 1) * ps].permute(1, 0, 2).reshape(-1)
            cache[page, n_kv * ps * hd:] = v[i * ps:(i + 1) * ps].permute(1, 2, 0).reshape(-1)
    rows = [(0, p) for p in (1020, 1021, 1022, 1023, 1024, 1025, 63, 64, 600)] + [(1, p) for p in (256, 255, 0)]
    pos = torch.tensor([p for _, p in rows], dtype=torch.int32)
    slots = torch.tensor([r for r, _ in rows], dtype=torch.int32)
    T = len(rows)
    q = torch.randn(T, n_heads * hd, generator=g)
    s = torch.randn(n_heads, generator=g) if sinks else None
    gates = torch.randn(T, n_heads if gate == "head" else n_heads * vd, generator=g) if gate else None
    want = torch.empty(T, n_heads, vd, dtype=torch.float64)
    for i, (r, p) in enumerate(rows):
        lo = p - p % chunk if chunk else 0
        for h in range(n_heads):
            kv = h // (n_heads // n_kv)
            sc = dense[r][0][lo:p + 1, kv] @ q[i].view(n_heads, hd)[h].double() / math.sqrt(hd)
            sc = cap * torch.tanh(sc / cap) if cap else sc
            e = torch.exp(sc - sc.max())
            o = e @ dense[r][1][lo:p + 1, kv] / (e.sum() + (torch.exp(s[h].double() - sc.max()) if sinks else 0))
            want[i, h] = o * (torch.sigmoid(gates[i, h] if gate == "head" else gates[i].view(n_heads, vd)[h]).double() if gate else 1)
    device = dict(sinks=s.to(DEV) if sinks else None, gate=gates.to(DEV) if gate == "head" else None, channel_gate=gates.to(DEV) if gate == "channel" else None)
    q, cache, pos, slots, table = (x.to(DEV) for x in (q, cache, pos, slots, table))

    def attend(**known):
        out = torch.full((T, n_heads * vd), float("nan"), device=DEV)
        return ops().attention_exact(q, cache, out, pos, slots, table, n_heads, n_kv, hd, page_size=ps, value_dim=vd, cap=cap, chunk=chunk, **device, **known)

    whole = attend()
    assert rel(whole, want.view(T, -1)) < 2e-6                                 # (as the test of one order of sums)
    for known in (dict(max_context=1030), dict(max_context=4096), dict(single_rows=True), dict(single_rows=True, max_context=1030)):
        assert torch.equal(attend(**known), whole), known


@pytest.mark.parametrize("n_heads,n_kv,hd,vd,window,chunk", [(32, 8, 64, 64, None, None), (16, 16, 48, 64, 300, None), (8, 8, 64, 16, None, 320), (6, 2, 64, 80, None, None), (34, 2, 128, 128, 520, None)])
def test_attention_exact_of_blocks_one_by_one(n_heads, n_kv, hd, vd, window, chunk):
    """32-bit: contexts around the ends of blocks of 64 and spans of 256 keys, shared out block by block (few rows), span by span (many) and not at all, rows of their own
    and rows of one request in a tile: the same bits, and the kernel of each number of rows is the one that the rule's line names."""
    ps, seen = 16, 1040
    pages = -(-seen // ps)
    g = torch.Generator(device=DEV).manual_seed(hd + vd)
    cache = torch.randn(2 * pages, n_kv * ps * (hd + vd), device=DEV, generator=g)
    cache[pages + 300 // ps].fill_(float("inf"))                               # met by the rows of the second request that see it
    table = torch.randperm(pages, device=DEV, generator=g).int()
    table = torch.stack([table, table + pages])
    picked = [0, 15, 16, 63, 64, 65, 127, 128, 255, 256, 257, 319, 320, 511, 512, 767, 1023, 1024, 1039]
    T = 160
    pos = torch.tensor([picked[i % len(picked)] for i in range(T)], dtype=torch.int32, device=DEV)
    slots = torch.tensor([i // len(picked) % 2 for i in range(T)], dtype=torch.int32, device=DEV)
    q = torch.randn(T, n_heads * hd, device=DEV, generator=g)
    sinks = torch.randn(n_heads, device=DEV, generator=g)

    def attend(first, n, **known):
        out = torch.full((n, n_heads * vd), 7.0, device=DEV)
        return ops().attention_exact(q[first:first + n], cache, out, pos[first:first + n], slots[first:first + n], table, n_heads, n_kv, hd, window, page_size=ps, value_dim=vd, cap=30.0,
                                     sinks=sinks, chunk=chunk, **known).view(torch.int32)

    wide = -(-min(seen, window or seen, chunk or seen) // 256) * 256           # as the wrapper asks
    spans = ops().lib().gi_attention_exact_spans(2, 2, n_heads, n_kv, hd, vd, ps, wide)

    def parts(n):                                                              # that a span of a (row, head) leaves
        return ops().lib().gi_attention_exact_part_floats(n, n, n_heads, n_kv, hd, vd, spans) // (n * n_heads * spans * (vd + 4))

    whole = attend(0, T, single_rows=True)
    small = hd <= 64 and vd <= 64
    few, many = 2, (1280 if not small else 1152 if spans <= 5 else 896) // (n_kv * 4 * (spans - 1)) + 1
    assert spans > 1 and parts(1) == parts(few) == 4 and parts(many) == (1 if small else 4)
    for n, known in ((1, dict(single_rows=True)), (few, dict(single_rows=True)), (19, dict(single_rows=True)), (many, dict(single_rows=True)), (19, dict()), (few + 19, dict(single_rows=few))):
        for first in (0, 18, T - n if n < T else 0):
            got = attend(first, n, max_context=seen, **known)
            assert torch.equal(got, whole[first:first + n]), (n, known, first)
    clean = torch.isfinite(whole.view(torch.float32)).all(1).tolist()
    assert clean[0] and any(clean[len(picked):2 * len(picked)]) and all(clean[:len(picked)]) and not all(clean)


@pytest.mark.parametrize("rows,n_heads,n_kv,hd,seen", [(3, 24, 8, 128, 600), (12, 32, 8, 64, 600)])
def test_attention_exact_without_room_for_blocks_goes_by_spans(rows, n_heads, n_kv, hd, seen, monkeypatch):
    """A device that has no room for what blocks of keys leave: spans leave a quarter of it, and the bits are the same."""
    ps, g = 16, torch.Generator(device=DEV).manual_seed(hd)
    pages = -(-seen // ps)
    cache, q = torch.randn(pages, n_kv * ps * 2 * hd, device=DEV, generator=g), torch.randn(rows, n_heads * hd, device=DEV, generator=g)
    table, slots = torch.arange(pages, dtype=torch.int32, device=DEV).view(1, -1), torch.zeros(rows, dtype=torch.int32, device=DEV)
    pos = torch.tensor([seen - 1 - 37 * i for i in range(rows)], dtype=torch.int32, device=DEV)
    attend = lambda: ops().attention_exact(q, cache, torch.full_like(q, 7.0), pos, slots, table, n_heads, n_kv, hd, page_size=ps, single_rows=True, max_context=seen)
    blocks, asked = attend(), []
    monkeypatch.setattr(ops(), "_room", lambda floats, device: asked.append(floats))
    spans = attend()
    assert torch.equal(spans, blocks) and asked == [4 * ops().lib().gi_attention_exact_span_floats(rows, n_heads, hd, ops()._exact_spans(rows, rows, n_heads, n_kv, hd, hd, ps, 768)[0])]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_finds_one_far_key(dtype):
    """Among 700 keys one is scaled so that its score stands out: the output must be its value."""
    from geneinfer_amd.parts import StepContext
    n_heads, n_kv, hd, ps = 4, 2, 64, 16
    cache, table, dense = build_paged([700], n_kv, hd, ps, dtype, seed=1)
    k, v = dense[0]
    target = 37
    q = (k[target].float().repeat_interleave(n_heads // n_kv, 0) * 3.0).reshape(1, n_heads * hd).to(dtype).to(DEV)
    pos = torch.tensor([699], dtype=torch.int32, device=DEV)
    slots = torch.tensor([1], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=1, dtype=dtype, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=[1], seg_start=[0],
                      seg_len=[1], seg_pos0=[699])
    out = torch.empty(1, n_heads * hd, dtype=dtype, device=DEV)
    ops().attention(q, cache, out, ctx, table, n_heads, n_kv, hd, None)
    want = plain_attention_rows(q, dense, [(0, 699)], n_heads, n_kv, hd, None)
    assert rel(out, want) < (2e-6 if dtype == torch.float32 else 8e-3)
    assert rel(out.view(n_heads, hd)[0], v[target, 0]) < 2e-2          # the softmax is nearly one-hot on the target


@pytest.mark.parametrize("hd", [32, 64, 96, 128])
@pytest.mark.parametrize("ps,window", [(16, None), (16, 19), (48, None)])
def test_decoded_rows_read_whole_blocks_of_keys(hd, ps, window):
    """Single rows whose ranges begin and end anywhere in a block of 16 positions, by whole cache lines or not; what lies beyond a row in its pages is NaN and reaches no result."""
    from geneinfer_amd.parts import StepContext
    contexts = list(range(1, 35)) + [47, 48, 49, 63, 64, 65, 129, 500]
    cache, table, dense = build_paged(contexts, 2, hd, ps, torch.bfloat16, seed=hd)
    T = len(contexts)
    q = randn(T, 6 * hd, dtype=torch.bfloat16, seed=3)
    pos = torch.tensor([n - 1 for n in contexts], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=torch.arange(1, T + 1, dtype=torch.int32, device=DEV),
                      seg_slot=list(range(1, T + 1)), seg_start=list(range(T)), seg_len=[1] * T, seg_pos0=[n - 1 for n in contexts])
    out = torch.full((T, 6 * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops().attention(q, cache, out, ctx, table, 6, 2, hd, window)
    want = plain_attention_rows(q, dense, [(i, n - 1) for i, n in enumerate(contexts)], 6, 2, hd, window)
    assert rel(out, want) < 8e-3, rel(out, want)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("rows", [2, 8, 21])
@pytest.mark.parametrize("n_heads,n_kv,hd,ps,window", [(6, 2, 64, 16, None), (6, 2, 128, 16, None), (40, 2, 64, 48, None), (20, 1, 128, 16, 200)])
def test_decoded_rows_that_share_their_pages(n_heads, n_kv, hd, ps, window, rows, fused):
    """Requests of two kinds in turn that each begin alike, on pages in common and on copies of them: keys and values come through the caches or past them, the bits are the same, and
    those of rows alone."""
    o = ops()
    from geneinfer_amd.parts import StepContext
    contexts = [530 + 37 * i for i in range(rows)]
    cache, table, dense = build_paged(contexts, n_kv, hd, ps, torch.bfloat16, seed=hd + rows)
    alike = 500 // ps                                                     # whole pages
    for i in range(2, rows):
        cache[table[i + 1, :alike].long()] = cache[table[1 + i % 2, :alike].long()]
    common = table.clone()
    for i in range(2, rows):
        common[i + 1, :alike] = table[1 + i % 2, :alike]
    if rows == 2:
        cache[table[2, :alike].long()], common[2, :alike] = cache[table[1, :alike].long()], table[1, :alike]
    pos, slots = torch.tensor([n - 1 for n in contexts], dtype=torch.int32, device=DEV), torch.arange(1, rows + 1, dtype=torch.int32, device=DEV)
    a, kvd = n_heads * hd, n_kv * hd
    qkv, angle = randn(rows, a + 2 * kvd, seed=31), randn(rows, hd // 2, seed=9)

    def made(table, first=0, n=rows, looks=True):
        seen, memo = cache.clone(), {}
        part = slice(first, first + n)
        out = torch.full((n, a), float("nan"), dtype=torch.bfloat16, device=DEV)
        plan = o.AttentionPlan(list(range(n)), [1] * n, [c - 1 for c in contexts[part]], list(range(first + 1, first + n + 1)), DEV)
        if fused:
            products = (qkv[part, :a], qkv[part, a:a + kvd], qkv[part, a + kvd:], torch.cos(angle[part]), torch.sin(angle[part]))
            o.attention_bf16(None, seen, out, plan, pos[part], slots[part], table, n_heads, n_kv, hd, window, products=products, memo=memo, in_common=looks)
        else:
            o.attention_bf16(qkv[part, :a].to(torch.bfloat16).contiguous(), seen, out, plan, pos[part], slots[part], table, n_heads, n_kv, hd, window, memo=memo, in_common=looks)
        return out, seen

    (own, cache_own), (shared, cache_shared), (unseen, cache_unseen) = made(table), made(common), made(common, looks=False)
    assert torch.equal(own, shared) and torch.equal(own, unseen) and not bool(torch.isnan(own.float()).any())
    assert all(torch.equal(torch.nan_to_num(cache_own, nan=-1.0), torch.nan_to_num(c, nan=-1.0)) for c in (cache_shared, cache_unseen))
    alone = torch.cat([made(table, i, 1)[0] for i in range(rows)])
    # (probabilities are rounded to bfloat16 about other maxima, 2^-9 of each at most on either side, and the results, 2^-8 between the two)
    assert rel(alone, own) < 2 * 2.0 ** -9 + 2.0 ** -8


@pytest.mark.parametrize("n_heads,n_kv,hd,ps,window", ATT_CASES)
@pytest.mark.parametrize("target_waves", [4096, 64])
def test_decode_attention_from_unrotated_products(n_heads, n_kv, hd, ps, window, target_waves, monkeypatch):
    """Single decoded rows whose keys and values are not in the cache yet: one kernel rotates q and k,
    attends (its own position included) and writes k and v to the right places, in one split and in several."""
    from geneinfer_amd.parts import StepContext
    shape = ops().decode_attention_shape
    monkeypatch.setattr(ops(), "decode_attention_shape", lambda *a, **k: shape(*a[:5], target_waves=target_waves))
    contexts = [300, 131, 1, 77, 530, 16, 17, 1200, 32, 33]           # the new row's position is the last of each
    gone = {slot: max(0, n - window) for slot, n in enumerate(contexts)} if window else None        # what a window has given back
    cache, table, dense = build_paged(contexts, n_kv, hd, ps, torch.bfloat16, seed=hd + n_heads + 1, gone_before=gone)
    T = len(contexts)
    pos = torch.tensor([n - 1 for n in contexts], dtype=torch.int32, device=DEV)
    slots = torch.arange(1, T + 1, dtype=torch.int32, device=DEV)
    a, kvd = n_heads * hd, n_kv * hd
    qkv = randn(T, a + 2 * kvd, seed=31)
    inv = torch.tensor([1.0 / (10000.0 ** (2 * k / hd)) for k in range(hd // 2)], dtype=torch.float64, device=DEV)
    cos, sin = torch.empty(T, hd // 2, device=DEV), torch.empty(T, hd // 2, device=DEV)
    ops().rope_cos_sin(pos, inv, cos, sin)

    def rotated(x, heads):
        x = x.double().cpu().view(T, heads, hd)
        c, s_ = torch.cat([cos, cos], -1).double().cpu()[:, None, :], torch.cat([sin, sin], -1).double().cpu()[:, None, :]
        return x * c + torch.cat([-x[..., hd // 2:], x[..., :hd // 2]], -1) * s_

    q_rot = rotated(qkv[:, :a], n_heads).to(torch.bfloat16).view(T, a)
    k_rot = rotated(qkv[:, a:a + kvd], n_kv).to(torch.bfloat16)
    v_new = qkv[:, a + kvd:].cpu().view(T, n_kv, hd).to(torch.bfloat16)
    want_cache = cache.clone()
    for i, n in enumerate(contexts):                                   # the row's own place: empty before, k and v after
        dense[i][0][n - 1], dense[i][1][n - 1] = k_rot[i], v_new[i]
        page, place = int(table[i + 1, (n - 1) // ps]), (n - 1) % ps
        cache[page, 0, :, place, :] = 0
        cache[page, 1].view(n_kv, hd, ps)[:, :, place] = 0
        want_cache[page, 0, :, place, :] = k_rot[i].to(DEV)
        want_cache[page, 1].view(n_kv, hd, ps)[:, :, place] = v_new[i].to(DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots,
                      seg_slot=list(range(1, T + 1)), seg_start=list(range(T)), seg_len=[1] * T, seg_pos0=[n - 1 for n in contexts])
    out = torch.full((T, a), float("nan"), dtype=torch.bfloat16, device=DEV)
    done = ops().attention_from_products(qkv[:, :a], qkv[:, a:a + kvd], qkv[:, a + kvd:], cos, sin, cache, out, ctx, table, n_heads, n_kv, hd, window)
    if not ops().attention_bf16_supports(hd, ps, False):
        assert done is False and bool(torch.isnan(out.float()).all())    # refused: the caller rotates and stores first
        return
    assert done is True
    want = plain_attention_rows(q_rot, dense, [(i, n - 1) for i, n in enumerate(contexts)], n_heads, n_kv, hd, window)
    assert rel(out, want) < 8e-3, rel(out, want)
    got_c, want_c = torch.nan_to_num(cache.float(), nan=-1.0), torch.nan_to_num(want_cache.float(), nan=-1.0)
    assert rel(got_c, want_c) < 1e-3                                  # a rotated key may round the other way in 32-bit
    assert float(((got_c - want_c).abs() > 0.02 * want_c.abs() + 1e-6).sum()) == 0
    # read-only use of another layer's pages (which now hold the rows' keys and values): the same output, the cache untouched
    out2, before = torch.full_like(out, float("nan")), cache.clone()
    assert ops().attention_from_products(qkv[:, :a], None, None, cos, sin, cache, out2, ctx, table, n_heads, n_kv, hd, window)
    assert rel(out2, want) < 8e-3
    assert torch.equal(torch.nan_to_num(cache, nan=-1.0), torch.nan_to_num(before, nan=-1.0))


@pytest.mark.parametrize("hd", [64, 128])
def test_decode_attention_shape_leaves_no_nearly_empty_round(hd):
    """The cut of the context over workgroups: whatever the number of rows, the context is either not cut at all (a workgroup of 4
    or 8 waves per row and group of heads, where the busiest compute unit is expected to be done no later than the chip's memory
    plus a merging kernel), or the workgroups fit the chip at once, or their last round is not a small remainder; pieces never
    fall under 64 positions and the waves cover the span."""
    o = ops()
    n_heads, n_kv, span = 32, 8, 4096
    uncut = 0
    for rows in list(range(17, 130)) + [192, 256, 500]:
        splits, n_waves = o.decode_attention_shape(rows, n_heads, n_kv, hd, span)
        assert 1 <= n_waves <= 8 and splits >= 1 and not 5 <= n_waves <= 7
        single = o._decode_single_split(rows * n_kv, span, hd, 8)
        if single is not None:
            assert (splits, n_waves) == single and splits == 1 and n_waves in (4, 8)
            uncut += 1
            continue
        assert splits * n_waves == 1 or o._decode_piece(span, splits * n_waves) >= 64
        rounds = rows * n_kv * splits / o._decode_places(hd, False, n_waves, 4)
        plain = o._decode_plain_shape(rows * n_kv, span, 8)
        if (splits, n_waves) != plain:
            assert rounds <= 1, (rows, splits, n_waves, rounds)
        else:
            assert rounds <= 1 or rounds - int(rounds) == 0 or rounds - int(rounds) >= 0.3, (rows, splits, n_waves, rounds)
    assert 30 <= uncut <= 100                              # (a workgroup for every compute unit, or a whole number of them: 32, 64, 96, 128 rows; not 40 or 65)
    assert o._decode_single_split(64 * n_kv, span, hd, 8) is not None and o._decode_single_split(65 * n_kv, span, hd, 8) is None
    assert o._decode_single_split(8 * n_kv, span, hd, 8) is None
    for rows in range(1, 17):                              # the kernel that also rotates and stores: the plain rule at 64 channels, one round at 128
        splits, n_waves = o.decode_attention_shape(rows, n_heads, n_kv, hd, span, fused=True)
        if hd == 64:
            assert (splits, n_waves) == o._decode_plain_shape(rows * n_kv, span, 8, small=True)
            assert o._decode_piece(span, splits * n_waves) >= 32 and (n_waves == 8) == (rows * n_kv <= 64 or splits == 1)
        else:
            assert rows * n_kv * splits <= o._decode_places(hd, True, n_waves, 4) or (splits, n_waves) == o._decode_plain_shape(rows * n_kv, span, 8)
            assert o._decode_piece(span, splits * n_waves) >= 64


def test_rope_store_writes_the_right_places():
    n_heads, n_kv, hd, ps = 4, 2, 32, 16
    n_pages = 5
    cache = torch.full((n_pages, 2, n_kv, ps, hd), -777.25, device=DEV)
    table = torch.tensor([[-1, -1, -1], [3, 0, 4]], dtype=torch.int32, device=DEV)
    T = 3
    pos = torch.tensor([15, 16, 17], dtype=torch.int32, device=DEV)     # the last place of a page, then the next page
    slots = torch.ones(T, dtype=torch.int32, device=DEV)
    qkv = randn(T, (n_heads + 2 * n_kv) * hd, seed=20)
    a, kvd = n_heads * hd, n_kv * hd
    inv = torch.tensor([1.0 / (10000.0 ** (2 * k / hd)) for k in range(hd // 2)], dtype=torch.float64, device=DEV)
    cos, sin = torch.empty(T, hd // 2, device=DEV), torch.empty(T, hd // 2, device=DEV)
    ops().rope_cos_sin(pos, inv, cos, sin)
    q_out = torch.empty(T, a, device=DEV)
    ops().rope_store(qkv[:, :a], qkv[:, a:a + kvd], qkv[:, a + kvd:], cos, sin, pos, slots, table, q_out, cache, n_heads, n_kv, hd)

    def rotate_half_form(x, heads):          # x*cos + rotate_half(x)*sin with cos/sin doubled over both halves (tests/verify_kernels.py:284-291)
        x = x.double().cpu().view(T, heads, hd)
        ang = pos.double().cpu()[:, None] * inv.cpu()[None, :]
        c, s_ = torch.cat([ang.cos(), ang.cos()], -1)[:, None, :], torch.cat([ang.sin(), ang.sin()], -1)[:, None, :]
        rot = torch.cat([-x[..., hd // 2:], x[..., :hd // 2]], -1)
        return x * c + rot * s_

    assert rel(q_out.view(T, n_heads, hd), rotate_half_form(qkv[:, :a], n_heads)) < 2e-6
    k_want = rotate_half_form(qkv[:, a:a + kvd], n_kv)
    v_want = qkv[:, a + kvd:].double().cpu().view(T, n_kv, hd)
    for t, (page, place) in enumerate([(3, 15), (0, 0), (0, 1)]):
        assert rel(cache[page, 0, :, place, :], k_want[t]) < 2e-6
        assert rel(cache[page, 1].view(n_kv, hd, ps)[:, :, place], v_want[t]) < 1e-7
    touched = torch.zeros_like(cache, dtype=torch.bool)
    for page, place in [(3, 15), (0, 0), (0, 1)]:
        touched[page, 0, :, place, :] = True
        touched[page, 1].view(n_kv, hd, ps)[:, :, place] = True
    assert torch.all(cache[~touched] == -777.25), "rope_store wrote outside its places"


@pytest.mark.parametrize("m, n, k", [(131, 2048, 2048), (129, 2048, 8192), (300, 1028, 1024), (500, 3072, 512), (257, 4096, 512), (64, 2048, 2048), (40, 3072, 1024), (128, 132, 512)])
def test_product_onto_rows_that_makes_the_whole_norm(m, n, k):
    """Shares of k added up, onto the rows, and the rows' norm: what the product and the norm's kernel make one after the other, in bits."""
    assert ops().gemm_bf16_onto_norm_takes(m, n, k)
    a, w = randn(m, k, dtype=torch.bfloat16, seed=1), randn(n, k, dtype=torch.bfloat16, seed=2)
    x = randn(m, n, dtype=torch.float32, seed=3)
    g = (1 + 0.1 * randn(n, dtype=torch.float32, seed=4)).to(torch.bfloat16)
    want_x = x.clone()
    ops().gemm_bf16(a, w, want_x, accumulate=True)
    want = ops().rmsnorm(want_x, g, 1e-5, torch.empty(m, n, dtype=torch.bfloat16, device=DEV))
    got = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops().gemm_bf16_onto_norm(a, w, x, g.float(), 1e-5, got)
    assert torch.equal(x, want_x) and torch.equal(got, want)
    assert rel(x, randn(m, n, dtype=torch.float32, seed=3).double() + a.double() @ w.double().t()) < 1e-5
