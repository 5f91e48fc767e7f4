"""The Rigalorn design in the engine against the plain implementation (`plain_rigalorn.py`): each kernel alone, then whole models
of five small configurations under every way of cutting the work into steps, and generation through the entry point and the
scheduler.  In float32 the engine's logits must not depend on the cutting at all (equal bits); in bfloat16 they must lie as close
to the exact model as rounding alone explains."""
import math

import numpy as np
import pytest
import torch

import plain_rigalorn as P
from model_folders import assert_within_bfloat16_noise, relative_error
from rigalorn_folders import CONFIGS, PAGE_SIZE, stored_weights, write_model

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _prompt(cfg, n, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, cfg["vocab"], (n,), generator=g).tolist()


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    root = tmp_path_factory.mktemp("rigalorn")
    out = {}
    for name, cfg in CONFIGS.items():
        write_model(root / name, cfg, seed=17 + ord(name))
        out[name] = root / name
    return out


_plain_cache = {}


def plain_logits(folders, name, tokens, rounded=False, dtype=torch.float64):
    key = (name, tuple(tokens), rounded, dtype)
    if key not in _plain_cache:
        _plain_cache[key] = P.forward(CONFIGS[name], stored_weights(folders[name]), tokens, dtype, store=P.to_bfloat16_and_back if rounded else P.same)
    return _plain_cache[key]


def make_runner(folders, name, dtype, **kw):
    from geneinfer_amd.engine import Runner, load_model
    model = load_model(folders[name], dtype, DEV)
    kw.setdefault("page_size", PAGE_SIZE[name])
    kw.setdefault("max_tokens", 1024)
    kw.setdefault("max_requests", 4)
    return Runner(model, **kw)


def feed(runner, request, tokens, cuts):
    """The request's tokens in portions of the sizes in `cuts` (the rest one by one); logits of every position, on the host."""
    from geneinfer_amd.engine import StepEntry
    rows, at = [], 0
    sizes = list(cuts) + [1] * (len(tokens) - sum(cuts))
    for n in sizes:
        rows.append(runner.step([StepEntry(request, tokens[at:at + n], tuple(range(n)))]).cpu())
        at += n
    return torch.cat(rows)


def check_against_plain(folders, name, dtype, tokens, got, what):
    exact = plain_logits(folders, name, tokens)
    if dtype == "float32":            # within 4 times what the plain model itself loses in 32-bit
        single = plain_logits(folders, name, tokens, dtype=torch.float32)
        noise = max(relative_error(single[p], exact[p]) for p in range(len(tokens)))
        err = max(relative_error(got[p], exact[p]) for p in range(len(tokens)))
        assert err < 4 * noise + 1e-5, f"{what}: float32 logits differ from the plain implementation by {err:.2e} (the plain model in 32-bit: {noise:.2e})"
    else:
        rounded = plain_logits(folders, name, tokens, rounded=True)
        assert_within_bfloat16_noise({p: got[p] for p in range(len(tokens))}, lambda p: exact[p], lambda p: rounded[p], what)


# =============================================================================================== kernels alone
def test_the_library_and_the_planner_agree_on_the_state_size():
    from geneinfer_amd.kernels import ops
    for h, g, dk, dv, taps in ((1, 1, 1, 1, 1), (3, 1, 20, 72, 5), (6, 2, 48, 64, 4), (2, 2, 255, 129, 2)):
        assert ops.lib().gi_delta_state_floats(h, g, dk, dv, taps) == ops.delta_state_floats(h, g, dk, dv, taps)
        assert ops.lib().gi_delta_memory_floats(h, dk, dv) == ops.delta_memory_floats(h, dk, dv)
    assert ops.lib().gi_delta_max_key_dim() == ops.DELTA_MAX_KEY_DIM and ops.lib().gi_delta_max_taps() == ops.DELTA_MAX_TAPS


def test_activation_of_the_plain_feed_forward():
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(1)
    x = torch.cat([4 * torch.randn(7, 33, generator=g), torch.tensor([[0.0, -0.0, 1e-8, -1e-8, 30.0, -30.0, -90.0] + [0.5] * 26])])
    for p, q in ((0.3, -0.7), (-25.0, 24.0), (0.0, 0.0)):
        params = torch.tensor([p, q])
        want = P.xielu(x.double(), params[0].double(), params[1].double())
        out = torch.empty(8, 33, device=DEV)
        ops.xielu(x.to(DEV), out, params.to(DEV))
        assert relative_error(out, want) < 1e-6
        half = torch.empty(8, 33, device=DEV, dtype=torch.bfloat16)
        ops.xielu(x.to(DEV), half, params.to(DEV))
        assert torch.equal(half.cpu(), out.cpu().to(torch.bfloat16))


@pytest.mark.parametrize("rows, n, k, first", [(1, 416, 128, 320), (16, 320, 136, 3), (9, 1100, 2048, 0), (300, 8192, 256, 0), (131, 16400, 192, 0), (700, 8192, 512, 0), (1777, 8200, 320, 0),
                                               (2048, 6000, 1024, 0)])
def test_product_with_the_activation_of_the_plain_feed_forward(rows, n, k, first):
    """Against the product and the activation one after the other: the same sums and the same activation, so the same bits."""
    from geneinfer_amd.kernels import ops
    assert ops.gemm_bf16_xielu_takes(rows, n, k, first)
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    a = torch.randn(rows, k, device=DEV, generator=g).bfloat16()
    w = (torch.randn(n, k, device=DEV, generator=g) * 1.5 / k ** 0.5).bfloat16()
    a[0, :] = 0                                                          # (a row of zeros; one that leaves the range of exp; one of infinities)
    if rows > 2:
        a[1, :] *= 300
        a[2, 0] = float("inf")
    params = torch.tensor([0.3, -0.7], device=DEV)
    both = torch.empty(rows, n, device=DEV)
    ops.gemm_bf16(a, w, both)
    want = torch.empty(rows, n - first, dtype=torch.bfloat16, device=DEV)
    ops.xielu(both[:, first:], want, params)
    out = torch.full((rows, n), 7.0, device=DEV) if first else None
    mid = torch.full((rows + 1, n - first + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.gemm_bf16_xielu(a, w, params, mid[:rows, :n - first], out)
    assert (mid[rows] == 7).all() and (mid[:, n - first:] == 7).all()
    if first:
        assert torch.equal(out[:, :first].nan_to_num(nan=9.0), both[:, :first].nan_to_num(nan=9.0)) and (out[:, first:] == 7).all()
    got, want = mid[:rows, :n - first].float(), want.float()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.nan_to_num(nan=9.0), want.nan_to_num(nan=9.0))


@pytest.mark.parametrize("heads, kv, dk, dv, taps", [(4, 2, 16, 24, 4), (3, 3, 64, 64, 2), (2, 1, 130, 10, 5), (1, 1, 7, 201, 1), (5, 5, 3, 5, 3), (2, 2, 300, 6, 8), (1, 1, 20, 9, 13)])
def test_gated_delta_rule_kernels(heads, kv, dk, dv, taps):
    """Two requests of unequal length in one step; then the longer one again from a fresh slot in steps down to one and two rows:
    the memories and the convolutions' tails carry, and the bits do not change."""
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(dk + taps)
    n_conv = 2 * kv * dk + heads * dv
    lens, cols = [29, 90], n_conv + 2 * heads + 3
    conv_off, a_off, b_off = 3, 3 + n_conv, 3 + n_conv + heads
    proj = torch.randn(sum(lens), cols, generator=g)
    w_taps = 0.6 * torch.randn(n_conv, taps, generator=g)
    a_log, dt_bias = -1.0 + 0.8 * torch.randn(heads, generator=g), 0.5 * torch.randn(heads, generator=g)

    def plain(rows):
        x = rows.double()
        y = P.short_conv_silu(x[:, conv_off:conv_off + n_conv], w_taps.double())
        unit = lambda z: z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)
        q, k = unit(y[:, :kv * dk].view(-1, kv, dk)) * dk ** -0.5, unit(y[:, kv * dk:2 * kv * dk].view(-1, kv, dk))
        v = y[:, 2 * kv * dk:].view(-1, heads, dv)
        decay = torch.exp(-torch.exp(a_log.double()) * P.softplus(x[:, a_off:a_off + heads] + dt_bias.double()))
        beta = torch.sigmoid(x[:, b_off:b_off + heads])
        return torch.cat([P.delta_rule(q[:, h // (heads // kv)], k[:, h // (heads // kv)], v[:, h], beta[:, h], decay[:, h]) for h in range(heads)], dim=-1)

    want = torch.cat([plain(proj[:lens[0]]), plain(proj[lens[0]:])])
    state = torch.zeros(5, ops.delta_state_floats(heads, kv, dk, dv, taps) + 3, device=DEV)
    dev = lambda t: t.to(DEV)

    def run(rows, seg_lens, slots, pos0):
        n = rows.shape[0]
        starts = [sum(seg_lens[:i]) for i in range(len(seg_lens))]
        row_slot = torch.tensor([s for s, m in zip(slots, seg_lens) for _ in range(m)], dtype=torch.int32, device=DEV)
        row_pos = torch.tensor([p + i for p, m in zip(pos0, seg_lens) for i in range(m)], dtype=torch.int32, device=DEV)
        seg_start, seg_len = torch.tensor(starts, dtype=torch.int32, device=DEV), torch.tensor(seg_lens, dtype=torch.int32, device=DEV)
        qkv, gates, out = torch.empty(n, n_conv, device=DEV), torch.empty(n, 2 * heads, device=DEV), torch.empty(n, heads * dv, device=DEV)
        rows = dev(rows)
        ops.delta_prepare(rows, conv_off, a_off, b_off, dev(w_taps), dev(a_log), dev(dt_bias), row_slot, row_pos, state, qkv, gates, heads, kv, dk, dv, dk ** -0.5)
        ops.delta_tail(rows, conv_off, taps, seg_start, seg_len, row_slot, state, heads, kv, dk, dv)
        ops.delta_scan(qkv, gates, seg_start, seg_len, row_slot, state, out, heads, kv, dk, dv)
        return out.cpu().double()

    got = run(proj, lens, [2, 0], [0, 0])
    assert relative_error(got, want) < 3e-5
    second = proj[lens[0]:]
    cuts, pieces, at = [2, 1, 1, 40, 1, 2, 3, 38, 2], [], 0
    for c in cuts:
        pieces.append(run(second[at:at + c], [c], [4], [at]))
        at += c
    assert at == lens[1] and torch.equal(torch.cat(pieces), got[lens[0]:])
    # two requests that both go on, side by side in one step, each from its own slot
    state[1], state[3] = state[2], state[4]
    more = torch.randn(11, cols, generator=g)
    both = run(torch.cat([more[:4], more[4:]]), [4, 7], [1, 3], [lens[0], lens[1]])
    alone = torch.cat([run(more[:4], [4], [2], [lens[0]]), run(more[4:], [7], [4], [lens[1]])])
    assert torch.equal(both, alone)


@pytest.mark.parametrize("heads, kv, dk, dv, taps", [(8, 4, 64, 128, 4), (3, 3, 20, 65, 2), (2, 1, 64, 64, 3), (2, 2, 33, 130, 4), (2, 1, 16, 24, 5), (2, 1, 16, 24, 1)])
def test_what_the_delta_rule_reads_of_single_rows_and_of_prompts(heads, kv, dk, dv, taps):
    """A step of single rows, each with a tail before it, in the kernel that moves the tails on, and a long step of several requests (one goes on, one begins, one of a
    single row, more rows than a wave takes at the end): row by row in steps of their own, in bits."""
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(dk + taps)
    n_conv = 2 * kv * dk + heads * dv
    cols, lens = n_conv + 2 * heads + 1, [5, 60, 1, 9]
    n = sum(lens)
    proj = torch.randn(n, cols, generator=g).to(DEV)
    w_taps, a_log, dt_bias = (x.to(DEV) for x in (0.6 * torch.randn(n_conv, taps, generator=g), 0.3 * torch.randn(heads, generator=g), 0.5 * torch.randn(heads, generator=g)))
    first = torch.randn(6, ops.delta_state_floats(heads, kv, dk, dv, taps) + 3, generator=g).to(DEV)
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)

    def step(rows, slots, positions, state, single):
        qkv, gates = torch.full((len(rows), n_conv), float("nan"), device=DEV), torch.full((len(rows), 2 * heads), float("nan"), device=DEV)
        ops.delta_prepare(rows, 1, 1 + n_conv, 1 + n_conv - heads, w_taps, a_log, dt_bias, ints(slots), ints(positions), state, qkv, gates, heads, kv, dk, dv, dk ** -0.5, single)
        return qkv, gates

    slots = [s for s, m in zip((4, 0, 5, 2), lens) for _ in range(m)]
    positions = [p + i for p, m in zip((7, 0, 3, 11), lens) for i in range(m)]
    together = step(proj, slots, positions, first.clone(), False)
    state = first.clone()
    for t in range(n):                                           # one row at a time through the general kernels
        one = step(proj[t:t + 1], slots[t:t + 1], positions[t:t + 1], state, False)
        ops.delta_tail(proj[t:t + 1], 1, taps, ints([0]), ints([1]), ints(slots[t:t + 1]), state, heads, kv, dk, dv)
        assert torch.equal(together[0][t], one[0][0]) and torch.equal(together[1][t], one[1][0]), t
    at, moved, kept = [0, 3, 70, 74], first.clone(), first.clone()
    rows = proj[at].contiguous()
    single, general = step(rows, [3, 1, 0, 5], [9, 2, 4, 1], moved, True), step(rows, [3, 1, 0, 5], [9, 2, 4, 1], kept, False)
    ops.delta_tail(rows, 1, taps, ints([0, 1, 2, 3]), ints([1] * 4), ints([3, 1, 0, 5]), kept, heads, kv, dk, dv)
    assert torch.equal(single[0], general[0]) and torch.equal(single[1], general[1]) and torch.equal(moved, kept)


def _rule_in_its_order(qkv, gates, M, heads, kv, dk, dv, channel):
    """The rule over one run of rows in 32 bits, every sum in the kernel's order: of a key's rows those 16 apart are one chain of fused
    multiply-adds, the 16 chains meet as a tree (place i and its mirror image, in 16, then in 8, then two apart, then neighbours).
    M [heads, dk, dv] is moved on; the read-outs come back.  A fused multiply-add: 64 bits of mantissa, rounded once to 32-bit."""
    f = np.float32
    fma = lambda a, b, c: (a.astype(np.longdouble) * b.astype(np.longdouble) + np.asarray(c).astype(np.longdouble)).astype(f)

    def chains(x, y, rounded=False):                                      # [..., dk, columns] -> [..., columns]
        rows = -(-dk // 16)
        acc = np.zeros(x.shape[:-2] + (16, x.shape[-1]), f)
        for r in range(rows):
            n = min(16, dk - 16 * r)
            a, b = x[..., 16 * r:16 * r + n, :], y[..., 16 * r:16 * r + n, :]
            acc[..., :n, :] = acc[..., :n, :] + a * b if rounded else fma(a, b, acc[..., :n, :])
        i = np.arange(16)
        for other in (15 - i, i ^ 7, i ^ 2, i ^ 1):
            acc = acc + acc[..., other, :]
        return acc[..., 0, :]

    n, per = qkv.shape[0], heads // kv
    q, k = (np.repeat(qkv[:, at:at + kv * dk].reshape(n, kv, dk), per, 1)[..., None] for at in (0, kv * dk))
    v = qkv[:, 2 * kv * dk:2 * kv * dk + heads * dv].reshape(n, heads, dv)
    decay, step = gates[:, :-heads].reshape(n, heads, -1, 1), gates[:, -heads:, None]
    out = np.empty((n, heads, dv), f)
    for t in range(n):
        kt, qt = np.broadcast_to(k[t], M.shape), np.broadcast_to(q[t], M.shape)
        kq = chains(k[t], q[t], rounded=channel)
        if channel:
            M[:] = M * decay[t]
            sk, sq = chains(M, kt), chains(M, qt)
            w = step[t] * (v[t] - sk)
            M[:] = fma(kt, w[:, None], M)
            out[t] = fma(w, np.broadcast_to(kq, w.shape), sq)
        else:
            sk, sq, d = chains(M, kt), chains(M, qt), np.broadcast_to(decay[t][:, 0], v[t].shape)
            w = step[t] * fma(-d, sk, v[t])
            M[:] = fma(np.broadcast_to(decay[t], M.shape), M, kt * w[:, None])
            out[t] = fma(d, sq, w * kq)
    return out.reshape(n, -1)


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("heads, kv, dk, dv, spare", [(2, 1, 64, 9, 3), (2, 2, 64, 8, 1), (2, 1, 32, 4, 0), (1, 1, 128, 6, 2), (1, 1, 100, 5, 3), (2, 2, 256, 4, 0), (1, 1, 512, 3, 1), (1, 1, 300, 3, 0)])
def test_delta_rule_sums_in_one_order(heads, kv, dk, dv, spare, channel):
    """The rule's results in bits: whole keys that are loaded four channels at a time (32, 64, 128, 256, 512 at aligned rows) and others, whole
    blocks of tokens and their ends, one row alone."""
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(dk)
    width = 2 * kv * dk + heads * dv
    lens = [21, 1, 34]
    n = sum(lens)
    wide = torch.randn(n, width + spare, generator=g)
    unit = wide[:, :2 * kv * dk].view(n, 2 * kv, dk)
    unit /= unit.norm(dim=2, keepdim=True)
    gates = torch.cat([torch.exp(-0.5 * torch.rand(n, heads * (dk if channel else 1), generator=g)), torch.rand(n, heads, generator=g)], 1)
    start = torch.tensor([0, 21, 22], dtype=torch.int32, device=DEV)
    length = torch.tensor(lens, dtype=torch.int32, device=DEV)
    slot = torch.tensor([2] * 21 + [0] + [1] * 34, dtype=torch.int32, device=DEV)
    tiles = -(-dv // 4)
    first = torch.randn(3, heads, tiles, dk, 4, generator=g)
    state, out = first.clone().view(3, -1).to(DEV), torch.full((n, heads * dv), 7.0, device=DEV)
    ops.delta_scan(wide.to(DEV), gates.to(DEV), start, length, slot, state, out, heads, kv, dk, dv, channel=channel)
    one_state, one = first.clone().view(3, -1).to(DEV), torch.full((1, heads * dv), 7.0, device=DEV)
    ops.delta_scan(wide[21:22].to(DEV), gates[21:22].to(DEV), start[:1], length[1:2], slot[21:22], one_state, one, heads, kv, dk, dv, channel=channel, single_rows=True)
    at = 0
    for m, s in zip(lens, (2, 0, 1)):
        M = first[s].permute(0, 2, 1, 3).reshape(heads, dk, 4 * tiles)[:, :, :dv].numpy().copy()
        want = _rule_in_its_order(wide[at:at + m, :width].numpy(), gates[at:at + m].numpy(), M, heads, kv, dk, dv, channel)
        assert torch.equal(out[at:at + m].cpu(), torch.from_numpy(want))
        held = state[s].view(heads, tiles, dk, 4).permute(0, 2, 1, 3).reshape(heads, dk, 4 * tiles)[:, :, :dv].cpu()
        assert torch.equal(held, torch.from_numpy(M))
        at += m
    assert torch.equal(one, out[21:22]) and torch.equal(one_state[0], state[0])


@pytest.mark.parametrize("channel", [False, True])
def test_delta_rule_of_single_rows_needs_no_runs(channel):
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(9)
    heads, kv, dk, dv, n = 4, 2, 40, 10, 5
    qkv, gates = torch.randn(n, 2 * kv * dk + heads * dv, generator=g).to(DEV), torch.rand(n, heads * ((dk if channel else 1) + 1), generator=g).to(DEV)
    slot, rows = torch.tensor([3, 0, 5, 1, 2], dtype=torch.int32, device=DEV), torch.arange(n, dtype=torch.int32, device=DEV)
    first = torch.randn(6, ops.delta_memory_floats(heads, dk, dv), generator=g).to(DEV)
    got = []
    for runs in ((rows, torch.ones_like(rows)), (None, None)):
        state, out = first.clone(), torch.empty(n, heads * dv, device=DEV)
        ops.delta_scan(qkv, gates, *runs, slot, state, out, heads, kv, dk, dv, channel=channel, single_rows=True)
        got.append((state, out))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    with pytest.raises(ops.KernelError):
        ops.delta_scan(qkv, gates, None, None, slot, state, out, heads, kv, dk, dv, channel=channel)


@pytest.mark.parametrize("H,d,r,rank,n,half_split", [(32, 64, 32, 256, 5, False), (3, 40, 8, 36, 16, True), (1, 8, 0, 16, 1, False), (4, 136, 64, 500, 7, True)])
def test_queries_of_a_few_rows_are_folded_in_one_launch(H, d, r, rank, n, half_split):
    """The bits of the two launches, whole and ragged strips of 16 columns and pieces of 32 channels, with and without turned channels; what it does not take is left alone."""
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(4)
    q = torch.randn(n, H * (d + r) + 4, generator=g).to(DEV)[:, :H * (d + r)]
    w = (torch.randn(H, rank, d, generator=g) * d ** -0.5).to(DEV, torch.bfloat16)
    angle = torch.randn(n, max(r // 2, 1), generator=g).to(DEV)
    cos, sin = (torch.cos(angle), torch.sin(angle)) if r else (None, None)
    plain, want = torch.empty(n, H * d, dtype=torch.bfloat16, device=DEV), torch.full((n, H * (rank + r)), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.latent_queries(q, cos, sin, plain, want, H, d, r, rank, half_split)
    assert ops.heads_product(plain, w, want, H, rank + r)
    got = torch.full_like(want, 7.0)
    assert ops.latent_fold(q, cos, sin, w, got, H, d, r, rank, half_split) and torch.equal(got, want)
    many = torch.zeros(17, H * (d + r), device=DEV)
    assert not ops.latent_fold(many, cos, sin, w, torch.empty(17, H * (rank + r), dtype=torch.bfloat16, device=DEV), H, d, r, rank, half_split)


def _delta_inputs(lens, heads, kv, dv, seed, steps=None, spare=0):
    """Rows as `delta_prepare` leaves them: unit keys, queries of length 1/8, decays as at initialisation, and where given one step size for all."""
    g = torch.Generator().manual_seed(seed)
    n, dk = sum(lens), 64
    qkv = torch.nn.functional.silu(0.5 * torch.randn(n, 2 * kv * dk + heads * dv + spare, generator=g))
    unit = qkv[:, :2 * kv * dk].view(n, 2 * kv, dk)
    unit /= unit.norm(dim=2, keepdim=True)
    qkv[:, :kv * dk] *= dk ** -0.5
    size = torch.exp(torch.rand(heads, generator=g) * 4.6 - 6.9)
    decay = torch.exp(-(1 + 15 * torch.rand(heads, generator=g)) * torch.nn.functional.softplus(torch.log(torch.expm1(size)) + 0.5 * torch.randn(n, heads, generator=g)))
    step = torch.sigmoid(torch.randn(n, heads, generator=g)) if steps is None else torch.full((n, heads), steps)
    return qkv, torch.cat([decay, step], 1)


@pytest.mark.parametrize("lens, least, heads, kv, dv, spare, steps", [([1777], 65, 8, 4, 128, 0, None), ([200, 3, 64, 65, 129], 65, 4, 2, 128, 4, None), ([128, 1], 64, 3, 1, 16, 0, None),
                                                                      ([66] * 70, 1, 2, 2, 48, 0, None), ([1, 63, 64, 2], 1, 2, 1, 208, 12, None), ([500], 65, 2, 1, 64, 0, 1.0)])
def test_delta_rule_in_blocks(lens, least, heads, kv, dv, spare, steps):
    """Blocks of 64 rows against the rule in 64 bits and against the scan, whose distance to it the blocks may not exceed by more than rounding's own
    spread; runs below `least` are left alone."""
    from geneinfer_amd.kernels import ops
    dk, n, tiles = 64, sum(lens), dv // 4
    qkv, gates = _delta_inputs(lens, heads, kv, dv, dv + n, steps, spare)
    starts = [sum(lens[:i]) for i in range(len(lens))]
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    slots = list(range(len(lens)))[::-1]
    rows = (qkv.to(DEV), gates.to(DEV), ints(starts), ints(lens))
    slot = ints([s for s, m in zip(slots, lens) for _ in range(m)])
    first = 0.2 * torch.randn(len(lens), heads, tiles, dk, 4, generator=torch.Generator().manual_seed(n))
    state, out = first.clone().view(len(lens), -1).to(DEV), torch.full((n, heads * dv), 7.0, device=DEV)
    ops.delta_chunks(*rows, lens, least, slot, state, out, heads, kv, dk, dv)
    scan_state, scan = first.clone().view(len(lens), -1).to(DEV), torch.full((n, heads * dv), 7.0, device=DEV)
    ops.delta_scan(*rows, slot, scan_state, scan, heads, kv, dk, dv)
    below_state, below = first.clone().view(len(lens), -1).to(DEV), torch.full((n, heads * dv), 7.0, device=DEV)
    ops.delta_scan(*rows, slot, below_state, below, heads, kv, dk, dv, below=least)
    far = lambda x, y, want: (float((x.double() - want).norm() / want.norm()), float((y.double() - want).norm() / want.norm()))
    for at, m, s in zip(starts, lens, slots):
        if m < least:
            assert torch.all(out[at:at + m] == 7.0) and torch.equal(state[s].cpu(), first[s].view(-1))
            assert torch.equal(below[at:at + m], scan[at:at + m]) and torch.equal(below_state[s], scan_state[s])
            continue
        assert torch.all(below[at:at + m] == 7.0) and torch.equal(below_state[s].cpu(), first[s].view(-1))
        M = first[s].permute(0, 2, 1, 3).reshape(heads, dk, dv).double()
        x, e = qkv[at:at + m].double(), gates[at:at + m].double()
        q, k = (x[:, i * kv * dk:(i + 1) * kv * dk].view(m, kv, dk).repeat_interleave(heads // kv, 1) for i in (0, 1))
        v, want = x[:, 2 * kv * dk:2 * kv * dk + heads * dv].view(m, heads, dv), torch.empty(m, heads, dv, dtype=torch.float64)
        for t in range(m):
            M = M * e[t, :heads, None, None]
            M = M + k[t][:, :, None] * (e[t, heads:, None] * (v[t] - torch.matmul(k[t][:, None], M)[:, 0]))[:, None]
            want[t] = torch.matmul(q[t][:, None], M)[:, 0]
        ours, scans = far(out[at:at + m].cpu(), scan[at:at + m].cpu(), want.view(m, -1))
        held, scan_held = far(*(y[s].view(heads, tiles, dk, 4).permute(0, 2, 1, 3).reshape(heads, dk, dv).cpu() for y in (state, scan_state)), M)
        print(f"{m} rows, {heads} heads, dv {dv}: read-outs {ours:.2e} (scan {scans:.2e}), memories {held:.2e} (scan {scan_held:.2e})", flush=True)
        # (2e-8: a third of a rounding, what two orders of the same sums differ by in their distance over one or two rows)
        assert ours < 1.2 * scans + 2e-8 and held < 1.2 * scan_held + 2e-8


@pytest.mark.parametrize("what, value", [("k", float("nan")), ("v", float("inf")), ("decay", float("nan")), ("q", float("-inf")), ("memory", float("nan"))])
def test_delta_rule_in_blocks_with_no_numbers(what, value):
    """A number that is none reaches what it reaches in the scan: its own row and the rows behind it, of its own head and columns."""
    from geneinfer_amd.kernels import ops
    lens, heads, kv, dk, dv = [300, 130], 4, 2, 64, 32
    qkv, gates = _delta_inputs(lens, heads, kv, dv, 5)
    state = torch.zeros(2, ops.delta_memory_floats(heads, dk, dv))
    if what == "memory":
        state[0, 70] = value
    elif what == "decay":
        gates[100, 1] = value
    else:
        qkv[100, {"q": 5, "k": kv * dk + 5, "v": 2 * kv * dk + dv + 3}[what]] = value
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    slot = ints([0] * 300 + [1] * 130)
    got = []
    for blocks in (True, False):
        st, out = state.clone().to(DEV), torch.empty(sum(lens), heads * dv, device=DEV)
        if blocks:
            ops.delta_chunks(qkv.to(DEV), gates.to(DEV), ints([0, 300]), ints(lens), lens, 65, slot, st, out, heads, kv, dk, dv)
        else:
            ops.delta_scan(qkv.to(DEV), gates.to(DEV), ints([0, 300]), ints(lens), slot, st, out, heads, kv, dk, dv)
        got.append((out.cpu(), st.cpu()[:, :state.shape[1]]))
    assert not bool(torch.isfinite(got[1][0]).all())
    for ours, scans in zip(*got):
        assert torch.equal(torch.isfinite(ours), torch.isfinite(scans)) and torch.equal(ours.isnan(), scans.isnan())
        keep = torch.isfinite(scans)
        assert relative_error(ours[keep].double(), scans[keep].double()) < 2e-6


def test_a_prompt_without_room_for_the_blocks_goes_token_by_token(tmp_path, monkeypatch):
    """A device that has no room for what the blocks of a long prompt hand on: the scan's logits and memories, which need none."""
    from geneinfer_amd.engine import Runner, StepEntry, load_model
    from geneinfer_amd.kernels import ops
    layer = dict(type="delta", mlp=dict(kind="dense", ff=128), mixer=dict(heads=2, kv_heads=1, dim=64, vdim=64, conv=4))
    cfg = dict(architecture="Rigalorn", vocab=97, width=64, embedding=dict(scale=8.0), norm=dict(eps=1e-5), max_positions=1024, layers=[layer])
    write_model(tmp_path, cfg, seed=5)
    model, tokens = load_model(tmp_path, "bfloat16", DEV), _prompt(cfg, 400, 6)
    assert ops.delta_chunks_pay([400], 65, 2)
    got = {}
    for what in ("blocks", "no room", "scan"):
        with monkeypatch.context() as patch:
            if what == "no room":
                patch.setattr(ops, "_room", lambda floats, device: None)
            if what == "scan":
                patch.setattr(ops, "delta_chunks_pay", lambda *a: False)
            runner = Runner(model, page_size=16, max_tokens=1024, max_requests=2)
            runner.open("r")
            got[what] = [runner.step([StepEntry("r", tokens[:399], tuple(range(399)))]).cpu().clone(), runner.step([StepEntry("r", tokens[399:], (0,))]).cpu().clone()]
    assert all(torch.equal(x, y) for x, y in zip(got["no room"], got["scan"])) and not torch.equal(got["blocks"][0], got["scan"][0])
    assert relative_error(got["blocks"][0], got["scan"][0].double()) < 1e-2


def test_delta_rule_takes_very_wide_values():
    """More tiles of four value channels than half of what a launch's third dimension holds."""
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(4)
    n, dk, dv = 3, 8, 4 * 32768 + 3
    qkv = torch.randn(n, 2 * dk + dv, generator=g)
    gates = torch.rand(n, 2, generator=g)
    ints = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    state, out = torch.zeros(1, ops.delta_memory_floats(1, dk, dv), device=DEV), torch.empty(n, dv, device=DEV)
    ops.delta_scan(qkv.to(DEV), gates.to(DEV), ints(0), ints(n), ints(0, 0, 0), state, out, 1, 1, dk, dv)
    x = qkv.double()
    assert relative_error(out, P.delta_rule(x[:, :dk], x[:, dk:2 * dk], x[:, 2 * dk:], gates[:, 1].double(), gates[:, 0].double())) < 1e-5


def test_head_norm_with_shared_weights_and_a_silu_gate():
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(3)
    n, heads, dv, eps = 9, 3, 37, 1e-3
    o, gate, w = torch.randn(n, heads * dv, generator=g), 2 * torch.randn(n, heads * dv, generator=g), 1 + 0.1 * torch.randn(dv, generator=g)
    od = o.double().view(n, heads, dv)
    want = (od / torch.sqrt((od * od).mean(-1, keepdim=True) + eps) * w.double()).reshape(n, -1) * (gate.double() * torch.sigmoid(gate.double()))
    out = torch.empty(n, heads * dv, device=DEV)
    ops.head_norm_gate(o.to(DEV), gate.to(DEV), w.to(DEV), eps, out, heads, dv, gate_activation="silu")
    assert relative_error(out, want) < 1e-6


def _paged(T, page, n_numbers, dtype, seed):
    """Pages for one request of T positions in slot 1, in a shuffled order, and its table."""
    n_pages = -(-T // page)
    order = torch.randperm(n_pages + 3, generator=torch.Generator().manual_seed(seed))[:n_pages]
    table = torch.full((3, n_pages + 2), -1, dtype=torch.int32)
    table[1, :n_pages] = order.to(torch.int32)
    cache = torch.zeros(n_pages + 3, page * n_numbers, dtype=dtype, device=DEV)
    return cache, table.to(DEV)


def _ctx(T, pos0=0, slot=1):
    from geneinfer_amd.parts import StepContext
    pos = torch.arange(pos0, pos0 + T, dtype=torch.int32, device=DEV)
    slots = torch.full((T,), slot, dtype=torch.int32, device=DEV)
    return StepContext(n_rows=T, dtype=torch.float32, device=torch.device(DEV), tokens=slots, row_pos=pos, row_slot=slots, seg_slot=[slot], seg_start=[0],
                       seg_len=[T], seg_pos0=[pos0])


@pytest.mark.parametrize("T, window, far", [(300, None, 3), (300, 36, 264), (300, 36, 263), (131, 17, 114), (131, 17, 113), (70, 1, 69), (70, 64, 6), (70, 64, 5)])
def test_attention_with_biases_blended_values_and_one_key_that_stands_out(T, window, far):
    """The last row's query points at the key of position `far`, which is scaled up so that, if seen, it takes nearly all the
    weight: just inside the window, just outside it, or hundreds of positions back.  Biases, a rotation of a part of the head with
    lengthened cosines, and values blended with another layer's are all on."""
    from geneinfer_amd.kernels import ops
    heads, kv, dk, dv, rot, page, scale = 4, 2, 24, 10, 8, 4, 0.3
    g = torch.Generator().manual_seed(T + far)
    q, k, v = torch.randn(T, heads * dk, generator=g), torch.randn(T, kv * dk, generator=g), torch.randn(T, kv * dv, generator=g)
    qb, kb, vb = torch.randn(heads * dk, generator=g), torch.randn(kv * dk, generator=g), torch.randn(kv * dv, generator=g)
    other, blend = torch.randn(T, kv * dv, generator=g), torch.tensor([0.35])
    freqs, mag = P.rotary_frequencies(rot, 30.0, dict(factor=4.0, original=16, fast=2.0, slow=0.5))
    # the unrotated channels of key `far` and of the last query line up, large
    k.view(T, kv, dk)[far, :, rot:] = 3.0
    q.view(T, heads, dk)[T - 1, :, rot:] = 3.0
    qd, kd = (q + qb).double().view(T, heads, dk), (k + kb).double().view(T, kv, dk)
    vd = (1 - 0.35) * (v + vb).double() + 0.35 * other.double()
    want = P.softmax_attention(P.rotate_half_split(qd, freqs, mag), P.rotate_half_split(kd, freqs, mag), vd.view(T, kv, dv), scale, window)
    seen = window is None or T - 1 - far < window
    weight = torch.softmax((torch.einsum("hd,shd->hs", P.rotate_half_split(qd, freqs, mag)[T - 1], P.rotate_half_split(kd, freqs, mag).repeat_interleave(2, 1)) * scale)
                           .masked_fill(~P.window_mask(T, window)[T - 1][None], float("-inf")), -1)[:, far]
    assert (weight > 0.9).all() if seen else (weight == 0).all()          # (the test's premise: the key matters exactly when it is seen)

    cache, table = _paged(T, page, kv * (dk + dv), torch.float32, seed=far)
    ctx = _ctx(T)
    cos, sin = torch.empty(T, rot // 2, device=DEV), torch.empty(T, rot // 2, device=DEV)
    ops.rope_cos_sin(ctx.row_pos, torch.tensor(freqs, dtype=torch.float64, device=DEV), cos, sin, mag)
    q_ready, keep = torch.empty(T, heads * dk, device=DEV), torch.empty(T, kv * dv, device=DEV)
    dev = lambda t: t.to(DEV)
    ops.norm_rope_store(dev(q), dev(k), dev(v), None, None, 1e-6, cos, sin, rot, ctx.row_pos, ctx.row_slot, table, q_ready, cache, page, heads, kv, dk, dv,
                        biases=(dev(qb), dev(kb), dev(vb)), blend=(dev(other), dev(blend)), keep=keep)
    assert relative_error(keep, (v + vb).double()) < 1e-6
    out = torch.empty(T, heads * dv, device=DEV)
    ops.attention_general(q_ready, cache, out, ctx, table, heads, kv, dk, page_size=page, value_dim=dv, window=window, scale=scale)
    assert relative_error(out.view(T, heads, dv), want) < 2e-5
    assert relative_error(out.view(T, heads, dv)[T - 1], want[T - 1]) < 2e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, kv, dk, dv, rot, page, extras", [(4, 2, 64, 64, 32, 16, "all"), (6, 3, 24, 10, 8, 8, "all"), (2, 2, 4, 7, 0, 24, "biases"), (5, 1, 128, 128, 128, 4, "none"), (4, 2, 64, 33, 16, 16, "growth")])
def test_rows_of_prompts_are_turned_and_stored_as_rows_one_by_one(heads, kv, dk, dv, rot, page, extras, dtype):
    """Rows of three requests (one from the middle of eight positions on, one of a few rows that shares windows with both others, one from a multiple of eight) in the kernel
    for many rows and heads (10,000 together), and the same rows 100 at a time: queries, pages and kept values in bits."""
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(dk + dv)
    lens, firsts = [875, 4, 890], [5, 863, 16]
    n = sum(lens)
    q, k, v, other = (torch.randn(n, width, generator=g).to(DEV) for width in (heads * dk, kv * dk, kv * dv, kv * dv))
    biases = tuple(torch.randn(width, generator=g).to(DEV) for width in (heads * dk, kv * dk, kv * dv)) if extras in ("all", "biases") else None
    blend = (other, torch.tensor([0.35], device=DEV)) if extras == "all" else None
    pos = torch.cat([torch.arange(p, p + m) for p, m in zip(firsts, lens)]).to(DEV, torch.int32)
    slot = torch.cat([torch.full((m,), s) for s, m in zip((2, 0, 1), lens)]).to(DEV, torch.int32)
    pages = 3 * -(-906 // page)
    assert n * (heads + 2 * kv) >= 10000 > 100 * (heads + 2 * kv)
    table = torch.randperm(pages, generator=g).view(3, -1).to(DEV, torch.int32)
    cos, sin = (torch.randn(n, rot // 2, generator=g).to(DEV) for _ in range(2)) if rot else (None, None)
    got = []
    for step in (n, 100):
        cache = torch.full((pages, kv * (dk + dv) * page), 9.0, dtype=dtype, device=DEV).view(pages, 1, kv * (dk + dv), page)
        q_out, keep = torch.empty(n, heads * dk, dtype=dtype, device=DEV), torch.empty(n, kv * dv, device=DEV) if extras == "all" else None
        for a in range(0, n, step):
            b = min(n, a + step)
            cut = lambda x: None if x is None else x[a:b]
            ops.norm_rope_store(q[a:b], k[a:b], v[a:b], None, None, 1e-6, cut(cos), cut(sin), rot, pos[a:b], slot[a:b], table, q_out[a:b], cache, page, heads, kv, dk, dv, biases=biases,
                                blend=None if blend is None else (other[a:b], blend[1]), keep=cut(keep), v_scale=0.7 if extras == "biases" else 1.0,
                                query_growth=(0.1, 20.0) if extras == "growth" else None)
        got.append((q_out, cache, keep))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and (got[0][2] is None or torch.equal(got[0][2], got[1][2]))
    assert bool((got[0][1] != 9.0).any())


def test_queries_of_many_rows_may_be_turned_in_their_own_place():
    """32-bit queries written over themselves, heads of 24 channels, whose pairs lie in two waves now and then: the numbers of queries written elsewhere."""
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(3)
    n, heads, kv, dk, page, rot = 600, 21, 1, 24, 8, 24
    q, k, v = (torch.randn(n, width * dk, generator=g).to(DEV) for width in (heads, kv, kv))
    cos, sin = (torch.randn(n, rot // 2, generator=g).to(DEV) for _ in range(2))
    pos, slot, table = torch.arange(n, dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV), torch.arange(n // page, dtype=torch.int32, device=DEV).view(1, -1)
    got = []
    for out in (torch.empty_like(q), q):
        cache = torch.zeros(n // page, 1, 2 * kv * dk, page, device=DEV)
        ops.norm_rope_store(q, k, v, None, None, 1e-6, cos, sin, rot, pos, slot, table, out, cache, page, heads, kv, dk, dk)
        got.append((out, cache))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("T, window, far", [(200, None, 2), (200, 50, 150), (200, 50, 149), (45, 16, 29), (45, 16, 30)])
def test_attention_through_latents_against_keys_and_values_made_in_full(T, window, far):
    """The kernels around the latent cache and the attention over it, with the up projections folded into query and output by hand
    here, against the plain layer that makes every head's keys and values of every position."""
    from geneinfer_amd.kernels import ops
    H, d, r, dv, q_rank, rank, page, scale, eps = 3, 12, 6, 7, 20, 18, 4, 0.3, 1e-5
    g = torch.Generator().manual_seed(T + far)
    m = dict(heads=H, dim=d, rot_dim=r, vdim=dv, kv_rank=rank, q_rank=q_rank, scale=scale, rot=dict(dims=r, base=40.0), mask=None if window is None else dict(size=window))
    hidden = 16
    w = {"dq": torch.randn(q_rank, hidden, generator=g) * 0.3, "dq.norm": 1 + 0.1 * torch.randn(q_rank, generator=g), "uq": torch.randn(H * (d + r), q_rank, generator=g) * 0.3,
         "dkv": torch.randn(rank + r, hidden, generator=g) * 0.3, "dkv.norm": 1 + 0.1 * torch.randn(rank, generator=g), "uk": torch.randn(H * d, rank, generator=g) * 0.3,
         "uv": torch.randn(H * dv, rank, generator=g) * 0.3, "o": torch.eye(H * dv)}
    h = torch.randn(T, hidden, generator=g)
    h[far] *= 6.0                                                        # a position whose latent is long: its scores are large either way
    want = P.latent_attention(h.double(), {k: v.double() for k, v in w.items()}, m, eps)

    dev = lambda t: t.to(DEV)
    cache, table = _paged(T, page, 2 * rank + r, torch.float32, seed=far)
    ctx = _ctx(T)
    f, _ = P.rotary_frequencies(r, 40.0)
    cos, sin = torch.empty(T, r // 2, device=DEV), torch.empty(T, r // 2, device=DEV)
    ops.rope_cos_sin(ctx.row_pos, torch.tensor(f, dtype=torch.float64, device=DEV), cos, sin)
    down = dev(torch.cat([h @ w["dq"].T, h @ w["dkv"].T], dim=1).contiguous())
    cq = torch.empty(T, q_rank, device=DEV)
    ops.latent_prepare(down, q_rank, rank, r, dev(w["dq.norm"]), dev(w["dkv.norm"]), eps, cos, sin, ctx.row_pos, ctx.row_slot, table, cq, cache, page)
    q = (cq @ dev(w["uq"]).T).contiguous()
    plain_part, folded = torch.empty(T, H * d, device=DEV), torch.empty(T, H * (rank + r), device=DEV)
    ops.latent_queries(q, cos, sin, plain_part, folded, H, d, r, rank)
    uk = dev(w["uk"]).view(H, d, rank)
    folded.view(T, H, rank + r)[:, :, :rank] = torch.einsum("thd,hdr->thr", plain_part.view(T, H, d), uk)
    att = torch.empty(T, H * rank, device=DEV)
    ops.attention_general(folded, cache, att, ctx, table, H, 1, rank + r, page_size=page, value_dim=rank, window=window, scale=scale)
    got = torch.einsum("thr,hvr->thv", att.view(T, H, rank), dev(w["uv"]).view(H, dv, rank)).reshape(T, H * dv)
    assert relative_error(got, want) < 3e-5


@pytest.mark.parametrize("H, kd, vd, window, lens, pos0", [(20, 152, 136, 44, [1, 1, 1], [700, 43, 0]), (8, 80, 64, None, [130, 1], [0, 300]), (32, 288, 256, 100, [70], [50]),
                                                          (3, 24, 16, 17, [33, 2, 1], [15, 16, 17]), (16, 96, 64, 1, [20], [0]), (16, 576, 512, 48, [40, 1], [30, 200]),
                                                          (5, 296, 264, None, [3], [60]), (16, 576, 512, 48, [100, 1], [30, 200]), (20, 152, 136, 44, [130, 70, 1], [700, 0, 5]),
                                                          (40, 80, 64, None, [90], [10]), (8, 288, 256, 300, [129, 200], [77, 0]), (130, 32, 16, 20, [80], [3])])
def test_matrix_core_attention_over_latent_pages(H, kd, vd, window, lens, pos0):
    """Requests at other positions each, on shuffled pages: single rows whose context is shared out over several waves, and
    portions of prompts; heads that fill one and a half matrix instructions; keys that are no multiple of 32 channels.  One key
    just inside every row's window stands out."""
    from geneinfer_amd.kernels import ops
    from geneinfer_amd.parts import StepContext
    g = torch.Generator().manual_seed(H + kd)
    page, scale = 16, 0.2
    total = [p + n for p, n in zip(pos0, lens)]
    n_pages = sum(-(-t // page) for t in total)
    order = torch.randperm(n_pages + 2, generator=g).tolist()
    table = torch.full((len(lens) + 1, max(-(-t // page) for t in total) + 1), -1, dtype=torch.int32)
    cache = torch.zeros(n_pages + 2, page * (kd + vd), dtype=torch.bfloat16)
    keys = []
    for s, t in enumerate(total):
        k = torch.randn(t, kd, generator=g).to(torch.bfloat16)
        keys.append(k)
        for i in range(-(-t // page)):
            pg = order.pop()
            table[s, i] = pg
            block = k[i * page:(i + 1) * page]
            cache[pg, :block.shape[0] * kd] = block.reshape(-1)
            values = torch.zeros(vd, page, dtype=torch.bfloat16)
            values[:, :block.shape[0]] = block[:, :vd].T
            cache[pg, page * kd:] = values.reshape(-1)
    q = torch.randn(sum(lens), H * kd, generator=g)
    row = 0
    want = []
    for s, (p0, n) in enumerate(zip(pos0, lens)):
        kf = keys[s].double()
        for i in range(n):
            p = p0 + i
            lo = 0 if window is None else max(0, p - window + 1)
            q.view(-1, H, kd)[row + i, :, :8] = 4.0 * kf[lo, :8] / kf[lo, :8].norm()        # the oldest key the row sees stands out
        qb = q[row:row + n].to(torch.bfloat16).double().view(n, H, kd)
        scores = torch.einsum("thd,sd->hts", qb, kf) * scale
        i_, j_ = torch.arange(p0, p0 + n)[:, None], torch.arange(total[s])[None, :]
        seen = (j_ <= i_) & ((i_ - j_ < window) if window is not None else True)
        pr = torch.softmax(scores.masked_fill(~seen[None], float("-inf")), -1)
        want.append(torch.einsum("hts,sd->thd", pr, kf[:, :vd]).reshape(n, H * vd))
        row += n
    want = torch.cat(want)
    T = sum(lens)
    starts = [sum(lens[:i]) for i in range(len(lens))]
    pos = torch.tensor([p + i for p, n in zip(pos0, lens) for i in range(n)], dtype=torch.int32, device=DEV)
    slots = torch.tensor([s for s, n in enumerate(lens) for _ in range(n)], dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=slots, row_pos=pos, row_slot=slots, seg_slot=list(range(len(lens))),
                      seg_start=starts, seg_len=list(lens), seg_pos0=list(pos0))
    assert ops.latent_attention_bf16_supports(kd, vd, page)
    out = torch.empty(T, H * vd, dtype=torch.bfloat16, device=DEV)
    ops.latent_attention_bf16(q.to(DEV, torch.bfloat16), cache.to(DEV), out, ctx, table.to(DEV), H, kd, vd, page, window, scale)
    assert relative_error(out, want) < 1.5e-2                                   # (probabilities and outputs are kept in bfloat16)
    exact = torch.empty(T, H * vd, dtype=torch.bfloat16, device=DEV)
    ops.attention_general(q.to(DEV, torch.bfloat16), cache.to(DEV), exact, ctx, table.to(DEV), H, 1, kd, page_size=page, value_dim=vd, window=window, scale=scale)
    assert relative_error(exact, want) < 6e-3 and relative_error(out, exact.double()) < 1.5e-2


@pytest.mark.parametrize("H, kd, vd, window, lens, pos0", [(32, 288, 256, 1000, [270], [900]), (64, 88, 56, None, [140, 33], [0, 40]), (96, 160, 128, 33, [65], [7]), (256, 24, 16, 20, [70], [3]),
                                                          (32, 256, 248, 31, [100, 1], [31, 9]), (160, 96, 64, None, [66], [0])])
def test_matrix_core_attention_over_latent_pages_with_heads_in_groups_of_32(H, kd, vd, window, lens, pos0):
    """A wave per row and 32 heads: one to eight groups, numbers of groups that leave waves without a row, keys and values shorter than the kernel's."""
    test_matrix_core_attention_over_latent_pages(H, kd, vd, window, lens, pos0)


@pytest.mark.parametrize("H, kd, vd", [(32, 288, 256), (64, 160, 128), (32, 88, 56)])
@pytest.mark.parametrize("window, pos0, n", [(None, 0, 70), (None, 47, 33), (5, 31, 66), (33, 96, 40), (100, 200, 17), (1, 15, 34)])
def test_prompt_rows_over_latent_pages_of_any_size(H, kd, vd, window, pos0, n):
    """Tiles of 32 positions over pages of 16 (two a tile), 48 (one or two), 32 and 112, looked up a tile ahead: first and last tiles of which half is seen, walks of one, two and more
    tiles; the same numbers in the same order, so the same bits, and pages that no row sees hold no number at all."""
    from geneinfer_amd.kernels import ops
    from geneinfer_amd.parts import StepContext
    g = torch.Generator().manual_seed(pos0 + n + kd)
    total = pos0 + n
    k, q = torch.randn(total, kd, generator=g).to(torch.bfloat16), torch.randn(n, H * kd, generator=g).to(torch.bfloat16)
    pos = torch.arange(pos0, total, dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=n, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=torch.zeros_like(pos), seg_slot=[0], seg_start=[0], seg_len=[n], seg_pos0=[pos0])
    first, outs = max(0, pos0 - (window or total) + 1), []
    for page in (16, 48, 32, 112):
        pages = -(-total // page)
        cache = torch.full((pages + 1, page * (kd + vd)), float("nan"), dtype=torch.bfloat16)
        table = torch.full((1, pages), pages, dtype=torch.int32)                   # (pages behind every window are somebody else's)
        for i in range(first // page, pages):
            block = torch.zeros(page, kd, dtype=torch.bfloat16)
            block[:len(k[i * page:(i + 1) * page])] = k[i * page:(i + 1) * page]
            table[0, i] = pages - 1 - i
            cache[pages - 1 - i] = torch.cat([block.reshape(-1), block[:, :vd].T.reshape(-1)])
        out = torch.empty(n, H * vd, dtype=torch.bfloat16, device=DEV)
        outs.append(ops.latent_attention_bf16(q.to(DEV), cache.to(DEV), out, ctx, table.to(DEV), H, kd, vd, page, window, 0.2))
    i_, j_ = torch.arange(pos0, total)[:, None], torch.arange(total)[None]
    scores = torch.einsum("thd,sd->hts", q.double().view(n, H, kd), k.double()) * 0.2
    want = torch.einsum("hts,sd->thd", torch.softmax(scores.masked_fill(~((j_ <= i_) & (i_ - j_ < (window or total + 1)))[None], float("-inf")), -1), k[:, :vd].double()).reshape(n, -1)
    assert relative_error(outs[0], want) < 1.5e-2                                  # (as above)
    for out in outs[1:]:
        assert torch.equal(out, outs[0])


@pytest.mark.parametrize("n, H, context, window", [(40, 32, 500, None), (12, 32, 4000, None), (60, 32, 511, 300), (32, 32, 500, None), (65, 20, 333, None)])
def test_single_rows_over_latent_pages_in_more_waves_than_places(n, H, context, window):
    """Shares of one and two tiles, on both sides of a wave for every place of the chip: the kernels that ask for the values before and behind the scores give the
    same bits, and the right ones."""
    from geneinfer_amd.kernels import ops
    from geneinfer_amd.parts import StepContext
    kd, vd, page = 288, 256, 16
    g = torch.Generator(device=DEV).manual_seed(n)
    pages = -(-context // page)
    cache = torch.randn(n * pages, page * (kd + vd), generator=g, device=DEV).to(torch.bfloat16)
    keys = cache[:, :page * kd].reshape(n, pages * page, kd)
    cache[:, page * kd:] = keys.reshape(n * pages, page, kd)[:, :, :vd].transpose(1, 2).reshape(n * pages, -1)
    table = torch.arange(n * pages, dtype=torch.int32, device=DEV).view(n, pages)
    at = [context - 1 - (7 * i) % (context // 2) for i in range(n)]
    q = torch.randn(n, H, kd, generator=g, device=DEV).to(torch.bfloat16)
    pos, slots = torch.tensor(at, dtype=torch.int32, device=DEV), torch.arange(n, dtype=torch.int32, device=DEV)
    seen = []
    for known in (True, False):
        ctx = StepContext(n_rows=n, dtype=torch.bfloat16, device=torch.device(DEV), tokens=pos, row_pos=pos, row_slot=slots, seg_slot=list(range(n)), seg_start=list(range(n)), seg_len=[1] * n, seg_pos0=at)
        plan = ops._plan_of(ctx)
        plan.decode_positions = plan.decode_positions if known else None
        seen.append(torch.empty(n, H * vd, dtype=torch.bfloat16, device=DEV))
        ops.latent_attention_bf16(q.view(n, -1), cache, seen[-1], ctx, table, H, kd, vd, page, window, 0.06)
    assert torch.equal(*seen)
    for i in (0, 1, n // 2, n - 1):
        k = keys[i, max(0, at[i] - window + 1) if window else 0:at[i] + 1].double()
        want = torch.softmax(0.06 * (q[i].double() @ k.T), -1) @ k[:, :vd]
        assert relative_error(seen[0][i], want.reshape(-1).cpu()) < 1e-2


@pytest.mark.parametrize("page, window", [(16, None), (48, 130), (64, None)])
def test_latent_attention_with_scores_that_climb_along_the_context_and_sinks(page, window):
    """Scores grow along the context by 0 to 12 units a tile of 32 positions, up to 60 and more: a column's maximum moves in every tile, by less and by more than what
    it may lag behind, and a maximum applied wrongly once is a factor.  Some heads' sinks are larger than every score."""
    from geneinfer_amd.kernels import ops
    from geneinfer_amd.parts import StepContext
    H, kd, vd, T, p0, scale = 32, 288, 256, 150, 203, 0.1
    g = torch.Generator().manual_seed(page)
    total = p0 + T
    n_pages = -(-total // page)
    order = torch.randperm(n_pages + 2, generator=g).tolist()
    table = torch.full((1, n_pages + 1), -1, dtype=torch.int32)
    cache = torch.zeros(n_pages + 2, page * (kd + vd), dtype=torch.bfloat16)
    direction = torch.nn.functional.normalize(torch.randn(kd, generator=g), dim=0)
    height = torch.cumsum(torch.where(torch.arange(total) < 120, 0.02, torch.where(torch.arange(total) < 280, 0.35, -0.2)), 0)
    k = (0.3 * torch.randn(total, kd, generator=g) + height[:, None] / scale / 8 * direction).to(torch.bfloat16)
    for i in range(n_pages):
        block = k[i * page:(i + 1) * page]
        table[0, i] = pg = order.pop()
        cache[pg, :block.shape[0] * kd] = block.reshape(-1)
        values = torch.zeros(vd, page, dtype=torch.bfloat16)
        values[:, :block.shape[0]] = block[:, :vd].T
        cache[pg, page * kd:] = values.reshape(-1)
    q = (8 * direction + 0.3 * torch.randn(T, H, kd, generator=g)).to(torch.bfloat16)
    sinks = torch.where(torch.arange(H) % 5 == 0, 70.0, torch.randn(H, generator=g))
    scores = torch.einsum("thd,sd->hts", q.double(), k.double()) * scale
    i_, j_ = torch.arange(p0, total)[:, None], torch.arange(total)[None, :]
    seen = (j_ <= i_) & ((i_ - j_ < window) if window else True)
    scores = torch.cat([scores.masked_fill(~seen[None], float("-inf")), sinks.double()[:, None, None].expand(H, T, 1)], -1)
    assert float(scores[1].max()) > 50
    want = torch.einsum("hts,sd->thd", torch.softmax(scores, -1)[..., :-1], k[:, :vd].double()).reshape(T, H * vd)
    pos = torch.arange(p0, total, dtype=torch.int32, device=DEV)
    slots = torch.zeros(T, dtype=torch.int32, device=DEV)
    ctx = StepContext(n_rows=T, dtype=torch.bfloat16, device=torch.device(DEV), tokens=slots, row_pos=pos, row_slot=slots, seg_slot=[0], seg_start=[0], seg_len=[T], seg_pos0=[p0])
    out = torch.empty(T, H * vd, dtype=torch.bfloat16, device=DEV)
    ops.latent_attention_bf16(q.view(T, -1).to(DEV), cache.to(DEV), out, ctx, table.to(DEV), H, kd, vd, page, window, scale, sinks.to(DEV))
    assert relative_error(out, want) < 1.5e-2                                   # (probabilities and outputs are kept in bfloat16)


@pytest.mark.parametrize("rows, H, k, n", [(1, 8, 32, 128), (37, 3, 72, 40), (300, 32, 64, 256), (16, 2, 256, 64), (5, 1, 8, 7),
                                           (300, 3, 72, 40), (575, 21, 64, 36), (577, 19, 40, 100), (13, 65, 64, 512), (16, 64, 40, 500)])
def test_every_head_s_product_in_one_launch(rows, H, k, n):
    from geneinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(rows + k)
    a, w = torch.randn(rows, H * k, generator=g).to(torch.bfloat16), torch.randn(H, n, k, generator=g).to(torch.bfloat16)
    want = torch.einsum("thk,hnk->thn", a.double().view(rows, H, k), w.double())
    for dtype, stride, tol in ((torch.float32, n, 1e-5), (torch.bfloat16, n + 24, 5e-3)):
        out = torch.zeros(rows, H * stride, dtype=dtype, device=DEV)
        assert ops.heads_product(a.to(DEV), w.to(DEV), out, H, stride)
        got = out.view(rows, H, stride)
        assert relative_error(got[:, :, :n], want) < tol and (got[:, :, n:] == 0).all()
    assert not ops.heads_product(a.to(DEV)[:, 1:], w.to(DEV), out, H, n)           # operands it does not take: the caller goes head by head


@pytest.mark.parametrize("rows, n", [(2, 65535 * 16), (2, 65535 * 16 + 5), (17, 65535 * 16 + 5)])
def test_a_head_s_product_of_more_columns_than_a_grid_has_strips_of_16(rows, n):
    from geneinfer_amd.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(rows)
    a, w = torch.randn(rows, 8, generator=g, device=DEV).to(torch.bfloat16), torch.randn(1, n, 8, generator=g, device=DEV).to(torch.bfloat16)
    out = torch.zeros(rows, n + 3, device=DEV)
    assert ops.heads_product(a, w, out[:, :n], 1)
    assert relative_error(out[:, :n], a.double() @ w[0].double().T) < 1e-5 and (out[:, n:] == 0).all()


# =============================================================================================== whole models
def _portions(n, sizes=(7, 2, 5, 3, 2, 11, 1, 4, 2, 19)):
    out, i = [], 0
    while sum(out) + sizes[i % len(sizes)] <= n:
        out.append(sizes[i % len(sizes)])
        i += 1
    return out


CUTS = {"whole": lambda n: [n], "singly": lambda n: [], "most then singly": lambda n: [n - 9], "portions": _portions, "twos": lambda n: [2] * (n // 2)}


@pytest.mark.parametrize("name", list(CONFIGS))
def test_float32_logits_match_the_plain_model_and_do_not_depend_on_the_cut(folders, name):
    tokens = _prompt(CONFIGS[name], 75, 5)
    runner = make_runner(folders, name, "float32")
    got = {}
    for what, cuts in CUTS.items():
        runner.open(what)
        got[what] = feed(runner, what, tokens, cuts(len(tokens)))
        runner.close(what)
    check_against_plain(folders, name, "float32", tokens, got["whole"], f"{name} whole")
    for what in CUTS:
        assert torch.equal(got[what], got["whole"]), f"{name}: the logits of '{what}' differ from those of the whole prompt"


@pytest.mark.parametrize("name", list(CONFIGS))
def test_bfloat16_logits_lie_within_rounding_noise(folders, name):
    tokens = _prompt(CONFIGS[name], 90, 6)
    runner = make_runner(folders, name, "bfloat16")
    for what in ("whole", "portions", "most then singly"):
        runner.open(what)
        got = feed(runner, what, tokens, CUTS[what](len(tokens)))
        runner.close(what)
        check_against_plain(folders, name, "bfloat16", tokens, got, f"{name} {what}")


@pytest.mark.parametrize("name, dtype", [("A", "float32"), ("B", "float32"), ("D", "float32"), ("E", "float32"), ("A", "bfloat16"), ("C", "bfloat16")])
def test_mixed_batches_on_a_pool_that_is_used_again(folders, name, dtype):
    """Up to four live requests, portions of some beside single tokens of others, through a pool that holds less than all requests
    together and four state slots: pages and slots are freed and used again.  Every request's logits against itself alone."""
    import random
    import traces
    from geneinfer_amd.engine import StepEntry
    cfg = CONFIGS[name]
    rng = random.Random(8)
    requests = {f"q{i}": [rng.randrange(cfg["vocab"]) for _ in range(n)] for i, n in enumerate([50, 1, 33, 77, 40, 9, 2, 61])}
    steps = traces.mixed(requests, seed=5)
    runner = make_runner(folders, name, dtype, max_tokens=traces.peak_tokens(steps, 64), max_requests=4)
    got = {}
    where = traces.wanted_positions(steps)
    for s in steps:
        for e in s["entries"]:
            if not runner.is_open(e["id"]):
                runner.open(e["id"])
        logits = runner.step([StepEntry(e["id"], e["tokens"], e["want"]) for e in s["entries"]])
        if logits is not None:
            for key, row in zip(where[s["step"]], logits.cpu()):
                got[key] = row.clone()
        for rid in s["end"]:
            runner.close(rid)
    runner.cache.check_consistency()
    alone = make_runner(folders, name, dtype)
    for rid, tokens in requests.items():
        mine = {p: row for (r, p), row in got.items() if r == rid}
        assert len(mine) == len(tokens)
        if dtype == "float32":
            alone.open(rid)
            ref = feed(alone, rid, tokens, [len(tokens)])
            alone.close(rid)
            assert all(torch.equal(mine[p], ref[p]) for p in mine), f"{name} {rid}: a mixed batch changed the logits"
        else:
            exact, rounded = plain_logits(folders, name, tokens), plain_logits(folders, name, tokens, rounded=True)
            assert_within_bfloat16_noise(mine, lambda p: exact[p], lambda p: rounded[p], f"{name} mixed {rid}")


@pytest.mark.parametrize("name, dtype", [("C", "bfloat16"), ("C", "float32"), ("B", "float32")])
def test_long_portions_beside_single_rows(folders, name, dtype):
    """Steps that hold portions of a hundred rows and more of some requests (the kernels that take the rows of prompts tile by tile)
    beside single rows and short portions of others, every request at another position."""
    from geneinfer_amd.engine import StepEntry
    cfg = CONFIGS[name]
    tokens = {r: _prompt(cfg, n, 70 + n) for r, n in (("a", 330), ("b", 150), ("c", 171), ("d", 40))}
    schedule = [[("a", 100), ("c", 70)], [("a", 130), ("b", 1), ("c", 1)], [("b", 140), ("a", 1), ("c", 99), ("d", 3)], [("a", 99), ("b", 2), ("c", 1), ("d", 37)], [("b", 7)]]
    runner = make_runner(folders, name, dtype, max_tokens=1024, max_requests=4)
    at, got = {r: 0 for r in tokens}, {r: [] for r in tokens}
    for step in schedule:
        entries = []
        for r, n in step:
            if not runner.is_open(r):
                runner.open(r)
            entries.append(StepEntry(r, tokens[r][at[r]:at[r] + n], tuple(range(n))))
        logits = runner.step(entries).cpu()
        row = 0
        for r, n in step:
            got[r].append(logits[row:row + n])
            row += n
            at[r] += n
    assert all(at[r] == len(t) for r, t in tokens.items())
    alone = make_runner(folders, name, dtype)
    for r, t in tokens.items():
        mine = torch.cat(got[r])
        if dtype == "float32":
            alone.open(r)
            assert torch.equal(mine, feed(alone, r, t, [len(t)])), f"{name} {r}: a mixed step changed the logits"
            alone.close(r)
        check_against_plain(folders, name, dtype, t, mine, f"{name} {r} in mixed steps")


def test_long_decoding_carries_state_and_passes_windows(folders):
    """A short prompt and 300 tokens decoded one by one through the captured decode step: the memories carry, and every window
    passes over decoded tokens only."""
    tokens = _prompt(CONFIGS["A"], 312, 9)
    for dtype in ("float32", "bfloat16"):
        runner = make_runner(folders, "A", dtype)
        runner.open("r")
        got = feed(runner, "r", tokens, [12])
        assert runner.steps_replayed > 250
        check_against_plain(folders, "A", dtype, tokens, got, f"A decoding ({dtype})")


@pytest.mark.parametrize("n", [2, 20, 131, 300])
def test_a_traced_prompt_makes_the_numbers_of_an_untraced_one(folders, n, monkeypatch):
    """bfloat16, with layers whose two halves end in one product: the rows behind every layer and the last position's logits, in bits (with every row's logits wanted the last norm is
    handed on, which a traced pass does not do); the trace is shown the same rows."""
    from geneinfer_amd.engine import StepEntry
    runner = make_runner(folders, "A", "bfloat16")
    layers = runner.model.layers
    assert sum(layer._last is not None for layer in layers) >= 2
    tokens, got, seen, behind = _prompt(CONFIGS["A"], n, 5), [], [], []

    def watched(forward):
        def run(x, *args, **kw):
            out = forward(x, *args, **kw)
            behind.append(x.clone())
            return out
        return run

    for layer in layers:
        monkeypatch.setattr(layer, "forward", watched(layer.forward))
    for trace in (None, lambda tag, entry, rows: seen.append((tag, entry, rows.clone()))):
        runner.model.set_trace(trace)
        runner.open("r")
        got.append(runner.step([StepEntry("r", tokens, (n - 1,))]).cpu())
        runner.close("r")
    assert torch.equal(got[0], got[1]) and len(behind) == 2 * len(layers)
    assert [(tag, entry) for tag, entry, _ in seen if tag.endswith("_out")] == [(tag, i) for i in range(len(layers)) for tag in ("attn_out", "ffn_out")]
    rows = {(tag, entry): x for tag, entry, x in seen}
    for i in range(len(layers)):
        assert torch.equal(behind[i], behind[len(layers) + i]) and torch.equal(behind[i], rows["ffn_out", i]), i
        assert rows["attn_out", i].shape == (n, CONFIGS["A"]["width"]) and not torch.equal(rows["attn_out", i], behind[i - 1] if i else rows["embedding", -1])


def test_first_layer_of_a_family_of_blended_values_may_come_anywhere(folders, tmp_path):
    """The same layers in another order: the family's first layer is now the model's last-but-one, and a layer that does not blend
    lies between."""
    import copy
    cfg = copy.deepcopy(CONFIGS["B"])
    cfg["layers"] = [cfg["layers"][i] for i in (4, 1, 3, 2, 0, 5)]
    cfg["layers"][2]["mixer"]["vdim"], cfg["layers"][2]["mixer"]["kv_heads"], cfg["layers"][2]["mixer"]["heads"] = 48, 3, 3
    write_model(tmp_path / "m", cfg, seed=4)
    from geneinfer_amd.engine import Runner, load_model
    tokens = _prompt(cfg, 40, 2)
    want = P.forward(cfg, stored_weights(tmp_path / "m"), tokens)
    runner = Runner(load_model(tmp_path / "m", "float32", DEV), page_size=8, max_tokens=256, max_requests=2)
    runner.open("r")
    got = feed(runner, "r", tokens, [13, 2])
    assert relative_error(got, want) < 5e-5


# =============================================================================================== entry points
@pytest.mark.parametrize("name", ["A", "D"])
def test_greedy_generation_through_the_entry_point_and_the_scheduler(folders, name):
    """Greedy tokens of several prompts, one by one through `LLM.generate` and together through the scheduler (more requests than
    it runs at once, prompts in portions), against the plain model's, as far as the plain model's two best logits are clearly apart."""
    import geneinfer_amd as gi
    from geneinfer_amd.engine import EngineConfig, EngineRequest
    from geneinfer_amd.sampling import SamplerConfig
    cfg, w = CONFIGS[name], stored_weights(folders[name])
    prompts = [_prompt(cfg, n, 30 + n) for n in (5, 23, 1, 40)]
    want, sure = [], []
    for p in prompts:
        tokens = P.greedy(cfg, w, p, 8)
        top2 = torch.topk(P.forward(cfg, w, p + tokens)[len(p) - 1:-1], 2, dim=-1).values
        clear = [bool(c) for c in (top2[:, 0] - top2[:, 1] > 1e-3)]
        want.append(tokens)
        sure.append(clear.index(False) if False in clear else len(clear))
    assert sum(sure) >= 24
    llm = gi.LLM(str(folders[name]), dtype="float32", page_size=PAGE_SIZE[name], max_tokens=512, max_running=2)
    assert type(llm.model.config).__name__ == "RigalornConfig"
    for p, t, n in zip(prompts, want, sure):
        assert llm.generate(p, steps=len(p) + 7, temperature=0.0).generated_tokens[:n] == t[:n]
    eng = llm.engine(EngineConfig(max_running=2, step_rows=16, prefill_chunk=6))
    ids = [eng.submit(EngineRequest(p, len(p) + 7, SamplerConfig(0.0))) for p in prompts]
    eng.run_until_idle()
    for i, t, n in zip(ids, want, sure):
        assert eng.result(i).generated_tokens[:n] == t[:n]


@pytest.mark.parametrize("dtype, mode", [("float32", "mixed"), ("bfloat16", "mixed"), ("float32", "portions")])
def test_replay_through_the_command_line(folders, tmp_path, dtype, mode):
    """bin/trace_run as a child process on a Rigalorn folder: up to four live requests, portions beside single tokens, a pool that
    holds less than all requests together, so that pages and state slots are used again."""
    import json
    import random
    import subprocess
    from pathlib import Path
    import numpy as np
    import traces
    root = Path(__file__).resolve().parent.parent
    cfg = CONFIGS["B"]
    rng = random.Random(4)
    requests = {f"q{i}": [rng.randrange(cfg["vocab"]) for _ in range(n)] for i, n in enumerate([50, 1, 33, 77, 40, 9])}
    steps = traces.mixed(requests, seed=3) if mode == "mixed" else traces.portions(requests)
    out = tmp_path / "out"
    cmd = [str(root / "bin" / "trace_run"), "--model", str(folders["B"]), "--dtype", dtype, "--out", str(out), "--max-tokens", str(traces.peak_tokens(steps, 64)),
           "--page-size", "8"]
    proc = subprocess.Popen(cmd, stdin=subprocess.PIPE, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    try:
        for s in steps:
            proc.stdin.write(json.dumps(s) + "\n")
            proc.stdin.flush()
            line = proc.stdout.readline().strip()
            assert line == f"done {s['step']}", (line, proc.stderr.read() if proc.poll() is not None else "")
        proc.stdin.close()
        assert proc.wait(timeout=60) == 0, proc.stderr.read()
    finally:
        if proc.poll() is None:
            proc.kill()
    got = {}
    for step, rows in traces.wanted_positions(steps).items():
        data = np.fromfile(out / f"{step}.f32", dtype="<f4").reshape(len(rows), cfg["vocab"])
        for key, row in zip(rows, data):
            got[key] = torch.from_numpy(row.copy())
    for rid, tokens in requests.items():
        mine = {p: row for (r, p), row in got.items() if r == rid}
        assert len(mine) > 0
        exact = plain_logits(folders, "B", tokens)
        if dtype == "float32":
            single = plain_logits(folders, "B", tokens, dtype=torch.float32)
            noise = max(relative_error(single[p], exact[p]) for p in mine)
            assert max(relative_error(row, exact[p]) for p, row in mine.items()) < 4 * noise + 1e-5
        else:
            rounded = plain_logits(folders, "B", tokens, rounded=True)
            assert_within_bfloat16_noise(mine, lambda p: exact[p], lambda p: rounded[p], f"replay {mode} {rid}")


def test_generation_from_the_command_line_on_random_weights():
    """bin/gi_generate on the shipped example configuration, random weights, greedy: runs, and twice the same."""
    import subprocess
    from pathlib import Path
    root = Path(__file__).resolve().parent.parent
    cmd = [str(root / "bin" / "gi_generate"), "--config", str(root / "configs" / "rigalorn-small.json"), "--random-seed", "3", "--prompt-ids", "5 17 3 999 4",
           "--steps", "24", "--temperature", "0"]
    runs = [subprocess.run(cmd, capture_output=True, text=True, timeout=280) for _ in range(2)]
    assert all(r.returncode == 0 for r in runs), runs[0].stderr[-2000:]
    assert runs[0].stdout == runs[1].stdout and len(runs[0].stdout.split()) >= 20


def test_the_new_parts_serve_other_designs():
    """The parts are not Rigalorn's own: a model put together by hand, a pre-norm layer around the gated delta rule and a SiLU-gated
    feed-forward, and a parallel layer around a plain Llama attention and the feed-forward without a gate, through the same step
    function; against a plain computation from the plain implementations' functions."""
    from geneinfer_amd.config import (AttentionSpec, DenseMlpSpec, GatedDeltaSpec, LayerSpec, ModelSpec, RmsNormSpec, RotarySpec, RunEntry, SwiGluSpec)
    from geneinfer_amd.engine import Runner
    from geneinfer_amd.engine.model import DecoderModel
    from geneinfer_amd.parts import model_tensor_needs
    from geneinfer_amd.weights import random_tensors
    from plain_llama import causal_attention, rms_norm, rope_inverse_frequencies, rope_rotate, swiglu
    d, vocab, eps = 64, 100, 1e-5
    norm = lambda name: RmsNormSpec(d, eps, name)
    delta = GatedDeltaSpec(d, 2, 1, 8, 24, 3, eps, "m.q", "m.k", "m.v", "m.qc", "m.kc", "m.vc", "m.a", "m.al", "m.dt", "m.b", "m.g", "m.n", "m.o")
    spec = ModelSpec(architecture="by hand", vocab_size=vocab, hidden_size=d, max_positions=256, embedding="emb", final_norm=norm("fn"), lm_head="head", layers=(
        LayerSpec(mixer=delta, feed_forward=SwiGluSpec(d, 80, "g.g", "g.u", "g.d"), mixer_norm=norm("p1"), feed_forward_norm=norm("p2"), block="prenorm"),
        LayerSpec(mixer=AttentionSpec(d, 4, 2, 16, "a.q", "a.k", "a.v", "a.o", RotarySpec(16, 10000.0)), feed_forward=DenseMlpSpec(d, 96, "f.u", "f.d", "xielu", "f.act"),
                  mixer_norm=norm("n1"), feed_forward_norm=None, block="parallel")),
        run_order=(RunEntry(0), RunEntry(1)))
    host = random_tensors(model_tensor_needs(spec), seed=5, dtype="float32", std=0.2)
    model = DecoderModel(spec, {k: v.to(DEV) for k, v in host.items()}, torch.float32, DEV)
    runner = Runner(model, page_size=4, max_tokens=256, max_requests=2)
    tokens = _prompt(dict(vocab=vocab), 45, 2)
    got = {}
    for what, cuts in (("whole", [45]), ("cut", [3, 20, 2])):
        runner.open(what)
        got[what] = feed(runner, what, tokens, cuts)
        runner.close(what)
    assert torch.equal(got["whole"], got["cut"])

    w = {k: v.double() for k, v in host.items()}
    T, pos = len(tokens), torch.arange(len(tokens))
    x = w["emb"][torch.tensor(tokens)]
    h = rms_norm(x, w["p1"], eps)
    m = dict(heads=2, kv_heads=1, dim=8, vdim=24)
    names = {"q": "m.q", "k": "m.k", "v": "m.v", "q.conv": "m.qc", "k.conv": "m.kc", "v.conv": "m.vc", "a": "m.a", "A_log": "m.al", "dt_bias": "m.dt", "b": "m.b",
             "g": "m.g", "norm": "m.n", "o": "m.o"}
    x = x + P.delta(h, {k: w[v] for k, v in names.items()}, m, eps)
    x = x + swiglu(rms_norm(x, w["p2"], eps), w["g.g"], w["g.u"], w["g.d"])
    h = rms_norm(x, w["n1"], eps)
    f = rope_inverse_frequencies(16, 10000.0)
    q, k = rope_rotate((h @ w["a.q"].T).view(T, 4, 16), pos, f), rope_rotate((h @ w["a.k"].T).view(T, 2, 16), pos, f)
    y = causal_attention(q, k, (h @ w["a.v"].T).view(T, 2, 16)).reshape(T, 64) @ w["a.o"].T
    x = x + y + P.dense_mlp(h, w["f.u"], w["f.d"], w["f.act"])
    want = rms_norm(x, w["fn"], eps) @ w["head"].T
    assert relative_error(got["whole"], want) < 5e-5
