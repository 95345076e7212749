"""The products' kernels at the edges of their dispatch rules: every kernel that serves a shape gives
what float64 gives, and where the order of the sums is fixed, the same bits."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# N and K: one part and several, a last part that is short, K no multiple of a stage of 32 (528), of a
# block of 16 (1000: the kernel of any length), more parts than the norm kernel adds is out of reach here
@pytest.mark.parametrize("N,K", [(70, 528), (896, 4864), (130, 1000), (64, 48), (1000, 896)])
def test_float32_rows_have_the_same_bits_in_every_kernel(N, K):
    """Up to 16 rows, 17 to 32, tiles of 64, tiles of 32, planes of partial sums: a row alone and among
    others, and the planes added in order."""
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(300, K, device=DEV, generator=gen)
    w = torch.randn(N, K, device=DEV, generator=gen)
    b = torch.randn(N, device=DEV, generator=gen)
    want = x.double() @ w.double().t()
    whole = ops.linear(x, w, b)
    # a sum of 16 rounds at 4 units at most and the sums of 16 are added one by one: sqrt(16) + sqrt(K / 16) roundings
    # of values of about sqrt(K), in 2^-24; ten times their spread over all elements
    bound = 10 * (4 + math.sqrt(K / 16)) * math.sqrt(K) * 2.0 ** -24
    assert float((whole.double() - want - b.double()).abs().max()) < bound
    plain = ops.linear(x, w)
    for rows in (1, 15, 16, 17, 32, 33, 64, 65, 256, 257):
        part = x[:rows].contiguous()
        assert torch.equal(ops.linear(part, w, b), whole[:rows]), rows
        for reader_adds in (False, True):
            got = ops.linear(part, w, partial_ok=True, portions_partial_ok=reader_adds)
            if isinstance(got, ops.PartialSums):
                assert reader_adds
                got = got.sum()
            assert torch.equal(got, plain[:rows]), rows


def test_float32_infinities_stay_in_their_rows_and_columns():
    """What lies past K is not multiplied: an infinite weight or input reaches its own outputs only."""
    from clockwork_amd import ops

    x, w = torch.ones(40, 528, device=DEV), torch.ones(70, 528, device=DEV)
    x[39, 527] = float("inf")
    w[69, 0] = float("inf")
    for rows in (slice(0, 40), slice(30, 40)):
        got = ops.linear(x[rows].contiguous(), w)
        assert bool(torch.isinf(got[-1]).all()) and bool(torch.isinf(got[:, 69]).all())
        assert bool((got[:-1, :69] == 528).all())


def _kept_cdf(row, temp, k, p, slack):
    """Which tokens stay and the running sums of their weights in index order, in float64, by the sampler's definition: ties at
    the k-th value survive, a token stays while the mass strictly above it is at most p (+ slack) of what top-k left."""
    v = row / temp
    keep = torch.ones_like(v, dtype=torch.bool)
    if 0 < k < v.numel():
        keep = v >= row.topk(k).values[-1] / temp
    w = torch.where(keep, torch.exp(v.double() - v.max().double()), 0.0)
    if p < 1.0:
        values, group = torch.unique(v, return_inverse=True)   # ascending
        mass = torch.zeros(values.numel(), dtype=torch.float64, device=row.device).index_add_(0, group, w)
        above = mass.flip(0).cumsum(0).flip(0) - mass
        keep &= (above <= (p + slack) * mass.sum())[group]
        w = torch.where(keep, w, 0.0)
    cdf = w.cumsum(0)
    return keep, cdf / cdf[-1]


# odd sizes (rows that do not begin at 16 bytes), values in steps of a half (thousands of equal logits in a bin, more
# than a workgroup's list and a row's list hold), nearly flat rows, spread ones, all equal, all but some masked by -inf or by
# the lowest value, a third of the row in a cluster that is narrower than any bin
@pytest.mark.parametrize("V,kind", [(1, "spread"), (70, "spread"), (511, "spread"), (2049, "steps"), (33333, "flat"), (151936, "steps"), (151936, "spread"),
                                    (151936, "flat"), (40001, "equal"), (151936, "masked"), (151936, "lowest"), (151936, "cluster")])
def test_sampling_lists_bins_and_chunks(V, kind):
    """Every option against its definition in float64, and the same tokens however many rows share the launch
    (which sets how a row is cut)."""
    from clockwork_amd import ops
    from tests.plain import qwen2_plain as plain

    gen = torch.Generator(device=DEV).manual_seed(V)
    n, draws_each = 24, 8
    logits = torch.randn(n, V, device=DEV, generator=gen) * {"spread": 5.0, "steps": 2.0, "flat": 0.01, "equal": 0.0}.get(kind, 3.0)
    if kind == "steps":
        logits = (2.0 * logits).round() / 2.0
    logits += 0.0   # no -0: the sampler's order has it below 0, while they compare equal
    if kind in ("masked", "lowest"):
        hidden = torch.rand(n, V, device=DEV, generator=gen) > torch.linspace(0.0003, 0.5, n, device=DEV)[:, None]
        hidden[:, 5] = False
        logits[hidden] = -float("inf") if kind == "masked" else torch.finfo(torch.float32).min
    if kind == "cluster":
        logits[:, ::3] = 1.0 + 1e-5 * logits[:, ::3]
    temps = torch.tensor([0.7, 1.0, 2.5, 0.0] * 5 + [0.05, 0.05, 0.05, 4.0], device=DEV)
    ks = [-1] * 4 + [7] * 4 + [-1] * 4 + [max(1, V // 2)] * 4 + [30] * 4 + [50, -1, max(1, V // 2), -1]   # the fourth four: the nucleus ends far above the k-th token
    ps = [1.0] * 8 + [0.8] * 4 + [0.3] * 4 + [0.97] * 4 + [1.0, 0.9, 0.9, 0.9]
    top_k, top_p = torch.tensor(ks, dtype=torch.int32, device=DEV), torch.tensor(ps, device=DEV)
    seeds = torch.arange(n, dtype=torch.int64, device=DEV) + 11
    each = torch.arange(n, device=DEV).repeat_interleave(draws_each)
    draws = torch.arange(draws_each, dtype=torch.int64, device=DEV).repeat(n)
    args = temps[each], top_k[each], top_p[each], seeds[each]
    got = ops.sample(logits[each], *args, draws).view(n, draws_each)
    for i in range(n):
        one = slice(i, i + 1)
        both = ks[i] > 0 and ps[i] < 1.0
        alone = ops.sample(logits[one].contiguous(), temps[one], top_k[one], top_p[one], seeds[one], draws[:1],
                           any_top_k=ks[i] > 0, any_top_p=ps[i] < 1.0, any_both=both)
        assert int(alone) == int(got[i, 0])
        if float(temps[i]) == 0.0:
            assert bool((got[i] == logits[i].argmax()).all())
            continue
        # weights are float32 exponentials (a few units of 2^-24 each, so that running sums of up to 151,936 of them are off by less
        # than 1e-6 of the whole) and rounded down to 2^-40; a nucleus that ends within 1e-6 of p may end on either side
        ways = [_kept_cdf(logits[i], temps[i], ks[i], float(top_p[i]), slack) for slack in (-1e-6, 1e-6)]
        for d, token in enumerate(got[i].tolist()):
            u = plain.uniform01(int(seeds[i]), d)
            assert any(bool(keep[token]) and (0.0 if token == 0 else float(cdf[token - 1])) - 2e-6 <= u <= float(cdf[token]) + 2e-6
                       for keep, cdf in ways), (i, d, token, u)
    many = 300
    if V <= 40001:
        rows = torch.arange(many, device=DEV) % n
        again = ops.sample(logits[rows], temps[rows], top_k[rows], top_p[rows], seeds[rows], draws[:1].expand(many).contiguous())
        assert torch.equal(again, got[rows, 0])


def test_sampling_with_flags_that_say_nothing():
    """The C entry's flags 3, some row may have top-k and some top-p: rows with both are drawn too."""
    from clockwork_amd import ops

    V, n = 5000, 4
    logits = 3.0 * torch.randn(n, V, device=DEV, generator=torch.Generator(device=DEV).manual_seed(2))
    temps, ps = torch.ones(n, device=DEV), torch.full((n,), 0.3, device=DEV)
    ks = torch.full((n,), V // 2, dtype=torch.int32, device=DEV)   # the nucleus ends far above the k-th token
    seeds, draws = (torch.arange(n, dtype=torch.int64, device=DEV) for _ in range(2))
    out = torch.full((n,), -7, dtype=torch.int32, device=DEV)
    lib = ops._load("sampling")
    ws = torch.empty(int(lib.cw_sample_workspace_bytes(n, V)), dtype=torch.uint8, device=DEV)
    args = (ops._ptr(t) for t in (temps, ks, ps, seeds, draws, out, ws))
    assert lib.cw_sample(ops._ptr(logits), V, n, V, *args, ws.numel(), 3, ops._stream()) == 0
    assert torch.equal(out, ops.sample(logits, temps, ks, ps, seeds, draws)) and bool((out >= 0).all())


def test_sampling_takes_as_long_for_flat_and_peaked_rows():
    """The bins follow the row's spread: rows that are nearly flat, rows far apart and masked rows take the time of
    others. (A row whose bin did not fit its list took 15 to 40 times as long.)"""
    from clockwork_amd import ops

    V, rows = 151936, 8
    gen = torch.Generator(device=DEV).manual_seed(1)
    noise = torch.randn(rows, V, device=DEV, generator=gen)
    masked = torch.where(torch.rand(rows, V, device=DEV, generator=gen) < 0.01, 3.0 * noise, -float("inf"))

    def us(logits, temperature, k, p):
        full = lambda v, dtype=torch.float32: torch.full((rows,), v, dtype=dtype, device=DEV)  # noqa: E731
        args = (logits, full(temperature), full(k, torch.int32), full(p), torch.arange(rows, device=DEV), torch.zeros(rows, dtype=torch.int64, device=DEV))
        ops.sample(*args)
        times = []
        for _ in range(15):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(5):
                ops.sample(*args)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end) * 200)
        return sorted(times)[len(times) // 2]

    for k, p in ((-1, 0.9), (50, 1.0), (V // 2, 1.0), (V // 2, 0.9)):
        usual = us(3.0 * noise, 1.0, k, p)
        for logits, temperature in ((0.02 * noise, 1.0), (0.4 * noise, 1.0), (3.0 * noise, 5.0), (3.0 * noise, 0.05), (masked, 1.0)):
            assert us(logits, temperature, k, p) < 4 * usual, (k, p, temperature)


# rows and columns that end inside a tile, one tile, K of a single stage a run, runs of unequal length, every tile size
@pytest.mark.parametrize("bm", [64, 128])
@pytest.mark.parametrize("bn", [64, 128])
@pytest.mark.parametrize("M,N,K", [(65, 64, 256), (130, 194, 320), (257, 1536, 1536), (1, 70, 640)])
def test_tiles_between_the_narrow_and_the_wide(M, N, K, bm, bn):
    """Plain with a bias, gated with each activation, and partial sums over runs of K."""
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    want = x.float() @ w.float().t()
    # float32 sums of K products of about 1 / sqrt(K): a few units of 2^-24 times sqrt(K); then one rounding to bfloat16
    f32 = dict(rtol=1e-4, atol=1e-4)
    bf16 = dict(rtol=2.0 ** -8 + 1e-4, atol=1e-4)
    for planes in (1, 3, 4):
        got = ops.linear_mid(x, w, bm | bn << 10 | planes << 20, partial=True)
        assert got.parts.shape == (planes, M, N)
        torch.testing.assert_close(got.sum(), want, **f32)
        first = (K // 64 // planes) * 64   # the first run's elements: stages [0, stages / planes)
        torch.testing.assert_close(got.parts[0], x[:, :first].float() @ w[:, :first].float().t(), **f32)
    one = bm | bn << 10 | 1 << 20
    for bias in (None, torch.randn(N, device=DEV, generator=gen), torch.randn(N, device=DEV, generator=gen).to(torch.bfloat16)):
        got = ops.linear_mid(x, w, one, bias=bias)
        torch.testing.assert_close(got.float(), want + (0 if bias is None else bias.float()), **bf16)
    g, u = want[:, : N // 2], want[:, N // 2:]
    gated = {0.0: torch.nn.functional.silu(g) * u, ops.RELU_GATE: torch.relu(g) * u,
             0.5: torch.clamp(g, max=0.5) * torch.sigmoid(1.702 * torch.clamp(g, max=0.5)) * (torch.clamp(u, -0.5, 0.5) + 1.0)}
    for limit, ref in gated.items():
        torch.testing.assert_close(ops.linear_mid(x, w, one, swiglu=True, limit=limit).float(), ref, **bf16)


# every tile of the wide-tile kernel that test_tiles_between_the_narrow_and_the_wide leaves out
WIDE_TILES = {0: [(96, 96), (128, 96), (160, 128), (192, 160), (256, 160), (256, 192)],
              2: [(160, 96), (160, 128), (160, 160), (192, 160), (192, 192), (256, 192), (256, 288)],
              3: [(96, 96), (160, 128), (192, 160), (192, 192), (256, 128), (256, 192)]}


# one row tile with few rows and fewer stages than slots; rows and columns that end inside a tile; more tiles than one for each of 256
# workgroups, 264 of the widest: the next tile's first loads beside this one's end
@pytest.mark.parametrize("mode,bm,bn", [(mode, *t) for mode, tiles in WIDE_TILES.items() for t in tiles])
@pytest.mark.parametrize("M,N,K", [(1, 16, 256), (65, 48, 64), (321, 1168, 640), (2048, 5168, 320), (2048, 9504, 256)])
def test_tiles_of_the_wide_kernel(mode, bm, bn, M, N, K):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    want = x.float() @ w.float().t()
    # as above: float32 sums of K products of about 1 / sqrt(K), one rounding to bfloat16
    f32, bf16 = dict(rtol=1e-4, atol=1e-4), dict(rtol=2.0 ** -8 + 1e-4, atol=1e-4)
    one = bm | bn << 10 | 1 << 20
    if mode == 0:
        for bias in (None, torch.randn(N, device=DEV, generator=gen), torch.randn(N, device=DEV, generator=gen).to(torch.bfloat16)):
            torch.testing.assert_close(ops.linear_mid(x, w, one, bias=bias).float(), want + (0 if bias is None else bias.float()), **bf16)
    elif mode == 2:
        g, u = want[:, : N // 2], want[:, N // 2:]
        for limit, ref in {0.0: torch.nn.functional.silu(g) * u, ops.RELU_GATE: torch.relu(g) * u,
                           ops.GELU_GATE: torch.nn.functional.gelu(g, approximate="tanh") * u,
                           0.5: torch.clamp(g, max=0.5) * torch.sigmoid(1.702 * torch.clamp(g, max=0.5)) * (torch.clamp(u, -0.5, 0.5) + 1.0)}.items():
            torch.testing.assert_close(ops.linear_mid(x, w, one, swiglu=True, limit=limit).float(), ref, **bf16)
    else:
        for planes in (p for p in (1, 3, 5) if p <= K // 64):
            got = ops.linear_mid(x, w, bm | bn << 10 | planes << 20, partial=True)
            torch.testing.assert_close(got.sum(), want, **f32)
            first = (K // 64 // planes) * 64
            torch.testing.assert_close(got.parts[0], x[:, :first].float() @ w[:, :first].float().t(), **f32)


# 32 MB and more of W beside one or two row tiles: whole lines past the caches; few stages and several tiles a workgroup, many stages and one
@pytest.mark.parametrize("mode,bm,bn", [(mode, *t) for mode, tiles in WIDE_TILES.items() for t in tiles if t[0] * t[1] <= 32 * 1024])
@pytest.mark.parametrize("N,K", [(30016, 576), (8208, 2112)])
def test_tiles_of_a_matrix_that_is_read_once(mode, bm, bn, N, K):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(N + bm)
    w = (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    # as above: float32 sums of K products of about 1 / sqrt(K), one rounding to bfloat16
    f32, bf16 = dict(rtol=1e-4, atol=1e-4), dict(rtol=2.0 ** -8 + 1e-4, atol=1e-4)
    for M in (bm - 7, bm + 1, 2 * bm):
        x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
        want = x.float() @ w.float().t()
        if mode == 0:
            torch.testing.assert_close(ops.linear_mid(x, w, bm | bn << 10 | 1 << 20).float(), want, **bf16)
        elif mode == 2:
            ref = torch.nn.functional.silu(want[:, : N // 2]) * want[:, N // 2:]
            torch.testing.assert_close(ops.linear_mid(x, w, bm | bn << 10 | 1 << 20, swiglu=True).float(), ref, **bf16)
        else:
            for planes in (1, 3):
                torch.testing.assert_close(ops.linear_mid(x, w, bm | bn << 10 | planes << 20, partial=True).sum(), want, **f32)


@pytest.mark.parametrize("mode,N", [(0, 1001), (2, 2 * 1004), (3, 1002)])
def test_tiles_for_whole_rows_refuse_others(mode, N):
    """Results whose rows are no multiples of 16 bytes: refused where a tile takes whole rows only, and served by another."""
    from clockwork_amd import ops

    M, K = 200, 512
    gen = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    for bm, bn in WIDE_TILES[mode]:
        if (bm, bn) != (256, 192):
            with pytest.raises(ops.KernelError):
                ops.linear_mid(x, w, bm | bn << 10 | 1 << 20, swiglu=mode == 2, partial=mode == 3)
    want = x.float() @ w.float().t()
    bf16 = dict(rtol=2.0 ** -8 + 1e-4, atol=1e-4)
    if mode == 2:
        ref = torch.nn.functional.silu(want[:, : N // 2]) * want[:, N // 2:]
        torch.testing.assert_close(ops.linear_mid(x, w, 256 | 192 << 10 | 1 << 20, swiglu=True).float(), ref, **bf16)
        torch.testing.assert_close(ops.linear_swiglu(x, w).float(), ref, rtol=4 * 2.0 ** -8, atol=2e-2)
    else:
        got = ops.linear(x, w, partial_ok=mode == 3, portions_partial_ok=mode == 3)
        torch.testing.assert_close(got.sum() if mode == 3 else got.float(), want, **bf16)


# one row, rows and pairs that end inside a tile, heads of one, three and four blocks of 16 pairs, a head over several tiles, an odd number of heads
@pytest.mark.parametrize("M", [1, 65, 130, 333])
@pytest.mark.parametrize("nh,nkv,hd,K,bias_dtype", [(12, 2, 128, 1536, torch.bfloat16), (14, 2, 64, 896, torch.float32), (3, 1, 32, 256, None),
                                                    (3, 3, 96, 320, torch.bfloat16), (2, 1, 256, 512, None)])
def test_queries_keys_and_values_of_many_rows_in_one_kernel(M, nh, nkv, hd, K, bias_dtype):
    """Product, bias, rotation and cache write against the same in float64, rows without a slot and slots that no row has
    left as they are, and the table of angles against the rotation kernel's own."""
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + hd)
    width = (nh + 2 * nkv) * hd
    x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
    w = (torch.randn(width, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    bias = None if bias_dtype is None else torch.randn(width, device=DEV, generator=gen).to(bias_dtype)
    positions = torch.randint(0, 30000, (M,), dtype=torch.int32, device=DEV, generator=gen)
    inv_freq = (1.0 / 1e6 ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd)).to(DEV)
    slots = torch.randperm(M + 9, device=DEV, generator=gen)[:M].to(torch.int32)
    slots[::5] = -1
    slots[3::11] = M + 9   # beyond the cache
    kc = torch.full((M + 9, nkv, hd), 9.0, device=DEV, dtype=torch.bfloat16)
    vc = kc.clone()
    angles = ops.rope_angles(positions, inv_freq)
    q = ops.qkv_rope_rows(x, w, bias, angles, slots, nh, nkv, hd, kc, vc)
    # the table is what the rotation kernel turns a pair (1, 0) by
    ones = torch.zeros(M, 1, 2, hd // 2, device=DEV)
    ones[:, :, 0] = 1.0
    turned = ones.view(M, hd).contiguous()
    ops.rope_kv_write(turned, None, positions, None, inv_freq, hd, 1, 0, hd, None, None)
    assert torch.equal(turned.view(M, 2, hd // 2), angles)
    y = x.double() @ w.double().t()
    y = (y if bias is None else y + bias.double()).view(M, nh + 2 * nkv, hd)
    a, b = y.chunk(2, dim=2)
    cos, sin = (angles[:, j].double()[:, None, :] for j in (0, 1))
    want = torch.cat([a * cos - b * sin, b * cos + a * sin], dim=2)
    want[:, nh + nkv:] = y[:, nh + nkv:]
    # float32 sums of K products of about 1 / sqrt(K) and one rounding to bfloat16
    t = dict(rtol=2.0 ** -8 + 1e-4, atol=1e-4)
    torch.testing.assert_close(q.double().view(M, nh, hd), want[:, :nh], **t)
    live = (slots >= 0) & (slots < M + 9)
    rows = slots[live].long()
    torch.testing.assert_close(kc[rows].double(), want[live, nh:nh + nkv], **t)
    torch.testing.assert_close(vc[rows].double(), want[live, nh + nkv:], **t)
    rest = torch.ones(M + 9, dtype=torch.bool, device=DEV)
    rest[rows] = False
    assert bool((kc[rest] == 9.0).all()) and bool((vc[rest] == 9.0).all())


def test_products_of_a_portion_by_their_rule():
    """What the rule names runs and is the product, on every side of its lines."""
    from clockwork_amd import ops

    lib = ops._load("gemm_tile")
    gen = torch.Generator(device=DEV).manual_seed(3)
    for N, K in ((256, 1024), (896, 896), (200, 320)):
        w = (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
        for M in (64, 65, 100, 319, 700, 1030):
            x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
            want = x.float() @ w.float().t()
            got = ops.linear(x, w, partial_ok=True, portions_partial_ok=True)
            if M > 64:
                assert isinstance(got, ops.PartialSums) == bool(lib.cw_gemm_bf16_mid_choice(3, M, N, K, K, ops._compute_units(x.device)))
            got = got.sum() if isinstance(got, ops.PartialSums) else got.float()
            torch.testing.assert_close(got, want, rtol=2.0 ** -8 + 1e-4, atol=1e-4)
            torch.testing.assert_close(ops.linear(x, w).float(), want, rtol=2.0 ** -8 + 1e-4, atol=1e-4)
            h = ops.linear_swiglu(x, w).float()
            ref = torch.nn.functional.silu(want[:, : N // 2]) * want[:, N // 2:]
            # the library's path rounds the product to bfloat16 before the gate: two roundings of up to 2^-8 each side
            torch.testing.assert_close(h, ref, rtol=4 * 2.0 ** -8, atol=2e-2)
    assert lib.cw_gemm_bf16_mid_choice(3, 144, 1536, 8960 + 32, 8992, 256) == 0   # K no whole number of stages


@pytest.mark.parametrize("M", [100, 400])
def test_operands_that_only_the_library_takes(M):
    """Rows that do not begin at 16 bytes and biases of other shapes go to the library whatever the rule names for the
    sizes; a float32 bias, which the library refuses, stays refused."""
    from clockwork_amd import ops

    N, K = 1152, 512
    gen = torch.Generator(device=DEV).manual_seed(M)
    lib = ops._load("gemm_tile")
    assert all(lib.cw_gemm_bf16_mid_choice(mode, M, N, K, K, 256) for mode in (0, 2, 3))
    assert ops.wide_swiglu_pays(400, 2 * 8960, 1536, 1536)
    wide = torch.randn(2 * 8960 * 1536 + 1, device=DEV, generator=gen).to(torch.bfloat16)

    def odd(*shape):
        return wide[1:1 + math.prod(shape)].view(shape)

    tol = dict(rtol=4 * 2.0 ** -8, atol=2e-2)   # two roundings of up to 2^-8 each side
    x, w = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16), (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    for a, b in ((odd(M, K), w), (x, odd(N, K) / K ** 0.5), (odd(M, K), odd(N, K))):
        b = odd(N, K).copy_(b) if b is not w else b
        want = a.float() @ b.float().t()
        for got in (ops.linear(a, b), ops.linear(a, b, partial_ok=True, portions_partial_ok=True)):
            torch.testing.assert_close(got.float(), want, **tol)
        g, u = want[:, : N // 2], want[:, N // 2:]
        torch.testing.assert_close(ops.linear_swiglu(a, b).float(), torch.nn.functional.silu(g) * u, rtol=4 * 2.0 ** -8, atol=0.03 * float((g * u).abs().max()))
    if M == 400:
        a, b = torch.randn(M, 1536, device=DEV, generator=gen).to(torch.bfloat16), odd(2 * 8960, 1536)
        assert ops.linear_swiglu(a, b).shape == (M, 8960)
    one = torch.full((1,), 3.0, device=DEV, dtype=torch.bfloat16)
    torch.testing.assert_close(ops.linear(x, w, one).float(), x.float() @ w.float().t() + 3.0, **tol)
    with pytest.raises(RuntimeError):
        ops.linear(x, w, torch.zeros(N, device=DEV))


def test_gate_up_of_a_captured_step_by_its_rows_and_tiles():
    """Steps of 1 to 24 padded single tokens beside a portion padded to 384 rows are steps of 385 to 408 rows: all of them
    take the wide tiles, no step of fewer rows does, whatever it is a multiple of."""
    from clockwork_amd import ops

    two_i, K = 2 * 8960, 1536
    assert all(ops.wide_swiglu_pays(M, two_i, K, K) for M in (384, 385, 386, 388, 392, 400, 408, 448, 450, 512, 1000))
    assert not any(ops.wide_swiglu_pays(M, two_i, K, K) for M in (256, 257, 264, 272, 288, 304, 320, 352, 576, 640))
    # several rounds: 345 tiles of 2048 x 22016 (the library served 700 rows, 97 us against 86)
    assert all(ops.wide_swiglu_pays(M, 22016, 2048, 2048) for M in (385, 512, 700, 768, 832)) and not ops.wide_swiglu_pays(640, 22016, 2048, 2048)
    gen = torch.Generator(device=DEV).manual_seed(4)
    w = (torch.randn(two_i, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    x = torch.randn(385, K, device=DEV, generator=gen).to(torch.bfloat16)
    h = x.float() @ w.float().t()
    want = torch.nn.functional.silu(h[:, :8960]) * h[:, 8960:]
    ran, real = [], ops.linear_tiled
    try:
        ops.linear_tiled = lambda *a, **k: (ran.append(a[0].shape[0]), real(*a, **k))[1]
        torch.testing.assert_close(ops.linear_swiglu(x, w).float(), want, rtol=4 * 2.0 ** -8, atol=2e-2)   # two roundings each side
        assert not ran   # a step that is not captured
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = ops.linear_swiglu(x, w)
        assert ran == [385]
    finally:
        ops.linear_tiled = real
    for _ in range(2):
        got.zero_()
        graph.replay()
        torch.testing.assert_close(got.float(), want, rtol=2.0 ** -8 + 1e-4, atol=1e-3)   # one rounding


# 16 requests at the edges of a wave's tile of 32 keys, of the turns of four and eight waves and of the line where
# eight take over (128 keys a split); 24 keys a page and 16; a group of more than 16 heads
@pytest.mark.parametrize("hd,nh,nkv,bs", [(32, 4, 2, 16), (64, 14, 2, 16), (96, 6, 3, 24), (128, 12, 2, 16), (128, 20, 1, 24), (160, 4, 2, 16)])
@pytest.mark.parametrize("splits,fixed", [(1, True), (1, False), (2, True), (5, True), (5, False)])
def test_decode_attention_at_the_turns_of_its_waves(hd, nh, nkv, bs, splits, fixed):
    from clockwork_amd import ops

    lens = [1, 2, 31, 32, 33, 127, 128, 129, 255, 256, 257, 511, 512, 513, 640, 700]
    gen = torch.Generator().manual_seed(hd + splits)
    width = -(-max(lens) // bs)
    tables = torch.randperm(len(lens) * width, generator=gen).view(len(lens), width)
    k, v = (torch.randn(len(lens) * width, bs, nkv, hd, generator=gen).bfloat16() for _ in range(2))
    q = torch.randn(len(lens), nh * hd, generator=gen).bfloat16()
    ws = None
    if splits > 1:
        ws = torch.full((ops.decode_attention_workspace_floats(hd, len(lens), nh, nkv, splits),), float("nan"), device=DEV)
    out = torch.empty(len(lens), nh * hd, dtype=torch.bfloat16, device=DEV)
    ints = lambda t: torch.as_tensor(t, dtype=torch.int32, device=DEV)  # noqa: E731
    items = ints([x for r in range(len(lens)) for x in (r, 0, 1, 0)])
    # what no request holds is poison: a key past a length that is counted shows
    kd, vd = (t.clone() for t in (k, v))
    for r, n in enumerate(lens):
        for page in range(width):
            kd[tables[r, page], max(0, min(bs, n - page * bs)):] = float("nan")
            vd[tables[r, page], max(0, min(bs, n - page * bs)):] = float("nan")
    extra = dict(identity=True, split_keys=32 * -(-(-(-max(lens) // splits)) // 32), max_ctx=max(lens)) if fixed else {}
    ops.attention_decode(q=q.to(DEV), q_stride=nh * hd, out=out, k_cache=kd.to(DEV), v_cache=vd.to(DEV), block_tables=ints(tables),
                         ctx_lens=ints(lens), cu_q=ints(range(len(lens) + 1)), items=items, n_items=len(lens), nh=nh, nkv=nkv,
                         hd=hd, block_size=bs, n_splits=splits, window=0, scale=hd ** -0.5, workspace=ws,
                         n_tokens=len(lens), n_requests=len(lens), **extra)
    got = out.view(len(lens), nh, hd).double().cpu()
    for r, n in enumerate(lens):
        kr = k[tables[r]].reshape(-1, nkv, hd)[:n].double().repeat_interleave(nh // nkv, 1)
        vr = v[tables[r]].reshape(-1, nkv, hd)[:n].double().repeat_interleave(nh // nkv, 1)
        p = torch.softmax(torch.matmul(kr.transpose(0, 1), q[r].double().view(nh, hd, 1)).squeeze(-1) * hd ** -0.5, -1)
        want = (p[..., None] * vr.transpose(0, 1)).sum(1)
        # the probabilities and the result are rounded to bfloat16: half of 2^-8 of each term and of the sum
        bound = 2.0 ** -8 * ((p[..., None] * vr.transpose(0, 1)).abs().sum(1) + want.abs()) + 1e-4
        assert bool(((got[r] - want).abs() <= bound).all()), (r, n)


# rows of pieces of 4: one piece, a part of a wave, around 256 pieces, the most that registers hold and one more; no
# multiple of 4 (the kernel of any length)
@pytest.mark.parametrize("H", [4, 100, 1020, 1024, 1028, 1536, 2048, 2052, 4096, 4100, 1535])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_in_pieces_of_four(H, dtype):
    """Residual add + LayerNorm with each kind of pending branch, the mean of two RMS norms, the q / k norm with its
    cache rows and the gated GELU, against float64."""
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(H)
    rand = lambda *shape, dt=dtype: torch.randn(*shape, device=DEV, generator=gen).to(dt)  # noqa: E731
    T, f64 = 5, torch.float64
    # values of a few units: the result's own rounding, and float32 sums of H terms
    tol = dict(atol=0.03, rtol=0.01) if dtype == torch.bfloat16 else dict(atol=2e-5, rtol=2e-5)
    w, b, zb, x = rand(H), rand(H), rand(2 * H), rand(T, H, dt=torch.float32)
    one, two, z, planes = rand(T, H), rand(T, H), rand(T, 2 * H), ops.PartialSums(rand(6, T, H, dt=torch.float32))
    gates = torch.sigmoid(z.to(f64) + zb.to(f64))
    for pending, extra in ((None, 0), ((None, None, one, None), one.to(f64)), ((z[:, :H].contiguous(), None, one, None), torch.sigmoid(z[:, :H].to(f64)) * one.to(f64)),
                           ((z, zb, one, two), gates[:, :H] * one.to(f64) + gates[:, H:] * two.to(f64)),
                           ((None, None, one, planes), one.to(f64) + planes.parts.to(f64).sum(0)),
                           ((z, zb, one, planes), gates[:, :H] * one.to(f64) + gates[:, H:] * planes.parts.to(f64).sum(0))):
        total = x.to(f64) + extra
        want = torch.nn.functional.layer_norm(total, (H,), w.to(f64), b.to(f64), 1e-5)
        branches = None if pending is None else ops.GatedBranches(*pending)
        pick = torch.tensor([4, 1], dtype=torch.int32, device=DEV)
        resid = x.clone()
        got = ops.add_layernorm(resid, branches, w, b, 1e-5, torch.empty(2, H, dtype=dtype, device=DEV), rows=pick)
        torch.testing.assert_close(got.to(f64), want[[4, 1]], **tol)
        assert torch.equal(resid, x)
        got = ops.add_layernorm(resid, branches, w, b, 1e-5, torch.empty(T, H, dtype=dtype, device=DEV))
        torch.testing.assert_close(got.to(f64), want, **tol)
        torch.testing.assert_close(resid.to(f64), total, atol=1e-5, rtol=1e-5)
        if branches is not None:
            torch.testing.assert_close(ops.gated_residual_add(x.clone(), branches).to(f64), total, atol=1e-5, rtol=1e-5)
    rms = lambda t, u: t.to(f64) * torch.rsqrt(t.to(f64).square().mean(-1, keepdim=True) + 1e-5) * u.to(f64)  # noqa: E731
    u, v = rand(H), rand(H)
    torch.testing.assert_close(ops.rms_mean2(one, two, u, v, 1e-5).to(f64), 0.5 * (rms(one, u) + rms(two, v)), **tol)
    torch.testing.assert_close(ops.rms_mean2(one, None, u, None, 1e-5).to(f64), rms(one, u), **tol)
    nk, nv = H // 12 * 4 + 4, H // 20 * 4 + 4
    proj, uk = rand(T, H + nk + nv), rand(nk)
    kc, vc = torch.zeros(9, nk, dtype=dtype, device=DEV), torch.zeros(9, nv, dtype=dtype, device=DEV)
    before, slots = proj.clone(), torch.tensor([3, -1, 0, 8, 9], dtype=torch.int32, device=DEV)
    ops.qk_rownorm_store(proj, 0, H, H + nk, H, nk, nv, u, uk, 1e-5, slots, kc, vc)
    torch.testing.assert_close(proj[:, :H].to(f64), rms(before[:, :H], u), **tol)
    assert torch.equal(proj[:, H:], before[:, H:])
    for t, slot in ((0, 3), (2, 0), (3, 8)):
        torch.testing.assert_close(kc[slot].to(f64), rms(before[t, H:H + nk], uk), **tol)
        assert torch.equal(vc[slot], before[t, H + nk:])
    assert not kc[[1, 2, 4, 5, 6, 7]].any() and not vc[[1, 2, 4, 5, 6, 7]].any()
    gu = torch.cat([torch.tensor([-200.0, -9.0, 0.0, 30.0], device=DEV), rand(T * 2 * H - 4, dt=torch.float32) * 4]).view(T, 2 * H).to(dtype)
    want = torch.nn.functional.gelu(gu[:, :H].to(f64), approximate="tanh") * gu[:, H:].to(f64)
    torch.testing.assert_close(ops.gelu_tanh_mul(gu, torch.empty(T, H, dtype=dtype, device=DEV)).to(f64), want, **tol)


# four columns a thread: 1 to 64 threads a row, rows that fill the last run and rows that do not, ranks in pieces of 4
# and not; 24 columns: a column a thread
@pytest.mark.parametrize("dim,vdim,rank", [(64, 128, 32), (40, 64, 16), (5, 4, 3), (128, 256, 20), (100, 32, 5), (1, 16, 1), (40, 24, 16)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_recurrence_of_few_tokens(dim, vdim, rank, dtype):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(dim + vdim)
    heads, lens, f64 = 3, [1, 17, 0, 2], torch.float64
    T, width = sum(lens), 3 * (2 * dim + 2 * vdim) + rank
    width += -width % 8
    proj = (torch.randn(T, width, device=DEV, generator=gen) * 0.7).to(dtype)
    a2 = (torch.randn(heads * dim, rank, device=DEV, generator=gen) * 0.5).to(dtype)
    a2b, bonus = (torch.randn(heads * dim, device=DEV, generator=gen) for _ in range(2))
    norm = torch.rand(vdim, device=DEV, generator=gen) + 0.5
    start = torch.randn(6, heads, dim, vdim, device=DEV, generator=gen)
    slots = torch.tensor([4, 0, 2, 5], dtype=torch.int32, device=DEV)
    cu = torch.tensor([0, 1, 18, 18, 20], dtype=torch.int32, device=DEV)
    offs = (0, heads * dim, 2 * heads * dim, 2 * heads * dim + heads * vdim, 2 * heads * dim + 2 * heads * vdim)
    for with_bonus in (False, True):
        state = start.clone()
        got = ops.linear_recurrence(proj, *offs, a2, a2b, norm, state, slots, cu, 4, heads, dim, vdim, dim ** -0.5, 16.0, 1e-5,
                                    bonus=bonus if with_bonus else None)
        cols = lambda at, n: proj[:, at:at + heads * n].to(f64).view(T, heads, n)  # noqa: E731
        q, k, v, g = cols(offs[0], dim) * dim ** -0.5, cols(offs[1], dim), cols(offs[2], vdim), cols(offs[3], vdim)
        z = proj[:, offs[4]:offs[4] + rank].to(f64) @ a2.to(f64).t() + a2b.to(f64)
        decay = torch.sigmoid(z).pow(1 / 16.0).view(T, heads, dim)
        want, at = torch.zeros(T, heads, vdim, dtype=f64, device=DEV), 0
        after = start.to(f64)
        for r, n in enumerate(lens):
            for t in range(at, at + n):
                S, kv = after[int(slots[r])], k[t, :, :, None] * v[t, :, None, :]
                if with_bonus:
                    want[t] = (q[t, :, :, None] * (S + bonus.to(f64).view(heads, dim, 1) * kv)).sum(1)
                S = decay[t, :, :, None] * S + kv
                if not with_bonus:
                    want[t] = (q[t, :, :, None] * S).sum(1)
                after[int(slots[r])] = S
            at += n
        want = want * torch.rsqrt(want.square().mean(-1, keepdim=True) + 1e-5) * norm.to(f64) * torch.nn.functional.silu(g)
        # 17 steps and sums of up to 128 float32 terms; the result's own rounding
        tol = dict(atol=0.02, rtol=0.01) if dtype == torch.bfloat16 else dict(atol=1e-4, rtol=1e-4)
        torch.testing.assert_close(got.to(f64).view(T, heads, vdim), want, **tol)
        torch.testing.assert_close(state.to(f64), after, atol=1e-4, rtol=1e-4)


# keys whose last run of rows is padded
@pytest.mark.parametrize("dim,vdim", [(5, 256), (100, 128)])
@pytest.mark.parametrize("with_bonus", [False, True])
def test_recurrence_of_infinite_values(dim, vdim, with_bonus):
    """An infinite value makes its own column infinite, with the sign of its terms, and no other; rows that only pad a thread's
    run add nothing to it."""
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(dim)
    proj = torch.rand(2, 2 * dim + vdim + 16, device=DEV, generator=gen) + 0.5   # q, k, v, the decay's input
    proj[0, 2 * dim + 3], proj[0, 2 * dim + 6] = float("inf"), -float("inf")
    state = torch.zeros(1, 1, dim, vdim, device=DEV)
    ints = lambda *t: torch.tensor(t, dtype=torch.int32, device=DEV)  # noqa: E731
    got = ops.linear_recurrence(proj, 0, dim, 2 * dim, -1, 2 * dim + vdim, torch.rand(dim, 16, device=DEV, generator=gen), None, None, state,
                                ints(0), ints(0, 2), 1, 1, dim, vdim, 1.0, 16.0, 1e-5,
                                bonus=torch.ones(1, dim, device=DEV) if with_bonus else None)
    assert bool((got[:, 3] == float("inf")).all()) and bool((got[:, 6] == -float("inf")).all())
    rest = [c for c in range(vdim) if c not in (3, 6)]
    assert bool(torch.isfinite(got[:, rest]).all()) and bool(torch.isfinite(state[..., rest]).all())
    assert bool((state[0, 0, :, 3] == float("inf")).all()) and bool((state[0, 0, :, 6] == -float("inf")).all())


# the matrix-core kernels' sizes (one to eight tiles of 16 channels, columns for one wave to four of four tiles each, waves
# without columns), and two that the walks take; requests of less than a chunk, of whole and of broken segments
@pytest.mark.parametrize("dim,vdim,rank", [(64, 128, 32), (16, 16, 5), (32, 256, 16), (128, 64, 8), (128, 192, 24), (64, 48, 3), (100, 32, 5), (64, 40, 8)])
@pytest.mark.parametrize("form", ["sigmoid_power", "bonus", "double_exp"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_recurrence_in_segments(dim, vdim, rank, form, dtype):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(dim + vdim)
    heads, lens, f64 = 2, [70, 0, 33, 5, 64], torch.float64
    T, width = sum(lens), 2 * (2 * dim + 2 * vdim) + rank
    width += -width % 8
    proj = (torch.randn(T, width, device=DEV, generator=gen) * 0.7).to(dtype)
    a2 = (torch.randn(heads * dim, rank, device=DEV, generator=gen) * 0.5).to(dtype)
    a2b, bonus = (torch.randn(heads * dim, device=DEV, generator=gen) for _ in range(2))
    if form == "double_exp":
        a2b[::3] = 6.0   # decays that vanish (exp(-400)): zeros, not infinities
    norm = torch.rand(vdim, device=DEV, generator=gen) + 0.5
    start = torch.randn(6, heads, dim, vdim, device=DEV, generator=gen)
    ints = lambda *t: torch.tensor(t, dtype=torch.int32, device=DEV)  # noqa: E731
    slots, cu = [4, 0, 2, 5, 1], [0, 70, 70, 103, 108, 172]
    items = [(r, t, min(32, n - t), t // 32) for r, n in enumerate(lens) for t in range(0, n, 32)]
    first = [sum(-(-n // 32) for n in lens[:r]) for r in range(6)]
    offs = (0, heads * dim, 2 * heads * dim, 2 * heads * dim + heads * vdim, 2 * heads * dim + 2 * heads * vdim)
    state = start.clone()
    got = ops.linear_recurrence_segments(proj, *offs, a2, a2b, norm, state, ints(*slots), ints(*cu), ints(*sum(items, ())), len(items), 32,
                                         ints(*first), 5, heads, dim, vdim, dim ** -0.5, 16.0, 1e-5,
                                         decay="double_exp" if form == "double_exp" else "sigmoid_power", bonus=bonus if form == "bonus" else None)
    cols = lambda at, n: proj[:, at:at + heads * n].to(f64).view(T, heads, n)  # noqa: E731
    q, k, v, g = cols(offs[0], dim) * dim ** -0.5, cols(offs[1], dim), cols(offs[2], vdim), cols(offs[3], vdim)
    z = proj[:, offs[4]:offs[4] + rank].to(f64) @ a2.to(f64).t() + a2b.to(f64)
    decay = (torch.exp(-torch.exp(z)) if form == "double_exp" else torch.sigmoid(z).pow(1 / 16.0)).view(T, heads, dim)
    want, after = torch.zeros(T, heads, vdim, dtype=f64, device=DEV), start.to(f64)
    for r, slot in enumerate(slots):
        S = after[slot]
        for t in range(cu[r], cu[r + 1]):
            kv = k[t, :, :, None] * v[t, :, None, :]
            if form == "bonus":
                want[t] = (q[t, :, :, None] * (S + bonus.to(f64).view(heads, dim, 1) * kv)).sum(1)
            S = decay[t, :, :, None] * S + kv
            if form != "bonus":
                want[t] = (q[t, :, :, None] * S).sum(1)
        after[slot] = S
    want = want * torch.rsqrt(want.square().mean(-1, keepdim=True) + 1e-5) * norm.to(f64) * torch.nn.functional.silu(g)
    # sums of up to 128 float32 terms over some 16 steps that have not decayed yet; the result's own rounding
    tol = dict(atol=0.02, rtol=0.01) if dtype == torch.bfloat16 else dict(atol=1e-4, rtol=1e-4)
    torch.testing.assert_close(got.to(f64).view(T, heads, vdim), want, **tol)
    torch.testing.assert_close(state.to(f64), after, atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("at", [0, 5, 16, 31, 40])
def test_recurrence_in_segments_with_an_infinite_value(at):
    """An infinite value makes its column infinite from its token on: no token before it, no other column."""
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(at)
    dim, vdim, T = 64, 128, 70
    proj = torch.rand(T, 2 * dim + vdim + 16, device=DEV, generator=gen) + 0.5
    proj[at, 2 * dim + 3] = float("inf")
    ints = lambda *t: torch.tensor(t, dtype=torch.int32, device=DEV)  # noqa: E731
    state = torch.zeros(1, 1, dim, vdim, device=DEV)
    got = ops.linear_recurrence_segments(proj, 0, dim, 2 * dim, -1, 2 * dim + vdim, torch.rand(dim, 16, device=DEV, generator=gen), None, None,
                                         state, ints(0), ints(0, T), ints(0, 0, 32, 0, 0, 32, 32, 1, 0, 64, 6, 2), 3, 32, ints(0, 3), 1, 1, dim, vdim,
                                         1.0, 16.0, 1e-5)
    assert bool((got[at:, 3] == float("inf")).all()) and bool(torch.isfinite(got[:at]).all())
    rest = [c for c in range(vdim) if c != 3]
    assert bool(torch.isfinite(got[:, rest]).all()) and bool(torch.isfinite(state[..., rest]).all())
    assert bool((state[0, 0, :, 3] == float("inf")).all())


@pytest.mark.parametrize("dim,vdim,lost", [(16, 64, 3), (64, 64, 7), (64, 128, 7), (64, 256, 7), (128, 128, 7), (128, 256, 7)])
def test_segments_of_the_recurrence_add_channels_in_several_chains(dim, vdim, lost):
    """A state of 2^24 in the first channel and of 1 in one of every four: added behind the large one each 1 is lost, and so is
    every one of the seven others in its chain of products, but none of the other chains'."""
    from clockwork_amd import ops

    T, rank = 40, 16
    ints = lambda *t: torch.tensor(t, dtype=torch.int32, device=DEV)  # noqa: E731
    proj = torch.zeros(T, 2 * dim + vdim + rank, device=DEV)
    proj[:, :dim] = 1.0                                  # queries; keys, values and decay inputs are zero
    state = torch.zeros(1, 1, dim, vdim, device=DEV)
    ones = [d for d in range(dim) if d % 16 < 4]
    state[0, 0, ones] = 1.0
    state[0, 0, 0] = 2.0 ** 24
    got = ops.linear_recurrence_segments(proj, 0, dim, 2 * dim, -1, 2 * dim + vdim, torch.zeros(dim, rank, device=DEV),
                                         torch.full((dim,), -60.0, device=DEV), None, state, ints(0), ints(0, T),
                                         ints(0, 0, 32, 0, 0, 32, 8, 1), 2, 32, ints(0, 2), 1, 1, dim, vdim, 1.0, 16.0, 1e-5,
                                         decay="double_exp")  # exp(-exp(-60)): decays of 1
    want = 2.0 ** 24 + len(ones) - 1
    assert bool(((want - got.double() >= 0) & (want - got.double() <= lost + 1)).all())


# runs of 32, 50 and 128 keys; mixed heads over one, two (two kernels) and three key/value heads (three kernels), no
# mixing over four; sizes that are read in pieces and one by one, more columns than threads, groups of more than 16 heads
@pytest.mark.parametrize("heads,kv,dim,vdim,talk", [(12, 2, 128, 128, True), (6, 2, 20, 24, True), (3, 1, 40, 24, True), (6, 3, 64, 64, True),
                                                    (8, 4, 64, 96, False), (20, 1, 32, 300, True), (4, 4, 16, 16, False)])
@pytest.mark.parametrize("sk", [32, 50, 128])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sink_decode_runs(heads, kv, dim, vdim, talk, sk, dtype):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(heads * sk)
    rand = lambda *shape, dt=dtype: torch.randn(*shape, device=DEV, generator=gen).to(dt)  # noqa: E731
    lens, window, bs, f64 = [1, 31, 32, 33, 200, 333, 700], 300, 16, torch.float64
    R, pages = len(lens), -(-max(lens) // bs)
    tables = torch.randperm(R * pages, device=DEV, generator=gen).view(R, pages).int()
    kc, vc = rand(R * pages, bs, kv, dim), rand(R * pages, bs, kv, vdim)
    stride = heads * dim + 8
    q = rand(R, stride)
    r1, r2, sink = (torch.rand(heads, device=DEV, generator=gen) for _ in range(3))
    mix = torch.eye(heads, device=DEV) + 0.2 * rand(heads, heads, dt=torch.float32) if talk else None
    out = torch.full((R, heads * vdim), float("nan"), device=DEV).to(dtype)
    ints = lambda t: torch.as_tensor(t, dtype=torch.int32, device=DEV)  # noqa: E731
    kd, vd = kc.clone(), vc.clone()
    for r, n in enumerate(lens):  # what no request holds is poison
        for page in range(pages):
            kd[tables[r, page], max(0, min(bs, n - page * bs)):] = float("nan")
            vd[tables[r, page], max(0, min(bs, n - page * bs)):] = float("nan")
    ops.sink_attention_decode(q, stride, out, kd, vd, tables, ints(lens), ints(range(R + 1)), R, sk, -(-window // sk), r1, r2, sink, mix,
                              heads, kv, dim, vdim, bs, window, dim ** -0.5)
    for r, n in enumerate(lens):
        lo = max(0, n - window)
        keys = kc[tables[r].long()].reshape(-1, kv, dim)[lo:n].to(f64).repeat_interleave(heads // kv, 1)
        values = vc[tables[r].long()].reshape(-1, kv, vdim)[lo:n].to(f64).repeat_interleave(heads // kv, 1)
        scores = (q[r, : heads * dim].to(f64).view(heads, 1, dim) * keys.transpose(0, 1)).sum(-1) * dim ** -0.5
        away = n - 1 - torch.arange(lo, n, device=DEV, dtype=f64)
        scores = scores - r1.to(f64)[:, None] * torch.log1p(r2.to(f64)[:, None] * away)
        p = torch.softmax(torch.cat([scores, sink.to(f64)[:, None]], 1), 1)[:, :-1]
        if talk:
            p = mix.to(f64) @ p
        want = (p[:, :, None] * values.transpose(0, 1)).sum(1).view(-1)
        # float32 sums of up to 300 terms of a few units; bfloat16: the result's own rounding
        tol = dict(atol=0.005, rtol=0.005) if dtype == torch.bfloat16 else dict(atol=2e-5, rtol=2e-5)
        torch.testing.assert_close(out[r].to(f64), want, **tol)


@pytest.mark.parametrize("talk", [False, True])
def test_sink_decode_of_scores_that_are_no_numbers(talk):
    """A NaN reaches the result of its request (with mixing, of every head) and no other; keys whose scores are -inf weigh
    nothing, a whole run of them as well."""
    from clockwork_amd import ops

    heads, kv, dim, n, bs, sk = 4, 2, 32, 100, 16, 32
    gen = torch.Generator(device=DEV).manual_seed(6)
    pages = -(-n // bs)
    tables = torch.arange(3 * pages, dtype=torch.int32, device=DEV).view(3, pages)
    k, v = (torch.randn(3 * pages, bs, kv, dim, device=DEV, generator=gen) for _ in range(2))
    q = torch.rand(3, heads * dim, device=DEV, generator=gen) + 0.5
    q[0, 0] = float("nan")                     # head 0 of request 0
    k[pages:pages + 3] = -float("inf")         # the first 48 keys of request 1: a run and a half
    mix = torch.eye(heads, device=DEV) + 0.2 if talk else None
    out = torch.zeros(3, heads * dim, device=DEV)
    ints = lambda t: torch.as_tensor(t, dtype=torch.int32, device=DEV)  # noqa: E731
    ops.sink_attention_decode(q, heads * dim, out, k, v, tables, ints([n] * 3), ints(range(4)), 3, sk, -(-n // sk), None, None, None, mix,
                              heads, kv, dim, dim, bs, 0, dim ** -0.5)
    assert bool(torch.isnan(out[0] if talk else out[0, :dim]).all()) and bool(torch.isfinite(out[1:]).all())
    for r, first in ((0, 0), (1, 48), (2, 0)):
        keys, values = (t[r * pages:(r + 1) * pages].reshape(-1, kv, dim)[first:n].double().repeat_interleave(2, 1) for t in (k, v))
        p = torch.softmax((q[r].double().view(heads, 1, dim) * keys.transpose(0, 1)).sum(-1) * dim ** -0.5, 1)
        p = mix.double() @ p if talk else p
        want = (p[:, :, None] * values.transpose(0, 1)).sum(1).view(-1)
        if r == 0:
            if talk:
                continue
            want, got = want[dim:], out[r, dim:]
        else:
            got = out[r]
        torch.testing.assert_close(got.double(), want, atol=2e-5, rtol=2e-5)   # float32 sums of 100 terms of a few units


# rows of the streaming kernels (one and several), of the tiles between and of the wide tiles; sizes that each takes
@pytest.mark.parametrize("M,K,I", [(1, 96, 64), (8, 1536, 8960), (33, 256, 512), (130, 1536, 8960), (400, 1536, 8960), (1100, 1536, 8960), (9, 100, 36)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gate_up_products_with_gelu(M, K, I, dtype):
    from clockwork_amd import ops

    if dtype == torch.float32 and M > 130:
        pytest.skip("float32 has no epilogue of its own")
    gen = torch.Generator(device=DEV).manual_seed(M)
    x, w = (torch.randn(*s, device=DEV, generator=gen).to(dtype) for s in ((M, K), (2 * I, K)))
    w *= 2.0 * K ** -0.5
    h = x.double() @ w.double().t()
    want = torch.nn.functional.gelu(h[:, :I], approximate="tanh") * h[:, I:]
    got = ops.linear_swiglu(x, w, limit=ops.GELU_GATE).double()
    # a product is off by its float32 sum (sums of K terms that come to about 2: 2^-19) and, where it is written before
    # the gate is applied, by its rounding (2^-8 of it in bfloat16's 8 bits); the gate's slope is at most 1.13, and the result is
    # rounded once more
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    g, u = h[:, :I].abs(), h[:, I:].abs()
    off_g, off_u = half * g + 2.0 ** -19, half * u + 2.0 ** -19
    bound = 1.13 * (off_g * (u + off_u) + g * off_u) + (half + 2.0 ** -20) * want.abs()
    assert bool(((got - want).abs() <= bound).all())


# both kernels of several products (tiles of their own with 4, 8 and 16 waves, and streamed), outputs that end inside a tile, the ends of
# the rows that each takes; the last has more steps than the streaming kernel of several products is built for
@pytest.mark.parametrize("K,widths", [(8, (1, 17)), (520, (16, 33, 1, 100)), (1032, (3000, 1000)), (1536, (2048, 4640, 3072)), (1536, (1536, 1535, 5120)),
                                      (4096, (8000, 300)), (4360, (8000, 300))])
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("same", [True, False])
def test_several_products_in_one_launch(M, K, widths, same):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + K)
    xs = [torch.randn(M, K, device=DEV, generator=gen).bfloat16()] * len(widths)
    if not same:
        xs = [(x * (i + 1)).contiguous() for i, x in enumerate(xs)]
    ws = [(torch.randn(n, K, device=DEV, generator=gen) * K ** -0.5).bfloat16() for n in widths]
    got = ops.linear_several(xs, ws)
    tiles = sum(-(-n // 16) for n in widths)
    if got is None:
        assert M > 16 and (not same or tiles < 256 or K < 1024 or K >= 4096)
        return
    assert M <= 16 or same
    for x, w, y in zip(xs, ws, got):
        want = x.double() @ w.double().t()
        # K terms that come to a unit, in float32 (2^-24 each step of sums of some 60 at most), then one rounding
        assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -17 * float(x.abs().max())).all())


# one part of K and several, a K of the most blocks, heads of one tile and of many, a step of one row and of the most
@pytest.mark.parametrize("M", [1, 7, 16])
@pytest.mark.parametrize("nh,nkv,hd,K", [(14, 2, 64, 896), (1, 1, 16, 16), (3, 1, 48, 560), (12, 2, 128, 1536), (2, 2, 32, 1920)])
@pytest.mark.parametrize("with_bias", [True, False])
def test_float32_queries_keys_and_values_rotated_by_their_product(M, nh, nkv, hd, K, with_bias):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + K)
    N, rows = (nh + 2 * nkv) * hd, 40
    x, w = torch.randn(M, K, device=DEV, generator=gen), torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5
    b = torch.randn(N, device=DEV, generator=gen) if with_bias else None
    slots = torch.randperm(rows, device=DEV, generator=gen)[:M].int()
    if M > 3:
        slots[1], slots[2] = -1, rows   # no row, and one past the cache
    positions = torch.randint(0, 30000, (M,), device=DEV, generator=gen, dtype=torch.int32)
    for freq in (torch.zeros(hd // 2, device=DEV), 1.0 / 10000.0 ** (torch.arange(0, hd, 2, device=DEV) / hd)):
        caches = [torch.full((rows, nkv, hd), 7.0, device=DEV) for _ in range(4)]
        assert ops.qkv_rope_fused_supported(x, w, hd, hd, nh, nkv)
        q = ops.qkv_rope_fused(x, w, b, positions, slots, freq, nh, nkv, hd, caches[0], caches[1])
        apart = ops.linear(x, w)
        ops.rope_kv_write(apart, b, positions, slots, freq, hd, nh, nkv, hd, caches[2], caches[3])
        for got, want in ((q, apart[:, : nh * hd]), (caches[0], caches[2]), (caches[1], caches[3])):
            if not bool(freq.any()):
                assert torch.equal(got, want)   # turned by nothing: the same sums
            # two products and a sum of values of up to 6 units, contracted or not: a unit in the last place of each
            assert bool(((got - want).abs() <= 3 * 6 * 2.0 ** -24).all())
    assert not ops.qkv_rope_fused_supported(x, w, hd - 2, hd, nh, nkv) and not ops.qkv_rope_fused_supported(x[:, : K - 8], w[:, : K - 8], hd, hd, nh, nkv)


# few tiles and more than two a workgroup, an output and a K that end inside a tile and a step, the most planes
@pytest.mark.parametrize("N,K", [(896, 896), (768, 512), (1544, 8968), (4096, 4096), (5128, 1000), (64, 8192)])
@pytest.mark.parametrize("M", [17, 32, 33, 64])
def test_planes_of_17_to_64_rows(M, N, K):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, device=DEV, generator=gen).bfloat16()
    w = (torch.randn(N, K, device=DEV, generator=gen) * K ** -0.5).bfloat16()
    planes = ops._load("gemm").cw_gemm_bf16_skinny_planes(M, N, K)
    got = ops.linear(x, w, partial_ok=True, portions_partial_ok=True)
    assert isinstance(got, ops.PartialSums) == (planes > 1) and (planes == 1 or got.parts.shape == (planes, M, N))
    if planes > 1:
        # float32 sums of K terms that come to a unit
        torch.testing.assert_close(got.sum().double(), x.double() @ w.double().t(), rtol=0, atol=2.0 ** -17)
    # a reader that adds no planes inside its kernel gets what it got
    assert not isinstance(ops.linear(x, w, portions_partial_ok=True), ops.PartialSums)


# four and eight rows of the state a thread; requests of one token and of several, a request without a slot, keys of one run and of many
@pytest.mark.parametrize("heads,dim,r_vdim,rank", [(14, 64, 64, 16), (12, 128, 128, 32), (10, 64, 64, 5)])
@pytest.mark.parametrize("q_lens", [(1,), (1, 1, 1, 1, 1), (1, 7, 1)])
def test_a_recurrence_beside_the_runs_of_single_tokens(heads, dim, r_vdim, rank, q_lens):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(heads + len(q_lens))
    rand = lambda *s: torch.randn(*s, device=DEV, generator=gen)  # noqa: E731
    ints = lambda t: torch.as_tensor(t, dtype=torch.int32, device=DEV)  # noqa: E731
    R, T, kv, bs, pages, sk = len(q_lens), sum(q_lens), 2, 16, 20, 32
    ctx = [300 - 70 * r for r in range(R)]
    k, v = (rand(R * pages, bs, kv, dim).bfloat16() for _ in range(2))
    tables, cu = torch.arange(R * pages, device=DEV, dtype=torch.int32).view(R, pages), ints([0, *torch.tensor(q_lens).cumsum(0).tolist()])
    q = rand(T, heads * dim).bfloat16()
    sink = (rand(heads).abs(), rand(heads).abs(), rand(heads), torch.eye(heads, device=DEV) + 0.2 * rand(heads, heads))
    runs = -(-max(ctx) // sk)
    assert ops.sink_decode_takes_beside(torch.bfloat16, runs, heads, kv, True)
    assert not ops.sink_decode_takes_beside(torch.float32, runs, heads, kv, True) and not ops.sink_decode_takes_beside(torch.bfloat16, runs, heads, kv, False)
    qk, vv = heads * 64, heads * r_vdim
    proj = rand(T, 2 * qk + 2 * vv + rank).bfloat16()
    a2, bias, norm = rand(qk, rank).bfloat16(), rand(qk), rand(r_vdim)
    first = rand(R + 1, heads, 64, r_vdim)
    slots = ints([R - r if r != 1 else -1 for r in range(R)])

    def both(beside):
        state, out = first.clone(), torch.zeros(T, heads * dim, device=DEV, dtype=torch.bfloat16)
        args = (proj, 0, qk, 2 * qk, 2 * qk + vv, 2 * qk + 2 * vv, a2, bias, norm, state, slots, cu, R, heads, 64, r_vdim, 0.125, 16.0, 1e-6)
        y, launch = ops.linear_recurrence(*args, prepare=True) if beside else (ops.linear_recurrence(*args), None)
        assert (launch is not None) == beside
        ops.sink_attention_decode(q, heads * dim, out, k, v, tables, ints(ctx), cu, R, sk, runs, *sink, heads, kv, dim, dim, bs, 200, dim ** -0.5,
                                  beside=launch)
        return y, state, out

    apart, together = both(False), both(True)
    rows = torch.cat([torch.arange(int(cu[r]), int(cu[r + 1]), device=DEV) for r in range(R) if r != 1])   # a request without a slot has no outputs
    assert torch.equal(apart[0][rows], together[0][rows]) and torch.equal(apart[1], together[1]) and torch.equal(apart[2], together[2])


# K: 16, 23.25, 24 and 28 steps of 32 for 16 waves (idle waves, a step that K ends in); N: 512 tiles of gates and ups, or of 16
# outputs, and just more
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("K", [512, 744, 768, 896])
@pytest.mark.parametrize("N", [8192, 8208])
def test_streamed_products_of_fewer_steps_than_two_a_wave(M, K, N):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + K + N)
    x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    w[3, 0] = w[N - 1, K - 1] = float("inf")   # stay in their outputs, as infinities where x is not zero
    x[:, 0] = x[:, K - 1] = 1.0
    assert ops._load("gemm").cw_gemm_bf16_skinny_fast(1, M, N, K) == 1
    y = x.double() @ w.double().t()
    # float32 sums of K products of about 1 / sqrt(K): 2^-24 sqrt(K) of the result's spread at most, ten times that
    got = ops.linear(x, w, out_dtype=torch.float32)
    assert bool((got[:, [3, N - 1]] == float("inf")).all())
    rest = [i for i in range(N) if i not in (3, N - 1)]
    assert float((got.double() - y)[:, rest].abs().max()) < 10 * 2.0 ** -24 * K ** 0.5
    # and rounded once to bfloat16: 2^-9 of a value
    gated = ops.linear_swiglu(x, torch.cat([w, w.flip(0)]))
    assert ops._load("gemm").cw_gemm_bf16_skinny_fast(2, M, 2 * N, K) == 1
    want = torch.nn.functional.silu(y) * y.flip(1)
    keep = [i for i in rest if N - 1 - i in rest]
    torch.testing.assert_close(gated.double()[:, keep], want[:, keep], rtol=2.0 ** -8, atol=1e-5)


# K of 16 waves: an odd number of steps a wave and waves outside of K; 7 steps; 8, the last wave's cut; chunks of 5 and of 6 steps with
# a K that ends inside a pair. Partial sums of 64 MB and more: chunks of 4 and 5 steps, waves outside of K, a K that ends inside a pair
@pytest.mark.parametrize("M", [1, 16, 17, 40])
@pytest.mark.parametrize("N,K,partial", [(8208, 1408, False), (8192, 3592, False), (8192, 4056, False), (8192, 5016, False), (8192, 5912, False),
                                         (5120, 6560, True), (3584, 9384, True), (1536, 22016, True)])
def test_streams_of_whole_lines(M, N, K, partial):
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(M + K + N)
    x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    y = x.double() @ w.double().t()
    if partial:
        got = ops.linear(x, w, partial_ok=True)
        got = got.parts.sum(0) if isinstance(got, ops.PartialSums) else got
    else:
        got = ops.linear(x, w, out_dtype=torch.float32)
    # float32 sums of K products of about 1 / sqrt(K): 2^-24 sqrt(K) of the result's spread at most, ten times that; a library product, where the
    # kernels decline more than 16 rows, is rounded to bfloat16 once
    ours = got.dtype == torch.float32 if partial else M <= 16 or ops._load("gemm").cw_gemm_bf16_skinny_fast(1, M, N, K)
    bound = 10 * 2.0 ** -24 * K ** 0.5 if ours else 2.0 ** -8 * float(y.abs().max())
    assert float((got.double() - y).abs().max()) < bound
    # an infinite weight stays one, the outputs beside it finite (K in one set of fragments a wave; or in the last columns, which the waves outside of K read)
    if partial or K <= 4096:
        w[3, K - 1] = float("inf")
        x[:, K - 1] = 1.0
        again = ops.linear(x, w, partial_ok=True) if partial else ops.linear(x, w, out_dtype=torch.float32)
        again = again.parts.sum(0) if isinstance(again, ops.PartialSums) else again
        assert bool((again[:, 3] == float("inf")).all()) and bool(torch.isfinite(again[:, [2, 4]]).all())


# N, K: workgroups of 8 outputs by 8 waves (K up to 2048, the last one short), of 4, of up to 8 and up to 16 outputs by 16 waves, pieces
# of a row no multiple of four, a K that ends inside an operand's pieces
@pytest.mark.parametrize("N,K,most", [(900, 264, 16), (1536, 1536, 16), (896, 4864, 15), (1000, 2504, 16), (1537, 8960, 8), (2052, 600, 16), (3584, 3584, 16)])
@pytest.mark.parametrize("norm_dtype", [torch.bfloat16, torch.float32])
def test_products_that_join_the_stream_and_begin_a_norm(N, K, most, norm_dtype):
    """The stream, the rows times the norm's weights and the sums of squares against float64, and the two products that
    take such rows against themselves on rows that were normed before."""
    from clockwork_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(N + K)
    w = (torch.randn(N, K, device=DEV, generator=gen) / K ** 0.5).to(torch.bfloat16)
    norm = (1 + 0.1 * torch.randn(N, device=DEV, generator=gen)).to(norm_dtype)
    assert not ops.linear_join_ok(17, w, norm) and not ops.linear_join_ok(1, w[:, :200].contiguous(), norm)
    width = N // 8 * 8   # the readers take rows in pieces of 16 bytes
    hd, nh, nkv = 32, 5, 2
    gate_up = (torch.randn(2 * 4104, width, device=DEV, generator=gen) / width ** 0.5).to(torch.bfloat16)
    qkv = (torch.randn((nh + 2 * nkv) * hd, width, device=DEV, generator=gen) / width ** 0.5).to(torch.bfloat16)
    inv_freq = 1.0 / 1e4 ** (torch.arange(0, hd, 2, device=DEV, dtype=torch.float32) / hd)
    for M in (1, 2, most):
        x = torch.randn(M, K, device=DEV, generator=gen).to(torch.bfloat16)
        before = torch.randn(M, N, device=DEV, generator=gen)
        resid = before.clone()
        assert ops.linear_join_ok(M, w, norm)
        begun = ops.linear_join(x, w, resid, norm, 1e-6)
        want = before.double() + x.double() @ w.double().t()
        # float32 sums of K products of about 1 / sqrt(K): sqrt(K) roundings of 2^-24 at most, ten times that
        assert float((resid.double() - want).abs().max()) < 10 * 2.0 ** -24 * K ** 0.5
        torch.testing.assert_close(begun.x.double(), want * norm.double(), rtol=2.0 ** -8, atol=1e-5)
        torch.testing.assert_close(begun.squares.double().sum(1), want.square().sum(1), rtol=1e-5, atol=0)
        if N != width:
            continue
        # x by its norm in float64, rounded once: what the readers differ by is where the factor joins, 2^-9 of each of
        # ``width`` products of about 1 / sqrt(width) on either side, and the rounding of the result
        normed = want * torch.rsqrt(want.square().mean(-1, keepdim=True) + 1e-6) * norm.double()
        y = normed @ gate_up.double().t()
        inner = torch.nn.functional.silu(y[:, :4104]) * y[:, 4104:]
        got = ops.linear_swiglu(begun, gate_up).double()
        assert float((got - inner).norm() / inner.norm()) < 4 * 2.0 ** -9
        positions = torch.arange(M, dtype=torch.int32, device=DEV) * 7
        slots = torch.arange(M, dtype=torch.int32, device=DEV) * 2 + 1
        caches = [torch.zeros(2 * M + 2, nkv, hd, dtype=torch.bfloat16, device=DEV) for _ in range(4)]
        q = ops.qkv_rope_fused(begun, qkv, None, positions, slots, inv_freq, nh, nkv, hd, *caches[:2])
        q2 = ops.qkv_rope_fused(normed.to(torch.bfloat16), qkv, None, positions, slots, inv_freq, nh, nkv, hd, *caches[2:])
        for a, b in ((q, q2), (caches[0], caches[2]), (caches[1], caches[3])):
            assert float((a.double() - b.double()).norm() / b.double().norm()) < 6 * 2.0 ** -9
    with pytest.raises(ops.KernelError):
        ops.linear_swiglu(ops.BegunNorm(torch.zeros(17, 1024, dtype=torch.bfloat16, device=DEV), torch.zeros(17, 4, device=DEV), 1e-6),
                          torch.zeros(64, 1024, dtype=torch.bfloat16, device=DEV))


@pytest.mark.parametrize("widths,T,chosen", [((1536,), 1, [0]), ((1536, 1024, 896, 8), 300, [299, 0, 0, 17]), ((7, 3), 40, [39]), ((4097, 2), 5, [4, 3])])
def test_chosen_rows_of_several_matrices(widths, T, chosen):
    from clockwork_amd import ops

    rows = torch.tensor(chosen, dtype=torch.int32, device=DEV)
    matrices = [torch.randn(T, n, device=DEV).to(torch.float32 if i % 2 == 0 else torch.bfloat16) for i, n in enumerate(widths)]
    for got, m in zip(ops.take_rows(rows, *matrices), matrices):
        assert torch.equal(got, m[rows.long()])
    with pytest.raises(ops.KernelError):
        ops.take_rows(rows, matrices[0], torch.zeros(T + 1, 8, device=DEV))
    with pytest.raises(ops.KernelError):
        ops.take_rows(rows.long(), matrices[0])


# 40 tokens, of which one, two, 16, half and more have logits: up to half are made alone behind the last mixer, in a block of a
# pair no more than 16 of so few; three blocks of one mixer, pairs with and without a feed-forward (gates of one branch and of two); models of
# one block make all
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("wanted", [[39], [0, 33], list(range(16)), list(range(20)), list(range(21))], ids=len)
@pytest.mark.parametrize("config", ["B", "one", "FA", "FC", "long"])
def test_the_last_block_makes_the_rows_that_are_asked_for(tmp_path, monkeypatch, dtype, wanted, config):
    """Logits of rows that the last block makes alone against those of all rows; and the token after them, which reads the last
    block's pages and state."""
    from clockwork_amd.engine.batch import StepEntry
    from clockwork_amd.parts import block
    from clockwork_amd.weights.random_init import write_random_model
    from tests import replay
    from tests.configs import FUVAVIK_A, FUVAVIK_C, FUVAVIK_LONG, TINY_B

    cfg = {"B": TINY_B, "one": dict(TINY_B, num_hidden_layers=1), "FA": FUVAVIK_A, "FC": FUVAVIK_C, "long": FUVAVIK_LONG}[config]
    kind = block.PreNormBlock if config in ("B", "one") else block.ParallelBlock
    model_dir = write_random_model(tmp_path / "model", cfg, 5)
    tokens = torch.randint(0, cfg.get("vocab_size", cfg.get("vocab")), (41,), generator=torch.Generator().manual_seed(2)).tolist()
    made, forward_rows = [], kind.forward_rows
    monkeypatch.setattr(kind, "forward_rows", lambda self, resid, *a: made.append(resid.shape[0]) or forward_rows(self, resid, *a))

    def logits(rows):
        runner = replay.make_runner(model_dir, dtype, 8, 16)
        runner.reserve("r", 0, 40)
        first = runner.step([StepEntry("r", 0, tokens[:40], rows)]).clone()
        runner.reserve("r", 40, 1)
        return first, runner.step([StepEntry("r", 40, tokens[40:], [0])]).clone()

    all_rows, after = logits(list(range(40)))
    assert not made
    got, then = logits(wanted)
    taken = config not in ("one", "FC") and len(wanted) <= (20 if kind is block.PreNormBlock else 16)
    assert made == ([40] if taken else [])
    bound = dict(rtol=1e-5, atol=1e-5) if dtype == "float32" else dict(rtol=2e-2, atol=2e-2)   # roundings of bfloat16 in another kernel
    torch.testing.assert_close(got, all_rows[wanted], **bound)
    torch.testing.assert_close(then, after, **bound)


@pytest.mark.parametrize("n", [1, 5, 64])
def test_draw_counts_that_come_with_the_launch(n):
    """Counts as a list of ints and as a device tensor draw the same tokens; a sampler whose batch comes again draws what a new
    one does, on the same stream and on another; more rows than go with a launch."""
    from types import SimpleNamespace

    from clockwork_amd import ops
    from clockwork_amd.engine.sequence import SamplingParams
    from clockwork_amd.sampling.sampler import Sampler

    gen = torch.Generator(device=DEV).manual_seed(n)
    logits = torch.randn(n, 5003, device=DEV, generator=gen)
    temperature = torch.full((n,), 0.9, device=DEV)
    top_k = torch.arange(n, dtype=torch.int32, device=DEV) * 7 - 1
    top_p = torch.full((n,), 0.95, device=DEV)
    seeds = torch.arange(n, dtype=torch.int64, device=DEV) + 3
    counts = [(i * 977 + 5) % 100000 for i in range(n)]
    want = ops.sample(logits, temperature, top_k, top_p, seeds, torch.tensor(counts, device=DEV))
    assert torch.equal(ops.sample(logits, temperature, top_k, top_p, seeds, counts), want)
    for bad in (counts + [1], [-1] * n, [1 << 32] * n):
        with pytest.raises(ops.KernelError):
            ops.sample(logits, temperature, top_k, top_p, seeds, bad)
    more = ops.SAMPLE_COUNTED_ROWS + 1
    with pytest.raises(ops.KernelError):
        ops.sample(logits[:1].expand(more, -1).contiguous(), torch.ones(more, device=DEV), torch.zeros(more, dtype=torch.int32, device=DEV),
                   torch.ones(more, device=DEV), torch.zeros(more, dtype=torch.int64, device=DEV), [0] * more)

    seqs = [SimpleNamespace(seq_id=str(i), sampling_params=SamplingParams(temperature=0.8, top_k=40, seed=i), output_token_ids=[]) for i in range(n)]
    kept, other = Sampler(torch.device(DEV)), torch.cuda.Stream()
    for turn in range(4):
        fresh = Sampler(torch.device(DEV)).launch(logits, seqs, pending=turn % 2)
        assert torch.equal(kept.launch(logits, seqs, pending=turn % 2), fresh)
        other.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(other):
            again = kept.launch(logits, seqs, pending=turn % 2)
        other.synchronize()
        assert torch.equal(again, fresh)
        for s in seqs:
            s.output_token_ids.append(turn)


@pytest.mark.parametrize("temp", [1.3, 1.7, 1.9999999, 2.5, 3.0, 0.7, 0.3])
def test_ties_that_dividing_by_the_temperature_makes(temp):
    """Top-k of 1 keeps every token whose logit / T, rounded once to float32, is the largest's: of neighbouring floats some are
    tied so and some are not, and which, the drawn tokens say."""
    from clockwork_amd import ops

    t = torch.tensor(temp, dtype=torch.float32)
    near = torch.from_numpy((torch.tensor(7.3).view(torch.int32) + torch.arange(4000)).to(torch.int32).numpy()).view(torch.float32)
    equal = (near[1:] / t) == (near[:-1] / t)
    pairs = [i for kind in (True, False) for i in (equal == kind).nonzero().flatten()[:32].tolist()]
    n, V, tries = len(pairs), 4099, 24
    logits = torch.full((n, V), torch.finfo(torch.float32).min)
    logits[:, ::7] = float("-inf")
    logits[:, 11], logits[:, 4001] = near[pairs], near[[i + 1 for i in pairs]]
    logits = logits.to(DEV)
    seen = torch.zeros(n, V, dtype=torch.bool)
    for i in range(tries):
        got = ops.sample(logits, torch.full((n,), temp, device=DEV), torch.ones(n, dtype=torch.int32, device=DEV), torch.ones(n, device=DEV),
                         torch.arange(n, dtype=torch.int64, device=DEV), [i] * n).cpu()
        seen[torch.arange(n), got.long()] = True
    assert bool(seen[:, 4001].all()) and int(seen.sum()) == int(seen[:, [11, 4001]].sum())
    # a tied pair weighs the same: 24 draws miss one of the two once in 2^23
    assert torch.equal(seen[:, 11], equal[pairs])
