"""The sampling kernel against temperature, top-k, top-p and draw in float64:
descending order is by value, then by index.

Bound: weights are 2^-40 fixed point of a float exponential (2^-22 of the
weight), so that sums and boundaries lie within 1e-6 of the float64 ones."""

import pytest
import torch

import hyperspot.ops as ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EPS = 1e-6


def _row(kind, v, g):
    x = torch.randn(v, generator=g)
    if kind == "peaked":
        x[torch.randint(0, v, (9,), generator=g)] += 14
    elif kind == "ties":
        x = (x * 2).round()
    elif kind == "masked":
        x[torch.rand(v, generator=g) < 0.9] = float("-inf")
    elif kind == "equal":
        x.fill_(-3.0)
    elif kind == "wide":
        x = x * 1e4
    elif kind == "huge":
        x = torch.where(torch.rand(v, generator=g) < 0.5, -3e38, 3e38)
    return x


def _allowed(x, t, p, k, u):
    """Whether a token may be drawn, by its place in the running sum."""
    if t == 0:
        return x == x.max(), None
    y = (x.double() - x.max().double()) / max(t, 1e-6)
    if 0 < k < len(y):
        y = y.masked_fill(x < x.topk(k).values[-1], float("-inf"))
    w = y.softmax(-1)
    slack = EPS
    if p < 1:
        s, at = w.sort(descending=True, stable=True)
        before = s.cumsum(-1) - s
        w[at[before >= p]] = 0
        near = (before - p).abs() < EPS
        slack += float(s[near].sum())
    c = w.cumsum(-1)
    z = float(c[-1])
    return (c + slack * 2 > u * z) & (c - w - slack * 2 <= u * z) \
        & (w + slack > 0), w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [1, 7, 1000, 8193, 50257, 128256])
def test_sample_against_float64(vocab, dtype):
    g = torch.Generator().manual_seed(vocab)
    kinds = ["normal", "peaked", "ties", "masked", "equal", "wide", "huge"]
    options = [(1.0, 1.0, 0), (0.7, 0.9, 0), (1.3, 0.5, 40), (0.0, 1.0, 0),
               (1.0, 1.0, 5), (0.8, 0.999, vocab), (2.0, 0.95, 600),
               (1e-3, 0.9, 0), (0.9, 1e-7, 3)]
    rows, want = [], []
    for kind in kinds:
        for t, p, k in options:
            rows.append(_row(kind, vocab, g))
            want.append((t, p, k))
    x = torch.stack(rows).to(dtype)
    t, p, k = (torch.tensor(c) for c in zip(*want))
    u = torch.rand(len(rows), generator=g)
    u[::7] = 0.0
    u[3::7] = 1 - 2.0 ** -24
    args = [a.to(DEV) for a in (x, t, p, k.int(), u)]
    out = ops.sample(*args)
    assert torch.equal(out, ops.sample(*args))        # no order in its sums
    for b in range(len(rows)):
        row = x[b].float().clamp(max=torch.finfo(torch.float32).max)
        if not torch.isfinite(row).any():
            continue
        ok, _ = _allowed(row, float(t[b]), float(p[b]), int(k[b]),
                         float(u[b]))
        i = int(out[b])
        assert ok[i], (kinds[b // len(options)], want[b], i, float(u[b]))
        if t[b] == 0:
            assert i == int(row.argmax())


def test_rows_without_a_choice():
    x = torch.full((3, 16), float("-inf"), device=DEV)
    x[2] = torch.arange(16.0)
    ones = torch.ones(3, device=DEV)
    out = ops.sample(x, torch.tensor([0.0, 1.0, 1.0], device=DEV),
                     torch.tensor([1.0, 1.0, 0.0], device=DEV),
                     torch.zeros(3, dtype=torch.int32, device=DEV), ones / 2)
    assert out.tolist() == [0, 15, 15]


@pytest.mark.parametrize("vocab", [130, 1025, 8192, 50257])
def test_what_stays_is_few_or_not(vocab):
    """Around the most that are listed, and shares that fill the list or not."""
    g = torch.Generator().manual_seed(vocab)
    options = [(t, p, k) for t in (0.3, 1.0, 3.0) for p in (1.0, 0.97, 0.3)
               for k in (0, 1, 127, 128, 129, 256, 257, 513)]
    x = torch.stack([_row(kind, vocab, g) * 3 for kind in
                     ("normal", "peaked", "ties", "masked")
                     for _ in options]).bfloat16()
    t, p, k = (torch.tensor(c).repeat(4) for c in zip(*options))
    u = torch.rand(len(x), generator=g)
    out = ops.sample(*(a.to(DEV) for a in (x, t, p, k.int(), u)))
    for b, row in enumerate(x.float()):
        ok, _ = _allowed(row, float(t[b]), float(p[b]), int(k[b]),
                         float(u[b]))
        assert ok[int(out[b])], (b // len(options), options[b % len(options)])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [1001, 8192])
def test_nan_is_not_drawn(vocab, dtype):
    """As if it were -inf, beside infinities too."""
    g = torch.Generator().manual_seed(vocab)
    options = [(0.0, 1.0, 0), (1.0, 1.0, 0), (0.7, 0.9, 0), (1.0, 1.0, 5),
               (3.0, 0.8, 300)]
    x = torch.stack([_row(kind, vocab, g) for kind in
                     ("normal", "peaked", "ties", "wide") for _ in options])
    x[::3, 77] = float("inf")
    gone = torch.rand(x.shape, generator=g) < 0.3
    gone[:, :16] = True                        # a thread's whole load
    gone[-1] = True
    t, p, k = (torch.tensor(c).repeat(4) for c in zip(*options))
    u = torch.rand(len(x), generator=g)
    nan, low = (ops.sample(*(a.to(DEV) for a in (
        x.masked_fill(gone, fill).to(dtype), t, p, k.int(), u)))
        for fill in (float("nan"), float("-inf")))
    assert torch.equal(nan, low)
    assert not gone[:-1].gather(1, nan[:-1, None].cpu()).any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [7, 1001, 8192, 50257, 128256])
def test_rows_whole_and_in_slices(vocab, dtype):
    """The same rows in a batch that is not divided and in one that is: both
    against float64, NaN as -inf and infinities as the largest value."""
    g = torch.Generator().manual_seed(vocab)
    kinds = ["normal", "peaked", "ties", "masked", "wide"]
    options = [(1.0, 1.0, 0), (0.7, 0.9, 0), (1.3, 0.5, 40), (0.0, 1.0, 0),
               (1.0, 1.0, 5), (2.0, 0.95, 600)]
    pick = [(i, o) for i in range(2 * len(kinds)) for o in range(len(options))]
    x = torch.stack([_row(kind, vocab, g) for kind in kinds * 2])
    x[len(kinds):].masked_fill_(torch.rand(len(kinds), vocab, generator=g) < .3,
                                float("nan"))
    x[2::3, vocab // 2] = float("inf")
    x = x.to(dtype)
    t, p, k = (torch.tensor(c) for c in zip(*(options[o] for _, o in pick)))
    u = torch.rand(len(pick), generator=g)
    which = torch.tensor([i for i, _ in pick])
    least = -(-vocab // 32768)
    all_rows = torch.arange(len(pick)).repeat(513 // (least * len(pick)) + 1)
    assert len(all_rows) * least > 512 >= 20 * least
    args = [a.to(DEV) for a in (x, t, p, k.int(), u, which)]

    def draw(a):
        x, t, p, k, u, which = args
        a = a.to(DEV)
        return ops.sample(x[which[a]], t[a], p[a], k[a], u[a])
    whole = draw(all_rows)[:len(pick)].tolist()
    sliced = torch.cat([draw(a) for a in all_rows[:len(pick)].split(20)]) \
        .tolist()
    for b, (i, o) in enumerate(pick):
        row = x[i].float().nan_to_num(
            float("-inf"), posinf=torch.finfo(torch.float32).max,
            neginf=float("-inf"))
        if not torch.isfinite(row).any():
            continue
        ok, _ = _allowed(row, *options[o], float(u[b]))
        assert ok[whole[b]] and ok[sliced[b]], (i, o, whole[b], sliced[b])


@pytest.mark.parametrize("vocab,rows", [
    (16384, 1), (32768, 100), (32776, 100), (65537, 40), (128256, 1),
    (128256, 30), (128256, 60), (128256, 129), (524288, 1), (524296, 1)])
def test_rows_in_slices(vocab, rows):
    """1 to 16 slices a row, one value more than a slice takes, and rows that
    are not divided; what is likely lies in one slice, at its end or anywhere."""
    g = torch.Generator().manual_seed(vocab + rows)
    options = [(0.0, 1.0, 0), (1.0, 1.0, 0), (0.7, 0.9, 0), (0.9, 1.0, 50),
               (0.8, 0.95, 40), (1.0, 0.5, 250), (1.0, 1.0, 300),
               (3.0, 0.9, 0)]
    x = torch.randn(8, vocab, generator=g)
    x[0, -3:] += 9
    x[1, :40] += 14
    x[2, torch.randint(0, vocab, (60,), generator=g)] += 18
    x[3] = (x[3] * 2).round()
    x[4, : vocab // 2] = float("-inf")
    x[5, 100:] = float("-inf")
    x[6] = 1.0
    x[7, vocab // 3] = float("inf")
    x = x.bfloat16()
    pick = [(i, o) for i in range(8) for o in range(8)]
    pick = (pick * (rows // 64 + 1))[:max(rows, 64) // rows * rows]
    u = torch.rand(len(pick), generator=g)
    t, p, k = (torch.tensor(c)
               for c in zip(*(options[o] for _, o in pick)))
    which = torch.tensor([i for i, _ in pick])
    out = torch.cat([
        ops.sample(*(c.to(DEV) for c in (x[which[a]], t[a], p[a], k[a].int(),
                                         u[a])))
        for a in torch.arange(len(pick)).split(rows)]).tolist()
    for b, (i, o) in enumerate(pick[:64]):
        row = x[i].float().clamp(max=torch.finfo(torch.float32).max)
        ok, _ = _allowed(row, *options[o], float(u[b]))
        assert ok[out[b]], (i, options[o], out[b], float(u[b]))
        if o == 0:
            assert out[b] == int(row.argmax())


@pytest.mark.parametrize("vocab", [8192, 50257, 128256])
def test_shares_of_more_values_than_are_listed_first(vocab):
    """Divided rows list 64 values for a share, then 128: shares of 1 to 200 equal
    or almost equal values, far above the others, at every part of the draw."""
    g = torch.Generator().manual_seed(vocab)
    counts = [1, 60, 63, 64, 65, 66, 80, 100, 127, 128, 129, 130, 200]
    pick = [(n, same, (i + 0.5) / 7) for n in counts for same in (0, 1)
            for i in range(7)]
    x = torch.randn(len(pick), vocab, generator=g) - 30
    for b, (n, same, _) in enumerate(pick):
        at = torch.randperm(vocab, generator=g)[:n]
        x[b, at] = 4.0 if same else 4 + torch.rand(n, generator=g)
    x = x.bfloat16()
    t, p = torch.ones(len(pick)), torch.full((len(pick),), 0.98)
    u = torch.tensor([v for _, _, v in pick])
    k = torch.zeros(len(pick), dtype=torch.int32)
    out = ops.sample(*(a.to(DEV) for a in (x, t, p, k, u))).tolist()
    for b, (n, same, _) in enumerate(pick):
        ok, _ = _allowed(x[b].float(), 1.0, 0.98, 0, float(u[b]))
        assert ok[out[b]], (n, same, float(u[b]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab,rows", [
    (8200, 64), (16384, 130), (50257, 40), (128256, 3), (128256, 60)])
def test_lists_of_slices(vocab, rows, dtype):
    """What 1 to 15 slices list of their largest values: these in one slice, in one
    wave or in none more than elsewhere, more equal ones than a list takes, weights
    about 2^-12 of the largest, and top_k and shares that just have a list or not."""
    g = torch.Generator().manual_seed(vocab + rows)
    x = torch.randn(8, vocab, generator=g)
    anywhere = torch.randperm(vocab, generator=g)
    x[0, 5:65] += 20                           # one wave has all
    x[1, anywhere[:300]] = 9.0                 # equal, more than are listed
    x[2, anywhere[:250]] = 9.0 + torch.rand(250, generator=g)
    x[3] = -torch.log(anywhere + 1.0) * 1.2    # a power law
    x[4] = 12 - 12 * 0.6931472 + 0.02 * x[4]   # many of 2^-12
    x[4, anywhere[:9]] = 12.0
    x[5, anywhere[20:]] = float("-inf")        # fewer values than top_k
    x[6, anywhere[:40]] = 60.0                 # and others without weight
    x[7, vocab // 2:] -= 30                    # slices far below the others
    x = x.to(dtype)
    options = [(1.0, 0.9, 0), (0.8, 0.999, 0), (1.0, 1.0, 0), (1.0, 1.0, 50),
               (0.7, 0.95, 128), (1.0, 1.0, 129), (1.0, 0.3, 1)]
    pick = [(i, o, (n + 0.5) / 5) for i in range(8)
            for o in range(len(options)) for n in range(5)]
    t, p, k = (torch.tensor(c) for c in zip(*(options[o] for _, o, _ in pick)))
    which = torch.tensor([i for i, _, _ in pick])
    u = torch.tensor([n for _, _, n in pick])
    out = torch.cat([
        ops.sample(*(c.to(DEV) for c in (x[which[a]], t[a], p[a], k[a].int(),
                                         u[a])))
        for a in torch.arange(len(pick)).split(rows)]).tolist()
    for b, (i, o, n) in enumerate(pick):
        ok, _ = _allowed(x[i].float(), *options[o], float(u[b]))
        assert ok[out[b]], (i, options[o], out[b], n)


@pytest.mark.parametrize("vocab,rows", [(8200, 64), (32768, 200), (50257, 40),
                                        (128256, 30)])
def test_slices_that_list_nothing(vocab, rows):
    """Slices whose values are too many for a list, or for a share of a list, and those
    that just have one: 230 to 300 equal ones in one wave, in one slice and all over, so
    many within 2^-7 of a largest, and nothing but equal values."""
    g = torch.Generator().manual_seed(vocab)
    x = torch.randn(8, vocab, generator=g)
    anywhere = torch.randperm(vocab, generator=g)
    x[0] = 1.5
    x[1] = torch.randint(0, 4, (vocab,), generator=g).float()
    x[2, 8:248] = 9.0                          # one wave
    x[3, :4 * 300:4] = 9.0                     # one slice
    x[4, anywhere[:230]] = 9.0
    for i, n in ((5, 250), (6, 270), (7, 2000)):
        x[i, anywhere[:n]] = 12 - 4 * torch.rand(n, generator=g)
        x[i, anywhere[0]] = 12.0
    x = x.bfloat16()
    options = [(1.0, 0.9, 0), (1.0, 0.2, 0), (1.0, 1.0, 50), (0.7, 0.95, 100),
               (1.0, 1.0, 101), (1.0, 1.0, 0)]
    pick = [(i, o, (n + 0.5) / 3) for i in range(8)
            for o in range(len(options)) for n in range(3)]
    t, p, k = (torch.tensor(c) for c in zip(*(options[o] for _, o, _ in pick)))
    which = torch.tensor([i for i, _, _ in pick])
    u = torch.tensor([n for _, _, n in pick])
    out = torch.cat([
        ops.sample(*(c.to(DEV) for c in (x[which[a]], t[a], p[a], k[a].int(),
                                         u[a])))
        for a in torch.arange(len(pick)).split(rows)]).tolist()
    for b, (i, o, n) in enumerate(pick):
        ok, _ = _allowed(x[i].float(), *options[o], float(u[b]))
        assert ok[out[b]], (i, options[o], out[b], n)


@pytest.mark.parametrize("vocab", [1000, 32768])
def test_zeros_of_either_sign_are_equal(vocab):
    """The first of the largest values is -0."""
    x = torch.full((2, vocab), -1.0)
    x[0, [vocab // 3, vocab - 1]] = torch.tensor([-0.0, 0.0])
    x[1, [vocab // 5, vocab // 5 + 1]] = torch.tensor([-0.0, 0.0])
    opt = torch.zeros(2, device=DEV)
    out = ops.sample(x.bfloat16().to(DEV), opt, opt + 1, opt.int(), opt + 0.5)
    assert out.tolist() == [vocab // 3, vocab // 5]


def _few_above(kind, vocab):
    """Rows whose top_k-th largest value is the smallest one, or nearly."""
    x = torch.full((vocab,), 1.0)
    if kind == "three":                      # above all others, which are equal
        x[[vocab // 5, vocab // 2, vocab - 1]] = 2.0
    elif kind == "tail":                     # smaller values in the last load
        x[vocab // 3] = 1.5
        x[vocab - vocab % 8 - 1:] = 0.0
    elif kind == "masked":                   # and others without weight
        x[vocab // 4:] = float("-inf")
        x[: min(9, vocab // 4)] = 2.0
    elif kind == "steps":                    # more values than are listed below
        x = (torch.arange(vocab) % 700).float() * -0.01
    elif kind == "end":                      # one value below all others
        x[vocab // 3] = 0.0
    return x


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab,rows", [
    (v, r) for v in (2, 5, 9, 40, 700, 8191, 8192, 32768, 32773)
    for r in (4, 1030)] + [(128256, 4)])
def test_the_smallest_values_may_stay(vocab, rows, dtype):
    """top_k where fewer values than that are above the smallest one: in slices
    (4 rows) and without, over uniforms that reach every part of a row."""
    kinds = ["three", "tail", "masked", "steps", "end"]
    options = [(1.0, 1.0, 50), (0.7, 1.0, 3), (1.0, 0.6, 50), (2.0, 1.0, 256),
               (1.0, 1.0, 1), (0.05, 1.0, 200)]
    x = torch.stack([_few_above(kind, vocab) for kind in kinds]).to(dtype)
    pick = [(i, o, (n + 0.5) / 8) for i in range(len(kinds))
            for o in range(len(options)) for n in range(8)]
    t, p, k = (torch.tensor(c) for c in
               zip(*(options[o] for _, o, _ in pick)))
    which = torch.tensor([i for i, _, _ in pick])
    u = torch.tensor([n for _, _, n in pick])
    out = torch.cat([
        ops.sample(*(c.to(DEV) for c in (x[which[a]], t[a], p[a], k[a].int(),
                                         u[a])))
        for a in torch.arange(len(pick)).repeat(
            -(-rows // len(pick))).split(rows)])[:len(pick)].tolist()
    for b, (i, o, n) in enumerate(pick):
        if not torch.isfinite(x[i].float()).any():
            continue
        ok, _ = _allowed(x[i].float(), *options[o], float(u[b]))
        assert ok[out[b]], (kinds[i], options[o], out[b], n)


def test_one_option_for_all_rows():
    """Options of one element count for every row; top_k of 64 bits."""
    g = torch.Generator().manual_seed(1)
    x = torch.randn(9, 500, generator=g).to(DEV)
    u = torch.rand(9, generator=g).to(DEV)
    one = [torch.tensor([c], device=DEV) for c in (0.7, 0.9)]
    k = torch.tensor([1 << 40], device=DEV)
    ref = ops.sample(x, *(t.expand(9).contiguous() for t in one),
                     torch.zeros(9, dtype=torch.int32, device=DEV), u)
    assert torch.equal(ops.sample(x, *one, k, u), ref)


@pytest.mark.parametrize("vocab", [1, 7, 32768, 128256])
def test_no_rows(vocab):
    none = torch.empty(0, device=DEV)
    for dtype in (torch.bfloat16, torch.float32):
        out = ops.sample(torch.empty(0, vocab, dtype=dtype, device=DEV), none,
                         none, none.int(), none)
        assert out.shape == (0,) and out.dtype == torch.long


def test_a_vocabulary_beyond_the_kernel():
    v = (1 << 23) + 8
    x = torch.zeros(2, v, device=DEV, dtype=torch.bfloat16)
    x[:, v - 3] = 40
    f = lambda *c: torch.tensor(c, device=DEV)
    for t, p, k in ((0.0, 1.0, 0), (1.0, 1.0, 0), (1.0, 0.9, 50)):
        out = ops.sample(x, f(t, 0.0), f(p, p), f(k, k).int(), f(0.3, 0.6))
        assert out.tolist() == [v - 3] * 2
