"""Attention over the paged pool: the step plan (CPU) and the kernels against
a plain fp32 attention over the gathered rows (GPU)."""

import numpy as np
import pytest
import torch

from deepspeed_amd.inference.ragged import PagedKVCache
from deepspeed_amd.ops import _loader, paged_attention as plans
from deepspeed_amd.ops.paged_attention import StepPlan

# (slots with the new rows of each, kept tokens by slot)
STEPS = {
    "decode": ([(0, 1), (1, 1), (2, 1)], [0, 31, 700]),
    "portion": ([(0, 70)], [33]),
    "first": ([(0, 129), (1, 129)], [0, 0]),
    "packed": ([(0, 1), (2, 45), (1, 1), (2, 3)], [64, 1, 500]),
    "long": ([(0, 1)], [5000]),
}


def _rows(step, lens):
    """Slots and positions of the rows; a slot's later runs go on behind its
    earlier ones."""
    slots, pos, at = [], [], list(lens)
    for s, m in step:
        slots += [s] * m
        pos += range(at[s], at[s] + m)
        at[s] += m
    return slots, np.array(pos), at


@pytest.mark.parametrize("lens,rows,kv_heads", [
    ([1], 1, 8), ([127] * 3, 1, 8), ([16000], 1, 8), ([16000] * 8, 1, 8),
    (range(1000, 3000, 63), 1, 8), ([2000] * 97, 1, 8), ([900] * 33, 1, 32),
    ([2000] * 24, 200, 8), ([200] * 15, 250, 8), ([30000] * 2, 7, 1)])
def test_splits_fill_whole_rounds(lens, rows, kv_heads):
    """Decoding requests beside a run of more rows: no more workgroups than whole
    rounds of those that the CUs hold, or than there are tiles; every key once."""
    lens = list(lens)
    slots = list(range(len(lens))) + [len(lens)] * (rows - 1)
    pos = np.array([*lens, *range(rows - 1)])
    tables = {s: list(range(500)) for s in range(len(lens) + 1)}
    plan = StepPlan.build(slots, pos, tables, 64, 4 * kv_heads, kv_heads, "cpu")
    meta = plan.meta.numpy()
    items = meta[:4 * plan.items].reshape(-1, 4)
    merges = meta[4 * (plan.items + plan.runs):][:2 * plan.merges].reshape(-1, 2)
    full = plans.ROUND[plan.nq]
    ends = [abs(items[f + n - 1][3]) for f, n in merges]
    if sum(ends) * kv_heads < plans.KEYS * full:
        full = plans.FEWER
    tiles = -(-plan.merges * kv_heads // full)
    assert plan.items * kv_heads <= tiles * full or plan.items == plan.merges
    for first, n in merges:
        at = 0
        for it in items[first:first + n]:
            assert it[2] == at < abs(it[3])
            at = abs(it[3])
    assert {*map(int, ends)} >= {n + 1 for n in lens}


@pytest.mark.parametrize("lens,rows,heads,split", [
    # tiles for all workgroups, and a few less
    ([2000] * 128, 1, (32, 8), False), ([2000, 3000] * 55, 1, (32, 8), True),
    ([382] * 9, 93, (256, 32), False), ([382] * 9, 40, (256, 32), True),
    # evenly long, a round and a quarter: each in two
    ([15828] * 2, 319, (64, 8), True)])
def test_many_tiles_and_even_ones(lens, rows, heads, split):
    slots = list(range(len(lens))) + [len(lens)] * (rows - 1)
    pos = np.array([*lens, *range(lens[0], lens[0] + rows - 1)])
    tables = {s: list(range(500)) for s in range(len(lens) + 1)}
    plan = StepPlan.build(slots, pos, tables, 64, *heads, "cpu")
    assert plan.any_merge == split
    if rows == 319:
        assert plan.items == 2 * plan.merges


@pytest.mark.parametrize("lens,heads,parts", [
    # whole, since a merge takes longer, and cut
    ([125] * 3, (32, 8), 1), ([150] * 24, (32, 8), 1), ([2000] * 32, (32, 8), 1),
    ([500], (32, 8), 1), ([16000] * 8, (32, 8), 3), ([11000], (16, 1), 86),
    # a tile of columns of 64 requests: as many as the first line takes, one more
    ([4000] * 64, (32, 8), 1), ([9000] * 65, (32, 8), 1)])
def test_cuts_by_what_they_take(lens, heads, parts):
    tables = {s: list(range(300)) for s in range(len(lens))}
    plan = StepPlan.build(list(range(len(lens))), np.array(lens), tables, 64,
                          *heads, "cpu")
    assert plan.any_merge == (plan.items > plan.merges)
    if len(lens) * heads[1] <= plans.FEWER:
        assert plan.items == parts * len(lens)
        end, n = np.array(lens) + 1, np.full(len(lens), parts)
        whole = plans._cost(end, np.ones_like(n), heads[1], plan.nq)
        assert plans._cost(end, n, heads[1], plan.nq) <= whole


@pytest.mark.parametrize("bs,parts", [(16, 3), (24, 3), (32, 1), (64, 1)])
def test_cuts_by_blocks(bs, parts):
    """Cuts by what the parts take are for blocks that hold a whole tile of keys."""
    need = -(-1881 // bs)
    tables = {s: list(range(s * need, (s + 1) * need)) for s in range(31)}
    args = (list(range(31)), np.full(31, 1880, np.int64), tables, bs, 32, 8)
    for items in (StepPlan.build(*args, "cpu").items, plans._planned(*args)[1]):
        assert items == 31 * parts


@pytest.mark.parametrize("heads", [(8, 8), (14, 2), (32, 8), (16, 1)])
def test_step_plan_equals_numpys(heads):
    """Single rows and runs of every length, slots that come again, tables of any
    kind, ties in length and long histories."""
    ext = _loader.get_ext()
    if ext is None:
        pytest.skip("the native plan is the extension's")
    rng = np.random.default_rng(0)
    seen = set()
    for case in range(200):
        bs = int(rng.choice([1, 16, 24, 64]))
        slots, pos, ends = [], [], {}
        for _ in range(rng.integers(1, 40)):
            s = int(rng.integers(0, 30))
            n = int(rng.choice([1, 1, 2, 17, 64, 300]))
            at = int(rng.choice([0, 5, 130, 500, 500, 4000]))
            slots += [s] * n
            pos += range(at, at + n)
            ends[s] = max(ends.get(s, 0), at + n)
        if case % 5 == 0:       # long runs only: tiles of 128 columns
            slots, pos = [0] * 300 + [1] * 70, [*range(900, 1200), *range(70)]
            pos[300:] = [p + 13 * case for p in pos[300:]]
            ends = {0: 1200, 1: 70 + 13 * case}
        tables = {s: rng.integers(0, 1000, -(-n // bs)) for s, n in ends.items()}
        if case % 2:
            tables = {s: t.tolist() for s, t in tables.items()}
        args = slots, np.array(pos), tables, bs, *heads
        want, *counts = plans._planned(*args)
        got, *native = ext.step_plan(*args, plans._lines(), False)
        assert torch.equal(got, want) and native == counts
        items, runs, merges, any_merge, nq, head = counts
        plan = StepPlan.build(*args, "cpu")
        assert torch.equal(plan.meta, want) and torch.equal(plan.dst, want[head:])
        assert (plan.items, plan.runs, plan.merges, plan.any_merge, plan.nq) == \
            (items, runs, merges, any_merge, nq)
        seen.add(nq)
    assert seen >= {2, 8}


@pytest.mark.parametrize("slots,pos", [
    ([], []), ([0], [64]), ([0, 1], [1]), ([0], [-1]), ([0, 2], [0, 128]),
    # in the next request's blocks, after rows of its own and in a run
    ([0, 2], [64, 0]), ([0, 2], [100, 0]), ([2, 0, 0], [5, 63, 64])])
@pytest.mark.parametrize("native", [True, False])
def test_no_step(slots, pos, native, monkeypatch):
    """Refused alike with the extension and on a host without it."""
    if native and _loader.get_ext() is None:
        pytest.skip("no extension")
    if not native:
        monkeypatch.setattr(_loader, "get_ext", lambda: None)
    pos, tables = np.array(pos, np.int64), {0: [3], 1: [], 2: [7, 8]}
    with pytest.raises((ValueError, IndexError)):
        StepPlan.build(slots, pos, tables, 64, 8, 8, "cpu")
    if len(slots) == len(pos) > 0:
        with pytest.raises(IndexError):
            StepPlan.rows(slots, pos, tables, 64)


@pytest.mark.parametrize("name", list(STEPS))
@pytest.mark.parametrize("bs", [16, 24, 64])
@pytest.mark.parametrize("heads", [(8, 8), (14, 2), (32, 8)])
def test_step_plan_covers_every_key_once(name, bs, heads):
    step, lens = STEPS[name]
    slots, pos, end = _rows(step, lens)
    rng = np.random.default_rng(0)
    free = list(rng.permutation(1000))
    tables = {s: [int(free.pop()) for _ in range(-(-n // bs))]
              for s, n in enumerate(end)}
    plan = StepPlan.build(slots, pos, tables, bs, *heads, "cpu")
    meta = plan.meta.numpy()
    items = meta[:4 * plan.items].reshape(-1, 4)
    runs = meta[4 * plan.items:][:4 * plan.runs].reshape(-1, 4)
    merges = meta[4 * (plan.items + plan.runs):][:2 * plan.merges]
    merges = merges.reshape(-1, 2)
    table = meta[4 * (plan.items + plan.runs) + 2 * plan.merges:]
    G = heads[0] // heads[1]
    for i, (s, p) in enumerate(zip(slots, pos)):
        assert plan.dst[i] == tables[s][p // bs] * bs + p % bs
        r = next(r for r in runs if r[0] <= i < r[0] + r[1])
        assert r[2] - r[1] + i - r[0] == p
        assert list(table[r[3]:r[3] + p // bs + 1]) == \
            tables[s][:p // bs + 1]
    for first, n in merges:
        run, tile = items[first][:2]
        ncols = runs[run][1] * G
        last = (min((tile + 1) * 16 * plan.nq, ncols) - 1) // G
        want = runs[run][2] - runs[run][1] + last + 1
        at = 0
        for it in items[first:first + n]:
            assert tuple(it[:2]) == (run, tile) and it[2] == at
            assert it[2] % 32 == 0 and (it[3] < 0) == (n == 1)
            at = abs(it[3])
            assert at > it[2]
        assert at == want
    tiles = sorted((int(items[f][0]), int(items[f][1])) for f, _ in merges)
    assert tiles == [(r, t) for r in range(len(runs))
                     for t in range(-(-runs[r][1] * G // (16 * plan.nq)))]
    assert plan.items == merges[:, 1].sum()


def test_mask_and_places_are_made_once_a_step(monkeypatch):
    """Every layer of a step reads the same mask and row places; the mask can be
    set, for the step, and both are new in the next one."""
    made = []
    rows = StepPlan.rows
    monkeypatch.setattr(StepPlan, "rows",
                        lambda *a: made.append(0) or rows(*a))
    cache = PagedKVCache(3, 2, 2, 32, 8, block_size=4)
    assert cache.last_mask is None
    for step, n in enumerate((5, 1, 6)):
        cache.begin_step([1, 0], n)
        mask = cache.last_mask
        lo = int(cache._starts[0])
        assert mask.shape == (2, 1, n, lo + n)
        assert torch.equal(mask[0, 0].sum(1), lo + 1 + torch.arange(n))
        k = torch.randn(3, 2, 2, n, 8)
        for layer in range(3):
            assert cache.last_mask is mask
            got, _ = cache.update(layer, k[layer], k[layer])
            assert torch.equal(got[:, :, lo:], k[layer])
        assert len(made) == step + 1
        cache.last_mask = other = ~mask
        assert cache.last_mask is other
        cache.last_mask = None
        assert cache.last_mask is None
        cache.end_step()
        assert cache.last_mask is None


@pytest.mark.parametrize("which", [0, 1, 2, None])
def test_rope_attention_leaves_gradients_alone(which, monkeypatch):
    """With a gradient for queries, keys or values the caller's own path, which
    has one, is taken."""
    cache = PagedKVCache(1, 1, 2, 64, 128)
    monkeypatch.setattr(cache, "_eligible", lambda *a: True)
    monkeypatch.setattr(cache, "_attend", lambda *a: "kernels")
    qkv = [torch.zeros(1, 3, h, 128) for h in (4, 2, 2)]
    if which is not None:
        qkv[which].requires_grad_()
    want = None if which is not None else "kernels"
    assert cache.rope_attention(0, *qkv, None, None) == want
    with torch.no_grad():
        assert cache.rope_attention(0, *qkv, None, None) == "kernels"
        # a mask of the caller's own is for the path that has one
        cache.begin_step([0], 3)
        cache.last_mask
        assert cache.rope_attention(0, *qkv, None, None) == "kernels"
        cache.last_mask = torch.ones(1, 1, 3, 3, dtype=torch.bool)
        assert cache.rope_attention(0, *qkv, None, None) is None
        cache.end_step()
        assert cache.rope_attention(0, *qkv, None, None) == "kernels"


@pytest.mark.parametrize("name", ["update", "decode_attention"])
def test_caches_with_methods_of_their_own(name, monkeypatch):
    """A subclass's or an instance's update and decode_attention are called."""
    own = type("Own", (PagedKVCache,), {name: lambda self, *a: None})
    qkv = [torch.zeros(1, 1, 2, 128)] * 3
    for cls in (own, PagedKVCache):
        cache = cls(1, 1, 2, 64, 128)
        monkeypatch.setattr(cache, "_eligible", lambda *a: True)
        monkeypatch.setattr(cache, "_attend", lambda *a: "kernels")
        assert cache.rope_attention(0, *qkv, None, None) == \
            (None if cls is own else "kernels")
    setattr(cache, name, lambda *a: None)
    assert cache.rope_attention(0, *qkv, None, None) is None


def test_kernels_get_aligned_tensors(monkeypatch):
    """16-byte accesses: a slice at an odd offset, or a pool of another layout
    than the cache's own, is laid out anew; a misaligned cache is left to the
    general path."""
    from deepspeed_amd.ops import paged_attention as P
    seen = []

    class Ext:
        def __getattr__(self, name):
            def call(*args):
                seen.append(name)
                for t in args:
                    if torch.is_tensor(t) and t.dtype is torch.bfloat16:
                        assert t.is_contiguous() and t.data_ptr() % 16 == 0
                return args[0]
            return call

    monkeypatch.setattr(P, "get_ext", Ext)

    def odd(*shape):
        n = int(np.prod(shape))
        return torch.randn(n + 1).bfloat16()[1:].view(shape)

    q, k, v = odd(1, 1, 4, 128), odd(1, 1, 2, 128), odd(1, 1, 2, 128)
    pool = odd(3, 2, 64, 128)
    P.paged_decode_attention(q[0], pool, pool, torch.zeros(1, 1),
                             torch.ones(1))
    cache = PagedKVCache(1, 1, 2, 64, 128, dtype=torch.bfloat16)
    cache.begin_step([0], 1)
    assert torch.equal(cache._attend(0, q, k, v), q)
    assert seen == ["paged_decode", "paged_append", "paged_rows"]

    class OnGpu(torch.Tensor):
        is_cuda = True

    q = torch.zeros(1, 1, 4, 128, dtype=torch.bfloat16).as_subclass(OnGpu)
    for p, want in ((torch.zeros(3, 2, 64, 128).bfloat16(), True),
                    (pool, False)):
        cache.k[0], cache.v[0] = p.as_subclass(OnGpu), p
        assert cache._eligible(0, q, q, q) is want
        cache.k[0], cache.v[0] = cache.v[0].as_subclass(OnGpu), pool
        assert cache._eligible(0, q, q, q) is False


def _reference(q, k, v, pos, scale):
    """q [m, H, D] at positions ``pos`` over k, v [L, Hkv, D], in fp64."""
    G = q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(G, 1).transpose(0, 1)
            for t in (k, v))
    s = torch.matmul(q.double().transpose(0, 1),
                     k.transpose(1, 2).contiguous()) * scale
    hidden = torch.arange(k.shape[1], device=q.device)[None] > pos[:, None]
    return torch.matmul(torch.softmax(s.masked_fill(hidden, -np.inf), -1),
                        v).transpose(0, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(STEPS))
@pytest.mark.parametrize("bs", [16, 24, 64])
@pytest.mark.parametrize("heads", [(1, 1), (8, 8), (14, 2), (32, 8), (16, 1)])
def test_paged_attention_gpu(name, bs, heads):
    """Rotation, cache write and attention of every kind of step. The pool's
    other rows hold NaN: nothing outside a request's own rows is used."""
    H, Hkv = heads
    step, lens = STEPS[name]
    slots, pos, end = _rows(step, lens)
    g = torch.Generator().manual_seed(H * 100 + bs)

    def rand(*shape):
        return torch.randn(shape, generator=g).to(torch.bfloat16).cuda()

    cache = PagedKVCache(1, 3, Hkv, 8192, 128, dtype=torch.bfloat16,
                         device="cuda", block_size=bs,
                         num_blocks=sum(-(-n // bs) for n in end) + 5)
    cache.free_blocks = torch.randperm(cache.num_blocks, generator=g).tolist()
    for t in (cache.k[0], cache.v[0]):
        t.fill_(float("nan"))
    kept = []
    for s, n in enumerate(lens):
        cache._ensure_blocks(s, n)
        rows = rand(n, Hkv, 128), rand(n, Hkv, 128)
        p = torch.arange(n, device="cuda")
        blk = torch.tensor(cache.block_table[s], dtype=torch.long,
                           device="cuda")
        for pool, x in zip((cache.k[0], cache.v[0]), rows):
            pool[blk[p // bs], :, p % bs] = x
        kept.append(rows)
    cache.lens[:] = torch.tensor(lens + [0] * (3 - len(lens)))
    T = len(slots)
    q, k, v = rand(T, 1, H, 128), rand(T, 1, Hkv, 128), rand(T, 1, Hkv, 128)
    ang = torch.rand(8192, 64, generator=g) * 6.28
    cos, sin = ang.cos().cuda(), ang.sin().cuda()
    positions = torch.tensor(pos, dtype=torch.int32, device="cuda")[:, None]
    cache.begin_step(slots, 1, offsets=[int(p) - lens[s] for s, p in
                                        zip(slots, pos)])
    got = cache.rope_attention(0, q, k, v, cos, sin, positions)
    from deepspeed_amd.ops.rope import apply_rope
    q2, k2 = (apply_rope(x, cos, sin, positions) for x in (q, k))
    cache.end_step()
    for s, n in enumerate(lens):
        mine = [i for i, t in enumerate(slots) if t == s]
        if not mine:
            continue
        kk = torch.cat([kept[s][0], k2[mine, 0]])
        vv = torch.cat([kept[s][1], v[mine, 0]])
        at = torch.tensor(pos[mine], device="cuda")
        want = _reference(q2[mine, 0], kk, vv, at, 128 ** -0.5)
        # one rounding to bf16 (2^-9 of the value) of sums whose terms carry
        # 2^-18 (split probabilities) and fp32 rounding
        err = (got[mine, 0].double() - want).abs()
        # 2^-13 a unit of the values; rotations rounded another way move the
        # result by some 2^-9 of the new rows' share, a value's 2^-8 at most
        assert (err <= 2.0 ** -7 * want.abs() + 2.0 ** -10).all(), err.max()
        blk = torch.tensor(cache.block_table[s], device="cuda")
        # fp32 rounding of the rotation may turn one rounding to bf16
        torch.testing.assert_close(cache.k[0][blk[at // bs], :, at % bs],
                                   k2[mine, 0], rtol=2.0 ** -7,
                                   atol=2.0 ** -20)
        assert torch.equal(cache.v[0][blk[at // bs], :, at % bs], v[mine, 0])


@pytest.mark.gpu
@pytest.mark.parametrize("device", ["cuda", "cpu"])
def test_lengths_kept_on_the_gpu(device):
    """The cache's lengths may lie beside its pool."""
    res = []
    for lens in ("cpu", "cuda"):
        torch.manual_seed(0)
        cache = PagedKVCache(1, 2, 2, 64, 128, dtype=torch.bfloat16,
                             device=device)
        cache.lens = cache.lens.to(lens)
        for n in (3, 1):
            cache.begin_step([1, 0], n)
            q, k, v = (torch.randn(2, n, h, 128).bfloat16().to(device)
                       for h in (4, 2, 2))
            o = cache.decode_attention(0, q, k, v)
            if o is None:
                o, _ = cache.update(0, k.transpose(1, 2), v.transpose(1, 2))
            cache.end_step()
        res.append(o)
    assert torch.equal(*res)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.05, -0.05, 0.0])
@pytest.mark.parametrize("splits", [None, 1, 5])
def test_paged_decode_scales_and_splits(scale, splits):
    from deepspeed_amd.ops.paged_attention import paged_decode_attention
    torch.manual_seed(1)
    lens = torch.tensor([0, 1, 33, 200], dtype=torch.int32, device="cuda")
    table = torch.randperm(16)[:16].view(4, 4).int().cuda()
    kp, vp = (torch.randn(16, 2, 64, 128, device="cuda").bfloat16()
              for _ in range(2))
    q = (4 * torch.randn(4, 14, 128, device="cuda")).bfloat16()
    got = paged_decode_attention(q, kp, vp, table, lens, splits, scale)
    assert not got[0].any()
    for i in range(1, 4):
        n = int(lens[i])
        kk, vv = (p[table[i].long()].transpose(1, 2).reshape(-1, 2, 128)[:n]
                  for p in (kp, vp))
        want = _reference(q[i:i + 1], kk, vv,
                          torch.tensor([n - 1], device="cuda"), scale)
        err = (got[i:i + 1].double() - want).abs()
        assert (err <= 2.0 ** -8 * want.abs() + 2.0 ** -13).all(), err.max()


@pytest.fixture
def blocks(monkeypatch):
    """Every run's items have 128 columns."""
    from deepspeed_amd.ops import paged_attention as P
    monkeypatch.setattr(P, "BLOCK", 1)
    monkeypatch.setattr(P, "BLOCK_WORK", 0)


@pytest.mark.parametrize("name", list(STEPS))
@pytest.mark.parametrize("heads", [(14, 2), (32, 8)])
def test_block_plan_covers_every_key_once(name, heads, blocks):
    test_step_plan_covers_every_key_once(name, 64, heads)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(STEPS))
@pytest.mark.parametrize("bs", [24, 64])
@pytest.mark.parametrize("heads", [(1, 1), (14, 2), (32, 8)])
def test_block_attention_gpu(name, bs, heads, blocks):
    test_paged_attention_gpu(name, bs, heads)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.05, -0.05, 0.0])
def test_block_scales(scale, blocks):
    """Splits in which a column sees no key, and every key alike at scale 0."""
    from deepspeed_amd.ops.paged_attention import paged_attention
    torch.manual_seed(1)
    slots, pos, _ = _rows([(0, 300)], [130])
    table = torch.randperm(9)[:7]
    plan = StepPlan.build(slots, pos, {0: table.tolist()}, 64, 14, 2, "cuda")
    assert plan.nq == 8 and plan.any_merge
    kp, vp = (torch.randn(9, 2, 64, 128, device="cuda").bfloat16()
              for _ in range(2))
    q = (4 * torch.randn(300, 14, 128, device="cuda")).bfloat16()
    got = paged_attention(plan, q, kp, vp, scale)
    kk, vv = (p[table.cuda()].transpose(1, 2).reshape(-1, 2, 128)[:430]
              for p in (kp, vp))
    want = _reference(q, kk, vv, torch.tensor(pos, device="cuda"), scale)
    err = (got.double() - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 2.0 ** -13).all(), err.max()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["rows", "blocks"])
@pytest.mark.parametrize("kept", [0, 130])
def test_scale_that_is_no_number(kind, kept, request):
    """Gives no numbers, whichever kernel the step's runs take and whether their
    keys are split."""
    from deepspeed_amd.ops.paged_attention import paged_attention
    if kind == "blocks":
        request.getfixturevalue("blocks")
    slots, pos, _ = _rows([(0, 100)], [kept])
    plan = StepPlan.build(slots, pos, {0: [3, 1, 0, 2]}, 64, 14, 2, "cuda")
    assert (plan.nq == 8) == (kind == "blocks")
    assert plan.any_merge == (kept > 0)
    kp, vp = (torch.randn(4, 2, 64, 128, device="cuda").bfloat16()
              for _ in range(2))
    q = torch.randn(100, 14, 128, device="cuda").bfloat16()
    assert paged_attention(plan, q, kp, vp, float("nan")).isnan().all()


@pytest.mark.gpu
def test_plans_made_ahead_of_the_gpu():
    """The host goes on while a plan is on its way: later ones do not touch it."""
    plans, want = [], []
    a = torch.randn(4096, 4096, device="cuda")
    for _ in range(20):
        a = a @ a * 1e-2
    for n in range(1, 9):
        args = ([0] * n, np.arange(5, 5 + n), {0: [n, 7]}, 16, 8, 2)
        plans.append(StepPlan.build(*args, "cuda"))
        want.append(StepPlan.build(*args, "cpu"))
    for p, w in zip(plans, want):
        assert torch.equal(p.meta.cpu(), w.meta)
        assert torch.equal(p.dst.cpu(), w.dst)
