"""The slice kernels (routed experts and a shared expert's rows of blocks of up to 256 tokens) against 64-bit products, on numbers and through
work lists that the ordinary cases do not reach."""
import ctypes as C

import numpy as np
import pytest
import torch

from gpu_helpers import ctx, launches_of, tfk

pytestmark = pytest.mark.gpu
TOP_K = 8


def affine(gen, rows, cols, fp16, size=1.0):
    """Codes, scales and biases, and the exact weights in 64 bits: zero-mean groups, weights of about 0.06 `size`."""
    W = torch.randint(0, 256, (rows, cols // 2), dtype=torch.uint8, device="cuda", generator=gen)
    s = (torch.rand((rows, cols // 64), device="cuda", generator=gen) * 0.016 + 0.004) * size
    b = s * -7.5 + (torch.rand(s.shape, device="cuda", generator=gen) - 0.5) * 0.02 * size
    s, b = (t.to(torch.float16 if fp16 else torch.bfloat16) for t in (s, b))
    q = torch.stack([W & 15, W >> 4], 2).reshape(rows, cols).double()
    return (W, s, b), q * s.double().repeat_interleave(64, 1) + b.double().repeat_interleave(64, 1)


def gelu(v):
    return v / (1 + torch.exp(-2 * (0.7978845608028654 * (v + 0.044715 * v ** 3)).clamp(-20, 20)))


def half(v):
    return v.half().double()


class Experts:
    """A pool of experts, their exact weights, and a work list of `tokens` rows over them."""

    def __init__(self, seed, tokens, experts, d, f, fp16=False, size=(1.0, 1.0), edit=None):
        self.gen = gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        self.tokens, self.experts, self.d, self.f, self.fp16, self.n = tokens, experts, d, f, fp16, tokens * TOP_K
        mats = [[affine(gen, *shape, fp16, s) for shape, s in (((f, d), size[0]), ((f, d), size[0]), ((d, f), size[1]))] for _ in range(experts)]
        if edit:
            edit(mats)
        self.weights = [[m[1] for m in e] for e in mats]
        offsets, at = [], 0
        for t in (t for m in mats[0] for t in m[0]):
            offsets.append(at)
            at = (at + t.numel() * t.element_size() + 15) // 16 * 16
        self.off, self.stride = tfk.ExpertOffsets(*offsets), (at + 255) // 256 * 256
        self.pool = torch.zeros((experts, self.stride), dtype=torch.uint8, device="cuda")
        for row, e in zip(self.pool, mats):
            for o, t in zip(offsets, (t for m in e for t in m[0])):
                raw = t.contiguous().view(torch.uint8).ravel()
                row[o:o + raw.numel()] = raw
        self.idx = torch.rand((tokens, experts), device="cuda", generator=gen).add(torch.linspace(1, 0, experts, device="cuda") ** 4).topk(TOP_K).indices.int().contiguous()
        self.wts = torch.rand((tokens, TOP_K), device="cuda", generator=gen).half()
        i32 = dict(dtype=torch.int32, device="cuda")
        self.capacity = experts + self.n // 128 + 1
        self.pairs, self.count = torch.zeros((self.n, 4), **i32), torch.zeros(1, **i32)
        self.chunks = torch.zeros((self.capacity, 3), **i32)
        offs, counts = torch.zeros(experts, **i32), torch.zeros(experts, **i32)
        k = ctx()
        k.check(k.lib.tf_prefill_group_pairs_device(k.handle, None, self.idx.data_ptr(), self.wts.data_ptr(), tokens, TOP_K, experts, self.pairs.data_ptr(),
                                                    offs.data_ptr(), counts.data_ptr(), self.chunks.data_ptr(), self.count.data_ptr()))
        torch.cuda.synchronize()

    def run(self, x, stride=None, pairs=None, chunks=None, count=None, capacity=None, pair_count=None):
        n = pair_count or self.n
        acts, partials = torch.zeros((n, self.f), dtype=torch.float16, device="cuda"), torch.zeros((self.n, self.d), dtype=torch.float16, device="cuda")
        pairs, chunks, count = (self.pairs if pairs is None else pairs), (self.chunks if chunks is None else chunks), (self.count if count is None else count)
        k = ctx()
        k.check(k.lib.tf_prefill_grouped_routed_moe_resident(k.handle, None, x.data_ptr(), 0, stride or self.d, pairs.data_ptr(), chunks.data_ptr(), count.data_ptr(),
                                                             capacity or self.capacity, n, self.pool.data_ptr(), self.stride, self.experts, C.byref(self.off),
                                                             acts.data_ptr(), partials.data_ptr(), self.d, self.f, TOP_K, tfk.TF_FP16 if self.fp16 else tfk.TF_BF16))
        torch.cuda.synchronize()
        return acts, partials.view(self.tokens, TOP_K, self.d)

    def exact_acts(self, x):
        """What the gate / up launch is to leave, pair by pair, before its rounding."""
        out = torch.empty((self.n, self.f), dtype=torch.float64, device="cuda")
        for e in range(self.experts):
            rows = (self.pairs[:, 1] == e).nonzero().ravel()
            if rows.numel():
                v = x[self.pairs[rows, 0].long()].double()
                out[rows] = gelu(v @ self.weights[e][0].T.contiguous()) * (v @ self.weights[e][1].T.contiguous())
        return out

    def exact_partials(self, acts):
        """What the down launch is to leave for these activations."""
        out = torch.empty((self.tokens, TOP_K, self.d), dtype=torch.float64, device="cuda")
        for e in range(self.experts):
            rows = (self.pairs[:, 1] == e).nonzero().ravel()
            if rows.numel():
                out[self.pairs[rows, 0].long(), self.pairs[rows, 2].long()] = acts[rows].double() @ self.weights[e][2].T.contiguous()
        return out


def check_rounded(got, want):
    # Rounding to fp16 is off by 2^-11 of a value at most, or by 2^-25 where it is subnormal.  The sums before it, of nibbles that the matrix unit
    # reads as fp16 subnormals, have a deviation of 2e-6 to 7e-6 of the outputs' norm (measured against 64-bit sums, at outputs near zero); the largest of
    # some hundred thousand is 3e-5 off, a half of what is allowed here.  An operand rounded to the step of a subnormal number costs 3e-4 and more.
    off, rms = (got.double() - want).abs(), float(want.norm()) / want.numel() ** 0.5
    bound = want.abs() * 2.0 ** -11 + 2.0 ** -25 + 4 * 2.0 ** -16 * rms
    assert torch.all(off <= bound), float((off / bound).max())


@pytest.mark.parametrize("size", [1e-3, 1e-4, 1e-5])
@pytest.mark.parametrize("tokens,experts,d,f,fp16", [(80, 8, 1344, 320, False), (24, 48, 1280, 704, True)])
def test_small_activations_keep_their_bits(tokens, experts, d, f, fp16, size):
    # Rows of 1e-3 to 1e-5, most of whose numbers are below fp16's normal range (6e-5) or would be after a division by sixteen; weights so
    # large that the results are of ordinary size.
    e = Experts(0x51CE + tokens, tokens, experts, d, f, fp16, size=(0.3 / size, 1.0))
    x = (torch.randn((tokens, d), device="cuda", generator=e.gen) * size).half()
    acts, _ = e.run(x)
    check_rounded(acts, e.exact_acts(x))
    e = Experts(0x52CE + tokens, tokens, experts, d, f, fp16, size=((size / 4) ** 0.5, 0.3 / size))       # activations of about `size`
    x = torch.randn((tokens, d), device="cuda", generator=e.gen).half()
    acts, partials = e.run(x)
    assert 0.1 * size < float(acts.double().norm() / acts.numel() ** 0.5) < 10 * size
    check_rounded(partials, e.exact_partials(acts))


def shared_block(x, mats, d, f, fp16, x_stride=None):
    k, rows = ctx(), x.shape[0]
    y = torch.full((rows, d), float("nan"), dtype=torch.float16, device="cuda")
    scratch = torch.zeros(f, dtype=torch.float16, device="cuda")
    gate, up, down = (tfk.projection(*m[0], r, c) for m, (r, c) in zip(mats, ((f, d), (f, d), (d, f))))
    k.check(k.lib.tf_prefill_shared_expert_int4_block(k.handle, None, x.data_ptr(), 0, y.data_ptr(), 0, C.byref(gate), C.byref(up), C.byref(down),
                                                      *(v for _ in range(3) for v in (scratch.data_ptr(), 0, f * 2)), rows, d, f, x_stride or d, d, 4,
                                                      tfk.TF_FP16 if fp16 else tfk.TF_BF16))
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("size", [1e-3, 1e-4, 1e-5])
@pytest.mark.parametrize("stage", ["gate / up", "down"])
@pytest.mark.parametrize("rows,d,f,fp16", [(97, 1344, 1088, False), (192, 1280, 704, True), (256, 2688, 704, False)])
def test_shared_expert_keeps_the_bits_of_small_activations(rows, d, f, fp16, stage, size):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + d)
    first, last = (0.3 / size, 1.0) if stage == "gate / up" else ((size / 4) ** 0.5, 0.3 / size)
    mats = [affine(gen, *shape, fp16, s) for shape, s in (((f, d), first), ((f, d), first), ((d, f), last))]
    x = (torch.randn((rows, d), device="cuda", generator=gen) * (size if stage == "gate / up" else 1.0)).half()
    y = shared_block(x, mats, d, f, fp16)
    # the stage boundary: gate, up and their product leave as fp16
    product = lambda a, m: a @ m[1].T.contiguous()
    want = product(half(gelu(half(product(x.double(), mats[0]))) * half(product(x.double(), mats[1]))), mats[2])
    # besides the last rounding one activation in some hundred may be a rounding step off (its gate, its up or itself): one percent of 2^-10 or so
    # of the sums
    assert float((y.double() - want).norm() / want.norm()) < 3.5e-4


def cut(pairs, run, empty_every=0):
    """The pairs' work list in runs of at most `run`, a chunk without pairs behind every `empty_every`-th."""
    expert, chunks, at = pairs[:, 1].tolist(), [], 0
    while at < len(expert):
        end = at
        while end < len(expert) and end - at < run and expert[end] == expert[at]:
            end += 1
        chunks.append((expert[at], at, end - at))
        at = end
        if empty_every and len(chunks) % empty_every == 0:
            chunks.append((3, at, 0))
    return chunks


@pytest.mark.parametrize("tokens,experts,d,f", [(24, 48, 1344, 320), (110, 16, 1280, 704)])
def test_results_do_not_depend_on_the_work_list(tokens, experts, d, f):
    # The kernels hold 256 chunks of a list at a time.  Lists of more room than they fill, of more than 256 chunks, of chunks without pairs in front, between
    # and behind: the same bits.
    e = Experts(0x53CE + tokens, tokens, experts, d, f)
    x = torch.randn((tokens, d), device="cuda", generator=e.gen).half()
    acts, partials = e.run(x)
    lists = [(cut(e.pairs, 128), 0), (cut(e.pairs, 128), 1000), (cut(e.pairs, 1), 0), (cut(e.pairs, 3, 2), 40), ([(1, 0, 0)] * 300 + cut(e.pairs, 40, 3) + [(2, 0, 0)] * 300, 0),
             (cut(e.pairs, 5) + [(0, 0, 0)] * 256, 1)]
    for chunks, room in lists:
        table = torch.full((len(chunks) + room, 3), 0x7FFFFFFF, dtype=torch.int32, device="cuda")      # what lies behind the list is never used
        table[:len(chunks)] = torch.tensor(chunks, dtype=torch.int32)
        got_acts, got = e.run(x, chunks=table, count=torch.tensor([len(chunks)], dtype=torch.int32, device="cuda"), capacity=len(chunks) + room)
        assert torch.equal(got_acts, acts) and torch.equal(got, partials), (len(chunks), room)
    check_rounded(acts, e.exact_acts(x))


@pytest.mark.parametrize("tokens,experts,d,f,pad", [(60, 16, 512, 128, 0), (300, 16, 1280, 256, 0),      # matrix-core tiles
                                                    (6, 64, 1280, 256, 0),                                # quad kernels
                                                    (6, 64, 1280, 256, 4)])                               # rows off 16 bytes: a row at a time, the next pair fetched ahead
def test_other_kernels_pass_over_chunks_without_pairs(tokens, experts, d, f, pad):
    # A list of the same runs with chunks of no pairs in front, between and behind, these ones starting where the pairs end
    e = Experts(0x56CE + tokens + pad, tokens, experts, d, f)
    x = torch.randn((tokens, d + pad), device="cuda", generator=e.gen).half()
    acts, partials = e.run(x, stride=d + pad)
    runs = cut(e.pairs, 128)
    chunks = [(1, 0, 0)] + [c for run in runs for c in (run, (2, run[1] + run[2], 0))] + [(0, e.n, 0)] * 3
    table = torch.tensor(chunks, dtype=torch.int32, device="cuda")
    got_acts, got = e.run(x, stride=d + pad, chunks=table, count=torch.tensor([len(chunks)], dtype=torch.int32, device="cuda"), capacity=len(chunks))
    assert torch.equal(got_acts, acts) and torch.equal(got, partials)
    assert float((acts.double() - e.exact_acts(x[:, :d])).norm() / acts.double().norm()) < 1e-3 and float((partials.double() - e.exact_partials(acts)).norm() / partials.double().norm()) < 1e-3


@pytest.mark.parametrize("tokens,experts,d,f,pad,shift", [(24, 48, 1344, 320, 8, 4), (90, 16, 1280, 704, 136, 12), (90, 16, 1280, 256, 0, 8)])
def test_padded_rows_and_pairs_off_sixteen_bytes(tokens, experts, d, f, pad, shift):
    # Rows of a longer stride, and a pair list that is aligned to four bytes as its entries are: the same bits.
    e = Experts(0x59CE + tokens + f, tokens, experts, d, f)
    x = torch.randn((tokens, d), device="cuda", generator=e.gen).half()
    acts, partials = e.run(x)
    padded = torch.full((tokens, d + pad), float("nan"), dtype=torch.float16, device="cuda")
    padded[:, :d] = x
    raw = torch.zeros(e.n * 4 + 8, dtype=torch.int32, device="cuda")
    moved = raw[shift // 4:shift // 4 + e.n * 4]
    moved.copy_(e.pairs.ravel())
    assert moved.data_ptr() % 16 == shift
    got_acts, got = e.run(padded, stride=d + pad, pairs=moved)
    assert torch.equal(got_acts, acts) and torch.equal(got, partials)
    check_rounded(acts, e.exact_acts(x))


@pytest.mark.parametrize("rows,d,f,pad", [(97, 1344, 1088, 8), (192, 1280, 704, 24), (256, 2688, 704, 40)])
def test_shared_expert_of_padded_rows(rows, d, f, pad):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + d + pad)
    mats = [affine(gen, *shape, False) for shape in ((f, d), (f, d), (d, f))]
    x = torch.randn((rows, d), device="cuda", generator=gen).half()
    padded = torch.full((rows, d + pad), float("nan"), dtype=torch.float16, device="cuda")
    padded[:, :d] = x
    assert torch.equal(shared_block(padded, mats, d, f, False, x_stride=d + pad), shared_block(x, mats, d, f, False))


@pytest.mark.parametrize("tokens,experts", [(24, 48), (32, 64), (32, 85)])
def test_few_tokens_are_their_three_calls(tokens, experts):
    e = Experts(0x54CE + tokens, tokens, experts, 1280, 256)
    gen, d = e.gen, e.d
    W, s, b = torch.randint(0, 256, (experts, d), dtype=torch.uint8, device="cuda", generator=gen), *(
        (torch.rand((experts, d // 64), device="cuda", generator=gen) * 0.02 * m).bfloat16() for m in (1, -127.5))
    eff, gain = torch.full((d,), d ** -0.5, device="cuda").bfloat16(), torch.ones(experts, device="cuda").bfloat16()
    x = torch.randn((tokens, d), device="cuda", generator=gen).half()
    i32, f16 = dict(dtype=torch.int32, device="cuda"), dict(dtype=torch.float16, device="cuda")
    router = [v for t in (W, s, b, x, eff, gain) for v in (t.data_ptr(), 0)]
    k, out = ctx(), []
    for one_call in (False, True):
        idx, wts, h2 = torch.zeros((tokens, TOP_K), **i32), torch.zeros((tokens, TOP_K), **f16), torch.zeros((tokens, d), **f16)
        acts, partials = torch.zeros((e.n, e.f), **f16), torch.zeros((e.n, d), **f16)
        head = (k.handle, None, *router, idx.data_ptr(), 0, wts.data_ptr(), 0, tokens, experts, d, TOP_K, d)
        if one_call:
            k.check(k.lib.tf_prefill_routed_moe_few_tokens(*head, x.data_ptr(), 0, d, e.pool.data_ptr(), e.stride, C.byref(e.off), acts.data_ptr(), partials.data_ptr(),
                                                           h2.data_ptr(), 0, e.f, tfk.TF_BF16))
        else:
            offs, counts = torch.zeros(experts, **i32), torch.zeros(experts, **i32)
            k.check(k.lib.tf_prefill_router_group_block(*head, e.pairs.data_ptr(), offs.data_ptr(), counts.data_ptr(), e.chunks.data_ptr(), e.count.data_ptr()))
            acts, partials = e.run(x)
            k.check(k.lib.tf_prefill_moe_reduce_token_major(k.handle, None, partials.data_ptr(), 0, wts.data_ptr(), 0, h2.data_ptr(), 0, tokens, TOP_K, d))
        torch.cuda.synchronize()
        out.append([t.reshape(-1) for t in (idx, wts, acts, partials, h2)])
    assert all(torch.equal(a, b) for a, b in zip(*out))


def test_a_number_of_pairs_that_is_no_number_of_tokens_goes_to_the_tiles():
    # 2396 pairs of top 8 are not those of a number of token rows: such a list may be of any length and goes, like the 300 rows it is taken from, to the tiles.
    tokens, n = 300, 300 * TOP_K - 4
    e = Experts(0x55CE, tokens, 16, 1280, 256)
    x = torch.randn((tokens, e.d), device="cuda", generator=e.gen).half()
    _, want = e.run(x)
    chunks = torch.tensor(cut(e.pairs[:n], 128), dtype=torch.int32, device="cuda")
    _, got = e.run(x, chunks=chunks, count=torch.tensor([len(chunks)], dtype=torch.int32, device="cuda"), capacity=len(chunks), pair_count=n)
    there = torch.zeros((tokens, TOP_K), dtype=torch.bool, device="cuda")
    there[e.pairs[:n, 0].long(), e.pairs[:n, 2].long()] = True
    assert torch.equal(got[there], want[there]) and not got[~there].any()


@pytest.mark.parametrize("tokens,experts,d,f,shared_f,launches", [
    (96, 16, 1280, 256, 1088, 2), (192, 16, 2560, 256, 1088, 2), (256, 16, 2688, 256, 1088, 2), (80, 128, 1280, 704, 2112, 2),      # in the slice launches
    (33, 16, 2816, 256, 1088, 2), (64, 40, 1280, 256, 1088, 2), (79, 47, 2816, 256, 1088, 2),        # few experts, up to 79 rows: its split tiles in the launches of the routed tiles
    (79, 64, 2560, 256, 1088, 2), (53, 84, 1280, 256, 1088, 2),                                      # and more experts of up to 2560 columns, from five pairs each on
    (53, 48, 2816, 256, 1088, 4), (79, 64, 2688, 256, 1088, 4), (53, 85, 1280, 704, 2112, 4),        # longer rows, fewer pairs: the slice kernels, and the split kernels behind them
    (257, 16, 2816, 256, 1088, 2), (193, 16, 2560, 256, 1088, 2),                                    # dense tiles in the launches of the routed tiles
    (96, 16, 1280, 192, 1088, 4),                                                                    # routed rows that only the tiles take: the slice kernels behind them
])
def test_what_a_shared_expert_rides_in(tokens, experts, d, f, shared_f, launches):
    n, k = tokens * TOP_K, ctx()
    i32, f16, u8 = (dict(dtype=t, device="cuda") for t in (torch.int32, torch.float16, torch.uint8))
    pool, x, acts, partials, y = torch.zeros(experts * 65536, **u8), torch.zeros((tokens, d), **f16), torch.zeros((n, f), **f16), torch.zeros((n, d), **f16), torch.zeros((tokens, d), **f16)
    pairs, chunks, count, cap = torch.zeros((n, 4), **i32), torch.zeros((experts + n // 128 + 1, 3), **i32), torch.zeros(1, **i32), experts + n // 128 + 1
    w, scratch, off = torch.zeros(d * shared_f, **u8), torch.zeros(shared_f, **f16), tfk.ExpertOffsets(*(4096 * i for i in range(9)))      # recorded, never run
    gate, up, down = tfk.projection(w, w, w, shared_f, d), tfk.projection(w, w, w, shared_f, d), tfk.projection(w, w, w, d, shared_f)
    assert launches_of(k, lambda stream: k.lib.tf_prefill_grouped_routed_moe_resident_shared(
        k.handle, stream, x.data_ptr(), 0, d, pairs.data_ptr(), chunks.data_ptr(), count.data_ptr(), cap, n, pool.data_ptr(), 65536, experts, C.byref(off), acts.data_ptr(),
        partials.data_ptr(), d, f, TOP_K, tfk.TF_BF16, x.data_ptr(), 0, y.data_ptr(), 0, C.byref(gate), C.byref(up), C.byref(down),
        *(v for _ in range(3) for v in (scratch.data_ptr(), 0, shared_f * 2)), tokens, shared_f, d, d, 4)) == launches


def same_kind(got, want):
    """Infinities of the same sign, and NaN, in the same places (a finite product beyond fp16's range is an infinity too); which are finite in both"""
    want = want.half()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got == float("inf"), want == float("inf")) and torch.equal(got == float("-inf"), want == float("-inf"))
    return want.isfinite()


def with_odd_rows(x):
    """Some rows get infinities and NaN: one, one of either sign far apart, two of one sign side by side, in the last columns; returns which rows."""
    x = x.clone()
    inf, nan = float("inf"), float("nan")
    edits = [{3: inf}, {700: -inf}, {5: nan}, {64: inf, x.shape[1] - 65: -inf}, {130: inf, 131: inf}, {x.shape[1] - 1: inf}, {x.shape[1] - 70: -inf, 0: nan}]
    odd = torch.zeros(x.shape[0], dtype=torch.bool, device="cuda")
    for i, edit in enumerate(edits):
        row = i * x.shape[0] // len(edits)
        odd[row] = True
        for column, v in edit.items():
            x[row, column] = v
    return x, odd


def one_huge_activation(mats, column=37):
    """Rows of gate and up so large that their product is beyond fp16's range where gelu lets it through"""
    for i in (0, 1):
        (W, s, b), w = mats[i]
        s[column] *= 4096
        b[column] *= 4096
        w[column] *= 4096


@pytest.mark.parametrize("tokens,experts,d,f,fp16", [(24, 48, 1344, 320, False), (90, 16, 1280, 704, True)])
def test_infinities_and_nan_stay_in_their_rows_and_keep_their_signs(tokens, experts, d, f, fp16):
    e = Experts(0x57CE + tokens, tokens, experts, d, f, fp16)
    x = torch.randn((tokens, d), device="cuda", generator=e.gen).half()
    acts, partials = e.run(x)
    odd_x, odd = with_odd_rows(x)
    odd_acts, odd_partials = e.run(odd_x)
    odd_pairs = odd[e.pairs[:, 0].long()]
    assert torch.equal(odd_acts[~odd_pairs], acts[~odd_pairs]) and torch.equal(odd_partials[~odd], partials[~odd])
    same_kind(odd_acts, e.exact_acts(odd_x))
    assert odd_acts[odd_pairs].isinf().any() and odd_acts[odd_pairs].isnan().any()
    # the down launch: activations of which one is an infinity
    e = Experts(0x58CE + tokens, tokens, experts, d, f, fp16, edit=lambda mats: [one_huge_activation(m) for m in mats])
    acts, partials = e.run(x)
    assert 0.2 < float(acts.isinf().any(1).float().mean()) < 0.8 and not acts.isnan().any()
    want = e.exact_partials(acts)
    finite = same_kind(partials, want)
    assert partials.isinf().any() and finite.any()
    small = e.pairs[acts.abs().amax(1) < 100]          # pairs without such an activation, in the units of those with one
    there = (small[:, 0].long(), small[:, 2].long())
    assert len(small) > 10
    check_rounded(partials[there], want[there])


@pytest.mark.parametrize("rows,d,f,fp16", [(97, 1344, 1088, False), (192, 1280, 704, True)])
def test_infinities_and_nan_through_a_shared_expert(rows, d, f, fp16):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + d)
    mats = [affine(gen, *shape, fp16) for shape in ((f, d), (f, d), (d, f))]
    x = torch.randn((rows, d), device="cuda", generator=gen).half()
    y = shared_block(x, mats, d, f, fp16)
    odd_x, odd = with_odd_rows(x)
    odd_y = shared_block(odd_x, mats, d, f, fp16)
    assert torch.equal(odd_y[~odd], y[~odd]) and not odd_y[odd].isfinite().any()
    one_huge_activation(mats)
    y = shared_block(x, mats, d, f, fp16)
    product = lambda a, m: a @ m[1].T.contiguous()
    same_kind(y, product(half(gelu(half(product(x.double(), mats[0]))) * half(product(x.double(), mats[1]))), mats[2]))
    assert y.isinf().any() and y.isfinite().any()
