"""Rows per expert at the edges of the GEMMs' blocks and m-tiles, against the CPU oracle.

Each token is routed to exactly one chosen local expert (its other seven picks lie in other groups), so
an expert's row count, and how many of its rows take exact products, are what the case says."""
import pytest
import torch

import moe_oracle as O
import moe_fp8
from moe_fp8 import workloads as W

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
ATOL, RTOL = 1e-2, 2e-2      # the operator's bar
E_LOCAL = 4


def cdiv(a, b):
    return -(-a // b)


def compute_units():
    return torch.cuda.get_device_properties(0).multi_processor_count


def gemm1_cut(counts, exact, I, slots):
    """The staged GEMM1's largest block height, and whether an expert's folded exact rows are cut tightly: of the four the
    one of fewest rounds of units, and of those the one of most blocks."""
    best = None
    for height, tight in ((128, False), (128, True), (160, False), (160, True)):
        blocks = 0
        for n, n2 in zip(counts, exact):
            n01, fold = n - n2, 1 <= n2 <= 32 and n > n2
            steps = cdiv(n01, 32) + (fold and not (tight and n2 <= 16 and (n01 - 1) % 32 < 16))
            k = cdiv(steps, height // 32)
            blocks += k + (fold and (height == 160 or not tight) and steps == k * (height // 32))
            blocks += 0 if fold else cdiv(n2, 32)
        rank = (cdiv(blocks * (I // 128), slots), -blocks)
        if best is None or rank < best[0]:
            best = (rank, height, tight)
    return best[1:]


def gemm2_kind(counts, exact, H, I, T, slots):
    """How GEMM2 takes a call of 64 < T <= 512: LDS-staged units, or the stream by chunks or by cost (rows take two
    terms of C where their products are exact)."""
    KB, NC = I // 128, H // 128
    unit_cost = lambda nt: 2 if nt <= 1 else 2 * nt - 1
    blocks, staged, weighted, planes = [], 0, 0, 0       # blocks: (m-tiles, number) of the stream's
    for n, n2 in zip(counts, exact):
        tiles = cdiv(n, 16)
        k = cdiv(tiles, 4)
        mine = [b for b in ((tiles // k + 1, tiles % k), (tiles // k, k - tiles % k)) if b[1]] if k else []
        blocks += mine
        staged += cdiv(n - n2, 128) + cdiv(n2, 128)
        weighted += (5 if n2 else 4) * sum(unit_cost(nt) * c for nt, c in mine)
        planes = max([planes] + [(2 if n2 else 1) * nt for nt, _ in mine])
    cost = sum(unit_cost(nt) * k for nt, k in blocks)
    if T >= 128 and cost:
        rounds = cdiv(staged * (H // 256), slots)
        fit, deep = 128 * 1024 // (planes * 16 * 256), 8 if planes <= 4 else 4      # K-blocks of C in LDS, in whole rings
        again = cdiv(KB, fit - fit % deep) - 1
        if weighted * NC * cdiv(KB, 8) * 8 + 4 * (8 + 32 * again) * slots >= 4 * rounds * (5 * KB + 20) * slots:
            return "staged"
    most = (cost * NC * KB + 13 * slots) // (slots * KB)
    for b in range(max(1, cdiv(cost * NC, slots)), most + 1):
        if sum(k * cdiv(NC, max(1, min(NC, b // unit_cost(nt)))) for nt, k in blocks) <= slots:
            return "chunks"
    return "cost"


def case_inputs(counts, exact, T, H, I, seed):
    """counts[e] rows for local expert e, the first exact[e] of them large (exact products); tokens past
    them have no local expert.  Tokens of the experts are interleaved."""
    g = torch.Generator().manual_seed(seed)
    owner = torch.full((T,), -1)
    order = torch.randperm(T, generator=g)
    big, at = torch.zeros(T, dtype=torch.bool), 0
    for e, n in enumerate(counts):
        owner[order[at:at + n]] = e
        big[order[at:at + exact[e]]] = True
        at += n
    logits = torch.full((T, 256), -8.0) + 0.1 * torch.randn(T, 256, generator=g)
    for base in (32, 33, 64, 65, 96, 97, 98, 99):          # eight remote picks in groups 1, 2, 3
        logits[:, base] = 2.0 + 0.1 * torch.randn(T, generator=g)
    local = owner >= 0
    logits[torch.nonzero(local).squeeze(1), owner[local]] = 4.0
    hidden = torch.randn(T, H, generator=g)
    hidden[big] *= 60.0
    hs, hss = W.quantize_rows_1x128(hidden)
    return logits, torch.zeros(256, dtype=torch.bfloat16), hs, hss


def check(counts, exact, T, H, I, seed):
    act = case_inputs(counts, exact, T, H, I, seed)
    weights = W.make_weights(len(counts), H, I, device="cpu", seed=91)
    args = (*act, *weights, 0, W.RSF)
    dbg = {}
    out = moe_fp8.run(*(a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args), debug=dbg)
    torch.cuda.synchronize()
    assert dbg["expert_offsets"].cpu().diff().tolist() == list(counts)
    ref32, _ = O.moe_forward(*args)
    err = (out.float().cpu() - ref32).abs()
    bad = int((err > ATOL + RTOL * ref32.abs()).sum())
    assert bad == 0, f"{bad} elements outside the bar, max abs err {float(err.max()):.3e}"
    none = torch.ones(T, dtype=torch.bool)
    off = dbg["expert_offsets"].cpu()
    none[dbg["permuted_tokens"].cpu()[:off[-1]].long()] = False
    assert torch.all(out.cpu()[none] == 0)


@pytest.mark.parametrize("T", [0, 1100])           # just the rows (at least 140 tokens), and past 1024 tokens
@pytest.mark.parametrize("counts", [(1, 15, 16, 17), (31, 32, 33, 0), (63, 64, 65, 2), (95, 96, 97, 3),
                                    (127, 128, 129, 4), (159, 160, 161, 5), (191, 193, 0, 224), (255, 256, 257, 33),
                                    (319, 320, 321, 48)])
def test_rows_per_expert(counts, T):
    T = max(T, sum(counts), 140)
    print(f"[rows] {counts} T={T}", flush=True)
    check(counts, (0,) * E_LOCAL, T, 512, 256, seed=sum(counts))


@pytest.mark.parametrize("T", [0, 1100])
@pytest.mark.parametrize("counts,exact", [((1, 2, 16, 17), (1, 1, 16, 16)), ((33, 48, 49, 64), (1, 16, 17, 32)),
                                          ((97, 128, 129, 160), (1, 17, 32, 32)), ((161, 193, 225, 300), (33, 32, 16, 40)),
                                          ((128, 129, 113, 98), (16, 16, 17, 1)), ((96, 104, 256, 273), (1, 8, 16, 17)),
                                          ((290, 320, 40, 35), (1, 32, 40, 3))])
def test_exact_rows_per_expert(counts, exact, T):
    """1 to 32 exact rows fold into an expert's last block, more get blocks of their own."""
    T = max(T, sum(counts), 140)
    print(f"[exact rows] {counts} exact {exact} T={T}", flush=True)
    check(counts, exact, T, 512, 256, seed=7 + sum(counts))


@pytest.mark.parametrize("counts,exact", [((5, 40, 70, 130), (0, 3, 0, 33)), ((64, 128, 16, 17), (0, 64, 16, 0))])
@pytest.mark.parametrize("H,I", [(256, 128), (768, 384), (256, 1152), (2048, 640)])
def test_odd_shapes(H, I, counts, exact):
    """One, three, nine and five K-blocks in GEMM2 (nine: more than one or both terms of a tall block's C hold
    in LDS at once); two to sixteen in GEMM1."""
    print(f"[shapes] H={H} I={I} {counts}", flush=True)
    check(counts, exact, 300, H, I, seed=H + I)


@pytest.mark.parametrize("T", [65, 255, 256, 257, 511, 512, 513, 769])
def test_token_block_edges(T):
    """The permutation's 256-token blocks: one, two (counted by the placing launch itself) and three or four."""
    print(f"[token blocks] T={T}", flush=True)
    counts = (T // 3, T // 4, 5, T - T // 3 - T // 4 - 6)
    check(counts, (T // 9, 0, 1, 3), T, 512, 256, seed=T)


@pytest.mark.parametrize("counts,exact,cut", [
    ((129, 144, 145, 159, 160), (0,) * 5, (160, False)),
    ((128, 131, 133, 160, 190), (33, 40, 33, 64, 33), (160, False)),      # exact-product blocks beside them
    ((112, 144, 113, 160, 129, 145), (16, 0, 17, 0, 0, 0), (160, False)),
    ((96, 320, 160, 300), (32, 32, 0, 0), (160, False)),
    ((98, 160, 112, 150), (1, 0, 15, 0), (160, True)),                    # folded in the free half of a step
    ((128, 288, 160, 129, 300), (16, 16, 0, 0, 31), (160, True)),
    ((320, 288, 304, 160), (32, 16, 0, 0), (160, True)),
    ((108, 100, 128, 112), (8, 10, 16, 1), (128, True)),
    ((128, 128, 96, 104), (16, 1, 32, 8), (128, False))])
def test_gemm1_cuts(counts, exact, cut):
    """32 experts of eight GEMM1 units per block, so that the rounds of units differ between the cuts: blocks of up to 160
    or 128 class 0/1 rows, folded exact rows tightly or loosely."""
    counts, exact = (counts * 8)[:32], (exact * 8)[:32]
    print(f"[cuts] {counts[:6]} exact {exact[:6]} {cut}", flush=True)
    assert gemm1_cut(counts, exact, 1024, compute_units()) == cut
    check(counts, exact, sum(counts), 256, 1024, seed=sum(counts) + sum(exact))


@pytest.mark.parametrize("T,H,I,counts,exact,kind", [
    (65, 256, 128, (65,), (0,), "chunks"),
    (127, 256, 1152, (48, 64, 15), (0, 0, 0), "chunks"),          # nine K-blocks: a tall block's in two passes,
    (127, 256, 1152, (100, 27), (3, 27), "chunks"),               # in three with both terms
    (127, 512, 2176, (33, 49, 17, 28), (0, 49, 0, 1), "chunks"),
    (127, 256, 2048, (127,), (40,), "cost"),
    (127, 2048, 384, (17, 16, 1) * 3, (0, 16, 1) * 3, "chunks"),
    (200, 2048, 2048, (16,) * 8, (0, 1) * 4, "chunks"),
    (200, 2048, 2048, (5,) * 20, (0, 2) * 10, "cost"),
    (500, 512, 2048, (15, 16, 17) * 10, (0,) * 30, "cost"),
    (500, 512, 2048, (15, 16, 17) * 10, (0, 16, 1) * 10, "cost"),     # (the staged units would be two blocks per expert)
    (512, 512, 256, (159, 160, 161, 5), (0, 0, 33, 5), "chunks"),     # one round of units
    (512, 2048, 256, (33, 17, 49) * 5, (0, 5, 49) * 5, "staged"),
    (512, 4096, 512, (129, 160, 145), (0, 33, 5), "staged"),
    (500, 2048, 640, (33,) * 15, (0,) * 15, "staged"),
    (256, 512, 4096, (80, 17, 3, 128), (0, 17, 0, 64), "staged"),     # eight passes over K in the stream
    (440, 512, 2048, (65, 80) * 3, (0,) * 6, "chunks"),               # two, four with both terms
    (440, 512, 2048, (65, 80) * 3, (0, 33) * 3, "staged"),
    (512, 2048, 2048, (128, 127, 129, 128), (0, 127, 1, 33), "staged")])
def test_gemm2_kinds(T, H, I, counts, exact, kind):
    """Each way that GEMM2 takes a call of up to 512 tokens, as its rule on the experts' rows chooses."""
    print(f"[gemm2] T={T} H={H} I={I} {counts[:4]} exact {exact[:4]} {kind}", flush=True)
    assert gemm2_kind(counts, exact, H, I, T, compute_units()) == kind
    check(counts, exact, T, H, I, seed=T + H + I)


@pytest.mark.parametrize("big", [0, 1])
@pytest.mark.parametrize("H,I", [(512, 256), (256, 128), (768, 640), (2048, 1152)])
@pytest.mark.parametrize("counts", [(1, 2, 3, 4), (5, 7, 8, 9), (15, 16, 17, 8), (24, 25, 1, 0), (0, 0, 64, 0)])
def test_two_terms_small_batch(counts, H, I, big):
    """Up to 64 tokens, every m-tile on both terms of C: 1 to 8 rows (hi and lo rows of one tile) and 9 to 16
    (steps of their own).  C in one f16 term errs by 2^-11 / sqrt(3) = 2.8e-4 of each element (rms over its binade
    and over the sum about 1.5e-4 of a row), in two by 2^-22, below the fp32 sums' own 1e-6 to 1e-5."""
    print(f"[two terms] {counts} H={H} I={I} big={big}", flush=True)
    T = min(64, sum(counts) + 3)
    act = case_inputs(counts, counts if big else (0,) * E_LOCAL, T, H, I, seed=3 + sum(counts) + I)
    logits, bias, hs, hss = act
    weights = list(W.make_weights(E_LOCAL, H, I, device="cpu", seed=91))
    if not big:
        hss = hss * 16.0
    args = (logits, bias, hs, hss, *weights, 0, W.RSF)
    out = moe_fp8.run(*(a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args), output_dtype=torch.float32)
    torch.cuda.synchronize()
    ref32, _ = O.moe_forward(*args)
    err = float((out.cpu() - ref32).norm() / ref32.norm())
    assert err < 5e-5, f"relative error {err:.2e}"
