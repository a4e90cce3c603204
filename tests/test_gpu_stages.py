"""GPU parity of each stage of the hot path against the CPU oracle, through the C ABI.

Integer results (expert choice, counts, offsets, pos) must be bit-exact; floating
point results must be within max-abs 2e-2 and mean-rel 1e-3 of the fp32 oracle.
"""
import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_REL = 2e-2, 1e-3


def _say(msg):
    print(msg, flush=True)


def dev(t):
    return t.cuda()


# ------------------------------------------------------------------ gate
@pytest.mark.parametrize("T,d,E,k,dtype,seed", [
    (64, 256, 4, 1, torch.float16, 0),
    (333, 768, 32, 1, torch.float16, 1),
    (512, 1024, 8, 2, torch.float16, 2),
    (129, 4096, 8, 2, torch.float16, 3),
    (100, 2048, 64, 2, torch.float16, 4),
    (77, 512, 70, 4, torch.float16, 5),
    (512, 256, 4, 1, torch.float32, 6),
    (300, 1032, 70, 3, torch.float32, 8),
    (64, 8, 2, 2, torch.float16, 7),
    (1, 8, 1, 1, torch.float16, 9),
    (3, 64, 1024, 8, torch.float16, 10),
    (70, 16384, 4, 2, torch.float16, 11),
    (5, 136, 17, 8, torch.float16, 12),
])
def test_gate_bit_exact(T, d, E, k, dtype, seed):
    from ccfuser_amd import ops
    _say(f"gate T={T} d={d} E={E} k={k} {dtype} seed={seed}")
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, d, generator=g).to(dtype)
    wg = (torch.randn(E, d, generator=g) * 0.02).to(dtype)
    bg = (torch.randn(E, generator=g) * 0.02).to(dtype)
    idx_ref, score_ref, logits_ref = O.naive_gate(x, wg, bg, k)
    idx, score, logits = ops.gate_topk_softmax(dev(x), dev(wg), dev(bg), k, return_logits=True)
    torch.cuda.synchronize()
    assert torch.equal(logits.cpu(), logits_ref), "logits differ bitwise"
    assert torch.equal(idx.cpu(), idx_ref), "expert choice differs"
    assert (score.cpu().float() - score_ref.float()).abs().max() <= 1e-3
    assert torch.allclose(score.float().sum(-1).cpu(), torch.ones(T), atol=2e-3)


@pytest.mark.parametrize("T,d,E,k", [(1, 8, 8, 2), (9, 136, 9, 1), (2049, 128, 16, 2), (2055, 1160, 33, 3), (4097, 256, 8, 1),
                                     (4127, 520, 64, 2), (4100, 2048, 65, 8), (100, 128, 130, 2)])
def test_gate_fp32_tiles(T, d, E, k):
    """Every tile of the fp32 gate (8, 16 or 32 tokens by 8 to 64 experts), ragged in tokens and experts, with
    fewer parts of K than wavefronts, more, and a short last part: the oracle's bits."""
    from ccfuser_amd import ops
    _say(f"fp32 gate T={T} d={d} E={E} k={k}")
    g = torch.Generator().manual_seed(T + d + E)
    x, wg, bg = torch.randn(T, d, generator=g), torch.randn(E, d, generator=g) * 0.05, torch.randn(E, generator=g) * 0.05
    idx_ref, score_ref, logits_ref = O.naive_gate(x, wg, bg, k)
    idx, score, logits = ops.gate_topk_softmax(dev(x), dev(wg), dev(bg), k, return_logits=True)
    assert torch.equal(logits.cpu(), logits_ref), "logits differ bitwise"
    assert torch.equal(idx.cpu(), idx_ref), "expert choice differs"
    assert torch.allclose(score.cpu(), score_ref, rtol=1e-5, atol=1e-7)
    idx2, _ = ops.gate_topk_softmax(dev(x), dev(wg), None, k)
    assert torch.equal(idx2.cpu(), O.naive_gate(x, wg, None, k)[0])


@pytest.mark.parametrize("scale", [1.0, 1e-20])
@pytest.mark.parametrize("T,d,E,k", [(4097, 8, 33, 2), (4127, 136, 64, 8), (4128, 1160, 70, 1), (8193, 648, 9, 2), (8256, 768, 16, 3),
                                     (8257, 1064, 17, 1), (16385, 1536, 32, 2),
                                     # part sums of two turns of the wavefronts at a time: 9, 16, 17 and 25 parts
                                     (4097, 1032, 40, 2), (4130, 2048, 64, 2), (4099, 2056, 65, 2), (8200, 3080, 20, 1)])
def test_gate_fp32_products_as_mfmas(T, d, E, k, scale):
    """Many tokens: the fp32 gate's products on the matrix cores, fewer parts of K than wavefronts and more, ragged in
    every direction, zeros of both signs, and operands whose products are subnormal or vanish: the oracle's bits."""
    from ccfuser_amd import ops
    _say(f"fp32 gate on MFMAs T={T} d={d} E={E} k={k} scale={scale}")
    g = torch.Generator().manual_seed(T + d + E)
    x, wg = torch.randn(T, d, generator=g) * scale, torch.randn(E, d, generator=g) * scale
    x[:, ::7], wg[::3, 1::5] = -0.0, 0.0
    bg = torch.randn(E, generator=g) * scale * scale
    idx_ref, score_ref, logits_ref = O.naive_gate(x, wg, bg, k)
    idx, score, logits = ops.gate_topk_softmax(dev(x), dev(wg), dev(bg), k, return_logits=True)
    assert torch.equal(logits.cpu().view(torch.int32), logits_ref.view(torch.int32)), "logits differ bitwise"
    assert torch.equal(idx.cpu(), idx_ref), "expert choice differs"
    assert torch.allclose(score.cpu(), score_ref, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("T,d,E,k", [(1, 4096, 1, 1), (512, 2056, 2, 2), (513, 2056, 2, 1), (341, 6152, 3, 3), (342, 6152, 3, 2), (300, 128, 33, 2), (513, 128, 33, 2),
                                     (1024, 64, 130, 2), (1025, 64, 130, 2), (40, 256, 200, 8), (100, 264, 130, 2),
                                     (5, 136, 1024, 2), (33, 8, 64, 1)])
def test_gate_fp32_wavefront_per_token(T, d, E, k):
    """Both sides of each line between a wavefront per token and the tiles: the oracle's bits, with and without a
    bias."""
    from ccfuser_amd import ops
    _say(f"fp32 gate T={T} d={d} E={E} k={k}")
    g = torch.Generator().manual_seed(T + d + E)
    x, wg, bg = torch.randn(T, d, generator=g), torch.randn(E, d, generator=g) * 0.05, torch.randn(E, generator=g) * 0.05
    for b in (bg, None):
        idx_ref, score_ref, logits_ref = O.naive_gate(x, wg, b, k)
        idx, score, logits = ops.gate_topk_softmax(dev(x), dev(wg), None if b is None else dev(b), k, return_logits=True)
        assert torch.equal(logits.cpu(), logits_ref), "logits differ bitwise"
        assert torch.equal(idx.cpu(), idx_ref), "expert choice differs"
        assert torch.allclose(score.cpu(), score_ref, rtol=1e-5, atol=1e-7)


_GATE_CASES = {}


def _gate_case(T, d, E, k):
    key = (T, d, E, k)
    if key not in _GATE_CASES:
        g = torch.Generator().manual_seed(T + E)
        x = torch.randn(T, d, generator=g).half()
        wg = (torch.randn(E, d, generator=g) * 0.05).half()
        bg = (torch.randn(E, generator=g) * 0.05).half()
        _GATE_CASES[key] = (x, wg, bg) + tuple(O.naive_gate(x, wg, bg, k))
    return _GATE_CASES[key]


@pytest.mark.parametrize("slots,waves,stream", [(0, 8, -1), (0, 8, 0), (1, 2, 0), (2, 1, 0), (4, 8, 0), (1, 8, 0),
                                                (0, 8, 1), (1, 8, 1), (2, 8, 1), (4, 8, 1)])
@pytest.mark.parametrize("T,d,E,k", [(5000, 512, 8, 2), (9000, 256, 32, 1), (40001, 128, 16, 2),
                                     (33000, 768, 32, 1), (300, 4096, 12, 2), (2100, 2048, 70, 4),
                                     (77, 8192, 8, 2), (130, 520, 40, 3)])
def test_gate_launch_shapes(slots, waves, stream, T, d, E, k):
    """Every way the gate spreads a problem over the machine gives the oracle's bits: 1, 2
    or 4 parts of K per wavefront (fewer tokens per workgroup), 1 to 8 wavefronts per
    workgroup (several rounds of parts when K is long) or every wavefront alone through all
    of K, both tile widths (16 and 32 experts, 1 to 3 tiles), a ragged last token group, a
    short last part."""
    from ccfuser_amd import ops
    _say(f"gate slots={slots} waves={waves} stream={stream} T={T} d={d} E={E} k={k}")
    x, wg, bg, idx_ref, score_ref, logits_ref = _gate_case(T, d, E, k)
    ops.set_option("gate_slots", slots)
    ops.set_option("gate_waves", waves)
    ops.set_option("gate_stream", stream)
    try:
        idx, score, logits = ops.gate_topk_softmax(dev(x), dev(wg), dev(bg), k, return_logits=True)
        torch.cuda.synchronize()
    finally:
        ops.set_option("gate_slots", 0)
        ops.set_option("gate_waves", 8)
        ops.set_option("gate_stream", -1)
    assert torch.equal(logits.cpu(), logits_ref), "logits differ bitwise"
    assert torch.equal(idx.cpu(), idx_ref), "expert choice differs"
    assert (score.cpu().float() - score_ref.float()).abs().max() <= 1e-3


@pytest.mark.parametrize("T,d,E,k", [
    (1, 8, 1, 1), (3, 136, 5, 3), (40, 200, 9, 8),         # one short part, a part and a bit, more lists than two
    (333, 4096, 8, 2), (512, 4096, 8, 1), (513, 4096, 8, 2),         # one round of workgroups, one workgroup more
    (5, 8192, 8, 2), (5, 8200, 8, 2),                      # as many chains as threads, one part more (MFMA tiles)
    (9, 4096, 16, 2), (2, 128, 512, 2), (2, 128, 513, 2),  # 512 chains of other shapes
    (100, 64, 3, 1), (2000, 768, 8, 2), (700, 1032, 7, 2), # several tokens at a time, ragged groups and parts
    (64, 32768, 1, 1), (64, 32768, 2, 1),                  # very long rows: LDS of a workgroup
])
def test_gate_of_few_tokens(T, d, E, k):
    """A thread per token, expert and part of K, and the sizes around it: the oracle's bits, with and without a bias,
    and what the MFMA tiles give."""
    from ccfuser_amd import ops
    _say(f"gate of few tokens T={T} d={d} E={E} k={k}")
    x, wg, bg, idx_ref, score_ref, logits_ref = _gate_case(T, d, E, k)
    idx, score, logits = ops.gate_topk_softmax(dev(x), dev(wg), dev(bg), k, return_logits=True)
    assert torch.equal(logits.cpu(), logits_ref), "logits differ bitwise"
    assert torch.equal(idx.cpu(), idx_ref), "expert choice differs"
    assert (score.cpu().float() - score_ref.float()).abs().max() <= 1e-3
    bare = ops.gate_topk_softmax(dev(x), dev(wg), None, k, return_logits=True)
    ops.set_option("gate_stream", 0)
    try:
        tiles = ops.gate_topk_softmax(dev(x), dev(wg), dev(bg), k, return_logits=True)
        bare_tiles = ops.gate_topk_softmax(dev(x), dev(wg), None, k, return_logits=True)
    finally:
        ops.set_option("gate_stream", -1)
    for a, b in zip((idx, score, logits, *bare), (*tiles, *bare_tiles)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T", [1, 5, 70])
@pytest.mark.parametrize("d,E,k", [(136, 9, 1), (136, 9, 2), (136, 9, 3), (64, 3, 3), (256, 8, 8), (64, 300, 5), (1024, 16, 8)])
def test_gate_of_few_tokens_orders_ties_infinities_and_nan(T, d, E, k):
    """Experts whose logits tie, are infinite or NaN, up to lists that NaN leave short, and rows of NaN: the choice, the
    scores and the routing of the form for few tokens are those of the MFMA tiles and of the routing on its own."""
    from ccfuser_amd import ops
    _say(f"gate order T={T} d={d} E={E} k={k}")
    g = torch.Generator().manual_seed(d + E)
    x, wg = torch.randn(T, d, generator=g), torch.randn(E, d, generator=g) * 0.05
    half = E // 2
    wg[half:2 * half] = wg[:half]                                        # ties, in pairs
    if T > 1:
        x[1] = float("nan")
    x, wg = x.half().cuda(), wg.half().cuda()
    nan, inf = float("nan"), float("inf")
    for bad in ([], [nan], [-inf], [inf], [-inf] * E, [nan] * E, [nan, -inf, inf, nan, -inf], [nan] * (E - 1), [nan] * (E - 2) + [-inf]):
        bg = torch.zeros(E)
        bad = bad[:E]
        bg[torch.randperm(E, generator=g)[:len(bad)]] = torch.tensor(bad)
        bg = bg.half().cuda()
        got = ops.gate_topk_softmax(x, wg, bg, k, return_logits=True)
        idx, score, routing = ops.gate_route(x, wg, bg, k, 2)
        ops.set_option("gate_waves", 7)                                  # the MFMA tiles
        try:
            ref = ops.gate_topk_softmax(x, wg, bg, k, return_logits=True)
        finally:
            ops.set_option("gate_waves", 8)
        for a, b in zip(got + (idx, score), ref + ref[:2]):
            assert torch.equal(a.nan_to_num(3.0, 4.0, 5.0) if a.is_floating_point() else a, b.nan_to_num(3.0, 4.0, 5.0) if b.is_floating_point() else b)
        r0 = ops.route(ref[0].reshape(-1), E, k, 2)
        n = int(r0["offsets"][-1])
        for name in ("counts", "offsets", "inv_pos", "idx_kept"):
            assert torch.equal(routing[name], r0[name]), name
        assert torch.equal(routing["pos"][:n], r0["pos"][:n])


@pytest.mark.parametrize("stream", [0, 1])
@pytest.mark.parametrize("E,k", [(32, 2), (8, 1), (70, 3)])
def test_gate_logits_that_are_nothing_but_rounding_error(E, k, stream):
    """Inputs whose exact logits are zero: inside every part of 128 the second half of the
    products repeats the first half, permuted and negated (weights are powers of two, so
    every product is exact).  What is left is the rounding error of the fp32 chain, which
    depends on the order of the additions and on every rounding being to nearest even;
    scaled into fp16's range it must equal the oracle's bit for bit."""
    from ccfuser_amd import ops
    _say(f"gate rounding residue E={E} k={k} stream={stream}")
    g = torch.Generator().manual_seed(E)
    T, d = 300, 512
    x = torch.empty(T, d)
    w = torch.empty(E, d)
    for p0 in range(0, d, 128):
        perm = torch.randperm(64, generator=g)
        xa = torch.randn(T, 64, generator=g) * 2.0 ** torch.randint(0, 7, (T, 64), generator=g)
        wa = 2.0 ** torch.randint(2, 8, (E, 64), generator=g) * (torch.randint(0, 2, (E, 64), generator=g) * 2 - 1)
        x[:, p0:p0 + 64] = xa
        w[:, p0:p0 + 64] = wa
        x[:, p0 + 64:p0 + 128] = -xa[:, perm]
        w[:, p0 + 64:p0 + 128] = wa[:, perm]
    x, w = x.half(), w.half()
    assert torch.equal((x.double() @ w.double().t()), torch.zeros(T, E, dtype=torch.float64))
    idx_ref, score_ref, logits_ref = O.naive_gate(x, w, None, k)
    assert (logits_ref != 0).float().mean() > 0.5          # the residue is there
    ops.set_option("gate_stream", stream)
    try:
        idx, score, logits = ops.gate_topk_softmax(dev(x), dev(w), None, k, return_logits=True)
        torch.cuda.synchronize()
    finally:
        ops.set_option("gate_stream", -1)
    assert torch.equal(logits.cpu(), logits_ref), "rounding residue differs"
    assert torch.equal(idx.cpu(), idx_ref)


def test_gate_random_shapes():
    """Thirty seeded random shapes (1..2500 tokens, K a multiple of 8 up to 3000, 1..140
    experts, any top-k the shape allows) under random launch shapes, all bitwise."""
    from ccfuser_amd import ops
    import random
    rng = random.Random(20240607)
    try:
        for case in range(30):
            T = rng.choice([1, 2, 15, 16, 17, 63, 64, 65, rng.randint(66, 2500)])
            d = 8 * rng.randint(1, 375)
            E = rng.choice([1, 2, 3, 8, 15, 16, 17, 31, 32, 33, 64, rng.randint(65, 140)])
            k = rng.randint(1, min(E, 8))
            slots, waves = rng.choice([0, 1, 2, 4]), rng.randint(1, 8)
            stream = (case * 7 + 1) % 3 - 1
            _say(f"gate random case {case}: T={T} d={d} E={E} k={k} slots={slots} waves={waves} stream={stream}")
            g = torch.Generator().manual_seed(case)
            x = (torch.randn(T, d, generator=g) * 2.0 ** rng.randint(-3, 3)).half()
            wg = (torch.randn(E, d, generator=g) * 0.05).half()
            bg = (torch.randn(E, generator=g) * 0.05).half() if case % 3 else None
            idx_ref, score_ref, logits_ref = O.naive_gate(x, wg, bg, k)
            ops.set_option("gate_slots", slots)
            ops.set_option("gate_waves", waves)
            ops.set_option("gate_stream", stream)
            idx, score, logits = ops.gate_topk_softmax(dev(x), dev(wg), None if bg is None else dev(bg), k,
                                                       return_logits=True)
            torch.cuda.synchronize()
            assert torch.equal(logits.cpu(), logits_ref), f"case {case}: logits differ bitwise"
            assert torch.equal(idx.cpu(), idx_ref), f"case {case}: expert choice differs"
            assert (score.cpu().float() - score_ref.float()).abs().max() <= 1e-3
    finally:
        ops.set_option("gate_slots", 0)
        ops.set_option("gate_waves", 8)
        ops.set_option("gate_stream", -1)


@pytest.mark.parametrize("tile", [32, 16])
def test_mfma_chain_equals_a_chain_of_fused_multiply_adds(tile):
    """What the fp16 gate rests on: a chain of K = 1 fp32 MFMAs gives, per output element,
    the bits of acc = fma(a, b, acc) step by step (round to nearest even), on operands that
    fp16 can hold with exponents spread over 16 binades, so that sums cancel and every
    rounding matters.  Products of such operands are exact in fp32, which lets numpy replay
    the chain with a multiply and an add.  Also pins which accumulator register of which lane
    holds which element, as the gate kernel assumes it."""
    import numpy as np
    from ccfuser_amd import _lib
    _say(f"mfma chain probe tile={tile}")
    steps, blocks, regs = 768, 64 // tile, 32 if tile == 32 else 16
    g = torch.Generator().manual_seed(tile)

    def operands():
        v = torch.randn(steps, 64, generator=g) * 2.0 ** torch.randint(-8, 9, (steps, 64), generator=g).float()
        return v.half().float()                                      # representable in fp16

    for trial in range(6):
        a, b = operands(), operands()
        out = torch.full((regs, 64), float("nan"), dtype=torch.float32, device="cuda")
        a_dev, b_dev = a.cuda(), b.cuda()
        assert _lib.probe_lib().ccf_probe_mfma_chain(a_dev.data_ptr(), b_dev.data_ptr(), steps, tile,
                                                     out.data_ptr(), None) == 0
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        an, bn = a.numpy(), b.numpy()
        for blk in range(blocks):
            ab, bb = an[:, blk * tile:(blk + 1) * tile], bn[:, blk * tile:(blk + 1) * tile]
            acc = np.zeros((tile, tile), np.float32)
            for s_ in range(steps):
                acc = acc + ab[s_][:, None] * bb[s_][None, :]
            for v in range(regs):
                if (v >> 4 if tile == 32 else v >> 2) != blk:
                    continue
                for lane in range(64):
                    if tile == 32:
                        row, col = 8 * ((v & 15) >> 2) + 4 * (lane >> 5) + (v & 3), lane & 31
                    else:
                        row, col = 4 * (lane >> 4) + (v & 3), lane & 15
                    assert got[v, lane] == acc[row, col], (trial, blk, v, lane)


def test_gate_ties_go_to_lower_expert():
    from ccfuser_amd import ops
    x = torch.ones(8, 64, dtype=torch.float16)
    wg = torch.zeros(6, 64, dtype=torch.float16)
    wg[1] = 0.5
    wg[4] = 0.5          # experts 1 and 4 tie for first, 0,2,3,5 tie for the rest
    idx, score = ops.gate_topk_softmax(dev(x), dev(wg), None, 3)
    assert idx.cpu().tolist() == [[1, 4, 0]] * 8
    ref_idx, ref_score, _ = O.naive_gate(x, wg, None, 3)
    assert torch.equal(idx.cpu(), ref_idx)
    assert (score.cpu().float() - ref_score.float()).abs().max() <= 1e-3


# --------------------------------------------------------------- routing
@pytest.mark.parametrize("n,E,k,cap,seed", [
    (1, 4, 1, -1, 0), (63, 4, 1, -1, 1), (1024, 8, 2, -1, 2), (1025, 8, 1, -1, 3),
    (16384, 8, 2, 2560, 4), (32768, 32, 1, -1, 5), (5000, 70, 2, 40, 6), (4096, 1000, 2, -1, 7),
    (3000, 3, 1, 0, 8),
    (70000, 600, 2, -1, 9),        # a table of counts too large for the pos launch to sum: the scan launch runs
    (40000, 900, 1, 30, 10),       # the same with a capacity
])
def test_route_bit_exact(n, E, k, cap, seed):
    from ccfuser_amd import ops
    _say(f"route n={n} E={E} k={k} cap={cap} seed={seed}")
    g = torch.Generator().manual_seed(seed)
    # skewed ids with some already-dropped entries
    p = torch.rand(E, generator=g) ** 3 + 1e-3
    idx = torch.multinomial(p / p.sum(), n, replacement=True, generator=g)
    idx[torch.rand(n, generator=g) < 0.05] = -1
    kept_ref = O.limit_by_capacity(idx, E, cap)
    counts_ref = O.expert_count(kept_ref, E)
    pos_ref, off_ref = O.assign_pos(kept_ref, E)
    r = ops.route(dev(idx), E, k, cap)
    torch.cuda.synchronize()
    R = int(off_ref[-1])
    assert torch.equal(r["counts"].cpu(), counts_ref)
    assert torch.equal(r["offsets"].cpu(), off_ref)
    assert torch.equal(r["idx_kept"].cpu(), kept_ref)
    assert torch.equal(r["pos"].cpu()[:R], pos_ref)
    assert torch.equal(r["src_row"].cpu()[:R].long(), pos_ref // k)
    assert torch.equal(r["dst_row"].cpu()[:R].long(), pos_ref)
    assert torch.equal(r["inv_pos"].cpu(), O.inverse_pos(pos_ref, n))


def test_expert_count_and_assign_pos_mirror_the_reference_calls():
    """functions.py:85-103 call sequence through the mirrored extension functions."""
    from ccfuser_amd import mix_moe_hip
    g = torch.Generator().manual_seed(11)
    E, n = 16, 8192
    gate = torch.randint(0, E, (n // 2, 2), generator=g)
    gate[torch.rand(n // 2, 2, generator=g) < 0.1] = -1
    cnt = torch.zeros(E, dtype=torch.int32, device="cuda")
    mix_moe_hip.expert_count(dev(gate), cnt)
    mix_moe_hip.expert_count(dev(gate), cnt)            # accumulates
    ref = O.expert_count(gate, E)
    assert torch.equal(cnt.cpu(), 2 * ref)
    lec_cum = torch.cumsum(ref.long(), 0).int().cuda()
    pos = torch.empty(int(lec_cum[-1]), dtype=torch.long, device="cuda")
    mix_moe_hip.assign_pos(lec_cum, dev(gate), pos)
    pos_ref, off_ref = O.assign_pos(gate, E)
    assert torch.equal(pos.cpu(), pos_ref)
    assert torch.equal(lec_cum.cpu(), off_ref[:-1])      # cum_count ends at the segment starts


def _count_cases():
    import os
    import numpy as np
    g = torch.Generator().manual_seed(5)
    table = np.load(os.path.join(os.path.dirname(__file__), "golden", "ref_all_expert_count.npy"))
    cases = [row.tolist() for row in table]                       # the reference's skewed 4x64 table
    cases += [[0, 0, 0], [63], [64], [65], [1, 64, 0, 128, 130, 5], [64] * 7, [3] * 9,
              [700, 0, 1, 0, 64, 63, 1000],                       # more full blocks than tails
              [1] * 40 + [128],                                   # more tails than full blocks
              torch.randint(0, 300, (1000,), generator=g).tolist(),
              torch.randint(0, 3, (1024,), generator=g).tolist()]
    return cases


@pytest.mark.parametrize("case", range(15))
def test_plan_blocks_matches_divide_into_block(case):
    """Device block planner against the oracle's divide_into_block, every array bit-exact."""
    from ccfuser_amd import ops
    counts = _count_cases()[case]
    _say(f"plan_blocks case={case} E={len(counts)} rows={sum(counts)}")
    ref = O.divide_into_block(counts, 64)
    got = ops.plan_blocks(torch.tensor(counts, dtype=torch.int32, device="cuda"), sum(counts), 64)
    total, remote = got["block_nums"].tolist()
    assert (total, remote) == (ref["total_block_num"], ref["remote_block_num"])
    for k in ("expert_ids", "ranks", "lens", "start_addrs", "expert_block_ids"):
        assert got[k][:total].tolist() == ref[k], k
        assert got[k].numel() >= total
    assert got["expert_block_id_idxs"].tolist() == ref["expert_block_id_idxs"]
    got32 = ops.plan_blocks(torch.tensor(counts, dtype=torch.int32, device="cuda"), sum(counts), 32, rank=3)
    ref32 = O.divide_into_block(counts, 32)
    t32 = int(got32["block_nums"][0])
    assert t32 == ref32["total_block_num"]
    assert got32["start_addrs"][:t32].tolist() == ref32["start_addrs"]
    assert got32["ranks"][:t32].tolist() == [3] * t32


@pytest.mark.parametrize("n_seg,E,seed", [(64, 8, 0), (1, 1, 1), (700, 37, 2), (3000, 200, 3), (5, 1024, 4)])
def test_segments_to_rows(n_seg, E, seed):
    """(start, len, expert) triples -> counts, offsets and the row list grouped by expert, rows of
    an expert in the order of the triple list and then row order (what the reference's kernels do
    per block through start_addrs / lens / expert_ids, mix_gemm.cu:296-301).  Triples with no
    rows or with an expert outside 0..E-1 are skipped.  Many triples, empty experts, bit for bit."""
    from ccfuser_amd import ops
    import numpy as np
    _say(f"segments_to_rows n_seg={n_seg} E={E} seed={seed}")
    rng = np.random.default_rng(seed)
    seg_len = rng.integers(0, 40, n_seg).astype(np.int32)
    seg_len[rng.random(n_seg) < 0.1] = 0
    seg_expert = rng.integers(0, E, n_seg).astype(np.int32)
    bad = rng.random(n_seg) < 0.05
    seg_expert[bad] = rng.choice([-1, E, E + 5], bad.sum())
    total = int(seg_len.sum())
    seg_start = (np.cumsum(seg_len) - seg_len).astype(np.int32)
    order = rng.permutation(n_seg)                       # the list is in no particular order
    seg_start, seg_len, seg_expert = seg_start[order], seg_len[order], seg_expert[order]
    counts_ref = np.zeros(E, dtype=np.int32)
    per = [[] for _ in range(E)]
    for st, ln, e in zip(seg_start, seg_len, seg_expert):
        if 0 <= e < E and ln > 0:
            counts_ref[e] += ln
            per[e].extend(range(st, st + ln))
    offsets_ref = np.concatenate([[0], np.cumsum(counts_ref)]).astype(np.int32)
    rows_ref = np.array([r for e in range(E) for r in per[e]], dtype=np.int32)
    counts, offsets, rows = ops.segments_to_rows(dev(torch.from_numpy(seg_start)), dev(torch.from_numpy(seg_len)),
                                                 dev(torch.from_numpy(seg_expert)), E, max(total, 1))
    torch.cuda.synchronize()
    assert np.array_equal(counts.cpu().numpy(), counts_ref)
    assert np.array_equal(offsets.cpu().numpy(), offsets_ref)
    assert np.array_equal(rows.cpu().numpy()[:len(rows_ref)], rows_ref)


# ------------------------------------------------- row moves and combine
def test_local_scatter_gather_with_reference_pos_vector():
    """The reference's own scatter check: index_select(input, 0, pos) with its
    pos.pt (csrc/test.cpp:405-449), M=4096 rows, N=1024."""
    import numpy as np, os
    from ccfuser_amd import ops
    pos = torch.from_numpy(np.load(os.path.join(os.path.dirname(__file__), "golden", "ref_pos_div2.npy")))
    g = torch.Generator().manual_seed(0)
    x = torch.randn(4096, 1024, generator=g).half()
    out = ops.local_scatter(dev(x), dev(pos.int()))
    assert torch.equal(out.cpu(), torch.index_select(x, 0, pos))
    # gather is the inverse move on a permutation
    perm = torch.randperm(4096, generator=g)
    back = ops.local_gather(dev(x), dev(perm.int()), 4096)
    ref = torch.zeros_like(x)
    ref.index_copy_(0, perm, x)
    assert torch.equal(back.cpu(), ref)


@pytest.mark.parametrize("T,k,d", [(100, 1, 64), (257, 2, 1024), (64, 4, 256)])
def test_combine(T, k, d):
    from ccfuser_amd import ops
    g = torch.Generator().manual_seed(T)
    y = torch.randn(T * k, d, generator=g).half()
    s = torch.softmax(torch.randn(T, k, generator=g), -1).half()
    inv = torch.arange(T * k, dtype=torch.int32)
    inv[torch.rand(T * k, generator=g) < 0.2] = -1
    y_masked = y.clone()
    y_masked[inv < 0] = 0
    ref = O.combine(y_masked.float(), s.float(), k)
    out = ops.combine(dev(y), dev(s), k, dev(inv))
    assert (out.cpu().float() - ref).abs().max() <= 2e-3 * max(1.0, float(ref.abs().max()))
    if k == 1:      # closed form: out = score * y
        assert torch.equal(ops.combine(dev(y), dev(torch.ones(T, 1).half()), 1).cpu(), y)


# ------------------------------------------------------------ expert FFN
def _ffn_case(R, d, f, E, seed, skew=False):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(R, d, generator=g).half()
    w1 = (torch.randn(E, f, d, generator=g) * 0.02).half()
    b1 = (torch.randn(E, f, generator=g) * 0.02).half()
    w2 = (torch.randn(E, d, f, generator=g) * 0.02).half()
    b2 = (torch.randn(E, d, generator=g) * 0.02).half()
    if skew:
        p = torch.rand(E, generator=g) ** 4 + 1e-4
    else:
        p = torch.ones(E)
    e_of_row = torch.multinomial(p / p.sum(), R, replacement=True, generator=g)
    return x, w1, b1, w2, b2, e_of_row


@pytest.mark.usefixtures("gemm_form")
@pytest.mark.parametrize("variant", [0, 1, 2, 3])
@pytest.mark.parametrize("R,d,f,E,skew,seed", [
    (512, 256, 1024, 4, False, 0),
    (700, 768, 3072, 32, True, 1),
    (1000, 1024, 512, 3, True, 2),
    (64, 64, 64, 1, False, 3),
    (1, 128, 192, 2, False, 4),
])
def test_ffn_stages(variant, R, d, f, E, skew, seed):
    from ccfuser_amd import ops
    _say(f"ffn variant={variant} R={R} d={d} f={f} E={E} skew={skew}")
    ops.set_option("gemm_variant", variant)
    try:
        x, w1, b1, w2, b2, e_of_row = _ffn_case(R, d, f, E, seed, skew)
        # rows arrive in token order; route them as a top-1 layer would
        pos_ref, off_ref = O.assign_pos(e_of_row, E)
        buf = O.local_scatter(x, pos_ref, 1)
        r = ops.route(dev(e_of_row), E, 1)
        h = ops.ffn1(dev(x), r["src_row"], r["offsets"], R, dev(w1), dev(b1), gelu=True)
        torch.cuda.synchronize()
        # FFN1 + GELU against fp32
        off = off_ref.tolist()
        h_ref = torch.zeros(R, f)
        for e in range(E):
            lo, hi = off[e], off[e + 1]
            if hi > lo:
                h_ref[lo:hi] = O.gelu_exact(buf[lo:hi].float() @ w1[e].float().t() + b1[e].float())
        assert O.max_abs_err(h.cpu(), h_ref) <= MAX_ABS
        assert O.mean_rel_err(h.cpu(), h_ref) <= MEAN_REL
        # FFN2 with the un-permute fused
        y = torch.zeros(R, d, dtype=torch.float16, device="cuda")
        ops.ffn2(h, r["dst_row"], r["offsets"], R, dev(w2), dev(b2), y)
        torch.cuda.synchronize()
        y_sorted = O.expert_ffn(buf, off_ref, w1, b1, w2, b2)
        y_ref = O.unpermute(y_sorted, pos_ref, R)
        assert O.max_abs_err(y.cpu(), y_ref) <= MAX_ABS
        assert O.mean_rel_err(y.cpu(), y_ref) <= MEAN_REL
    finally:
        ops.set_option("gemm_variant", -1)


@pytest.mark.parametrize("R,d,f,E,skew,seed", [
    (9000, 1024, 2048, 8, False, 50),          # several rounds of tiles per workgroup, ragged last tiles
    (3000, 768, 1536, 32, True, 51),           # many partly filled tiles (the eight-wavefront form computes their padding)
    (700, 256, 320, 5, False, 52),             # four K tiles, N no multiple of 256
])
def test_eight_wavefront_kernel_gives_the_four_wavefront_bits(R, d, f, E, skew, seed):
    """The persistent kernel with eight wavefronts per workgroup (one register buffer of token
    fragments, refilled row block by row block) adds over K in the same order with the same
    instruction as the four-wavefront form: both GEMMs must agree bit for bit."""
    from ccfuser_amd import ops
    x, w1, b1, w2, b2, e_of_row = _ffn_case(R, d, f, E, seed, skew)
    r = ops.route(dev(e_of_row), E, 1)
    _say(f"8 vs 4 wavefronts R={R} d={d} f={f} E={E} counts={r['counts'].tolist()[:10]}")
    res = {}
    ops.set_option("split_tail", 0)
    try:
        for variant in (2, 3):
            ops.set_option("gemm_variant", variant)
            h = ops.ffn1(dev(x), r["src_row"], r["offsets"], R, dev(w1), dev(b1), gelu=True)
            y = torch.zeros(R, d, dtype=torch.float16, device="cuda")
            ops.ffn2(h, r["dst_row"], r["offsets"], R, dev(w2), dev(b2), y)
            torch.cuda.synchronize()
            res[variant] = (h.cpu(), y.cpu())
    finally:
        ops.set_option("gemm_variant", -1)
        ops.set_option("split_tail", 1)
    assert torch.isfinite(res[3][0].float()).all() and res[3][0].abs().sum() > 0
    assert torch.equal(res[2][0], res[3][0]), "first GEMM"
    assert torch.equal(res[2][1], res[3][1]), "second GEMM"


@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("E", [1, 8, 300, 1024])
@pytest.mark.parametrize("capacity", [-1, 3])
def test_route_of_few_indices(n, E, capacity):
    """One or two chunks of indices, counted by the launch that writes the positions, and the sizes next to them:
    the results of the three-launch form, also with indices that name no expert."""
    from ccfuser_amd import ops
    g = torch.Generator().manual_seed(n + E)
    idx = torch.randint(0, E, (n,), generator=g)
    idx[torch.rand(n, generator=g) < 0.1] = -1
    got = ops.route(dev(idx), E, 1, capacity)
    ops.set_option("route_rows_max", 0)
    try:
        ref = ops.route(dev(idx), E, 1, capacity)
    finally:
        ops.set_option("route_rows_max", 16384)
    kept = int(ref["offsets"][-1])
    for k, v in ref.items():
        m = kept if k in ("pos", "src_row", "dst_row") else v.numel()
        assert torch.equal(got[k][:m], v[:m]), k


@pytest.mark.parametrize("n", [1000, 1500, 2048, 5000])
def test_route_in_place(n):
    """``idx_kept`` written over the indices themselves: every index is counted before any is replaced."""
    from ccfuser_amd import _lib, ops
    E, capacity = 8, n // 20
    idx = dev(torch.randint(0, E, (n,), generator=torch.Generator().manual_seed(n)))
    ref = ops.route(idx, E, 1, capacity)
    got = {k: torch.empty_like(v) for k, v in ref.items()}
    got["idx_kept"] = idx.clone()
    nbytes = _lib.lib().ccf_route_workspace_bytes(n, E)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    _lib.call("ccf_route", got["idx_kept"].data_ptr(), n, E, 1, capacity, *[got[k].data_ptr() for k in
              ("counts", "offsets", "pos", "src_row", "dst_row", "inv_pos", "idx_kept")], ws.data_ptr(), nbytes,
              torch.cuda.current_stream().cuda_stream)
    kept = int(ref["offsets"][-1])
    assert kept < n
    for k, v in ref.items():
        m = kept if k in ("pos", "src_row", "dst_row") else v.numel()
        assert torch.equal(got[k][:m], v[:m]), k


@pytest.mark.parametrize("counts,N,K,pad", [
    ([1], 8, 64, 0),                                          # fewer K tiles than wavefronts, half a column tile
    ([1, 0, 1], 264, 448, 0),                                 # seven wavefronts with a K tile; a ragged last column tile
    ([0, 16, 0, 0], 40, 576, 0),                              # a full row block, nine K tiles
    ([17, 0, 15], 24, 1088, 0),                               # two row blocks, one row in the second
    ([0] * 70 + [3, 0, 1] + [0] * 60 + [2], 136, 1024, 9),    # experts over several passes of the search, spare rows
    ([1] * 32, 16, 2112, 0),
    ([0, 0], 16, 64, 4),                                      # no rows
])
def test_thin_rows_kernel(counts, N, K, pad):
    """K cut over the wavefronts of a workgroup for a few rows in all, through row indices, both epilogues: the fp32
    product within the error of the sums and one rounding to fp16, and a second call bit for bit; rows no index
    points at stay as they are."""
    from ccfuser_amd import ops
    _say(f"thin rows counts={len(counts)} N={N} K={K}")
    E, R = len(counts), sum(counts)
    g = torch.Generator().manual_seed(N + K)
    x = dev(torch.randn(R + 9, K, generator=g).half())
    w = dev((torch.randn(E, N, K, generator=g) * K ** -0.5).half())
    b = dev(torch.randn(E, N, generator=g).half())
    off = dev(torch.tensor([0] + counts).cumsum(0).int())
    src = dev(torch.cat([torch.randperm(R + 9, generator=g)[:R], torch.zeros(pad, dtype=torch.int64)]).int())
    dst = dev(torch.cat([torch.randperm(R + 3, generator=g)[:R], torch.zeros(pad, dtype=torch.int64)]).int())
    scale = dev(torch.rand(R + pad, generator=g).half())

    def outputs():
        y = torch.full((R + 3 + pad, N), 7.0, dtype=torch.float16, device="cuda")
        return (ops.ffn1(x, src, off, R + pad, w, b, gelu=True, out=y.clone(), dst_row=dst),
                ops.ffn2(x, dst, off, R + pad, w, b, y.clone(), src_row=src, row_scale=scale))

    ops.set_option("few_rows", 3)
    try:
        got, again = outputs(), outputs()
    finally:
        ops.set_option("few_rows", 1)
    e_of = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).cuda()
    xs, rows = x[src[:R].long()].double(), dst[:R].long()
    pre = torch.empty(R, N, dtype=torch.float64, device="cuda")
    for e in e_of.unique().tolist():
        pre[e_of == e] = xs[e_of == e] @ w[e].double().t() + b[e].double()
    refs = (torch.nn.functional.gelu(pre), pre * scale[:R, None].double())
    for out, second, ref in zip(got, again, refs):
        assert torch.equal(out, second)
        # K additions in fp32 of terms whose magnitudes sum to K^0.5 or so, the GELU's 6e-5, half a step of fp16
        tol = K * 2.0 ** -24 * K ** 0.5 + 6e-5
        assert ((out[rows].double() - ref).abs() <= tol + 2.0 ** -11 * ref.abs()).all()
        rest = torch.ones(out.shape[0], dtype=torch.bool, device="cuda")
        rest[rows] = False
        assert (out[rest] == 7.0).all()


@pytest.mark.parametrize("E,N,K,rows,thin", [
    (4, 1024, 1024, 32, True), (4, 1024, 1024, 33, False),         # 32 rows in all
    (4, 1024, 960, 16, False),                                     # two K tiles a wavefront
    (8, 1024, 2048, 16, True), (8, 1040, 2048, 16, False),         # two workgroups a CU
    (2, 4096, 1024, 2, False), (2, 2048, 1024, 2, True),           # two of few K tiles, one
    (1, 4096, 1024, 16, True), (1, 4096, 1024, 32, False),         # rows of an expert
    (1, 8192, 2048, 24, False), (1, 8192, 2048, 2, True),
    (4, 1024, 4096, 3, True), (4, 1024, 4096, 4, False),           # fewer rows than experts of a long contraction
])
def test_thin_rows_rule_takes_the_faster_form(E, N, K, rows, thin):
    """At most 32 rows: the form that cuts K over the wavefronts or tiles of few rows, told apart by the bits that their
    orders of the sum leave; both against fp32."""
    from ccfuser_amd import ops
    _say(f"thin rule E={E} N={N} K={K} rows={rows}")
    g = torch.Generator(device="cuda").manual_seed(N + K + rows)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    a, w, b = rnd(rows, K).half(), (rnd(E, N, K) * 0.02).half(), rnd(E, N).half()
    counts = [rows // E + (e < rows % E) for e in range(E)]
    off = torch.tensor([0] + counts).cumsum(0).int().cuda()
    out = {}
    try:
        for mode in (0, 1, 2, 3):
            ops.set_option("few_rows", mode)
            out[mode] = ops.ffn2(a, None, off, rows, w, b, torch.empty(rows, N, dtype=torch.float16, device="cuda"))
    finally:
        ops.set_option("few_rows", 1)
    assert torch.equal(out[1], out[3]) == (thin or rows > 32)
    if K < 4096:
        assert torch.equal(out[1], out[2]) != thin
    ref = torch.cat([a[off[e]:off[e + 1]].float() @ w[e].float().t() + b[e].float() for e in range(E)])
    for y in out.values():
        assert float((y.float() - ref).abs().max()) <= (2.0 ** -11 + K * 2.0 ** -24) * float(ref.abs().max()) + 1e-4


@pytest.mark.parametrize("shape", range(6))
@pytest.mark.parametrize("counts,N,K", [
    ([0, 1, 63, 64, 65, 127, 128, 129, 0], 264, 64),          # edges of both tile heights, a ragged last column tile
    ([300, 0, 17], 72, 320),                                  # several M tiles per expert; columns end inside the first tile
    ([2] * 70, 520, 192),                                     # more experts than lanes, several tiles per workgroup
    ([40], 8, 1024),                                          # one expert, the narrowest output
])
def test_few_rows_kernel(shape, counts, N, K):
    """Every tile shape of the kernel for few rows per expert, both weight layouts and all epilogues, through row
    indices: the bits of the 256-row tiles, which add over K in the same order, and the fp32 product."""
    from ccfuser_amd import ops
    g = torch.Generator().manual_seed(shape * 100 + N)
    E, R = len(counts), sum(counts)
    pad = 5                                                   # max_rows may exceed the rows
    _say(f"few rows shape={shape} E={E} R={R} N={N} K={K}")
    x = dev(torch.randn(R + 9, K, generator=g).half())
    w = dev((torch.randn(E, N, K, generator=g) * K ** -0.5).half())
    b = dev(torch.randn(E, N, generator=g).half())
    off = dev(torch.tensor([0] + counts).cumsum(0).int())
    src = dev(torch.cat([torch.randperm(R + 9, generator=g)[:R], torch.zeros(pad, dtype=torch.int64)]).int())
    dst = dev(torch.cat([torch.randperm(R, generator=g), torch.zeros(pad, dtype=torch.int64)]).int())
    wk = w.transpose(1, 2).contiguous()
    scale = dev(torch.rand(R + pad, generator=g).half())

    def outputs():
        res = [ops.ffn1(x, src, off, R + pad, w, b, gelu=True, out=torch.zeros(R, N, dtype=torch.float16, device="cuda"), dst_row=dst),
               ops.ffn1(x, src, off, R + pad, wk, b, gelu=True, out=torch.zeros(R, N, dtype=torch.float16, device="cuda"),
                        dst_row=dst, w_kn=True)]
        for ww, kn in ((w, False), (wk, True)):
            res.append(ops.ffn2(x, dst, off, R + pad, ww, b, torch.zeros(R, N, dtype=torch.float16, device="cuda"), src_row=src,
                                row_scale=scale, w_kn=kn))
        act, pre = ops.ffn1_keep(x, src, off, R + pad, w, b)
        torch.cuda.synchronize()
        return res + [act[:R], pre[:R]]

    ops.set_option("few_rows", 16 + shape)
    try:
        got = outputs()
        ops.set_option("few_rows", 0)
        ops.set_option("split_tail", 0)
        ops.set_option("skinny", 0)
        tiles = outputs()
    finally:
        ops.set_option("few_rows", 1)
        ops.set_option("split_tail", 1)
        ops.set_option("skinny", 1)
    for i, (a, t) in enumerate(zip(got, tiles)):
        assert torch.equal(a, t), f"output {i} differs from the 256-row tiles"
    e_of = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).cuda()
    pre = torch.cat([x[src[:R].long()][e_of == e].float() @ w[e].float().t() + b[e].float() for e in range(E)])
    assert O.mean_rel_err(got[5].cpu(), pre.cpu()) <= MEAN_REL
    plain = torch.zeros_like(pre)
    plain[dst[:R].long()] = pre * scale[:R, None].float()
    assert O.mean_rel_err(got[2].cpu(), plain.cpu()) <= MEAN_REL


@pytest.mark.parametrize("knob,value,default", [("gemm_variant", 3, -1), ("split_tail", 0, 1), ("split_parts", 2, 8),
                                                ("skinny", 0, 1), ("skinny_tail", 1, 0), ("split_inside", 0, 1)])
def test_tile_knobs_select_the_256_row_tiles(knob, value, default):
    """A knob of the 256-row tiles away from its default takes a GEMM of few rows back to them: the launch with a
    plan (``persistent_wgs`` is 0 where no plan is used)."""
    from ccfuser_amd import ops
    R, E, d, f = 512, 8, 256, 1024
    ws = ops.ffn_workspace(R, E, d, f, torch.empty(1, device="cuda")).zero_()
    form = lambda: [ops.ffn_plan_info(ws, R, E, d, f, which)["persistent_wgs"] for which in (1, 2)]
    assert form() == [0, 0]
    ops.set_option(knob, value)
    try:
        assert all(n > 0 for n in form())
    finally:
        ops.set_option(knob, default)
    assert form() == [0, 0]


@pytest.mark.parametrize("E,rows,d,f,which,few", [
    # FFN1 / FFN2 in microseconds, 256-row tiles against tiles of few rows
    (8, 256, 3072, 11008, 1, False),      # 184, 230
    (16, 128, 1536, 6144, 1, False),      # 100, 110
    (32, 128, 768, 3072, 1, False),       # 56, 62
    (16, 256, 1024, 4096, 1, False),      # 68, 72
    (4, 256, 3584, 12096, 1, False),      # 133, 154
    (4, 300, 2048, 8192, 2, False),       # 68, 81
    (2, 1, 4096, 14336, 2, False),        # 51, 60
    (2, 1, 4096, 14336, 1, True),         # 53, 38
    (8, 32, 4096, 14336, 1, True),        # 207, 179
    (8, 32, 4096, 14336, 2, True),        # 197, 175
    (4, 128, 256, 1024, 2, True),         # 29, 10
    (16, 64, 1024, 4096, 1, True),        # 38, 29
    (8, 110, 4096, 12288, 2, True),       # 234, 187
    (8, 230, 1024, 4096, 1, True),        # 44, 40
])
def test_few_row_rule_takes_the_faster_form(E, rows, d, f, which, few):
    """The form that a GEMM of evenly loaded experts runs in, at sizes where the other one measured slower
    (``persistent_wgs`` is 0 where no plan is used)."""
    from ccfuser_amd import ops
    R = E * rows
    ws = ops.ffn_workspace(R, E, d, f, torch.empty(1, device="cuda")).zero_()
    assert (ops.ffn_plan_info(ws, R, E, d, f, which)["persistent_wgs"] == 0) == few


@pytest.mark.usefixtures("gemm_form")
def test_ffn_special_cases():
    """Closed forms: zero weights give the bias path; a single expert is a dense MLP."""
    from ccfuser_amd import ops
    R, d, f = 300, 128, 256
    g = torch.Generator().manual_seed(5)
    x = torch.randn(R, d, generator=g).half()
    b1 = (torch.randn(1, f, generator=g)).half()
    b2 = (torch.randn(1, d, generator=g)).half()
    w1 = torch.zeros(1, f, d).half()
    w2 = torch.zeros(1, d, f).half()
    off = torch.tensor([0, R], dtype=torch.int32).cuda()
    h = ops.ffn1(dev(x), None, off, R, dev(w1), dev(b1), gelu=True)
    ref_h = O.gelu_exact(b1.float()).half().expand(R, f)
    assert (h.cpu().float() - ref_h.float()).abs().max() <= 2e-3
    y = torch.zeros(R, d, dtype=torch.float16, device="cuda")
    ops.ffn2(h, None, off, R, dev(w2), dev(b2), y)
    assert torch.equal(y.cpu(), b2.expand(R, d))
    # the GELU itself over [-8, 8] (zero weights: h = gelu(b1)); every fp16 value of the
    # sweep within one fp16 rounding step of the exact erf form
    f2 = 4096
    sweep = torch.linspace(-8.0, 8.0, f2).half().reshape(1, f2)
    h2 = ops.ffn1(dev(x), None, off, R, dev(torch.zeros(1, f2, d).half()), dev(sweep), gelu=True)
    exact = O.gelu_exact(sweep.float()).reshape(-1)
    got = h2[0].cpu().float()
    step = torch.maximum(exact.abs() * 2.0 ** -10, torch.tensor(6.2e-5))
    assert bool(((got - exact).abs() <= step).all()), float(((got - exact).abs() / step).max())
    assert torch.equal(h2[0], h2[R - 1])
    # pre-activation output
    w1 = (torch.randn(1, f, d, generator=g) * 0.05).half()
    pre = ops.ffn1(dev(x), None, off, R, dev(w1), dev(b1), gelu=False)
    ref = x.float() @ w1[0].float().t() + b1.float()
    assert O.max_abs_err(pre.cpu(), ref) <= MAX_ABS


@pytest.mark.usefixtures("gemm_form")
@pytest.mark.parametrize("R", [4, 300])
def test_gelu_of_every_fp16_value(R):
    """Zero weights, every fp16 value as a bias: within the fp32 form's bound (4e-6 of the argument) and half an fp16
    step of the exact function; infinities and NaN as the exact form has them; the same bits with the pre-activation kept."""
    from ccfuser_amd import ops
    d, f = 64, 65536
    v = torch.arange(f, dtype=torch.int32).to(torch.int16).view(torch.float16)
    x, w = torch.ones(R, d, dtype=torch.float16), torch.zeros(1, f, d, dtype=torch.float16)
    off = torch.tensor([0, R], dtype=torch.int32).cuda()
    h = ops.ffn1(dev(x), None, off, R, dev(w), dev(v[None]), gelu=True)
    kept, pre = ops.ffn1_keep(dev(x), None, off, R, dev(w), dev(v[None]))
    bits = lambda t: t.nan_to_num(nan=7.0).view(torch.int16)
    assert torch.equal(bits(h), bits(kept)) and torch.equal(bits(h), bits(h[:1].expand(R, f).contiguous()))
    assert torch.equal(bits(pre[R - 1].cpu()), bits(v + 0.0))
    got, u = h[R - 1].cpu().double(), v.double()
    exact = 0.5 * u * torch.erfc(-u / 2.0 ** 0.5)
    sane = torch.isfinite(u)
    bound = 4e-6 * u.abs() + exact.abs() * 2.0 ** -11 + 2.0 ** -25
    assert bool(((got - exact).abs() <= bound)[sane].all()), float(((got - exact).abs() / bound)[sane].max())
    assert torch.equal(torch.isnan(got), torch.isnan(u) | (u == float("-inf")))
    assert got[u == float("inf")] == float("inf")


@pytest.mark.parametrize("inside", [1, 0])
def test_split_k_tail_at_its_default_threshold(inside):
    """K = 4096 is where the split of the last round switches on by itself: 36 M tiles x 16 N
    tiles = 2.25 rounds of 256 workgroups, in both GEMMs, whole outputs against fp32.  The parts
    run inside the persistent launch (each workgroup one, behind its tiles) or as a launch of
    their own."""
    from ccfuser_amd import ops
    ops.set_option("split_inside", inside)
    g = torch.Generator().manual_seed(22)
    R, d, f, E = 8192, 4096, 4096, 6
    x = torch.randn(R, d, generator=g).half()
    w1 = (torch.randn(E, f, d, generator=g) * 0.02).half()
    b1 = (torch.randn(E, f, generator=g) * 0.05).half()
    w2 = (torch.randn(E, d, f, generator=g) * 0.02).half()
    b2 = (torch.randn(E, d, generator=g) * 0.05).half()
    idx = torch.randint(0, E, (R,), generator=g)
    r = ops.route(dev(idx), E, 1, -1)
    off, pos = r["offsets"].cpu(), r["pos"].cpu()
    _say(f"split-K tail by default R={R} d={d} f={f} E={E} counts={r['counts'].tolist()}")
    out = {}
    ops.set_option("skinny", 0)               # every row in 256-row tiles: the tile count this test is built on
    for mode in (1, 0):
        ops.set_option("split_tail", mode)
        try:
            h = ops.ffn1(dev(x), r["src_row"], r["offsets"], R, dev(w1), dev(b1), gelu=True)
            y = torch.zeros(R, d, dtype=torch.float16, device="cuda")
            ops.ffn2(h, r["dst_row"], r["offsets"], R, dev(w2), dev(b2), y)
            out[mode] = (h.cpu(), y.cpu())
        finally:
            ops.set_option("split_tail", 1)
    ops.set_option("skinny", 1)
    buf = x[pos].float()
    h_ref = torch.zeros(R, f)
    y_ref = torch.zeros(R, d)
    hq = out[1][0].float()
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        h_ref[lo:hi] = O.gelu_exact(buf[lo:hi] @ w1[e].float().t() + b1[e].float())
        y_ref[pos[lo:hi]] = hq[lo:hi] @ w2[e].float().t() + b2[e].float()
    assert O.max_abs_err(out[1][0], h_ref) <= MAX_ABS and O.mean_rel_err(out[1][0], h_ref) <= MEAN_REL
    assert O.max_abs_err(out[1][1], y_ref) <= MAX_ABS and O.mean_rel_err(out[1][1], y_ref) <= MEAN_REL
    # the split did run: bits differ from the unsplit kernels
    assert not torch.equal(out[1][0], out[0][0]) and not torch.equal(out[1][1], out[0][1])
    ops.set_option("split_inside", 1)


def test_split_k_tail_all_epilogues():
    """The last, partly filled round of tiles is cut along K and reduced by a separate kernel.
    By default that happens for K >= 4096 only; here it is forced on a small K so that the
    reduction's three epilogues (plain with row index and scale, GELU, GELU keeping the
    pre-activation) are compared with the oracle and with the unsplit kernels."""
    from ccfuser_amd import ops
    g = torch.Generator().manual_seed(21)
    R, d, f, E = 8192, 2048, 2048, 6           # 16+ M tiles x 8 N tiles: more tiles than workgroups, a ragged last round
    x = (torch.randn(R, d, generator=g)).half()
    w1 = (torch.randn(E, f, d, generator=g) * 0.05).half()
    b1 = (torch.randn(E, f, generator=g) * 0.05).half()
    w2 = (torch.randn(E, d, f, generator=g) * 0.02).half()
    b2 = (torch.randn(E, d, generator=g) * 0.05).half()
    idx = torch.randint(0, E, (R,), generator=g)
    r = ops.route(dev(idx), E, 1, -1)
    off = r["offsets"].cpu()
    pos = r["pos"].cpu()
    scale = (torch.rand(R, generator=g) + 0.5).half()
    _say(f"split-K tail R={R} d={d} f={f} E={E} counts={r['counts'].tolist()}")
    results = {}
    ops.set_option("skinny", 0)               # every row in 256-row tiles: the tile count this test is built on
    for mode in (0, 4, -4):                   # -4: as 4, the parts as a launch of their own
        ops.set_option("split_tail", abs(mode))
        ops.set_option("split_inside", 0 if mode < 0 else 1)
        try:
            h = ops.ffn1(dev(x), r["src_row"], r["offsets"], R, dev(w1), dev(b1), gelu=True)
            act, pre = ops.ffn1_keep(dev(x), r["src_row"], r["offsets"], R, dev(w1), dev(b1))
            y = torch.zeros(R, d, dtype=torch.float16, device="cuda")
            ops.ffn2(h, r["dst_row"], r["offsets"], R, dev(w2), dev(b2), y, row_scale=dev(scale))
            results[mode] = [t.cpu() for t in (h, act, pre, y)]
        finally:
            ops.set_option("split_tail", 1)
            ops.set_option("split_inside", 1)
    ops.set_option("skinny", 1)
    # the same parts and the same order of summation wherever they run
    assert all(torch.equal(a, b) for a, b in zip(results[4], results[-4]))
    buf = x[torch.div(pos, 1, rounding_mode="floor")].float()
    h_ref = torch.zeros(R, f)
    pre_ref = torch.zeros(R, f)
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        pre_ref[lo:hi] = buf[lo:hi] @ w1[e].float().t() + b1[e].float()
    h_ref = O.gelu_exact(pre_ref)
    for mode, (h, act, pre, y) in results.items():
        assert O.max_abs_err(h, h_ref) <= MAX_ABS and O.mean_rel_err(h, h_ref) <= MEAN_REL, mode
        assert torch.equal(h, act), mode
        assert O.max_abs_err(pre, pre_ref) <= MAX_ABS, mode
    y_ref = torch.zeros(R, d)
    hq = results[4][0].float()
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        y_ref[pos[lo:hi]] = (hq[lo:hi] @ w2[e].float().t() + b2[e].float()) * scale[lo:hi].float()[:, None]
    assert O.max_abs_err(results[4][3], y_ref) <= MAX_ABS and O.mean_rel_err(results[4][3], y_ref) <= MEAN_REL
    # split and unsplit differ only in summation order (and do differ: the split path ran)
    assert O.max_abs_err(results[4][3], results[0][3].float()) <= MAX_ABS
    assert O.max_abs_err(results[4][0], results[0][0].float()) <= MAX_ABS
    assert not torch.equal(results[4][3], results[0][3]) and not torch.equal(results[4][0], results[0][0])


# Forced cases are sized so that both GEMMs have at least as many worst-case tiles as the chip has
# CUs ((ceil(R / 256) + E) * ceil(N / 256) >= 256): only then does the persistent launch set
# workgroups aside for skinny tiles.  `expect`: which GEMMs must report skinny tiles actually run.
@pytest.mark.parametrize("R,d,f,E,skew,seed,mode,expect", [
    (8192, 4096, 4096, 6, False, 31, 1, ""),          # remainders of 56..122 rows: one or two skinny tiles each, if the plan wants them
    (8192 + 6 * 200, 4096, 4096, 6, False, 35, 1, ""),   # remainders of ~25 rows, long K: the plan's own choice
    (0, 256, 1024, 60, False, 32, -2, "1"),           # first GEMM with K = 256: four K tiles, the shortest the loop takes
    (2100, 1024, 2048, 70, True, 33, -1, "12"),       # most experts are nothing but a skinny tile, some are empty
    (1150, 512, 768, 3, False, 34, -3, ""),           # remainders of 127, 130 and 125 rows: none is skinny, nothing to do
    (15360, 1088, 832, 60, False, 36, -4, "12"),      # N no multiple of 256 in either GEMM (832, 1088)
    (8192, 4096, 4096, 6, False, 37, -5, "12"),       # as a launch of their own, cut along K: a workgroup's range inside one tile
    (0, 1536, 4160, 40, False, 38, -5, "12"),         # experts of 17..64 rows only: ranges of four tiles, N = 4160
    (8192, 4096, 4096, 6, False, 39, -6, "12"),       # cut along K inside the persistent launch, before / behind the 256-row tiles
    (0, 1536, 4160, 40, False, 40, -6, "12"),         # the same where most workgroups have no 256-row tile at all
    (20000, 2048, 2048, 12, False, 41, -6, "12"),     # several 256-row tiles per workgroup in front of / behind the ranges
])
def test_skinny_tiles(R, d, f, E, skew, seed, mode, expect):
    """Rows beyond an expert's full 256-row tiles (at most 64) run as 64-row tiles: in workgroups
    the plan sets aside beside the 256-row tiles (mode -n: forced, n workgroups per XCD) or as a
    launch of their own cut along K (mode -5: forced) or cut along K inside the persistent launch
    (mode -6: forced); mode 1 leaves the choice to the plan's cost model.  All three forward epilogues with that path on and off, each against fp32.
    Beside the 256-row tiles the path adds over K in the same order as they do and must agree
    bit for bit; cut along K it agrees within rounding.  The plan must report that skinny tiles
    really ran where the case is built for them."""
    from ccfuser_amd import ops
    counts = None
    if expect and not skew:
        # every expert: whole 256-row tiles (R / E rounded down to them) plus a remainder of 17..64 rows
        counts = torch.tensor([(R // E) // 256 * 256 + 17 + (e * 11) % 48 for e in range(E)])
        R = int(counts.sum())
    x, w1, b1, w2, b2, e_of_row = _ffn_case(R, d, f, E, seed, skew)
    g = torch.Generator().manual_seed(seed)
    if counts is not None:
        e_of_row = torch.repeat_interleave(torch.arange(E), counts)[torch.randperm(R, generator=g)]
    scale = (torch.rand(R, generator=g) + 0.5).half()
    r = ops.route(dev(e_of_row), E, 1)
    off, pos = r["offsets"].cpu().tolist(), r["pos"].cpu()
    rem = r["counts"].cpu() % 256
    _say(f"skinny mode={mode} R={R} d={d} f={f} E={E} remainders={rem.tolist()[:12]}")
    ws = ops.ffn_workspace(R, E, d, f, dev(x))
    res, info = {}, {}
    for m in (mode, 0):
        ops.set_option("skinny", m)
        # beside the 256-row tiles: keep those unsplit, the comparison is about the skinny path;
        # a launch of their own needs the split kernels launched (every K tile count allowed)
        ops.set_option("split_tail", 2 if mode <= -5 else 0)
        ops.set_option("skinny_tail", 1 if mode == -5 else 0)   # the launch of their own is off by default
        try:
            h = ops.ffn1(dev(x), r["src_row"], r["offsets"], R, dev(w1), dev(b1), gelu=True, workspace=ws)
            info[m, 1] = ops.ffn_plan_info(ws, R, E, d, f, 1)
            act, pre = ops.ffn1_keep(dev(x), r["src_row"], r["offsets"], R, dev(w1), dev(b1))
            y = torch.zeros(R, d, dtype=torch.float16, device="cuda")
            ops.ffn2(h, r["dst_row"], r["offsets"], R, dev(w2), dev(b2), y, row_scale=dev(scale), workspace=ws)
            info[m, 2] = ops.ffn_plan_info(ws, R, E, d, f, 2)
            torch.cuda.synchronize()
            res[m] = [t.cpu() for t in (h, act, pre, y)]
        finally:
            ops.set_option("skinny", 1)
            ops.set_option("split_tail", 1)
            ops.set_option("skinny_tail", 0)
    _say(f"  plan, first GEMM: {info[mode, 1]}")
    _say(f"  plan, second GEMM: {info[mode, 2]}")
    for which in (1, 2):
        i = info[mode, which]
        ran = i["skinny_tiles"] > 0 and (i["skinny_wgs_per_xcd"] > 0 or i["skinny_tail_steps"] != 0)
        if str(which) in expect:
            assert ran, (which, i)
            # steps > 0: as a launch of their own; < 0: inside the persistent launch
            assert (i["skinny_tail_steps"] > 0) == (mode == -5) and (i["skinny_tail_steps"] < 0) == (mode == -6), i
            assert i["skinny_wgs_per_xcd"] == (-mode if mode > -5 else 0), i
        if mode < 0:
            assert info[0, which]["skinny_tiles"] == 0
    buf = x[pos].float()
    pre_ref = torch.zeros(R, f)
    for e in range(E):
        lo, hi = off[e], off[e + 1]
        if hi > lo:
            pre_ref[lo:hi] = buf[lo:hi] @ w1[e].float().t() + b1[e].float()
    h_ref = O.gelu_exact(pre_ref)
    for m, (h, act, pre, y) in res.items():
        assert O.max_abs_err(h, h_ref) <= MAX_ABS and O.mean_rel_err(h, h_ref) <= MEAN_REL, m
        assert torch.equal(h, act), m
        assert O.max_abs_err(pre, pre_ref) <= MAX_ABS, m
        y_ref = torch.zeros(R, d)
        hq = h.float()
        for e in range(E):
            lo, hi = off[e], off[e + 1]
            if hi > lo:
                y_ref[pos[lo:hi]] = (hq[lo:hi] @ w2[e].float().t() + b2[e].float()) * scale[lo:hi].float()[:, None]
        assert O.max_abs_err(y, y_ref) <= MAX_ABS and O.mean_rel_err(y, y_ref) <= MEAN_REL, m
    same = [torch.equal(a, b) for a, b in zip(res[mode], res[0])]
    _say(f"  skinny on/off bitwise equal (h, act, pre, y): {same}")
    cut = any(info[mode, which]["skinny_tail_steps"] != 0 for which in (1, 2))   # the plan's own choice may be a K cut too
    if mode <= -5 or cut:
        # another summation order: close, and not identical where skinny tiles ran
        for a, b in zip(res[mode], res[0]):
            assert O.max_abs_err(a, b.float()) <= MAX_ABS
        assert not all(same)
    else:
        assert all(same)


def test_mfma_probe_runs_and_counts_its_flop():
    """ccf_probe_mfma: the MFMA-only loop bench.py times for its measured ceiling.  With zero
    operands every sum it leaves is zero; the flop count is the closed form."""
    import ctypes as C
    from ccfuser_amd import _lib
    probe = _lib.probe_lib()
    wgs, iters = 16, 10
    out = torch.full((wgs * 256,), 7.0, dtype=torch.float32, device="cuda")
    flop = C.c_double()
    for const in (1, 0):
        assert probe.ccf_probe_mfma(wgs, iters, const, out.data_ptr(), C.byref(flop), None) == 0
        torch.cuda.synchronize()
        assert flop.value == wgs * 4 * iters * 64 * 16 * 16 * 32 * 2
        assert bool(torch.isfinite(out).all())
        if const:
            assert not out.any()
    assert probe.ccf_probe_mfma(0, iters, 1, out.data_ptr(), C.byref(flop), None) == 1


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("T,d,E,k,capacity", [
    (1, 128, 8, 2, -1),                    # one workgroup of one token
    (333, 192, 4, 1, 20),                  # few experts: counts one at a time, capacity limit
    (1999, 768, 8, 2, -1),
    (515, 64, 3, 3, -1),                   # slots that do not tile the routing's chunks: counted by the routing
    (8192, 256, 64, 2, 300),               # the longest table there is room for in fp32
    (8193, 128, 64, 1, -1),                # one workgroup more than that
    (4096, 128, 36, 2, -1),                # four counts a load, experts that do not divide a wavefront
    (6000, 64, 9, 4, -1),                  # a long table of odd width
    (200, 64, 600, 2, -1),                 # more experts than threads
    (700, 64, 300, 2, -1),                 # the same in a table of counts
    (512, 256, 64, 2, -1), (513, 256, 64, 2, -1),    # 1024 indices, counted by the routing, and more
    (64, 1024, 32, 2, -1), (65, 1024, 32, 2, -1),    # fp16: 2048 counts, and more than the routing takes for 1024 indices
    (700, 4096, 2, 1, -1),                 # fp32: a wavefront per token, which leaves no counts
    (2, 4096, 8, 2, -1), (3, 4096, 8, 2, -1),        # fp16: gate and routing as one launch in two turns, one token more
    (8, 768, 8, 2, 3), (9, 768, 8, 2, 0),            # the same at four tokens a turn, capacity limits
    (32, 256, 4, 2, 9), (33, 256, 4, 2, -1),         # 64 indices, and more
    (7, 136, 9, 8, 4), (21, 8, 3, 3, -1), (1, 512, 128, 8, -1),
])
def test_gate_with_routing_is_the_gate_then_the_routing(T, d, E, k, capacity, dtype):
    """One call for both: the bits of the gate alone and of the routing on its choice; rows of NaN choose nothing."""
    from ccfuser_amd import ops
    _say(f"gate_route T={T} d={d} E={E} k={k} capacity={capacity} {dtype}")
    g = torch.Generator().manual_seed(T + E)
    x = torch.randn(T, d, generator=g)
    if T > 100:
        x[7] = float("nan")
    x, wg, bg = [t.to(dtype).cuda() for t in (x, torch.randn(E, d, generator=g) * 0.1, torch.randn(E, generator=g))]
    idx, score, r = ops.gate_route(x, wg, bg, k, capacity)
    idx0, score0 = ops.gate_topk_softmax(x, wg, bg, k)
    r0 = ops.route(idx0.reshape(-1), E, k, capacity)
    assert torch.equal(idx, idx0) and torch.equal(score.nan_to_num(3.0), score0.nan_to_num(3.0))
    n = int(r0["offsets"][-1])
    for name in ("counts", "offsets", "inv_pos", "idx_kept"):
        assert torch.equal(r[name], r0[name]), name
    for name in ("pos", "src_row", "dst_row"):
        assert torch.equal(r[name][:n], r0[name][:n]), name


@pytest.mark.parametrize("T,E,k", [(65536, 32, 8), (65537, 17, 8), (131075, 8, 8), (65536, 32, 4), (65536, 20, 5)])
def test_gate_workgroups_of_more_indices_than_a_routing_chunk(T, E, k):
    """Gate workgroups of 256 tokens: eight experts each are 2048 indices, twice a chunk of the routing, which then counts
    for itself; four fill a chunk.  Gate with routing and the layer call against the gate, then the routing."""
    from ccfuser_amd import ops
    _say(f"gate rows longer than a chunk T={T} E={E} k={k}")
    d = f = 64
    g = torch.Generator(device="cuda").manual_seed(T + k)
    rnd = lambda *s: (torch.randn(*s, generator=g, device="cuda") * 0.1).half()
    x, wg, bg = rnd(T, d), rnd(E, d), rnd(E)
    idx0, score0 = ops.gate_topk_softmax(x, wg, bg, k)
    r0 = ops.route(idx0.reshape(-1), E, k)
    idx, score, r = ops.gate_route(x, wg, bg, k)
    assert torch.equal(idx, idx0) and torch.equal(score, score0)
    for name in ("counts", "offsets", "pos", "src_row", "dst_row", "inv_pos", "idx_kept"):
        assert torch.equal(r[name], r0[name]), name
    _, m = ops.moe_forward(x, wg, bg, rnd(E, f, d), rnd(E, f), rnd(E, d, f), rnd(E, d), k, return_routing=True)
    for name in ("counts", "offsets", "pos"):
        assert torch.equal(m[name], r0[name]), name
    assert torch.equal(m["idx"].view(-1), idx0.view(-1)) and torch.equal(m["score"].view(-1), score0.view(-1))


def test_gate_hooks_run_where_the_routing_goes_with_the_gate():
    """A gate with a hook, a subclass and another number of experts are called as modules, the gate itself is not."""
    from ccfuser_amd.mix_moe.gates import NaiveGate
    from ccfuser_amd.mix_moe.transformer import AsyncExpertAssignment
    with torch.device("cuda"):
        gate = NaiveGate(64, 4, 1, 2).half()
    x = torch.randn(50, 64, dtype=torch.float16, device="cuda")
    assign = AsyncExpertAssignment(0, 1, 0, 4, 50)
    pos0, score0, infos0 = assign.process_data(gate, x, 4, 1)
    assert gate.calls_forward_only() and gate.has_loss
    seen = []
    handle = gate.register_forward_hook(lambda m, a, out: seen.append(out[0].shape))
    pos1, score1, infos1 = assign.process_data(gate, x, 4, 1)
    handle.remove()
    assert seen == [torch.Size([50, 2])]

    class Mine(NaiveGate):
        def forward(self, inp, return_all_scores=False):
            seen.append("mine")
            return super().forward(inp, return_all_scores)
    with torch.device("cuda"):
        mine = Mine(64, 4, 1, 2).half()
    mine.load_state_dict(gate.state_dict())
    pos2, score2, infos2 = assign.process_data(mine, x, 4, 1)
    assert seen[-1] == "mine"
    wide = assign.process_data(gate, x, 6, 1)[2]
    assert wide["counts"].numel() == 6 and torch.equal(wide["counts"][:4], infos0["counts"])
    n = int(infos0["offsets"][-1])
    for pos, score, infos in ((pos1, score1, infos1), (pos2, score2, infos2)):
        assert torch.equal(pos[:n], pos0[:n]) and torch.equal(score, score0) and torch.equal(infos["inv_pos"], infos0["inv_pos"])


@pytest.mark.parametrize("scored", [3, 6])
def test_gate_that_scores_another_number_of_experts_is_called_as_a_module(scored):
    """A router whose linear layer was replaced: the routing goes over the caller's experts, and a choice beyond them is
    nobody's."""
    from ccfuser_amd import ops
    from ccfuser_amd.mix_moe.gates import NaiveGate
    from ccfuser_amd.mix_moe.transformer import AsyncExpertAssignment
    with torch.device("cuda"):
        gate = NaiveGate(64, 4, 1, 2).half()
        gate.gate = torch.nn.Linear(64, scored).half()
    x = torch.randn(500, 64, dtype=torch.float16, device="cuda")
    pos, score, infos = AsyncExpertAssignment(0, 1, 0, 4, 500).process_data(gate, x, 4, 1)
    idx, score0 = gate(x)
    r = ops.route(idx.reshape(-1), 4, 2)
    n = int(r["offsets"][-1])
    assert torch.equal(score, score0) and torch.equal(pos[:n], r["pos"][:n])
    for name in ("counts", "offsets", "inv_pos", "idx_kept"):
        assert torch.equal(infos[name], r[name]), name


@pytest.mark.parametrize("kn", [False, True])
@pytest.mark.parametrize("counts", [[64, 1], [60, 200], [0, 128]])
def test_few_rows_of_large_weights(counts, kn):
    """Weights large enough for non-temporal loads, an expert of one M tile beside none, another or one of several: the
    bits of the 256-row tiles."""
    from ccfuser_amd import ops
    E, d, f = 2, 4096, 10304                                # 169 MB each way, a last column tile that is not full
    R = sum(counts)
    _say(f"few rows of large weights {counts} kn={kn}")
    g = torch.Generator(device="cuda").manual_seed(R)
    rnd = lambda *s: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, 0.05, generator=g)
    off = torch.tensor([0, counts[0], R], dtype=torch.int32, device="cuda")
    x, h = rnd(R, d), rnd(R, f)
    w1, w2 = (rnd(E, d, f), rnd(E, f, d)) if kn else (rnd(E, f, d), rnd(E, d, f))
    b1, b2 = rnd(E, f), rnd(E, d)
    rows = torch.randperm(R, generator=torch.Generator().manual_seed(R)).int().cuda()

    def both():
        y = torch.zeros(R, d, dtype=torch.float16, device="cuda")
        return ops.ffn1(x, rows, off, R, w1, b1, w_kn=kn), ops.ffn2(h, rows, off, R, w2, b2, y, w_kn=kn)

    ops.set_option("few_rows", 2)
    try:
        got = both()
        for name, value in (("few_rows", 0), ("split_tail", 0), ("skinny", 0)):
            ops.set_option(name, value)
        ref = both()
    finally:
        for name, value in (("few_rows", 1), ("split_tail", 1), ("skinny", 1)):
            ops.set_option(name, value)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kn", [False, True])
@pytest.mark.parametrize("counts", [[64, 0, 0, 0], [0, 5, 60, 0], [20, 1, 40, 64], [0, 200, 3, 0]])
def test_few_rows_of_large_weights_by_experts_with_rows(counts, kn):
    """Experts of 84 MB, of which non-temporal loads want four with rows, or two of a layer's alternating products: on
    both sides of either number the bits of the 256-row tiles."""
    from ccfuser_amd import ops
    E, d, f = 4, 4096, 10304
    R = sum(counts)
    _say(f"few rows by experts with rows {counts} kn={kn}")
    g = torch.Generator(device="cuda").manual_seed(R)
    rnd = lambda *s: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, 0.05, generator=g)
    off = torch.tensor([0] + counts).cumsum(0).int().cuda()
    x, h = rnd(R, d), rnd(R, f)
    w1, w2 = (rnd(E, d, f), rnd(E, f, d)) if kn else (rnd(E, f, d), rnd(E, d, f))
    b1, b2 = rnd(E, f), rnd(E, d)

    def both(in_layer):
        y = torch.zeros(R, d, dtype=torch.float16, device="cuda")
        return ops.ffn1(x, None, off, R, w1, b1, w_kn=kn, in_layer=in_layer), ops.ffn2(h, None, off, R, w2, b2, y, w_kn=kn, in_layer=in_layer)

    ops.set_option("few_rows", 2)
    try:
        got = both(False) + both(True)
        for name, value in (("few_rows", 0), ("split_tail", 0), ("skinny", 0)):
            ops.set_option(name, value)
        ref = both(False)
    finally:
        for name, value in (("few_rows", 1), ("split_tail", 1), ("skinny", 1)):
            ops.set_option(name, value)
    for a, b in zip(got, ref + ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("counts,N,K,apart", [
    ([64, 1], 10304, 4096, True),              # 169 MB, a last column tile that is not full; one M tile each
    ([100, 140], 6912, 6144, True),            # 170 MB; two M tiles of 128 rows for one of them
    ([0, 33, 0], 20608, 4096, True),           # one expert with rows among three: their number is not known on the host
    ([100, 157], 10304, 4096, False),          # more than 128 rows an expert on average
    ([64, 1], 10304, 4160, False),             # rows that do not lie 4 KB apart
    ([64, 1], 9728, 4096, False),              # 159 MB
])
def test_few_rows_of_weights_from_memory_start_at_places_of_their_own(counts, N, K, apart):
    """By the rule, the column tiles of large [E, N, K] weights start inside K and go around: other bits than in ascending
    order, and no further from the product in 64 bits (their errors' 2-norms within 5 %: both round about K sums of the
    same terms, and then to fp16, which dominates).  The same bits from every epilogue, in a layer or alone, and from a
    call with other rows beside them."""
    from ccfuser_amd import ops
    E, R = len(counts), sum(counts)
    _say(f"starts apart {counts} N={N} K={K}")
    g = torch.Generator(device="cuda").manual_seed(N + K + R)
    rnd = lambda *s, std=1.0: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=g)
    off = torch.tensor([0] + counts).cumsum(0).int().cuda()
    x, w, b = rnd(R, K), rnd(E, N, K, std=0.02), rnd(E, N)
    ref = torch.cat([x[off[e]:off[e + 1]].double() @ w[e].double().t() + b[e].double() for e in range(E)])
    new = lambda rows: torch.empty(rows, N, dtype=torch.float16, device="cuda")
    out, h = {}, {}
    try:
        for mode in (2, 1):
            ops.set_option("few_rows", mode)
            out[mode] = ops.ffn2(x, None, off, R, w, b, new(R))
            h[mode] = ops.ffn1(x, None, off, R, w, b)
    finally:
        ops.set_option("few_rows", 1)
    assert torch.equal(out[1], out[2]) != apart and torch.equal(h[1], h[2]) != apart
    err = {m: float((y.double() - ref).norm()) for m, y in out.items()}
    assert err[1] <= 1.05 * err[2], err
    assert torch.equal(out[1], ops.ffn2(x, None, off, R, w, b, new(R), in_layer=True))
    act, pre = ops.ffn1_keep(x, None, off, R, w, b)
    assert torch.equal(act, h[1]) and torch.equal(pre, out[1])
    if apart and counts[1] > 1:                # the last expert's rows without one of them
        e = max(i for i, c in enumerate(counts) if c)
        fewer = off.clone()
        fewer[e + 1:] -= 1
        assert torch.equal(ops.ffn2(x, None, fewer, R - 1, w, b, new(R - 1)), out[1][:R - 1])


def test_places_of_a_sum_go_by_the_column_alone():
    """Sums start where their column says: the same bits for an expert in another slot of the weights."""
    from ccfuser_amd import ops
    counts, N, K = [40, 24], 10304, 4096
    E, R = len(counts), sum(counts)
    _say("places by the column")
    g = torch.Generator(device="cuda").manual_seed(R)
    rnd = lambda *s, std=1.0: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=g)
    x, w, b = rnd(R, K), rnd(E, N, K, std=0.02), rnd(E, N)

    def product(x, counts, w, b):
        off = torch.tensor([0] + counts).cumsum(0).int().cuda()
        return ops.ffn2(x, None, off, len(x), w, b, torch.empty(len(x), N, dtype=torch.float16, device="cuda"))

    out = product(x, counts, w, b)
    ops.set_option("few_rows", 2)
    try:
        assert not torch.equal(out, product(x, counts, w, b))             # it is a call whose sums start inside K
    finally:
        ops.set_option("few_rows", 1)
    swapped = product(torch.cat([x[40:], x[:40]]), counts[::-1], w.flip(0).contiguous(), b.flip(0).contiguous())
    assert torch.equal(torch.cat([swapped[24:], swapped[:24]]), out)


def test_places_of_a_sum_for_fewer_rows_than_experts():
    """Whether sums start inside K goes by the weights that are there, not by how many rows might touch them: a row has the
    same bits alone in a call and beside others."""
    from ccfuser_amd import ops
    E, N, K = 2, 10304, 4096
    _say("places with fewer rows than experts")
    g = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s, std=1.0: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=g)
    x, w, b = rnd(3, K), rnd(E, N, K, std=0.02), rnd(E, N)

    def product(x, *counts):
        off = torch.tensor([0, *counts]).cumsum(0).int().cuda()
        return ops.ffn2(x, None, off, len(x), w, b, torch.empty(len(x), N, dtype=torch.float16, device="cuda"))

    out = product(x, 2, 1)
    for i, counts in enumerate(([1, 0], [1, 0], [0, 1])):
        assert torch.equal(product(x[i:i + 1].contiguous(), *counts), out[i:i + 1]), i


@pytest.mark.parametrize("K", [2048, 4096])
def test_places_of_a_sum_in_every_tile_shape(K):
    """Sums that start inside K, in tiles of all shapes with several tiles per workgroup, one and more M tiles an expert and
    a last column tile that is not full, with and without non-temporal loads: the same bits from every shape, other
    ones than in ascending order, and as near to the product in 64 bits as those (2-norms within 5 %: fp16 rounding dominates
    both)."""
    from ccfuser_amd import ops
    counts, N = [1, 64, 65, 130, 0, 128, 33, 5, 127, 16, 260, 48, 2, 70, 64, 20, 17, 100, 3], 4136
    E, R = len(counts), sum(counts)
    _say(f"places in every shape K={K}")
    g = torch.Generator(device="cuda").manual_seed(K)
    rnd = lambda *s, std=1.0: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=g)
    off = torch.tensor([0] + counts).cumsum(0).int().cuda()
    x, w, b, scale = rnd(R + 9, K), rnd(E, N, K, std=0.02), rnd(E, N), rnd(R)
    perm = lambda n: torch.randperm(n, generator=g, device="cuda")[:R].int()
    src, dst = perm(R + 9), perm(R)
    kn = w.transpose(1, 2).contiguous()

    def outputs(in_layer):
        y = torch.empty(R, N, dtype=torch.float16, device="cuda")
        plain = ops.ffn2(x, dst, off, R, w, b, y, row_scale=scale, src_row=src, in_layer=in_layer)
        act, pre = ops.ffn1_keep(x, src, off, R, w, b)
        return plain, ops.ffn1(x, src, off, R, w, b, in_layer=in_layer), act, pre

    out = {}
    try:
        for shape in range(6):
            ops.set_option("few_rows", 16 + shape)
            for places in (1, 0):
                ops.set_option("few_rows_places", places)
                out[shape, places] = outputs(False)
                for a, c in zip(outputs(True), out[shape, places]):
                    assert torch.equal(a, c), (shape, places)
                for a, c in zip(out[shape, places], out[0, places]):
                    assert torch.equal(a, c), (shape, places)
        ops.set_option("few_rows_places", 1)                      # [E, K, N] weights keep the ascending order
        assert torch.equal(ops.ffn1(x, src, off, R, kn, b, w_kn=True), out[0, 0][1])
    finally:
        ops.set_option("few_rows", 1)
        ops.set_option("few_rows_places", -1)
    for a, c in zip(out[0, 1], out[0, 0]):
        assert not torch.equal(a, c)
    xs = x[src.long()].double()
    pre = torch.cat([xs[off[e]:off[e + 1]] @ w[e].double().t() + b[e].double() for e in range(E)])
    err = [float((out[0, p][3].double() - pre).norm()) for p in (1, 0)]
    assert err[0] <= 1.05 * err[1], err
    assert torch.equal(out[0, 1][1], out[0, 1][2])


def test_places_of_a_sum_over_two_rounds_of_tiles():
    """A decoding batch's first product by the rule: each workgroup has a second column tile, whose places are other ones.
    No further from the product in 64 bits than the ascending sums (squares within 10 %: fp16 rounding dominates both), and
    their bits with the places switched off."""
    from ccfuser_amd import ops
    E, rows, N, K = 8, 32, 14336, 4096
    R = E * rows
    _say("places over two rounds")
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda *s, std=1.0: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=g)
    off = (torch.arange(E + 1) * rows).int().cuda()
    x, w, b = rnd(R, K), rnd(E, N, K, std=0.02), rnd(E, N)
    out = {}
    try:
        for mode, places in ((1, -1), (2, -1), (1, 0)):
            ops.set_option("few_rows", mode)
            ops.set_option("few_rows_places", places)
            out[mode, places] = ops.ffn2(x, None, off, R, w, b, torch.empty(R, N, dtype=torch.float16, device="cuda"))
    finally:
        ops.set_option("few_rows", 1)
        ops.set_option("few_rows_places", -1)
    assert torch.equal(out[1, 0], out[2, -1]) and not torch.equal(out[1, -1], out[1, 0])
    sq = {key: 0.0 for key in out}
    for e in range(E):
        at = slice(e * rows, (e + 1) * rows)
        ref = x[at].double() @ w[e].double().t() + b[e].double()
        for key, y in out.items():
            sq[key] += float((y[at].double() - ref).square().sum())
    assert sq[1, -1] <= 1.1 * sq[1, 0], sq


@pytest.mark.parametrize("counts,N,K", [
    ([513, 512, 511, 500, 257, 1, 0, 700], 3072, 768),       # remainders of one row, of none and of nearly a tile
    ([300] * 8, 3840, 256),                                  # the shortest K, two tiles an expert: just inside a round
    ([2040], 7168, 1024),
])
def test_one_round_of_tiles_has_no_skinny_tiles(counts, N, K):
    """256-row tiles that fill a round at most need no reduction launch: both weight layouts and the form that keeps the
    pre-activation against fp32 (sums of K terms, half an fp16 step), and the bits of the call without skinny tiles."""
    from ccfuser_amd import ops
    E, R = len(counts), sum(counts)
    _say(f"one round {counts} N={N} K={K}")
    g = torch.Generator(device="cuda").manual_seed(N + K + R)
    rnd = lambda *s, std=1.0: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=g)
    off = torch.tensor([0] + counts).cumsum(0).int().cuda()
    x, w, b = rnd(R, K), rnd(E, N, K, std=K ** -0.5), rnd(E, N)
    kn = w.transpose(1, 2).contiguous()
    ws = ops.ffn_workspace(R, E, K, N, x)
    res = {}
    try:
        ops.set_option("few_rows", 0)
        for skinny in (1, 0):
            ops.set_option("skinny", skinny)
            h = ops.ffn1(x, None, off, R, w, b, gelu=False, workspace=ws)
            assert ops.ffn_plan_info(ws, R, E, K, N, 1)["skinny_tiles"] == 0
            res[skinny] = (h, ops.ffn1(x, None, off, R, kn, b, gelu=False, w_kn=True), ops.ffn1_keep(x, None, off, R, w, b)[1])
    finally:
        ops.set_option("few_rows", 1)
        ops.set_option("skinny", 1)
    ref = torch.cat([x[off[e]:off[e + 1]].float() @ w[e].float().t() + b[e].float() for e in range(E)])
    for a, c in zip(res[1], res[0]):
        assert torch.equal(a, c)
        assert float((a.float() - ref).abs().max()) <= (2.0 ** -11 + K * 2.0 ** -24) * float(ref.abs().max()) + 1e-4


def _launches(fn):
    """Kernel launches of a call: the nodes of a graph that captures it."""
    import ctypes as C
    from ccfuser_amd import _lib
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        fn()
    n = C.c_size_t(0)
    get = _lib.lib().hipGraphGetNodes                         # of the HIP runtime that the library is linked to
    assert get(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(n)) == 0
    return n.value


def _zipf_counts(E, R, skew):
    w = torch.arange(1, E + 1).double() ** -skew
    counts = (w / w.sum() * R).floor().long()
    counts[0] += R - counts.sum()
    return counts[torch.randperm(E, generator=torch.Generator().manual_seed(E))].tolist()


@pytest.mark.parametrize("E,R,skew,N,K,one_round", [
    (8, 3998, 0.0, 3072, 768, True),           # a training step's first product
    (8, 3998, 0.0, 3328, 768, False),          # another column tile: two standard deviations beyond a round
    (8, 2400, 0.0, 3840, 256, True),           # the shortest K, just inside a round
    (8, 2400, 0.0, 4096, 256, False),
    (16, 3644, 1.5, 3072, 768, True),          # uneven loads of more than a round (300 tiles), K too short to cut
    (8, 3236, 0.0, 4096, 1024, True),          # where uneven loads might not fit: the last K that may, and the first that may not
    (8, 3236, 0.0, 4096, 1088, False),
    (16, 7000, 1.5, 1536, 3584, True),         # a long K whose uneven loads fit
    (32, 12762, 1.5, 896, 3136, False),        # and one whose uneven loads do not (284 tiles): 130 us in tiles only, 100 with skinny ones
])
def test_one_round_of_tiles_by_sizes(E, R, skew, N, K, one_round):
    """Which sizes of 256-row tiles plan neither skinny tiles nor a reduction launch, in both weight layouts; results
    against fp32 (sums of K terms, half an fp16 step)."""
    from ccfuser_amd import ops
    _say(f"one round E={E} R={R} skew={skew} N={N} K={K}")
    counts = _zipf_counts(E, R, skew)
    g = torch.Generator(device="cuda").manual_seed(N + K + R)
    rnd = lambda *s, std=1.0: torch.empty(*s, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=g)
    off = torch.tensor([0] + counts).cumsum(0).int().cuda()
    x, w, b = rnd(R, K), rnd(E, N, K, std=K ** -0.5), rnd(E, N)
    ws = ops.ffn_workspace(R, E, K, N, x)
    tiles = sum(-(-c // 256) for c in counts) * -(-N // 256)
    ref = torch.cat([x[off[e]:off[e + 1]].float() @ w[e].float().t() + b[e].float() for e in range(E)])
    ops.set_option("few_rows", 0)
    try:
        for weight, kn in ((w, False), (w.transpose(1, 2).contiguous(), True)):
            out = torch.empty(R, N, dtype=torch.float16, device="cuda")
            call = lambda: ops.ffn1(x, None, off, R, weight, b, gelu=False, out=out, workspace=ws, w_kn=kn)
            assert _launches(call) == (2 if one_round else 3), kn      # plan and product; with the reduction
            call()
            if skew and not one_round:                                 # the plan can still help loads of more than a round
                assert tiles > 256 and ops.ffn_plan_info(ws, R, E, K, N, 1)["skinny_tiles"] > 0
            tol = K * 2.0 ** -24 * K ** 0.5 + 2.0 ** -11 * ref.abs()
            assert ((out.float() - ref).abs() <= tol + 1e-6).all()
    finally:
        ops.set_option("few_rows", 1)
