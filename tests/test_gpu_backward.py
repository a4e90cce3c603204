"""GPU parity of the backward stages against the CPU oracle, through the C ABI.

Gradients are fp16 with fp32 accumulation.  Tolerance: max-abs error at most
2e-2 times max(1, largest reference magnitude) (weight gradients sum over an
expert's rows and exceed 1), and mean-rel (mean |err| / mean |ref|) at most 1e-3.
"""
import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu

MAX_ABS, MEAN_REL = 2e-2, 1e-3


def _say(msg):
    print(msg, flush=True)


def _close(got, ref, what):
    got, ref = got.float().cpu(), ref.float()
    bound = MAX_ABS * max(1.0, float(ref.abs().max()))
    err = O.max_abs_err(got, ref)
    assert err <= bound, (what, err, bound)
    if float(ref.abs().mean()) > 1e-6:
        assert O.mean_rel_err(got, ref) <= MEAN_REL, (what, O.mean_rel_err(got, ref))


def _case(T, d, f, E, k, seed, skew=False):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s, sc=1.0: (torch.randn(*s, generator=g) * sc).half()
    p = {"x": r(T, d), "wg": r(E, d, sc=0.05), "bg": r(E, sc=0.05), "w1": r(E, f, d, sc=0.05),
         "b1": r(E, f, sc=0.05), "w2": r(E, d, f, sc=0.05), "b2": r(E, d, sc=0.05)}
    if skew:                                   # most tokens to expert 0, expert 1 empty
        p["bg"][0] += 3.0
        p["bg"][1] -= 50.0
    return p


@pytest.mark.usefixtures("gemm_form")
@pytest.mark.parametrize("T,d,f,E,k,cap,skew,seed", [
    (300, 256, 512, 4, 2, -1, False, 0),
    (512, 512, 256, 8, 2, 100, False, 1),     # capacity drops slots
    (257, 256, 1024, 3, 1, -1, False, 2),
    (64, 256, 256, 16, 2, -1, False, 3),      # every expert far below one K tile of rows
    (700, 256, 512, 4, 2, -1, True, 4),       # one large expert, one empty
    (200, 320, 576, 4, 2, -1, False, 5),      # widths that are no multiple of 256: transposed-weight path, partial tiles
    (1500, 512, 768, 2, 1, -1, False, 6),     # several M tiles per expert
])
@pytest.mark.parametrize("transpose", [0, 1])
def test_ffn_backward_stages(T, d, f, E, k, cap, skew, seed, transpose):
    """transpose=0: input gradients read the stored weight as [K][N], and weight gradients the
    two activation matrices row-major, where the widths allow; transpose=1: always on transposed
    copies."""
    from ccfuser_amd import ops
    ops.set_option("dgrad_transpose", transpose)
    ops.set_option("wgrad_transpose", transpose)
    try:
        _ffn_backward_stages(T, d, f, E, k, cap, skew, seed)
    finally:
        ops.set_option("wgrad_transpose", 0)
        ops.set_option("dgrad_transpose", 0)


@pytest.mark.parametrize("transpose", [0, 1])
def test_ffn_backward_stages_with_split_last_round(transpose):
    """Input gradients with the last, partly filled round of tiles cut along K (forced on a
    short K; by default it takes K >= 4096): 36 M tiles x 8 N tiles on 256 workgroups, in both
    weight forms, against the oracle; and the split path did run (bits differ from unsplit)."""
    from ccfuser_amd import ops
    T, d, f, E, k = 4096, 2048, 2048, 6, 2
    ops.set_option("dgrad_transpose", transpose)
    ops.set_option("split_tail", 4)
    ops.set_option("skinny", 0)               # every row in 256-row tiles: the tile count this test is built on
    try:
        _ffn_backward_stages(T, d, f, E, k, -1, False, 7)
        g = torch.Generator().manual_seed(77)
        n = T * k
        rt = ops.route(torch.randint(0, E, (n,), generator=g).cuda(), E, k, -1)
        gy = torch.randn(n, d, generator=g).half().cuda()
        act = torch.randn(n, f, generator=g).half().cuda()
        w2 = (torch.randn(E, d, f, generator=g) * 0.05).half().cuda()
        ga_split = ops.ffn2_backward(gy, act, rt["dst_row"], rt["offsets"], n, w2)[0]
        ops.set_option("split_tail", 0)
        ga_whole = ops.ffn2_backward(gy, act, rt["dst_row"], rt["offsets"], n, w2)[0]
        assert O.max_abs_err(ga_split.cpu(), ga_whole.float().cpu()) <= MAX_ABS
        assert not torch.equal(ga_split, ga_whole)
    finally:
        ops.set_option("dgrad_transpose", 0)
        ops.set_option("split_tail", 1)
        ops.set_option("skinny", 1)


@pytest.mark.parametrize("T,k,E,seed", [(4096, 2, 8, 0), (300, 3, 64, 1), (1000, 8, 1024, 2), (257, 1, 5, 3), (1, 1, 1, 4)])
def test_gate_backward_of_softmax_and_selection(T, k, E, seed):
    """ccf_gate_backward against the oracle's formula (softmax over the k selected logits
    backwards, scattered into [T, E]; the bias gradient its column sums): the scattered values
    are the fp32 values rounded once, so they must match a float32 evaluation to one fp16 step;
    twice the same bits; and no bias gradient when none is asked for."""
    from ccfuser_amd import ops
    _say(f"gate backward T={T} k={k} E={E}")
    g = torch.Generator().manual_seed(seed)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    score = torch.softmax(torch.randn(T, k, generator=g), dim=-1).half()
    gs = torch.randn(T, k, generator=g).half()
    s32, g32 = score.float(), gs.float()
    g_val = s32 * (g32 - (s32 * g32).sum(-1, keepdim=True))
    ref = torch.zeros(T, E).scatter_add_(1, idx, g_val)
    gl, gb = ops.gate_backward(score.cuda(), gs.cuda(), idx.cuda(), E)
    gl2, gb2 = ops.gate_backward(score.cuda(), gs.cuda(), idx.cuda(), E)
    torch.cuda.synchronize()
    assert torch.equal(gl, gl2) and torch.equal(gb, gb2)
    assert float((gl.cpu().float() - ref).abs().max()) <= 2.0 ** -10 * max(1.0, float(ref.abs().max()))
    _close(gb, ref.sum(0), "grad_bias")
    gl3, none = ops.gate_backward(score.cuda(), gs.cuda(), idx.cuda(), E, want_bias=False)
    assert none is None and torch.equal(gl3, gl)


@pytest.mark.parametrize("T,d,E,k", [(1, 2, 1, 1), (63, 510, 8, 2), (65, 514, 9, 1), (257, 512, 16, 8), (1999, 768, 8, 2),
                                     (5000, 130, 16, 2), (1100, 16386, 5, 3)])
def test_gate_backward_products(T, d, E, k):
    """The gate's input, weight and bias gradients from the k selected experts only, against the dense products in
    fp64: each within one rounding of fp16 plus a fp32 sum; two runs give the same bits."""
    from ccfuser_amd import ops
    g = torch.Generator().manual_seed(T + d)
    x, w = torch.randn(T, d, generator=g).half(), (torch.randn(E, d, generator=g) * 0.1).half()
    idx = torch.rand(T, E, generator=g).topk(k, -1).indices
    score = torch.softmax(torch.randn(T, k, generator=g), -1).half()
    gs = torch.randn(T, k, generator=g).half()
    args = [t.cuda() for t in (score, gs, idx, x, w)]
    got = ops.gate_backward_products(*args)
    again = ops.gate_backward_products(*args)
    only_w = ops.gate_backward_products(*args, want_x=False, want_bias=False)
    torch.cuda.synchronize()
    s, q = score.double(), gs.double()
    val = s * (q - (s * q).sum(-1, keepdim=True))
    dense = torch.zeros(T, E, dtype=torch.float64).scatter_(1, idx, val)
    mag = torch.zeros(T, E, dtype=torch.float64).scatter_(1, idx, s * (q.abs() + (s * q).abs().sum(-1, keepdim=True)))
    # fp16 rounds by half a unit in 2^11 (absolute below 2^-14); a sum of n terms, and the cancellation inside val, by
    # n units in 2^24 of the sum of magnitudes
    for out, ref, terms, n in ((got[0], dense @ w.double(), mag @ w.double().abs(), k),
                               (got[1], dense.t() @ x.double(), mag.t() @ x.double().abs(), T),
                               (got[2], dense.sum(0), mag.sum(0), T)):
        err = (out.cpu().double() - ref).abs()
        bound = ref.abs() * 2.0 ** -11 + 2.0 ** -25 + terms * (min(n, 600) + 8) * 2.0 ** -24
        assert (err <= bound).all(), (err - bound).max()
    for a, b in zip(got, again):
        assert torch.equal(a, b)
    assert only_w[0] is None and only_w[2] is None and torch.equal(only_w[1], got[1])


@pytest.mark.parametrize("mode", [-1, -3, -5, -6, 1])
def test_input_gradient_with_skinny_tiles(mode):
    """The input-gradient GEMM on the stored [K][N] weight with every expert's remainder rows
    (17 .. 64 of them) in 64-row tiles: beside the 256-row tiles (1 or 3 workgroups per XCD),
    cut along K as a launch of their own (-5) or inside the persistent launch (-6), and as the
    plan's cost model chooses (1).  Against fp32 matmuls per expert, and against the call
    without skinny tiles: the same bits where a skinny tile runs over all of K in one piece,
    other bits (so the path did run) where it is cut along K."""
    from ccfuser_amd import ops
    E, d, f = 8, 2048, 2048
    counts = [1024 + 17 + (e * 11) % 48 for e in range(E)]
    n = sum(counts)
    g = torch.Generator().manual_seed(31)
    idx = torch.cat([torch.full((c,), e, dtype=torch.int64) for e, c in enumerate(counts)])
    idx = idx[torch.randperm(n, generator=g)]
    rt = ops.route(idx.cuda(), E, 1, -1)
    assert rt["counts"].cpu().tolist() == counts
    gy = torch.randn(n, d, generator=g).half().cuda()
    act = torch.randn(n, f, generator=g).half().cuda()
    w2 = (torch.randn(E, d, f, generator=g) * 0.05).half().cuda()
    _say(f"input gradient, skinny mode {mode}: {n} rows, counts {counts}")
    # cutting along K (the skinny tiles, and with them the last round of 256-row tiles) is forced on: K = 2048 is
    # below its default threshold; where bits are compared nothing is cut
    ops.set_option("split_tail", 0 if mode in (-1, -3) else 4)
    ops.set_option("skinny_tail", 1 if mode == -5 else 0)
    try:
        ops.set_option("skinny", 0)
        whole = ops.ffn2_backward(gy, act, rt["dst_row"], rt["offsets"], n, w2)[0]
        ops.set_option("skinny", mode)
        got = ops.ffn2_backward(gy, act, rt["dst_row"], rt["offsets"], n, w2)[0]
        torch.cuda.synchronize()
    finally:
        ops.set_option("skinny", 1)
        ops.set_option("split_tail", 1)
        ops.set_option("skinny_tail", 0)
    rows = gy[rt["dst_row"].long()].float()
    off = rt["offsets"].cpu().tolist()
    ref = torch.cat([rows[off[e]:off[e + 1]] @ w2[e].float() for e in range(E)])
    _close(got, ref.cpu(), "grad_act")
    if mode in (-1, -3):
        assert torch.equal(got, whole)
    elif mode in (-5, -6):
        assert not torch.equal(got, whole)
        assert O.max_abs_err(got.float().cpu(), whole.float().cpu()) <= MAX_ABS


def _ffn_backward_stages(T, d, f, E, k, cap, skew, seed):
    from ccfuser_amd import ops
    _say(f"ffn backward T={T} d={d} f={f} E={E} k={k} cap={cap} skew={skew}")
    p = _case(T, d, f, E, k, seed, skew)
    g = torch.Generator().manual_seed(1000 + seed)
    grad_out = torch.randn(T, d, generator=g).half()
    ref = O.moe_layer_backward(p["x"], p["wg"], p["bg"], p["w1"], p["b1"], p["w2"], p["b2"], k,
                               grad_out, capacity=cap)
    pos, offsets = ref["pos"], ref["offsets"]
    n = T * k
    idx_kept = O.limit_by_capacity(ref["idx"], E, cap)
    rt = ops.route(idx_kept.reshape(-1).cuda(), E, k, -1)
    assert torch.equal(rt["offsets"].cpu().long(), offsets.long())

    # combine backward on the fp16-rounded forward values
    y16, s16 = ref["y_flat_fwd"].half(), ref["score_fwd"].half()
    gy_ref, gs_ref = O.combine_backward(grad_out, y16, s16, k)
    kept = (O.inverse_pos(pos, n) >= 0)
    gy_ref = gy_ref * kept[:, None]
    gs_ref = gs_ref.reshape(-1) * kept
    gy, gs = ops.combine_backward(grad_out.cuda(), y16.cuda(), s16.reshape(-1).cuda(), k, rt["inv_pos"])
    _close(gy, gy_ref, "grad_y_flat")
    _close(gs, gs_ref, "grad_score")

    # second GEMM backward
    act16, gy16 = ref["act_fwd"].half(), gy_ref.half()
    a_pad = torch.zeros(n, f, dtype=torch.float16)
    a_pad[: act16.shape[0]] = act16
    ga_ref, gw2_ref, gb2_ref = O.ffn2_backward(gy16, act16, pos, offsets, p["w2"])
    ga, gw2, gb2 = ops.ffn2_backward(gy16.cuda(), a_pad.cuda(), rt["dst_row"], rt["offsets"], n, p["w2"].cuda())
    R = pos.numel()
    _close(ga[:R], ga_ref, "grad_act")
    assert float(ga[R:].abs().max()) == 0.0 if R < n else True
    _close(gw2, gw2_ref, "grad_w2")
    _close(gb2, gb2_ref, "grad_b2")
    # the same call taking the gradient through the GELU: act = gelu(h_pre)
    hp16 = ref["h_pre"].half()
    hp_pad = torch.zeros(n, f, dtype=torch.float16)
    hp_pad[:R] = hp16
    gh_ref = O.gelu_backward(ga_ref, hp16)
    gh_fused, gw2_b, _ = ops.ffn2_backward(gy16.cuda(), a_pad.cuda(), rt["dst_row"], rt["offsets"], n,
                                           p["w2"].cuda(), h_pre=hp_pad.cuda())
    _close(gh_fused[:R], gh_ref, "grad_h through the GELU")
    assert torch.equal(gw2_b, gw2)
    # and the forward that keeps the pre-activation
    act_k, hpre_k = ops.ffn1_keep(p["x"].cuda(), rt["src_row"], rt["offsets"], n, p["w1"].cuda(), p["b1"].cuda())
    _close(hpre_k[:R], ref["h_pre"], "h_pre")
    _close(act_k[:R], ref["act_fwd"], "act")

    # first GEMM backward
    gh16 = ref["h"].half()
    gh_pad = torch.zeros(n, f, dtype=torch.float16)
    gh_pad[:R] = gh16
    gin_ref, gw1_ref, gb1_ref = O.ffn1_backward(gh16, p["x"], pos, k, offsets, p["w1"])
    gx_flat, gw1, gb1 = ops.ffn1_backward(gh_pad.cuda(), p["x"].cuda(), rt["src_row"], rt["dst_row"],
                                          rt["offsets"], n, p["w1"].cuda(), n)
    ones = torch.ones(n, dtype=torch.float16, device="cuda")
    gin = ops.combine(gx_flat, ones, k, rt["inv_pos"])
    _close(gin, gin_ref, "grad_in")
    _close(gw1, gw1_ref, "grad_w1")
    _close(gb1, gb1_ref, "grad_b1")
    # the same through the GELU in one call: grad_act in, multiplied by gelu'(h_pre) in place
    ga_in = torch.zeros(n, f, dtype=torch.float16)
    ga_in[:R] = ga_ref.half()
    gh_want = O.gelu_backward(ga_ref.half(), hp16)                  # what the call must leave in grad_act
    gin_ref2, gw1_ref2, gb1_ref2 = O.ffn1_backward(gh_want.half(), p["x"], pos, k, offsets, p["w1"])
    ga_dev = ga_in.cuda()
    gx2, gw1_2, gb1_2 = ops.ffn1_backward(ga_dev, p["x"].cuda(), rt["src_row"], rt["dst_row"], rt["offsets"], n,
                                          p["w1"].cuda(), n, h_pre=hp_pad.cuda())
    _close(ga_dev[:R], gh_want, "grad_h left in place")
    _close(ops.combine(gx2, ones, k, rt["inv_pos"]), gin_ref2, "grad_in through the GELU")
    _close(gw1_2, gw1_ref2, "grad_w1 through the GELU")
    _close(gb1_2, gb1_ref2, "grad_b1 through the GELU")


@pytest.mark.usefixtures("gemm_form")
@pytest.mark.parametrize("T,d,f,E,k,cf,seed", [
    (384, 256, 512, 4, 2, None, 10),
    (512, 256, 512, 8, 2, 1.0, 11),          # capacity factor 1.0 drops slots
    (200, 512, 256, 4, 1, None, 12),
])
def test_module_backward_matches_oracle(T, d, f, E, k, cf, seed):
    """loss = <out, grad_out> through MixMOETransformerMLP (gate, two expert GEMMs with
    torch's GELU between them, combine) against the oracle's closed-form gradients."""
    from ccfuser_amd.mix_moe import MixMOETransformerMLP
    _say(f"module backward T={T} d={d} f={f} E={E} k={k} cf={cf}")
    p = _case(T, d, f, E, k, seed)
    g = torch.Generator().manual_seed(2000 + seed)
    grad_out = torch.randn(T, d, generator=g).half()
    mlp = MixMOETransformerMLP("naive", {"num_local_expert": E, "hidden_size": f}, d, 0, 1,
                               total_batch_size=T, top_k=k, capacity_factor=cf).half().cuda()
    with torch.no_grad():
        mlp.gate.gate.weight.copy_(p["wg"]); mlp.gate.gate.bias.copy_(p["bg"])
        mlp.experts.htoh4.weight[:E].copy_(p["w1"]); mlp.experts.htoh4.bias[:E].copy_(p["b1"])
        mlp.experts.h4toh.weight[:E].copy_(p["w2"]); mlp.experts.h4toh.bias[:E].copy_(p["b2"])
    x = p["x"].cuda().requires_grad_(True)
    out = mlp(x)
    out.backward(grad_out.cuda())
    cap = mlp._capacity(T)
    ref = O.moe_layer_backward(p["x"], p["wg"], p["bg"], p["w1"], p["b1"], p["w2"], p["b2"], k,
                               grad_out, capacity=cap)
    fwd = O.moe_layer_forward(p["x"], p["wg"], p["bg"], p["w1"], p["b1"], p["w2"], p["b2"], k, capacity=cap)
    assert O.max_abs_err(out.detach().cpu(), fwd["out"]) <= MAX_ABS
    _close(x.grad, ref["x"], "grad_x")
    _close(mlp.gate.gate.weight.grad, ref["wg"], "grad_wg")
    _close(mlp.gate.gate.bias.grad, ref["bg"], "grad_bg")
    _close(mlp.experts.htoh4.weight.grad[:E], ref["w1"], "grad_w1")
    _close(mlp.experts.htoh4.bias.grad[:E], ref["b1"], "grad_b1")
    _close(mlp.experts.h4toh.weight.grad[:E], ref["w2"], "grad_w2")
    _close(mlp.experts.h4toh.bias.grad[:E], ref["b2"], "grad_b2")
    assert float(mlp.experts.htoh4.weight.grad[E:].abs().max()) == 0.0     # slots of no expert
    # the path overlapped with a side stream differentiates the same way
    mlp.zero_grad()
    x2 = p["x"].cuda().requires_grad_(True)
    mlp.async_expert_assignment(x2)
    mlp(x2).backward(grad_out.cuda())
    _close(x2.grad, ref["x"], "grad_x (async)")
    _close(mlp.experts.h4toh.weight.grad[:E], ref["w2"], "grad_w2 (async)")
    # the reference's three steps (linear, torch GELU, linear) give the same gradients
    mlp.zero_grad()
    mlp.experts.fuse_training = False
    x3 = p["x"].cuda().requires_grad_(True)
    mlp(x3).backward(grad_out.cuda())
    _close(x3.grad, ref["x"], "grad_x (unfused)")
    _close(mlp.experts.htoh4.weight.grad[:E], ref["w1"], "grad_w1 (unfused)")
    _close(mlp.experts.htoh4.bias.grad[:E], ref["b1"], "grad_b1 (unfused)")
    mlp.close()


@pytest.mark.parametrize("name", ["c3_mixtral", "c5_skewed"])
def test_full_size_backward_properties(workloads, name):
    """At BASELINE sizes the oracle's weight gradients are too slow for a unit test, so
    check what does not depend on size: sampled entries of every gradient against their
    defining sums in float64, the bias gradients against column sums over each expert's
    rows, and linearity (doubling the incoming gradient doubles the weight gradient)."""
    from ccfuser_amd import ops
    wl = workloads(name)
    t = wl.tensors
    T, d, f, E, k = wl.tokens, wl.d_model, wl.d_ffn, wl.num_expert, wl.top_k
    _say(f"full size backward {name}")
    idx, _, _ = O.naive_gate(t["x"], t["wg"], t["bg"], k)
    pos, offsets = O.assign_pos(idx, E)
    off = offsets.tolist()
    n = T * k
    rt = ops.route(idx.reshape(-1).cuda(), E, k, -1)
    g = torch.Generator().manual_seed(77)
    gy = (torch.randn(n, d, generator=g) * 0.5).half()
    act = (torch.randn(n, f, generator=g) * 0.5).half()
    gh = (torch.randn(n, f, generator=g) * 0.5).half()
    w1, w2, x = t["w1"].half(), t["w2"].half(), t["x"].half()
    ga, gw2, gb2 = ops.ffn2_backward(gy.cuda(), act.cuda(), rt["dst_row"], rt["offsets"], n, w2.cuda())
    gx, gw1, gb1 = ops.ffn1_backward(gh.cuda(), x.cuda(), rt["src_row"], rt["dst_row"], rt["offsets"], n,
                                     w1.cuda(), n)
    torch.cuda.synchronize()
    ga, gw2, gb2, gx, gw1, gb1 = (v.cpu() for v in (ga, gw2, gb2, gx, gw1, gb1))
    for v in (ga, gw2, gb2, gx, gw1, gb1):
        assert torch.isfinite(v.float()).all()
    gy_sorted = gy[pos].double()                       # gradient rows in expert order
    src = torch.div(pos, k, rounding_mode="floor")
    expert_of = torch.bucketize(torch.arange(n), offsets[1:].long(), right=True)
    rnd = lambda hi: int(torch.randint(0, hi, (1,), generator=g))
    tol = lambda ref: MAX_ABS * max(1.0, abs(ref))
    for _ in range(24):
        e = rnd(E)
        lo, hi = off[e], off[e + 1]
        m, c = rnd(d), rnd(f)
        ref = float((gy_sorted[lo:hi, m] * act[lo:hi, c].double()).sum())       # grad_w2[e, m, c]
        assert abs(float(gw2[e, m, c]) - ref) <= tol(ref), ("gw2", e, m, c)
        ref = float((gh[lo:hi, c].double() * x[src[lo:hi], m].double()).sum())  # grad_w1[e, c, m]
        assert abs(float(gw1[e, c, m]) - ref) <= tol(ref), ("gw1", e, c, m)
        j = rnd(n)
        ej = int(expert_of[j])
        ref = float((gy_sorted[j] * w2[ej, :, c].double()).sum())               # grad_act[j, c]
        assert abs(float(ga[j, c]) - ref) <= tol(ref), ("ga", j, c)
        ref = float((gh[j].double() * w1[ej, :, m].double()).sum())             # grad of sorted row j, column m
        assert abs(float(gx[int(pos[j]), m]) - ref) <= tol(ref), ("gx", j, m)
    for e in range(E):
        lo, hi = off[e], off[e + 1]
        _close(gb2[e], gy_sorted[lo:hi].sum(0).float(), "grad_b2")
        _close(gb1[e], gh[lo:hi].double().sum(0).float(), "grad_b1")
    _, gw2_twice, _ = ops.ffn2_backward((gy * 2).cuda(), act.cuda(), rt["dst_row"], rt["offsets"], n, w2.cuda())
    _close(gw2_twice, gw2.float() * 2, "linearity of grad_w2")
    # no atomics anywhere: a second run gives the same bits
    _, gw2_again, gb2_again = ops.ffn2_backward(gy.cuda(), act.cuda(), rt["dst_row"], rt["offsets"], n, w2.cuda())
    assert torch.equal(gw2_again.cpu(), gw2) and torch.equal(gb2_again.cpu(), gb2)


def test_backward_without_rows():
    """No routed rows (every slot dropped): parameter gradients are zero, not left unwritten."""
    from ccfuser_amd import ops
    E, d, f = 4, 256, 512
    w1 = torch.randn(E, f, d).half().cuda()
    w2 = torch.randn(E, d, f).half().cuda()
    offsets = torch.zeros(E + 1, dtype=torch.int32, device="cuda")
    empty_f = torch.empty(0, f, dtype=torch.float16, device="cuda")
    empty_d = torch.empty(0, d, dtype=torch.float16, device="cuda")
    gw2 = torch.full_like(w2, 7.0)
    gb2 = torch.full((E, d), 7.0, dtype=torch.float16, device="cuda")
    ga, _, _ = ops.ffn2_backward(empty_d, empty_f, None, offsets, 0, w2, gw2, gb2)
    assert ga.shape == (0, f) and float(gw2.abs().max()) == 0.0 and float(gb2.abs().max()) == 0.0
    gw1 = torch.full_like(w1, 7.0)
    gb1 = torch.full((E, f), 7.0, dtype=torch.float16, device="cuda")
    gx, _, _ = ops.ffn1_backward(empty_f, empty_d, None, None, offsets, 0, w1, 0, gw1, gb1)
    assert gx.shape == (0, d) and float(gw1.abs().max()) == 0.0 and float(gb1.abs().max()) == 0.0


@pytest.mark.parametrize("E,d,f", [(3, 4160, 64), (70, 64, 512), (3, 64, 4160)])
def test_backward_without_rows_of_a_long_contraction(E, d, f):
    """No rows at sizes where the form of the input-gradient GEMM, or a cut along K, is decided by an estimate."""
    from ccfuser_amd import ops
    offsets = torch.zeros(E + 1, dtype=torch.int32, device="cuda")
    empty = lambda n: torch.empty(0, n, dtype=torch.float16, device="cuda")
    w2 = torch.ones(E, d, f, dtype=torch.float16, device="cuda")
    ga, gw, gb = ops.ffn2_backward(empty(d), empty(f), None, offsets, 0, w2)
    assert ga.shape == (0, f) and not gw.any() and not gb.any()
    w1 = torch.ones(E, f, d, dtype=torch.float16, device="cuda")
    gx, gw, gb = ops.ffn1_backward(empty(f), empty(d), None, None, offsets, 0, w1, 0)
    assert gx.shape == (0, d) and not gw.any() and not gb.any()


def _random_shapes(count, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda lo, hi: int(torch.randint(lo, hi + 1, (1,), generator=g))
    out = []
    for i in range(count):
        E = r(1, 9)
        out.append((r(1, 600), 64 * r(1, 10), 64 * r(1, 10), E, min(r(1, 3), E), [-1, -1, r(0, 200)][r(0, 2)], 100 + i))
    return out


@pytest.mark.usefixtures("gemm_form")
@pytest.mark.parametrize("T,d,f,E,k,cap,seed", _random_shapes(10, 4242))
def test_ffn_backward_random_shapes(T, d, f, E, k, cap, seed):
    """Widths from 64 to 640 in steps of 64 (one K tile, partial M and N tiles, both weight
    forms), 1 to 600 tokens, 1 to 9 experts, top-1 to top-3, with and without capacity."""
    _ffn_backward_stages(T, d, f, E, k, cap, False, seed)


@pytest.mark.parametrize("E,first,shape", [(5, 2, (8,)), (3, 3, (16, 8)), (4, 0, (24, 40)), (11, 8, (768, 64))])
def test_zero_tails(E, first, shape):
    from ccfuser_amd import ops
    a, b = torch.ones(E, *shape, dtype=torch.float16, device="cuda"), torch.ones(E, shape[0], dtype=torch.float16, device="cuda")
    ops.zero_tails(a, b, first)
    for t in (a, b):
        assert (t[:first] == 1).all() and (t[first:] == 0).all()


@pytest.mark.usefixtures("gemm_form")
@pytest.mark.parametrize("T,k,d,f,E,slots,capacity", [
    (700, 2, 256, 512, 4, 7, -1),           # both weight gradients in one launch, fewer tiles than compute units
    (700, 2, 512, 256, 4, 4, 90),           # wider input, dropped slots, no unused slot
    (1999, 2, 768, 3072, 8, 11, -1),        # more than one round of tiles
    (33, 1, 256, 256, 16, 19, -1),          # experts without rows, square widths
    (1, 2, 256, 256, 3, 6, -1),
    (300, 3, 256, 768, 1, 2, -1),           # one expert, three slots a token
    (300, 2, 320, 704, 4, 7, 100),          # widths that are no multiples of 256: the layers one after the other
    (70, 2, 256, 256, 520, 521, -1),        # more experts than one plan holds twice
    (70, 2, 256, 256, 512, 513, -1),        # as many as it holds
])
def test_backward_of_both_layers_in_one_call(T, k, d, f, E, slots, capacity):
    """Gradients of both expert layers from one call: the bits of the two layers' own calls and the sum over a token's
    slots, unused slots zero."""
    from ccfuser_amd import ops
    print(f"backward pair T={T} k={k} d={d} f={f} E={E} slots={slots} capacity={capacity}", flush=True)
    g = torch.Generator().manual_seed(T + d)
    rnd = lambda *s: (torch.randn(*s, generator=g) * 0.1).half().cuda()
    k_eff = min(k, E)
    idx = torch.rand(T, E, generator=g).topk(k_eff, dim=-1).indices
    if k_eff < k:
        idx = idx.repeat(1, k)[:, :k]
    r = ops.route(idx.reshape(-1).contiguous().cuda(), E, k, capacity)
    n = T * k
    x, gy = rnd(T, d), rnd(n, d)
    w1, b1, w2 = rnd(slots, f, d), rnd(slots, f), rnd(slots, d, f)
    act, pre = ops.ffn1_keep(x, r["src_row"], r["offsets"], n, w1[:E], b1[:E])
    torch.full((slots, f, d), float("nan"), dtype=torch.float16, device="cuda")          # freed at once
    got = ops.ffn_backward_pair(gy, x, act, pre, r["src_row"], r["dst_row"], r["inv_pos"], r["offsets"], w1, w2)
    ga, gw2, gb2 = ops.ffn2_backward(gy, act, r["dst_row"], r["offsets"], n, w2[:E])
    gf, gw1, gb1 = ops.ffn1_backward(ga, x, r["src_row"], r["dst_row"], r["offsets"], n, w1[:E], n, h_pre=pre)
    gx = ops.combine(gf, torch.ones(n, dtype=torch.float16, device="cuda"), k, r["inv_pos"])
    for name, a, b in zip(("x", "w1", "b1", "w2", "b2"), got, (gx, gw1, gb1, gw2, gb2)):
        tail = a[b.shape[0]:]
        assert torch.equal(a[:b.shape[0]], b), name
        assert torch.equal(tail, torch.zeros_like(tail)), name


def test_backward_with_parameters_that_are_contiguous_only_as_slices():
    """One expert of three slots that lie apart in memory: the layers' own calls on the slice, the gradients of the
    contiguous parameter."""
    from ccfuser_amd.mix_moe import MixMOETransformerMLP
    d, f, T = 256, 512, 100
    grads = []
    for apart in (False, True):
        torch.manual_seed(0)
        with torch.device("cuda"):
            mlp = MixMOETransformerMLP("naive", {"num_local_expert": 1, "hidden_size": f}, d, 0, 1, total_batch_size=T, top_k=1,
                                       popular_expert_num=2).half()
        if apart:
            for lin in (mlp.experts.htoh4, mlp.experts.h4toh):
                wide = torch.empty(3, 2, *lin.weight.shape[1:], dtype=torch.float16, device="cuda")
                wide[:, 0] = lin.weight.detach()
                lin.weight = torch.nn.Parameter(wide[:, 0])
            assert not mlp.experts.htoh4.weight.is_contiguous()
        x = torch.randn(T, d, dtype=torch.float16, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).requires_grad_(True)
        mlp(x).backward(torch.ones(T, d, dtype=torch.float16, device="cuda"))
        grads.append({"x": x.grad, **{n: p.grad[:1] for n, p in mlp.named_parameters() if n.startswith("experts")}})
    for name, g in grads[0].items():
        assert torch.equal(g, grads[1][name]), name
