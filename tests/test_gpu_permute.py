"""GPU parity of the permute path: HIP kernels (through the C ABI via the
drop-in wrappers) against the C/torch oracle on the same seeded inputs.

Bar: bit-exact for the row map, group sizes, permuted payload bytes, permuted
probs, permute_kv_and_lrs outputs and the unpermute (fp32 fma accumulation in
slot order, one rounding); fp32 rtol/atol 1e-5 for the backward reductions
whose summation order the reference leaves to the compiler.
"""
import pytest
import torch

from oracle import permute as OP
from tests.helpers import load_golden, routing_c2, topk_mask_like_reference_test
from uttt_amd.lact_moe_triton import triton_permute as TP

pytestmark = pytest.mark.gpu
DEV = "cuda"


def bits(t):
    t = t.detach().cpu()
    return t.view(torch.int16) if t.element_size() == 2 else t.view(torch.int32)


def test_row_id_map_kat_on_gpu():
    kat = load_golden("row_id_map_kat.json")
    m = torch.tensor(kat["routing_map_token_major"], dtype=torch.int32).t().unsqueeze(0)
    rm = TP.make_row_id_map(m.to(DEV), 1, 5, 3).cpu()
    assert rm[0].tolist() == kat["expected_full"]


@pytest.mark.parametrize(
    "B,T,E,k,mask_dtype,ragged",
    [
        (1, 65536, 16, 2, torch.bool, False),   # the permute microbench shape
        (2, 4097, 32, 2, torch.int32, True),
        (3, 255, 7, 3, torch.bool, True),
        (1, 1, 1, 1, torch.bool, False),
        (1, 1000, 128, 4, torch.int32, True),
        (2, 300, 5, 5, torch.bool, False),      # every expert selected
        # one-launch row map (contiguous bool mask, T % 16 == 0, T <= 4096, E <= 64)
        (1, 2048, 32, 2, torch.bool, False),    # one apply's routing at the 760M shape
        (2, 2048, 32, 2, torch.bool, True),
        (1, 2048, 16, 2, torch.bool, True),     # the 124M shape
        (2, 4096, 64, 3, torch.bool, True),     # largest one-launch case: 16 tiles, E = 64
        (1, 1040, 7, 2, torch.bool, True),      # partial last tile and 64-token segment
        (1, 16, 3, 1, torch.bool, False),
        (1, 4096, 65, 2, torch.bool, False),    # E = 65 and T = 4112 take the three launches
        (1, 4112, 8, 2, torch.bool, True),
        # expert counts below their kernel's compile-time bucket
        (1, 2048, 20, 2, torch.bool, True),     # one launch, 32-expert bucket
        (1, 4096, 40, 3, torch.bool, True),     # one launch, 64-expert bucket
        (2, 5000, 20, 2, torch.bool, True),     # two launches, count rows padded to 32
        (1, 70000, 24, 4, torch.int32, False),  # two launches, E = 24, two count-table chunks
    ],
)
def test_row_id_map_bit_exact(B, T, E, k, mask_dtype, ragged):
    g = torch.Generator().manual_seed(B + T + E)
    scores = torch.rand(B, E, T, generator=g)
    m = torch.zeros(B, E, T, dtype=torch.int32).scatter_(1, scores.topk(k, 1).indices, 1)
    if ragged:
        m = m * (torch.rand(B, E, T, generator=g) > 0.3).to(torch.int32)
        m[:, E // 2] = 0  # an empty expert
    gs = torch.empty(B, E, dtype=torch.int32, device=DEV)
    rm = TP.make_row_id_map(m.to(mask_dtype).to(DEV), B, T, E, group_sizes=gs)
    ref = OP.make_row_id_map(m)
    assert torch.equal(rm.cpu(), ref)
    assert torch.equal(gs.cpu(), m.sum(-1).to(torch.int32))


def test_row_id_map_strided_mask():
    # a [B, T, E] tensor viewed as [B, E, T]: the kernel honours strides
    g = torch.Generator().manual_seed(3)
    B, T, E = 2, 1500, 12
    m = torch.zeros(B, T, E, dtype=torch.int32).scatter_(2, torch.rand(B, T, E, generator=g).topk(2, 2).indices, 1)
    view = m.to(DEV).transpose(1, 2)
    assert not view.is_contiguous()
    rm = TP.make_row_id_map(view, B, T, E)
    assert torch.equal(rm.cpu(), OP.make_row_id_map(m.transpose(1, 2).contiguous()))


def test_row_id_map_deterministic():
    _, _, mask, _, _ = routing_c2(T=65536, E=16, k=2, seed=1)
    md = mask.to(DEV)
    a = TP.make_row_id_map(md, 1, 65536, 16)
    b = TP.make_row_id_map(md, 1, 65536, 16)
    assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,H", [(torch.bfloat16, 768), (torch.float32, 16), (torch.bfloat16, 900), (torch.float16, 130)])
def test_permute_fwd_bit_exact(dtype, H):
    T, E, k = (65536, 16, 2) if H == 768 else (2000, 6, 2)
    _, _, mask, gs, comb = routing_c2(T=T, E=E, k=k, seed=2)
    comb = comb.clone()
    comb[0, :, 5] = 0.0  # padding slots -> zero rows
    g = torch.Generator().manual_seed(7)
    x = torch.randn(1, T, H, generator=g).to(dtype)
    out, pp, rm = TP.permute_with_expert_mask(x.to(DEV), mask.to(DEV), comb.to(DEV), k)
    ref_rm = OP.make_row_id_map(mask)
    assert torch.equal(rm.cpu(), ref_rm)
    ref_out, ref_pp = OP.permute(x, ref_rm, comb, k * T)
    wr = OP.written_rows(ref_rm, k * T)
    assert torch.equal(bits(out)[wr], bits(ref_out)[wr])
    assert torch.equal(pp.cpu()[wr], ref_pp[wr])


def test_permute_without_probs_and_few_slots():
    # the reference test's mask keeps k-1 experts: tail rows stay unwritten
    g = torch.Generator().manual_seed(321)
    B, T, E, H, k = 2, 32, 4, 16, 2
    mask = topk_mask_like_reference_test(B, T, E, k, g)
    x = torch.randn(B, T, H, generator=g)
    out, pp, rm = TP.permute_with_expert_mask(x.to(DEV), mask.to(DEV), None, k)
    assert pp is None
    ref_rm = OP.make_row_id_map(mask)
    ref_out, _ = OP.permute(x, ref_rm, None, k * T)
    wr = OP.written_rows(ref_rm, k * T)
    assert torch.equal(out.cpu()[wr], ref_out[wr])


def test_unpermute_reference_invariant():
    # uttt_nvs/tests/test_triton_permute.py:32-53 on our kernels
    g = torch.Generator().manual_seed(321)
    B, T, E, H, k = 2, 32, 4, 16, 2
    mask = topk_mask_like_reference_test(B, T, E, k, g)
    x = torch.randn(B, T, H, generator=g)
    probs = torch.rand(B, E, T, generator=g) * mask
    xp, _, rm = TP.permute_with_expert_mask(x.to(DEV), mask.to(DEV), probs.to(DEV), k)
    merged = TP.unpermute_and_merge_with_probs(xp, rm, probs.to(DEV))
    ref = x * (probs * mask).sum(dim=1).unsqueeze(-1)
    torch.testing.assert_close(merged.cpu(), ref, atol=1e-3, rtol=1e-3)


@pytest.mark.parametrize("dtype,H,T,E", [(torch.bfloat16, 768, 65536, 16), (torch.float32, 48, 3000, 9)])
def test_unpermute_fwd_bit_exact(dtype, H, T, E):
    k = 2
    _, _, mask, gs, comb = routing_c2(T=T, E=E, k=k, seed=4)
    g = torch.Generator().manual_seed(9)
    rm = OP.make_row_id_map(mask)
    y = torch.randn(1, k * T, H, generator=g).to(dtype)
    out = TP.unpermute_and_merge_with_probs(y.to(DEV), rm.to(DEV), comb.to(DEV))
    ref = OP.unpermute(y, rm, comb, T)
    assert torch.equal(bits(out), bits(ref))


@pytest.mark.parametrize("dtype,H", [(torch.bfloat16, 256), (torch.float32, 36)])
def test_permute_unpermute_topk4_ragged(dtype, H):
    # top-4 with dropped slots: slots past the first two take the kernels'
    # general loop, tokens with 0..4 slots mix within one wave
    B, T, E, k = 2, 1537, 12, 4
    g = torch.Generator().manual_seed(17)
    scores = torch.rand(B, E, T, generator=g)
    mask = torch.zeros(B, E, T, dtype=torch.bool).scatter_(1, scores.topk(k, 1).indices, True)
    mask &= torch.rand(B, E, T, generator=g) > 0.25
    probs = torch.rand(B, E, T, generator=g) * mask
    probs[:, :, 3] = 0.0  # a token whose every gate is zero
    x = torch.randn(B, T, H, generator=g).to(dtype)
    out, pp, rm = TP.permute_with_expert_mask(x.to(DEV), mask.to(DEV), probs.to(DEV), k)
    ref_rm = OP.make_row_id_map(mask)
    assert torch.equal(rm.cpu(), ref_rm)
    ref_out, ref_pp = OP.permute(x, ref_rm, probs, k * T)
    wr = OP.written_rows(ref_rm, k * T)
    assert torch.equal(bits(out)[wr], bits(ref_out)[wr])
    assert torch.equal(pp.cpu()[wr], ref_pp[wr])
    y = torch.randn(B, k * T, H, generator=g).to(dtype)
    merged = TP.unpermute_and_merge_with_probs(y.to(DEV), rm, probs.to(DEV))
    assert torch.equal(bits(merged), bits(OP.unpermute(y, ref_rm, probs, T)))


def test_unpermute_strided_probs():
    # probs given as a [B, T, E] tensor viewed [B, E, T] (P:835-839)
    T, E, H, k = 1000, 8, 64, 2
    _, _, mask, _, comb = routing_c2(T=T, E=E, k=k, seed=5)
    g = torch.Generator().manual_seed(10)
    rm = OP.make_row_id_map(mask)
    y = torch.randn(1, k * T, H, generator=g).to(torch.bfloat16)
    pv = comb.transpose(1, 2).contiguous().to(DEV).transpose(1, 2)
    out = TP.unpermute_and_merge_with_probs(y.to(DEV), rm.to(DEV), pv)
    assert torch.equal(bits(out), bits(OP.unpermute(y, rm, comb, T)))


def test_permute_unpermute_backward():
    T, E, H, k = 3000, 8, 96, 2
    _, _, mask, _, comb = routing_c2(T=T, E=E, k=k, seed=6)
    g = torch.Generator().manual_seed(11)
    x = torch.randn(1, T, H, generator=g)
    xd = x.to(DEV).requires_grad_(True)
    pd = comb.to(DEV).requires_grad_(True)
    xp, pp, rm = TP.permute_with_expert_mask(xd, mask.to(DEV), pd, k)
    gy = torch.randn(1, k * T, H, generator=g)
    gpp = torch.randn(1, k * T, generator=g)
    (xp * gy.to(DEV)).sum().add((pp * gpp.to(DEV)).sum()).backward()
    rm_c = rm.cpu()
    gi, gp = OP.permute_bwd(gy, rm_c, gpp, T)
    torch.testing.assert_close(xd.grad.cpu(), gi, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(pd.grad.cpu(), gp, rtol=1e-5, atol=1e-5)

    y = torch.randn(1, k * T, H, generator=g)
    yd = y.to(DEV).requires_grad_(True)
    pd2 = comb.to(DEV).requires_grad_(True)
    out = TP.unpermute_and_merge_with_probs(yd, rm, pd2)
    go = torch.randn(1, T, H, generator=g)
    (out * go.to(DEV)).sum().backward()
    ag, gp2 = OP.unpermute_bwd(go, rm_c, y, comb)
    wr = OP.written_rows(rm_c, k * T)
    torch.testing.assert_close(yd.grad.cpu()[wr], ag[wr], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(pd2.grad.cpu(), gp2, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("kd,vd,lrd,H,T,E", [
    (torch.bfloat16, torch.bfloat16, torch.bfloat16, 768, 2048, 16),
    (torch.bfloat16, torch.float32, torch.float32, 1536, 2048, 32),
    (torch.float32, torch.float32, torch.float32, 50, 777, 5),
])
def test_permute_kv_and_lrs_bit_exact(kd, vd, lrd, H, T, E):
    k = 2
    _, _, mask, _, comb = routing_c2(T=T, E=E, k=k, seed=8)
    g = torch.Generator().manual_seed(12)
    kx = torch.randn(1, T, H, generator=g).to(kd)
    vx = torch.randn(1, T, H, generator=g).to(vd)
    lrs = [torch.sigmoid(torch.randn(1, T, generator=g)).mul(0.1).to(lrd) for _ in range(3)]
    outs = TP.permute_kv_and_lrs(kx.to(DEV), vx.to(DEV), *(l.to(DEV) for l in lrs),
                                 mask.to(torch.int32).to(DEV), comb.to(DEV), k)
    rm = OP.make_row_id_map(mask)
    refs = OP.permute_kv_lrs(kx, vx, *lrs, rm, comb, k * T)
    wr = OP.written_rows(rm, k * T)
    for o, r in zip(outs, refs):
        assert torch.equal(bits(o)[wr], bits(r)[wr])


def test_permute_kv_and_lrs_3d_lr_and_backward():
    T, E, H, k = 1500, 8, 64, 2
    _, _, mask, _, comb = routing_c2(T=T, E=E, k=k, seed=9)
    comb = comb.clone()
    comb[0, :, 11] = 0.0
    g = torch.Generator().manual_seed(13)
    kx = torch.randn(1, T, H, generator=g)
    vx = torch.randn(1, T, H, generator=g)
    lrs = [torch.rand(1, T, 1, generator=g) for _ in range(3)]
    kd, vd = kx.to(DEV).requires_grad_(True), vx.to(DEV).requires_grad_(True)
    lds = [l.to(DEV).requires_grad_(True) for l in lrs]
    pd = comb.to(DEV).requires_grad_(True)
    outs = TP.permute_kv_and_lrs(kd, vd, *lds, mask.to(DEV), pd, k)
    assert outs[2].shape == (1, k * T)
    grads = [torch.randn(o.shape, generator=g) for o in outs]
    sum((o * gg.to(DEV)).sum() for o, gg in zip(outs, grads)).backward()
    rm = OP.make_row_id_map(mask)
    grad_k, grad_v, grad_lr, gp = OP.permute_kv_lrs_bwd(grads[0], grads[1], grads[2:], rm, vx, comb, T)
    torch.testing.assert_close(kd.grad.cpu(), grad_k, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(vd.grad.cpu(), grad_v, rtol=1e-5, atol=1e-5)
    for ld, gr in zip(lds, grad_lr):
        assert ld.grad.shape == (1, T, 1)
        torch.testing.assert_close(ld.grad.cpu().squeeze(-1), gr, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(pd.grad.cpu(), gp, rtol=1e-5, atol=1e-4)


def test_permute_roundtrip_full_size_property():
    # full-size property check: unpermute(permute(x)) with unit-sum gates
    # reproduces x up to one bf16 rounding of sum_j x*p_j
    T, E, k, H = 65536, 16, 2, 768
    _, _, mask, _, comb = routing_c2(T=T, E=E, k=k, seed=10)
    g = torch.Generator().manual_seed(14)
    x = torch.randn(1, T, H, generator=g).to(torch.bfloat16).to(DEV)
    xp, _, rm = TP.permute_with_expert_mask(x, mask.to(DEV), comb.to(DEV), k)
    back = TP.unpermute_and_merge_with_probs(xp, rm, comb.to(DEV))
    torch.testing.assert_close(back.float(), x.float(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("T,E", [(1, 25), (9, 128), (63, 64), (64, 65), (65, 128), (129, 33),
                                 (512, 65), (513, 65), (4112, 48), (5000, 96), (32904, 30),
                                 (70001, 27)])
@pytest.mark.parametrize("form", ["bool", "uint8_values", "int32", "token_major"])
def test_row_map_from_64_token_tiles(T, E, form):
    """The general row map (E > 24, or too many tokens for one launch): every
    mask form it accepts, tokens with none to all experts, experts with no
    token; bit-exact, with the group sizes."""
    B = 2
    g = torch.Generator().manual_seed(T * 131 + E)
    n = torch.randint(0, 4, (B, 1, T), generator=g)
    if T > 2:
        n[:, :, 1] = E                                   # a token with every expert
    rank = torch.rand(B, E, T, generator=g).argsort(1).argsort(1)
    mask = rank < n
    mask[1, E // 2] = False
    ref = OP.make_row_id_map(mask)
    if form == "bool":
        m = mask.to(DEV)
    elif form == "uint8_values":
        m = (mask.to(torch.uint8) * torch.randint(1, 256, mask.shape, generator=g).to(torch.uint8)).to(DEV)
    elif form == "int32":
        m = (mask.to(torch.int32) * 256).to(DEV)
    else:
        m = mask.to(DEV).transpose(1, 2).contiguous().transpose(1, 2)
    gs = torch.empty(B, E, dtype=torch.int32, device=DEV)
    rm = TP.make_row_id_map(m, B, T, E, group_sizes=gs)
    assert torch.equal(rm.cpu(), ref)
    assert torch.equal(gs.cpu(), mask.sum(-1).to(torch.int32))


LANE_SIZES = [(B, T, E, k, H) for H in (8, 24, 192, 200, 384, 520, 768, 2048, 2056)
              for B, T, E, k in ((1, 1, 1, 1), (2, 65, 128, 4), (1, 700, 16, 2))] + [
    # token counts past which the lane groups take narrow rows, more slots and wide rows
    (1, 2049, 16, 2, 24), (2, 1030, 16, 2, 1024), (1, 4100, 48, 4, 264), (1, 8200, 9, 3, 136),
    (1, 16400, 9, 2, 1536), (1, 32775, 6, 2, 1032),
    # many short batches: waves past the end, full and nearly full 64s, 17 to 19 tokens
    (600, 9, 8, 6, 192), (300, 17, 6, 4, 520), (300, 17, 6, 4, 264), (300, 20, 6, 4, 1024),
    (512, 60, 8, 3, 24), (514, 51, 3, 3, 136)]


@pytest.mark.parametrize("B,T,E,k,H", LANE_SIZES)
def test_grouped_lane_kernels_of_16_bit_rows(B, T, E, k, H):
    """The 16-bit backward kernels and the k / v / lr permute at the edges of
    their lane groups (and past them: H = 2056), tokens with none to k + 1
    experts, gates of zero, rows past num_out.  k / v / lr outputs bit-exact.
    Backward: fp32 sums of the same bf16 values in slot order, one bf16 rounding
    (2^-8 relative); dot products in another order: H * 2^-24 of sum |x||y|."""
    g = torch.Generator().manual_seed(H + T)
    n = torch.randint(0, k + 2, (B, 1, T), generator=g).clamp(max=E)
    mask = torch.rand(B, E, T, generator=g).argsort(1).argsort(1) < n
    probs = torch.rand(B, E, T, generator=g) * mask
    probs[:, :, T // 2] = 0.0
    N = k * T
    rm = OP.make_row_id_map(mask)
    wr = OP.written_rows(rm, N)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    kx, vx, go, y = bf(B, T, H), bf(B, T, H), bf(B, T, H), bf(B, N, H)
    lrs = [torch.rand(B, T, generator=g).to(torch.bfloat16) for _ in range(3)]
    # rows past num_out stay unwritten, their slots absent
    refs = OP.permute_kv_lrs(kx, vx, *lrs, rm, probs, N)
    ins = [t.to(DEV).requires_grad_() for t in (kx, vx, *lrs, probs)]
    outs = TP.permute_kv_and_lrs(*ins[:5], mask.to(DEV), ins[5], k)
    for o, r in zip(outs, refs):
        assert torch.equal(bits(o)[wr], bits(r)[wr])
    gk, gv = bf(B, N, H), bf(B, N, H)
    gl = [torch.randn(B, N, generator=g).to(torch.bfloat16) for _ in range(3)]
    grads = torch.autograd.grad(outs, ins, [t.to(DEV).view(o.shape) for t, o in zip((gk, gv, *gl), outs)])
    close = lambda a, r: bool(((a.cpu().double() - r).abs() <= 2.0 ** -8 * r.abs() + 1e-5).all())
    slots = [(b, t, int(rm[b, t, j]), int(rm[b, t, E + j])) for b in range(B) for t in range(T)
             for j in range(int(rm[b, t, 2 * E])) if int(rm[b, t, j]) < N]
    b_, t_, r_, e_ = (torch.tensor(c, dtype=torch.long) for c in zip(*slots)) if slots else [torch.empty(0, dtype=torch.long)] * 4
    p_ = probs[b_, e_, t_].double()
    sum_rows = lambda rows: torch.zeros(B, T, *rows.shape[1:], dtype=torch.float64).index_put_((b_, t_), rows, accumulate=True)
    assert close(grads[0], sum_rows(gk[b_, r_].double()))
    assert close(grads[1], sum_rows(gv[b_, r_].double() * p_[:, None]))
    for q in range(3):
        assert close(grads[2 + q], sum_rows(gl[q][b_, r_].double()))
    tol = lambda a, c: H * 2.0 ** -24 * (a.double().abs() * c.double().abs()).sum(-1) + 1e-30

    def check_gp(got, a, c, zero_gate):
        ref, bound = torch.zeros(B, E, T, dtype=torch.float64), torch.zeros(B, E, T, dtype=torch.float64)
        live = (p_ != 0) if zero_gate else torch.ones_like(p_, dtype=torch.bool)
        ref[b_, e_, t_] = (a.double() * c.double()).sum(-1) * live
        bound[b_, e_, t_] = tol(a, c)
        assert bool(((got.cpu().double() - ref).abs() <= bound).all())

    check_gp(grads[5], gv[b_, r_], vx[b_, t_], True)
    # unpermute backward
    yd, pd = y.to(DEV).requires_grad_(), probs.to(DEV).requires_grad_()
    out = TP.unpermute_and_merge_with_probs(yd, rm.to(DEV), pd)
    gy, gp = torch.autograd.grad(out, [yd, pd], go.to(DEV))
    if slots:
        assert torch.equal(bits(gy)[b_, r_], bits((go[b_, t_].float() * p_.float()[:, None]).to(torch.bfloat16)))
    check_gp(gp, go[b_, t_], y[b_, r_], False)
    # permute backward
    xd, pd = kx.to(DEV).requires_grad_(), probs.to(DEV).requires_grad_()
    xp, pp, _ = TP.permute_with_expert_mask(xd, mask.to(DEV), pd, k)
    gpp = torch.randn(B, N, generator=g)
    gx, gp = torch.autograd.grad([xp, pp], [xd, pd], [gk.to(DEV), gpp.to(DEV)])
    assert close(gx, sum_rows(gk[b_, r_].double()))
    ref = torch.zeros(B, E, T)
    ref[b_, e_, t_] = gpp[b_, r_]
    assert torch.equal(gp.cpu(), ref)


@pytest.mark.parametrize("H", [24, 384])
def test_grouped_lane_kernels_keep_infinities_apart(H):
    """An infinity or NaN in one row reaches its token's sums and its own prob
    gradient only, also in the chunks that lanes past the row repeat."""
    B, T, E, k = 1, 2100, 16, 2
    g = torch.Generator().manual_seed(H)
    mask = torch.rand(B, E, T, generator=g).argsort(1).argsort(1) < k
    probs = (torch.rand(B, E, T, generator=g) * mask).to(DEV)
    rm = TP.make_row_id_map(mask.to(DEV), B, T, E)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    x, v, go, y, gk, gv = bf(B, T, H), bf(B, T, H), bf(B, T, H), bf(B, k * T, H), bf(B, k * T, H), bf(B, k * T, H)
    lr = [torch.rand(B, T, generator=g).to(DEV) for _ in range(3)]
    gl = [torch.rand(B, k * T, generator=g).to(DEV) for _ in range(3)]
    gpp = torch.rand(B, k * T, generator=g).to(DEV)

    def run():
        kv = TP._kv_fwd(x, v, *lr, rm, probs, k * T)
        kvb = TP._kv_bwd(gk, gv, *gl, v, probs, rm, T)
        pb = TP._permute_bwd(gk, rm, gpp, B, T, E, H)
        ub = TP._unpermute_bwd(go, rm, y, probs, B, T, E, k * T, H)
        return [kvb[0], kvb[1], pb[0]], [kvb[5], pb[1], ub[1]], [kv[0], kv[1], ub[0]]

    clean = run()
    t = T - 1
    rows = rm[0, t, :k].long()
    for a in (x, v, go):
        a[0, t, H - 1] = float("inf")
    for a in (y, gk, gv):
        a[0, rows[1], H - 1] = float("nan")
    bad = run()
    tok = torch.arange(T, device=DEV) != t
    out = torch.ones(k * T, dtype=torch.bool, device=DEV)
    out[rows] = False
    for a, c in zip(bad[0], clean[0]):
        assert torch.equal(a[0, tok], c[0, tok]) and bool(a[0, t, H - 1].isnan())
        assert bool(a[0, t, : H - 1].isfinite().all())
    for a, c in zip(bad[1], clean[1]):
        assert torch.equal(a[0, :, tok], c[0, :, tok])
    for a, c in zip(bad[2], clean[2]):
        assert torch.equal(a[0, out], c[0, out])
