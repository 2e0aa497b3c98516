"""The narrow-expert UPDATE kernels (csrc/narrow.hip: 64 hidden units x 128
tokens, stages of 32 k) against the general tiles, which the reference-layout
output and the backward without saved tensors take.  Both multiply in the same
order and round at the same places: stage 1, whose pointwise part has one way
to contract its multiply-adds, gives the same bits; the backward's may contract
differently, so an intermediate can land on the other side of a rounding tie
(one bf16 ulp, 2^-8, of a few elements)."""
import contextlib

import pytest
import torch

from uttt_amd import _lib as L
from uttt_amd.lact_moe_triton import _grouped as G
from uttt_amd.lact_moe_triton import _update_bwd as UB

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (group sizes per batch, D, I, N or None): one and several unit and token
# tiles, their remainders, a k tail, two stages (the smallest), the widest
CASES = {
    "tile_edges": ([[128, 129, 0, 127, 256, 31, 33, 1]], 192, 192, None),
    "ragged_two_batches": ([[70, 0, 130], [1, 199, 0]], 200, 104, None),
    "two_stages_one_unit_group": ([[5, 300, 2]], 40, 8, None),
    "widest": ([[33, 200]], 512, 512, None),
    "over_64_experts": ([[7 * (i % 5) for i in range(70)]], 64, 72, None),
    "slack_rows": ([[60, 40]], 384, 384, 160),
    "over_count": ([[60, 90, 70]], 96, 200, 140),
    "all_empty": ([[0, 0, 0]], 192, 64, 32),
    # from the tokens where the widest backward takes the general tiles, and one less
    "widest_many_tokens": ([[49111, 41]], 448, 512, None),
    "widest_one_token_less": ([[49110, 41]], 448, 512, None),
    # absent tiles between the batches': 256 tiles, and 192 where both may take a second round
    "many_batches_256": ([[256, 0, 255, 300]] * 16, 256, 256, 1024),
    "many_batches_192": ([[16, 0, 30, 18]] * 64, 192, 384, 64),
    "short_segments_wide": ([[200, 0, 193, 1, 300, 192]], 520, 776, None),
}


@pytest.mark.parametrize("lr_dtype", [torch.bfloat16, torch.float32, None])
@pytest.mark.parametrize("name", list(CASES))
def test_narrow_update_equals_general_tiles(name, lr_dtype):
    sizes, D, I, N = CASES[name]
    gs = torch.tensor(sizes, dtype=torch.int32, device=DEV)
    B, E = gs.shape
    N = int(gs.sum(1).max()) if N is None else N
    g = torch.Generator().manual_seed(N + D)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(torch.bfloat16).to(DEV)
    W02, gW02 = (rnd(B, E, 2 * I, D, scale=D ** -0.5) for _ in range(2))
    W1, gW1 = (rnd(B, E, D, I, scale=I ** -0.5) for _ in range(2))
    K, V = rnd(B, N, D), rnd(B, N, D)
    lrs = [None] * 3 if lr_dtype is None else \
        [torch.rand(B, N, generator=g).to(lr_dtype).to(DEV) for _ in range(3)]
    rows = torch.arange(N, device=DEV) < gs.sum(1, keepdim=True).clamp(max=N)  # [B, N] routed

    dy, hid, ys, dhs = G.update_stage1(W02, W1, K, V, *lrs, gs, True, save=True)
    dy_g, hid_g = G.update_stage1(W02, W1, K, V, *lrs, gs, False)
    for a, b in ((dy, dy_g), (hid, hid_g)):
        assert torch.equal(a[rows], b.transpose(1, 2)[rows])
    plain = G.update_stage1(W02, W1, K, V, *lrs, gs, True)
    assert torch.equal(plain[0][rows], dy[rows]) and torch.equal(plain[1][rows], hid[rows])
    if lr_dtype is None:
        return

    ours = UB._backward(W02, W1, K, V, *lrs, gs, gW02, gW1, ys, dhs)
    gen = UB._backward(W02, W1, K, V, *lrs, gs, gW02, gW1, None, None)
    # 2^-8 of the whole if every element of an intermediate were an ulp off; one
    # wrong token row of n would be n ** -0.5
    for a, b in zip(ours[:4], gen[:4]):
        if a.shape[:2] == (B, N):
            a, b = a[rows], b[rows]
        assert (a.double() - b.double()).norm() <= 2.0 ** -8 * b.double().norm()
    # one output rounding where a sum lands on the other side of a tie, and the
    # fp32 sums of I products of about one in two orders
    ulp = 2.0 ** -7 if lr_dtype == torch.bfloat16 else 0.0
    for a, b in zip(ours[4:], gen[4:]):
        a, b = a.double(), b.double()
        assert bool((a[~rows] == 0).all())
        scale = max(1.0, b.abs().max().item())
        assert bool(((a - b).abs() <= ulp * b.abs() + I * 2.0 ** -23 * scale).all())


def test_one_launch_stage1_allocates_its_outputs_alone():
    """No fp32 DH [B, N, I] beside them: the peak over the call is the outputs
    (and what the allocator rounds up, under 2 MiB for each of four tensors)."""
    B, E, I, D, N = 1, 4, 512, 512, 32768
    rnd = lambda *s: torch.randn(*s, device=DEV).to(torch.bfloat16)
    gs = torch.full((B, E), N // E, dtype=torch.int32, device=DEV)
    args = (rnd(B, E, 2 * I, D), rnd(B, E, D, I), rnd(B, N, D), rnd(B, N, D), None, None, None, gs)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    outs = G.update_stage1(*args, True)
    peak = torch.cuda.max_memory_allocated() - before
    assert peak < B * N * 3 * I * 2 + 4 * (2 << 20), (peak, [tuple(o.shape) for o in outs])


@contextlib.contextmanager
def general_tiles():
    """The 256-token tiles: a forced wave layout takes every product there."""
    prev = L.lib().uttt_debug_set_gemm_layout(2)
    try:
        yield
    finally:
        L.lib().uttt_debug_set_gemm_layout(prev)


@pytest.mark.parametrize("name", list(CASES))
def test_narrow_products_equal_general_tiles(name):
    """Gate/up (rows in expert order and gathered) and the plain and chained
    products (192 x 192 tiles): the same multiplications in the same order."""
    sizes, D, I, N = CASES[name]
    gs = torch.tensor(sizes, dtype=torch.int32, device=DEV)
    B, E = gs.shape
    N = int(gs.sum(1).max()) if N is None else N
    g = torch.Generator().manual_seed(N + I)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    W02, W1, W2 = rnd(B, E, 2 * I, D), rnd(B, E, D, I), rnd(B, E, D, I)
    X, H, H2, Y = rnd(B, N, D), rnd(B, N, I), rnd(B, N, I), rnd(B, N, 2 * I)
    rows = torch.arange(N, device=DEV) < gs.sum(1, keepdim=True).clamp(max=N)
    src = torch.randint(0, N, (B, N), generator=g, dtype=torch.int32).to(DEV)

    def products():
        out = [G.gate_up(W02, X, gs, token_major=True), G.gemm_nt(W1, H, gs), G.gemm_tn(W1, X, gs),
               G.gemm_tn(W02, Y, gs), G.gemm_nt2(W1, H, W2, H2, gs), G.gemm_tn2(W1, X, W2, X, gs)]
        if G.gate_up_gathers(N, E):
            out.append(G.gate_up_gather(W02, X, src, gs))
        return out

    ours = products()
    with general_tiles():
        general = products()
    for i, (a, b) in enumerate(zip(ours, general, strict=True)):
        assert torch.equal(a[rows], b[rows]), i


def test_short_segments_on_192_tiles_equal_general_tiles():
    """Experts past the narrow widths with at most 256 tokens each."""
    gs = torch.tensor([[200, 0, 193, 1, 300, 192]], dtype=torch.int32, device=DEV)
    B, E, D, I, N = 1, 6, 520, 776, 890
    g = torch.Generator().manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    W02, W1, W2 = rnd(B, E, 2 * I, D), rnd(B, E, D, I), rnd(B, E, D, I)
    X, H, Y = rnd(B, N, D), rnd(B, N, I), rnd(B, N, 2 * I)
    products = lambda: [G.gemm_tn(W02, Y, gs), G.gemm_nt2(W1, H, W2, H, gs),
                        G.gemm_tn2(W02, Y, W02, Y, gs)]
    ours = products()
    with general_tiles():
        general = products()
    n = int(gs.sum())
    for a, b in zip(ours, general):
        assert torch.equal(a[:, :n], b[:, :n])


@pytest.mark.parametrize("M,K,sizes", [
    (384, 16, [200000, 0, 3, 140001, 53333]),   # super-tiles that overhang the token tiles
    (1736, 8, [97] * 640),                       # ten row tiles in super-tiles of eight
])
def test_super_tiles_of_192_equal_general_tiles(M, K, sizes):
    """Grids of 4096 tiles and more."""
    gs = torch.tensor([sizes], dtype=torch.int32, device=DEV)
    E, N = len(sizes), sum(sizes)
    g = torch.Generator(device=DEV).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    W, Wt, X = rnd(1, E, K, M), rnd(1, E, M, K), rnd(1, N, K)
    products = lambda: [G.gemm_tn(W, X, gs), G.gemm_nt(Wt, X, gs)]
    ours = products()
    with general_tiles():
        general = products()
    for a, b in zip(ours, general):
        assert torch.equal(a, b)


def _same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(7.0), b.nan_to_num(7.0))


@pytest.mark.parametrize("D,I", [(192, 192), (200, 104), (512, 512)])
def test_infinities_and_nan_stay_with_their_tokens_and_experts(D, I):
    """An infinity in one token's rows, at the end of its expert's segment (the
    row that partial tiles repeat), and a NaN in another expert's weights: what
    has no part in them keeps its bits, the rest is the general tiles'."""
    sizes = [130, 65, 200, 31]
    gs = torch.tensor([sizes], dtype=torch.int32, device=DEV)
    E, N = len(sizes), sum(sizes)
    g = torch.Generator().manual_seed(D)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(torch.bfloat16).to(DEV)
    W02, gW02 = (rnd(1, E, 2 * I, D, scale=D ** -0.5) for _ in range(2))
    W1, gW1 = (rnd(1, E, D, I, scale=I ** -0.5) for _ in range(2))
    K, V, H, Y = rnd(1, N, D), rnd(1, N, D), rnd(1, N, I), rnd(1, N, 2 * I)
    lrs = [torch.rand(1, N, generator=g).to(DEV) for _ in range(3)]

    def run():
        s1 = G.update_stage1(W02, W1, K, V, *lrs, gs, True, save=True)
        bwd = UB._backward(W02, W1, K, V, *lrs, gs, gW02, gW1, *s1[2:])
        tok = [G.gate_up(W02, K, gs, token_major=True), G.gemm_nt(W1, H, gs), G.gemm_tn(W02, Y, gs),
               *s1, *bwd[2:]]
        return tok, [*G.wgrad_pair(Y, K, H, V, gs), *bwd[:2]]

    clean = run()
    bad_tok, bad_e = sizes[0] + sizes[1] - 1, 2
    for t in (K, V, H, Y):
        t[0, bad_tok] = float("inf")
    W02[0, bad_e, 5, 7] = W1[0, bad_e, 3, 2] = float("nan")
    ours = run()
    with general_tiles():
        general = run()
    e_of = torch.repeat_interleave(torch.arange(E), torch.tensor(sizes)).to(DEV)
    ok_rows = (e_of != bad_e) & (torch.arange(N, device=DEV) != bad_tok)
    for a, c in zip(ours[0], clean[0], strict=True):
        assert torch.equal(a[0, ok_rows], c[0, ok_rows])
    for a, b in zip(ours[0][:7], general[0][:7]):     # all but the backward: bit for bit
        assert _same(a, b)
    for a, b in zip(ours[0][7:], general[0][7:]):
        assert torch.equal(a.isfinite(), b.isfinite())
    clean_e = [0, 3]
    for a, c, b in zip(ours[1], clean[1], general[1], strict=True):
        assert torch.equal(a[0, clean_e], c[0, clean_e])
        assert torch.equal(a.isfinite(), b.isfinite())
