"""Single-pass chunked CE (smel.loss over include/smel_loss.h) on the GPU: the reference's own three tests
(tests/test_loss_single_pass.py:23-63: against full fp32 logits with and without softcapping at 1e-4, bf16 single
pass against the two-pass comparator, the int8 head against its dequantized weight) and the fp64 oracle
(oracle/loss_ref.py) at a larger bf16 shape; a vocabulary that is not a multiple of the chunk, several token chunks,
a target in every chunk position (first, last column)."""
import pytest
import torch

from oracle import loss_ref as LR

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lm():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from smel import loss, quant
    return loss, quant


def full_ref(h, W, tgt, softcap, denom):
    h = h.detach().clone().requires_grad_(True)
    lg = h @ W.float().t()
    if softcap:
        lg = softcap * torch.tanh(lg / softcap)
    loss = torch.nn.functional.cross_entropy(lg, tgt, reduction="sum") / denom
    loss.backward()
    return loss.detach(), h.grad


@pytest.mark.parametrize("softcap", [0.0, 30.0])
def test_fp32_matches_full_logits(lm, softcap):
    loss_mod, _ = lm
    torch.manual_seed(0)
    n, H, V = 37, 64, 1000                      # V is not a multiple of the vocab chunk
    h = torch.randn(n, H, device="cuda") * 0.5
    W = torch.randn(V, H, device="cuda") * 0.2
    tgt = torch.randint(0, V, (n,), device="cuda")
    tgt[0], tgt[1], tgt[2] = 0, V - 1, 127      # first column, last column, last column of a chunk
    head = loss_mod.LMHead(weight=W, vocab_chunk=128, softcap=softcap)
    loss_ref, grad_ref = full_ref(h, W, tgt, softcap, denom=n)
    h_ = h.clone().requires_grad_(True)
    loss = loss_mod.chunked_ce(h_, head, tgt, denom=n, token_chunk=16)
    loss.backward()
    assert abs(loss.item() - loss_ref.item()) < 1e-4 * max(1.0, abs(loss_ref.item()))
    assert (h_.grad - grad_ref).norm() / grad_ref.norm() < 1e-4
    l64, g64 = LR.full_ce(h, W, tgt, softcap, denom=n)
    assert abs(loss.item() - float(l64)) < 1e-4 * max(1.0, abs(float(l64)))
    assert (h_.grad.double().cpu() - g64).norm() / g64.norm() < 1e-4


def test_bf16_matches_two_pass(lm):
    loss_mod, _ = lm
    torch.manual_seed(1)
    n, H, V = 300, 128, 5000
    h = (torch.randn(n, H, device="cuda") * 0.5).bfloat16()
    W = (torch.randn(V, H, device="cuda") * 0.2).bfloat16()
    tgt = torch.randint(0, V, (n,), device="cuda")
    for softcap in (0.0, 30.0):
        head = loss_mod.LMHead(weight=W, vocab_chunk=1024, softcap=softcap)
        l1, g1 = loss_mod._ce_chunk(h, head, tgt, True)
        l2, g2 = loss_mod._ce_chunk_two_pass(h, head, tgt, True)
        assert abs(l1.item() - l2.item()) / abs(l2.item()) < 1e-3
        assert (g1 - g2).norm() / g2.norm() < 2e-2
        l64, g64 = LR.full_ce(h, W, tgt, softcap)
        assert abs(l1.item() - float(l64)) / abs(float(l64)) < 1e-3
        assert (g1.double().cpu() - g64).norm() / g64.norm() < 3e-2    # bf16 logits and probabilities


def test_int8_head_runs_and_matches_its_dequantized_weight(lm):
    loss_mod, quant = lm
    torch.manual_seed(2)
    n, H, V = 64, 96, 700
    h = torch.randn(n, H, device="cuda") * 0.5
    W = torch.randn(V, H, device="cuda") * 0.2
    tgt = torch.randint(0, V, (n,), device="cuda")
    q = {k: v.cuda() for k, v in quant.quantize_int8_rows(W).items()}
    w_dq = quant.dequant_int8_rows(q["q"], q["scale"], torch.float32)
    loss_q = loss_mod.chunked_ce(h, loss_mod.LMHead(int8=q, vocab_chunk=256), tgt, denom=n, token_chunk=32,
                                 need_grad=False)
    loss_dq = loss_mod.chunked_ce(h, loss_mod.LMHead(weight=w_dq), tgt, denom=n, token_chunk=32, need_grad=False)
    assert abs(loss_q.item() - loss_dq.item()) < 1e-3 * abs(loss_dq.item())


def test_repeatable_and_empty(lm):
    loss_mod, _ = lm
    torch.manual_seed(3)
    h = (torch.randn(130, 64, device="cuda")).bfloat16().requires_grad_(True)
    W = (torch.randn(777, 64, device="cuda") * 0.2).bfloat16()
    tgt = torch.randint(0, 777, (130,), device="cuda")
    head = loss_mod.LMHead(weight=W, vocab_chunk=100)
    a = loss_mod.chunked_ce(h, head, tgt, denom=130.0, token_chunk=64)
    a.backward()
    ga = h.grad.clone()
    h.grad = None
    b = loss_mod.chunked_ce(h, head, tgt, denom=130.0, token_chunk=64)
    b.backward()
    assert torch.equal(a, b) and torch.equal(ga, h.grad)
    e = loss_mod.chunked_ce(h[:0], head, tgt[:0], denom=1.0)
    assert e.item() == 0.0


def rounded_full_ce(h, W, tgt, softcap):
    """Comparator written for these tests: the full logits rounded to h's dtype (the library GEMM's output), capped
    in fp32, the exact softmax from their log-sum-exp, the softmax terms rounded to h's dtype before they meet W (the
    reference's p.to(h.dtype) @ W). Targets outside [0, V) contribute no target logit and no target row."""
    V = W.shape[0]
    z = (h @ W.t()).float()
    dz = torch.ones_like(z)
    if softcap:
        t = torch.tanh(z / softcap)
        z, dz = softcap * t, 1 - t * t
    lse = torch.logsumexp(z, -1)
    ok = (tgt >= 0) & (tgt < V)
    idx = torch.where(ok, tgt, torch.zeros_like(tgt))
    zt = torch.where(ok, z.gather(1, idx[:, None])[:, 0], torch.zeros_like(lse))
    p = torch.exp(z - lse[:, None])
    p[torch.arange(len(tgt), device=h.device)[ok], idx[ok]] -= 1.0
    g = ((p * dz).to(h.dtype) @ W).float()
    return (lse - zt).sum(), g


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("softcap", [0.0, 30.0])
def test_several_vocabulary_chunks(lm, dtype, softcap):
    """Vocabulary chunks of 4096 columns (16 logits tiles, 32 statistics windows) and a short last chunk of 100
    columns (one partly filled tile): the running maximum moves between chunks, so the accumulator and the window
    shifts are rescaled. Loss and gradient against the fp64 full-logit oracle and the rounded full-logit comparator."""
    loss_mod, _ = lm
    print(f"multi-chunk CE {dtype} softcap {softcap}", flush=True)
    torch.manual_seed(4)
    n, H, V = 300, 256, 2 * 4096 + 100
    h = (torch.randn(n, H, device="cuda") * 0.5).to(dtype)
    W = (torch.randn(V, H, device="cuda") * 0.2).to(dtype)
    tgt = torch.randint(0, V, (n,), device="cuda")
    tgt[:6] = torch.tensor([0, 127, 128, 4095, 4096, V - 1])           # window, tile, chunk edges, the last column
    head = loss_mod.LMHead(weight=W, vocab_chunk=4096, softcap=softcap)
    l1, g1 = loss_mod._ce_chunk(h, head, tgt, True)
    l64, g64 = LR.full_ce(h, W, tgt, softcap)
    lc, gc = rounded_full_ce(h, W, tgt, softcap)
    tol_l, tol_g = (1e-3, 3e-2) if dtype == torch.bfloat16 else (1e-5, 1e-4)
    assert abs(l1.item() - float(l64)) / abs(float(l64)) < tol_l
    assert (g1.double().cpu() - g64).norm() / g64.norm() < tol_g
    assert abs(l1.item() - lc.item()) / abs(lc.item()) < tol_l
    assert (g1 - gc).norm() / gc.norm() < (2e-2 if dtype == torch.bfloat16 else 1e-4)
    l2, g2 = loss_mod._ce_chunk_two_pass(h, head, tgt, True)           # the same sums without any rescaling
    assert abs(l1.item() - l2.item()) / abs(l2.item()) < tol_l
    assert (g1 - g2).norm() / g2.norm() < (2e-2 if dtype == torch.bfloat16 else 1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_wide_logit_range(lm, dtype):
    """Head rows of very different norms: windows whose maxima lie 100-400 below the row's maximum get shifts past
    the bf16 / fp32 range (their terms become zero, as exp underflows in the reference), others small shifts; a few
    rows put their target in such a window (a large loss). bf16 against the rounded full-logit comparator (logits of
    a few hundred carry bf16 steps of 0.5-2 in both), fp32 against the fp64 oracle."""
    loss_mod, _ = lm
    print(f"wide-range CE {dtype}", flush=True)
    torch.manual_seed(6)
    n, H, V = 96, 128, 3000
    h = torch.randn(n, H, device="cuda").to(dtype)
    scale = torch.ones(V, 1, device="cuda")
    scale[0:128] = 40.0            # window 0: logits of a few hundred
    scale[1024:1152] = 8.0         # a window at a moderate offset
    W = (torch.randn(V, H, device="cuda") * 0.1 * scale).to(dtype)
    tgt = torch.randint(0, V, (n,), device="cuda")
    tgt[:4] = torch.tensor([5, 1030, 2999, 700])
    head = loss_mod.LMHead(weight=W, vocab_chunk=1024)
    l1, g1 = loss_mod._ce_chunk(h, head, tgt, True)
    if dtype == torch.bfloat16:
        lc, gc = rounded_full_ce(h, W, tgt, 0.0)
        assert abs(l1.item() - lc.item()) / abs(lc.item()) < 1e-4
        assert (g1 - gc).norm() / gc.norm() < 2e-2
    else:
        l64, g64 = LR.full_ce(h, W, tgt)
        assert abs(l1.item() - float(l64)) / abs(float(l64)) < 1e-5
        assert (g1.double().cpu() - g64).norm() / g64.norm() < 1e-4


def test_several_row_passes(lm):
    """Passes of 16 rows (a caller's token_chunk bounds the rows of a pass): the loss accumulates over the passes and
    each pass writes its own gradient rows; equal to one pass over all rows."""
    loss_mod, _ = lm
    torch.manual_seed(7)
    n, H, V = 200, 64, 1500
    h = (torch.randn(n, H, device="cuda") * 0.5).bfloat16()
    W = (torch.randn(V, H, device="cuda") * 0.2).bfloat16()
    tgt = torch.randint(0, V, (n,), device="cuda")
    head = loss_mod.LMHead(weight=W, vocab_chunk=512)
    one = h.clone().requires_grad_(True)
    l_one = loss_mod.chunked_ce(one, head, tgt, denom=float(n))
    l_one.backward()
    many = h.clone().requires_grad_(True)
    l_many = loss_mod.chunked_ce(many, head, tgt, denom=float(n), token_chunk=16)
    (l_many * 2.0).backward()                                      # the incoming gradient scales the rows
    assert abs(l_one.item() - l_many.item()) < 1e-5 * abs(l_one.item())
    assert torch.equal(many.grad.float(), (2.0 * one.grad.float()).bfloat16().float())
    l64, g64 = LR.full_ce(h, W, tgt, denom=float(n))
    assert abs(l_many.item() - float(l64)) / abs(float(l64)) < 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("n", [1, 128, 129, 257, 384, 385])
def test_row_tiles_and_parts(lm, n, dtype):
    """Row counts around the 128- and 256-row tiles, with the gradient's contraction in several parts and a vocabulary of
    several chunks where the pass takes them (vocab_chunk 512), against the fp64 oracle: fp32 rows to 1e-4, 16-bit rows
    within their rounding (the softmax terms and the logits each rounded once: 2 x 2^-8, bf16)."""
    loss_mod, _ = lm
    torch.manual_seed(n)
    H, V = 328, 6007
    h = (torch.randn(n, H, device="cuda") * 0.5).to(dtype)
    W = (torch.randn(V, H, device="cuda") * 0.1).to(dtype)
    tgt = torch.randint(0, V, (n,), device="cuda")
    l64, g64 = LR.full_ce(h, W, tgt, 0.0, denom=n)
    for kw in ({"vocab_chunk": 512}, {}):
        for tc in ({}, {"token_chunk": 200}):
            x = h.clone().requires_grad_(True)
            loss = loss_mod.chunked_ce(x, loss_mod.LMHead(weight=W, **kw), tgt, denom=n, **tc)
            loss.backward()
            rel = float((x.grad.double().cpu() - g64).norm() / g64.norm())
            print(f"CE n={n} {dtype} {kw} {tc}: loss {loss.item():.6f} grad rel {rel:.2e}", flush=True)
            assert abs(loss.item() - float(l64)) < (1e-4 if dtype == torch.float32 else 2e-3) * abs(float(l64))
            assert rel < (1e-4 if dtype == torch.float32 else 1e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V,H", [(1, 8), (63, 72), (129, 64), (700, 328)])
def test_int8_rows_and_transpose_bits(lm, V, H, dtype):
    """smel_ce_dequant8 against dequant_int8_rows bit for bit, the transposed copy's padding columns zero, and the
    16-byte transpose of a dense head against torch's."""
    loss_mod, quant = lm
    from smel import _lib as L
    torch.manual_seed(V)
    q = {"q": torch.randint(-127, 128, (V, H), dtype=torch.int8, device="cuda"),
         "scale": (torch.rand(V, device="cuda") * 0.01).to(torch.bfloat16)}
    ref = quant.dequant_int8_rows(q["q"], q["scale"], dtype)
    Vp = (V + 7) // 8 * 8
    rows, wt = torch.empty_like(ref), torch.full((H, Vp), 7.0, dtype=dtype, device="cuda")
    sc = q["scale"].to(dtype)
    L.call("smel_ce_dequant8", L.ptr(q["q"]), L.ptr(sc), V, H, loss_mod._DT[dtype], L.ptr(rows), L.ptr(wt), Vp, L.stream())
    assert torch.equal(rows.view(torch.int16), ref.view(torch.int16))
    assert torch.equal(wt[:, :V], ref.t()) and not wt[:, V:].any()
    _, wt2 = loss_mod._rows_and_transpose(ref, True)
    assert torch.equal(wt2, wt)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("vc", [4097, 4160, 4128, 4161, 4224])
def test_gradient_windows_keep_their_shifts(lm, vc, dtype):
    """The gradient product against fp64 where neighbouring windows' shifts differ by up to twelve powers of two and the last
    window holds one k-step (vc % 128 in 1..64 for 16-bit rows, 1..32 for fp32) or more, for every number of parts: a
    block's k loop is rotated, so that it takes the last window's step right before the part's first."""
    from smel import _lib as L
    torch.manual_seed(vc)
    n, H, p = 512, 2048, L.ptr
    vcp = (vc + 255) // 256 * 256
    P = torch.zeros(n, vcp, device="cuda")
    P[:, :vc] = torch.rand(n, vc, device="cuda") * 0.5 + 0.5
    WT = torch.zeros(H, vcp, device="cuda")
    WT[:, :vc] = torch.randn(H, vc, device="cuda")
    P, WT = P.to(dtype), WT.to(dtype)
    nwin = vcp // 128
    r = torch.ones(n, device="cuda")
    shift = ((torch.arange(nwin, device="cuda") * 5 + 3) % 13).to(torch.uint8)   # the last window's is no part's first
    sh = shift[:, None].expand(nwin, n).contiguous()
    scale = torch.ldexp(torch.ones(nwin, device="cuda", dtype=torch.float64), -shift.int()).repeat_interleave(128)
    ref = (P.double() * scale) @ WT.double().t()
    for splits in range(1, 9):
        acc = torch.empty(splits, n, H, device="cuda")
        L.call("smel_ce_grad_split", p(WT), vcp, H, p(P), vcp, vc, p(sh), n, p(r), n, L_DT[dtype], 0, splits, p(acc),
               L.stream())
        # fp32 sums of about 4000 terms in some order: 2^-24 sqrt(4000) = 4e-6 of the result; the shifted terms stay exact
        # (an fp16 term of 0.5 at the largest shift is 2^-13)
        err = ((acc.double().sum(0) - ref).norm() / ref.norm()).item()
        assert err < 1e-5, (splits, err)


L_DT = {torch.bfloat16: 0, torch.float32: 1, torch.float16: 2}


@pytest.mark.parametrize("tail_level", [6.0, -6.0])
@pytest.mark.parametrize("V", [4097, 4160])
def test_short_last_window_of_the_vocabulary(lm, V, tail_level):
    """A vocabulary whose last window holds one k-step, its logits 6 above or below all others: the column of the gradient
    that only those rows of the head reach, against fp64."""
    loss_mod, _ = lm
    torch.manual_seed(V)
    n, H, m = 512, 2048, V - 4096
    h = torch.randn(n, H, device="cuda") * 0.1
    h[:, 0], h[:, 1] = 1.0, 0.0
    W = torch.randn(V, H, device="cuda") * 0.02
    W[:, :2] = 0.0
    W[4096:, 0], W[4096:, 1] = tail_level, 4.0
    h, W = h.bfloat16(), W.bfloat16()
    tgt = torch.randint(0, 4096, (n,), device="cuda")
    x = h.clone().requires_grad_(True)
    loss_mod.chunked_ce(x, loss_mod.LMHead(weight=W), tgt, denom=1.0).backward()
    p = torch.softmax(h.double() @ W.double().t(), -1)
    ref = 4.0 * p[:, 4096:].sum(-1)
    # a logit near 6 is rounded to bf16 steps of 2^-5 (half of one: 1.6 % of its term), the others' errors average out;
    # terms and the gradient round once more (2^-9 each)
    assert ((x.grad[:, 1].double() - ref).abs() <= 0.025 * ref).all()


def test_two_half_form_equals_two_parts(lm):
    """smel_ce_grad / smel_ce_finish (two halves, the second one's accumulator alternating between two buffers) against
    smel_ce_grad_split / _finish_split with two parts, over three chunks: bitwise."""
    from smel import _lib as L
    torch.manual_seed(3)
    n, H, vc, p = 200, 136, 768, L.ptr
    f = lambda *s: torch.empty(*s, device="cuda")
    P = torch.rand(n, vc, device="cuda").bfloat16()
    WT = torch.randn(H, vc, device="cuda").bfloat16()
    shift = torch.randint(0, 4, (vc // 128, n), dtype=torch.uint8, device="cuda")
    r = torch.full((n,), 0.5, device="cuda")
    acc, part, acc2 = f(n, H), f(2, n, H), f(2, n, H)
    for c in range(3):
        L.call("smel_ce_grad", p(WT), vc, H, p(P), vc, vc, p(shift), n, p(r), n, 0, c, p(acc), p(part), L.stream())
        L.call("smel_ce_grad_split", p(WT), vc, H, p(P), vc, vc, p(shift), n, p(r), n, 0, c, 2, p(acc2), L.stream())
    assert torch.equal(acc, acc2[0]) and torch.equal(part[0], acc2[1])
    m, s, tz, td, l1, l2 = (torch.ones(n, device="cuda") for _ in range(6))
    tgt = torch.randint(0, 10, (n,), device="cuda")
    trows = torch.randn(n, H, device="cuda").bfloat16()
    g1, g2 = f(n, H), f(n, H)
    L.call("smel_ce_finish", p(m), p(s), p(tz), p(td), p(acc), p(part[0]), None, 0, p(trows), p(tgt), 10, n, H, 0, 0.5,
           p(g1), H, 1, p(l1), L.stream())
    L.call("smel_ce_finish_split", p(m), p(s), p(tz), p(td), p(acc2), 2, None, 0, p(trows), p(tgt), 10, n, H, 0, 0.5,
           p(g2), H, 1, p(l2), L.stream())
    assert torch.equal(g1, g2) and torch.equal(l1, l2)


def test_token_chunk_bounds_pass_memory(lm):
    """token_chunk x vocab_chunk bounds a pass's scratch, as the reference promises for its peak memory: with
    token_chunk=256 over 4096 rows, one call allocates at most one 256-row pass (softmax terms 256 x vocab_chunk
    bf16, fp32 row state and accumulators) beyond its gradient output; left at the default, a pass takes all 4096
    rows and its terms alone are 16 times larger. Both give the same loss and gradient."""
    loss_mod, _ = lm
    torch.manual_seed(9)
    n, H, V, vc = 4096, 256, 65536, 32768
    h = torch.randn(n, H, device="cuda").bfloat16()
    W = (torch.randn(V, H, device="cuda") * 0.05).bfloat16()
    tgt = torch.randint(0, V, (n,), device="cuda")
    head = loss_mod.LMHead(weight=W, vocab_chunk=vc)

    def run(**kw):
        x = h.clone().requires_grad_(True)
        loss_mod.chunked_ce(x, head, tgt, denom=float(n), **kw)   # the head's transposed copy is made once, here
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        loss = loss_mod.chunked_ce(x, head, tgt, denom=float(n), **kw)
        loss.backward()
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - base, loss.detach(), x.grad

    peak_small, l_small, g_small = run(token_chunk=256)
    peak_dflt, l_dflt, g_dflt = run()
    tc = 256
    one_pass = tc * vc * 2 + tc * H * 4 * 3 + 2 * (vc // 128) * tc * 4 + (vc // 128) * tc + 6 * tc * 4
    bound = one_pass + 2 * n * H * 2 + (1 << 20)    # + the gradient output and x.grad (bf16), small tensors
    print(f"CE peak allocation: token_chunk=256 {peak_small / 2**20:.1f} MiB (bound {bound / 2**20:.1f}), default "
          f"{peak_dflt / 2**20:.1f} MiB", flush=True)
    assert peak_small <= bound
    assert peak_dflt > 8 * tc * vc * 2
    # the gradient GEMM splits its contraction by the number of row tiles of a pass, so the two pass sizes sum the
    # fp32 partials in different orders: equal up to the last bits
    assert abs(l_small.item() - l_dflt.item()) <= 1e-5 * abs(l_dflt.item())
    d = (g_small.float() - g_dflt.float()).abs().max().item()
    assert d <= 2**-7 * g_dflt.float().abs().max().item(), d


@pytest.mark.parametrize("tc,vc", [(128, 4096), (256, 4096), (64, 32768), (640, 8192)])
def test_accumulators_stay_in_the_pass_bound(lm, tc, vc):
    """A hidden size whose accumulators are most of a pass: 12 H bytes a row, or twice the bytes of its terms, beside the
    terms themselves and the row state."""
    loss_mod, _ = lm
    torch.manual_seed(tc)
    H, V = 2048, 2 * vc
    W = (torch.randn(V, H, device="cuda") * 0.05).bfloat16()
    tgt = torch.randint(0, V, (tc,), device="cuda")
    x = torch.randn(tc, H, device="cuda").bfloat16().requires_grad_(True)
    head = loss_mod.LMHead(weight=W, vocab_chunk=vc)

    def run():   # the head's transposed copy is made in the first one
        loss_mod.chunked_ce(x, head, tgt, denom=float(tc), token_chunk=tc).backward()
        x.grad = None
        torch.cuda.synchronize()

    run()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    run()
    peak = torch.cuda.max_memory_allocated() - base
    terms = tc * vc * 2
    bound = terms + max(tc * H * 12, 2 * terms) + (2 * (vc // 128) * 4 + vc // 128 + 24) * tc
    bound += 2 * tc * H * 2 + (1 << 18)   # gradients, small tensors
    print(f"CE peak at H {H}: {peak / 2**20:.1f} MiB (bound {bound / 2**20:.1f})", flush=True)
    assert peak <= bound


def test_qwen_head_full_size(lm):
    """The bench's shape (4092 rows, hidden 2048, vocabulary 248320, chunks of 32768, bf16): loss and gradient of
    chunked_ce against the rounded full-logit comparator run in fp32 torch on the GPU (the [4092, 248320] logits fit
    in memory there), and the same call twice gives bitwise equal results."""
    loss_mod, _ = lm
    print("CE full size", flush=True)
    torch.manual_seed(8)
    T, H, V = 4092, 2048, 248320
    h = torch.randn(T, H, device="cuda").bfloat16()
    W = (torch.randn(V, H, device="cuda") * 0.02).bfloat16()
    tgt = torch.randint(0, V, (T,), device="cuda")
    head = loss_mod.LMHead(weight=W)
    x = h.clone().requires_grad_(True)
    loss = loss_mod.chunked_ce(x, head, tgt, denom=float(T))
    loss.backward()
    g1 = x.grad.clone()
    x.grad = None
    loss2 = loss_mod.chunked_ce(x, head, tgt, denom=float(T))
    loss2.backward()
    assert torch.equal(loss, loss2) and torch.equal(g1, x.grad)
    lc, gc = rounded_full_ce(h, W, tgt, 0.0)
    lc, gc = lc / T, gc / T
    rel_l = abs(loss.item() - lc.item()) / abs(lc.item())
    rel_g = ((g1.float() - gc).norm() / gc.norm()).item()
    cos = torch.nn.functional.cosine_similarity(g1.float().flatten(), gc.flatten(), dim=0).item()
    print(f"full-size CE: loss rel err {rel_l:.2e}, grad rel err {rel_g:.2e}, cos {cos:.6f}", flush=True)
    assert rel_l < 1e-4 and rel_g < 2e-2 and cos > 0.9999


def test_targets_outside_the_vocabulary(lm):
    """A target outside [0, V) (e.g. an ignore index of -100 that a caller did not filter) matches no row: its loss
    term is the log-sum-exp alone and its gradient has no target row, as in the reference's _ce_chunk; no row of W is
    gathered for it."""
    loss_mod, _ = lm
    torch.manual_seed(5)
    n, H, V = 40, 64, 900
    h = torch.randn(n, H, device="cuda") * 0.5
    W = torch.randn(V, H, device="cuda") * 0.2
    tgt = torch.randint(0, V, (n,), device="cuda")
    tgt[3], tgt[7], tgt[11] = -100, V, V + 1000
    for softcap in (0.0, 30.0):
        head = loss_mod.LMHead(weight=W, vocab_chunk=256, softcap=softcap)
        l1, g1 = loss_mod._ce_chunk(h, head, tgt, True)
        lc, gc = rounded_full_ce(h, W, tgt, softcap)
        assert abs(l1.item() - lc.item()) < 1e-4 * abs(lc.item())
        assert (g1 - gc).norm() / gc.norm() < 1e-4


@pytest.mark.parametrize("n", [1, 128, 129, 256, 257, 384, 385, 512])
def test_tail_tile_edges(n):
    """Row counts at the edges of the short last token tile (its own kernel) through the public call: mean loss and gradient
    against the fp64 formula (the rows one by one: test_tail_tile_rows_against_whole_tiles)."""
    g = torch.Generator().manual_seed(n)
    H, V = 64, 700
    h = torch.randn(n, H, generator=g).to(torch.bfloat16)
    w = (torch.randn(V, H, generator=g) * 0.2).to(torch.bfloat16)
    tgt = torch.randint(0, V, (n,), generator=g)
    from smel.loss import LMHead, chunked_ce
    hd = h.cuda().requires_grad_(True)
    loss = chunked_ce(hd, LMHead(weight=w.cuda()), tgt.cuda(), n)
    loss.backward()
    h64 = h.double().requires_grad_(True)
    ref = torch.nn.functional.cross_entropy(h64 @ w.double().t(), tgt)
    ref.backward()
    # logits are rounded to bf16 (2^-9 of values of about 1.6, V of them averaged), gradients once more
    assert abs(loss.item() - ref.item()) < 1e-2 * abs(ref.item())
    assert (hd.grad.cpu().double() - h64.grad).norm() < 1.5e-2 * h64.grad.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 127, 128, 129, 255, 256, 257, 384, 385])
def test_tail_tile_rows_against_whole_tiles(lm, n, dtype):
    """The same row edges over several hidden tiles, rotated parts and a last window of one k-step: every row's loss and
    fp32 gradient against those of the row in a pass padded to whole 256-row tiles. The two passes take their fp32 sums
    (about V / 2 terms of a row) in other orders: 1e-5 of the row's size; the terms themselves are the same."""
    loss_mod, _ = lm
    torch.manual_seed(n)
    H, V, m = 776, 5003, (n + 255) // 256 * 256
    h = torch.randn(m, H, device="cuda").to(dtype)
    W = (torch.randn(V, H, device="cuda") * 0.1).to(dtype)
    tgt = torch.randint(0, V, (m,), device="cuda")
    head = loss_mod.LMHead(weight=W)

    def rows(k):
        x, t = loss_mod._prep(h[:k], tgt[:k])
        ps = loss_mod._Pass(k, H, head._kernel_chunks(), dtype, True, x.device)
        loss_mod._sweep(x, head, t, True, ps)
        return loss_mod._finish(x, head, t, ps, True), ps.loss

    g, l = rows(n)
    gw, lw = rows(m)
    assert ((l - lw[:n]).abs() <= 1e-5 * lw[:n].abs()).all()
    assert ((g - gw[:n]).abs().amax(1) <= 1e-5 * gw[:n].norm(dim=1)).all()
