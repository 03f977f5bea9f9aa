"""The fp32 path (float32 activations: the reference's fp32 models, whose _gmm falls to per-group matmuls for any
non-bf16 tensor, smel/moe.py:58-72, and whose own tests compare at 1e-5, tests/test_moe.py:10-36 and
tests/test_layer_major.py:86-134) against the oracle computed in fp64 and the reference's own fp32 golden outputs.

The bar is the reference's fp32 one: ||out - ref|| / ||ref|| <= 1e-5 (rel_err of smel/quant.py:108-110) for outputs,
dX and every LoRA gradient; the measured errors are printed."""
import itertools

import pytest
import torch

from helpers import LORA_NAMES, c1_layer, to_device_layer
from oracle import moe_ref as R

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 1e-5


def _say(msg):
    print(msg, flush=True)


def _check(out, ref, name, tol=TOL):
    e = R.rel_err(out.detach().cpu(), ref.detach().cpu())
    _say(f"  {name}: rel {e:.2e}")
    assert e <= tol, f"{name}: rel {e:.3e} > {tol}"
    return e


# ------------------------------------------------------------------------------------------------ GEMM primitives


def _int4_bank(E, R_, C, group, seed):
    g = torch.Generator().manual_seed(seed)
    return R.quantize_int4(torch.randn(E, R_, C, generator=g) * 0.05, group)


@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("kind", ["int4", "fp32", "sel", "int4_bf16"])
def test_gmm_f32_against_fp64(trans, kind, pad):
    """smel_gmm_f32 on a tile list of uneven groups (an empty one, one longer than a tile, rows not a multiple of 64,
    K not a multiple of 16, N not a multiple of 64), each weight kind, both orientations, with beta = 1 on top of a
    given C, against the fp64 per-group product."""
    from smel import _lib as L
    from smel import moe_f32 as F
    _say(f"gmm_f32 trans={trans} kind={kind} pad={pad}")
    torch.manual_seed(1)
    E, Rw, Cw, group = 5, 96, 136, 8     # one matrix [96][136]
    counts = [70, 0, 5, 130, 33]
    rows = sum(counts)
    q = _int4_bank(E, Rw, Cw, group, 3)
    if kind.startswith("int4"):
        deq = R.dequant_int4(q["q"], q["scale"], q["zero"], torch.bfloat16 if kind == "int4_bf16" else torch.float32)
        W = deq.double()
    else:
        Wf = torch.randn(E, Rw, Cw) * 0.05
        W = Wf.double()
    K, N = (Rw, Cw) if trans else (Cw, Rw)
    lda = K + pad                         # pad 3: not a multiple of 4, the scalar load path
    A = torch.randn(rows, lda)
    C0 = torch.randn(rows, N + 5)
    kconst = {"int4": L.KIND_INT4, "int4_bf16": L.KIND_INT4, "fp32": L.KIND_BF16, "sel": L.KIND_SEL}[kind]
    tl, _ = F.count_tiles(counts, kconst, DEV)
    if kind.startswith("int4"):
        dq = {k: v.to(DEV) for k, v in q.items()}
        w = F._ws(Rw, Cw, 1 << L.KIND_INT4, q4=L.ptr(dq["q"]), scale=L.ptr(dq["scale"]), zero=L.ptr(dq["zero"]))
        w.group = group
        w.q4_round_bf16 = int(kind == "int4_bf16")
    elif kind == "fp32":
        Wd = Wf.to(DEV)
        w = F._ws(Rw, Cw, 1 << L.KIND_BF16, wf=L.ptr(Wd))
    else:
        Wd = Wf.to(DEV)
        w = F._ws(Rw, Cw, 1 << L.KIND_SEL, wsel=L.ptr(Wd))
    Ad, Cd = A.to(DEV), C0.to(DEV)
    F.gmm(w, trans, tl, Ad, lda, Cd, N + 5, alpha=0.75, beta=1.0)
    torch.cuda.synchronize()
    ref = C0.double().clone()
    r = 0
    for e, c in enumerate(counts):
        We = W[e] if trans else W[e].t()
        ref[r:r + c, :N] += 0.75 * (A[r:r + c, :K].double() @ We)
        r += c
    _check(Cd.cpu(), ref, "C", tol=1e-6)


# (row counts of the groups, one matrix [R][C], int4 group): the tile shapes and load forms of smel_gmm_f32. The first
# has enough tiles for the 64 x 128 blocks (every number of 16-row slices, N and K over an edge); the next ones the
# 32 x 64 blocks (whole, with C not a multiple of 16, a group that is no power of two); then few output columns.
_MANY = [1, 16, 17, 33, 48, 49, 64, 65, 100, 0, 130, 5] * 6
GMM_SHAPES = [(_MANY, 840, 80, 16), ([40, 3, 70], 208, 144, 16), ([40, 3, 70], 132, 68, 4), ([65, 9], 192, 96, 48),
              ([70, 20], 1, 300, 4), ([33], 8, 2048, 64), ([64, 1], 16, 37 * 2, 2), ([50], 24, 132, 4),
              ([30, 17], 64, 512, 64)]


@pytest.mark.parametrize("kind", ["int4", "int4_bf16", "fp32"])
@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("shape", range(len(GMM_SHAPES)))
def test_gmm_f32_shapes_against_fp64(shape, trans, kind):
    """Every block shape and load form of smel_gmm_f32, forward and transposed, against the fp64 product; columns and
    rows outside the result stay untouched. Bound: sums of K <= 2048 fp32 products (rounded to 2^-24 each, errors adding
    as their square root against a sum that grows the same way) stay well inside 1e-6."""
    from smel import _lib as L
    from smel import moe_f32 as F
    counts, Rw, Cw, group = GMM_SHAPES[shape]
    if trans:
        Rw, Cw = (Cw, Rw) if kind == "fp32" or Rw % group == 0 else (Cw, (Rw + group - 1) // group * group)
    _say(f"gmm_f32 {Rw}x{Cw} trans={trans} kind={kind}")
    torch.manual_seed(shape)
    E, rows = len(counts), sum(counts)
    if kind.startswith("int4"):
        q = _int4_bank(E, Rw, Cw, group, shape)
        W = R.dequant_int4(q["q"], q["scale"], q["zero"],
                           torch.bfloat16 if kind == "int4_bf16" else torch.float32).double()
        dq = {k: v.to(DEV) for k, v in q.items()}
        w = F._ws(Rw, Cw, 1 << L.KIND_INT4, q4=L.ptr(dq["q"]), scale=L.ptr(dq["scale"]), zero=L.ptr(dq["zero"]))
        w.group, w.q4_round_bf16 = group, int(kind == "int4_bf16")
    else:
        Wf = torch.randn(E, Rw, Cw) * 0.05
        W, Wd = Wf.double(), Wf.to(DEV)
        w = F._ws(Rw, Cw, 1 << L.KIND_BF16, wf=L.ptr(Wd))
    K, N = (Rw, Cw) if trans else (Cw, Rw)
    tl, _ = F.count_tiles(counts, L.KIND_INT4 if kind.startswith("int4") else L.KIND_BF16, DEV)
    A, C0 = torch.randn(rows, K), torch.randn(rows + 1, N + 3)
    Ad = A.to(DEV)
    for beta in (0.0, 1.0):
        Cd = C0.to(DEV)
        F.gmm(w, trans, tl, Ad, K, Cd, N + 3, alpha=0.5, beta=beta)
        ref = C0.double().clone()
        ref[:rows, :N] *= beta
        r = 0
        for e, c in enumerate(counts):
            ref[r:r + c, :N] += 0.5 * (A[r:r + c].double() @ (W[e] if trans else W[e].t()))
            r += c
        got = Cd.cpu()
        _check(got[:rows, :N], ref[:rows, :N], "C", tol=1e-6)
        assert torch.equal(got[:, N:], C0[:, N:]) and torch.equal(got[rows], C0[rows])


# (N, K, group or 0 for fp32 weights, extra A columns) that need the forms for any alignment (quads with aligned rows and
# not, pairs, single elements), and short K (LoRA factors); enough tiles for the 64 x 128 blocks, and (counts of one group)
# the 32 x 64 ones
GMM_ANY = [(704, 104, 8, 0), (704, 100, 4, 1), (700, 74, 2, 0), (690, 70, 10, 3), (701, 77, 0, 0), (704, 80, 0, 1),
           (704, 192, 64, 1), (701, 16, 0, 0), (704, 48, 0, 0), (706, 32, 0, 0), (704, 8, 0, 0), (702, 96, 0, 0)]


@pytest.mark.parametrize("counts", [_MANY, [70, 3, 40]])
@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("shape", GMM_ANY)
def test_gmm_f32_any_alignment(shape, trans, counts):
    """The load forms of smel_gmm_f32 for any alignment and any group, and K of one or two steps, against the fp64 product:
    forward and transposed, beta 0 and 1, result rows on 8 bytes and not. K <= 192 fp32 products: inside 1e-6."""
    from smel import _lib as L
    from smel import moe_f32 as F
    N, K, group, pad = shape
    if group and trans:   # the group divides the matrix's columns, which are N here
        N = N // group * group
    Rw, Cw = (K, N) if trans else (N, K)
    E, rows = len(counts), sum(counts)
    g = torch.Generator().manual_seed(N + K)
    forms = [("fp32", 0)] if group == 0 else [("int4", 0), ("int4", 1)]
    for kind, rbf in forms:
        if kind == "int4":
            q = _int4_bank(E, Rw, Cw, group, K)
            W = R.dequant_int4(q["q"], q["scale"], q["zero"], torch.bfloat16 if rbf else torch.float32).double()
            dq = {k: v.to(DEV) for k, v in q.items()}
            w = F._ws(Rw, Cw, 1 << L.KIND_INT4, q4=L.ptr(dq["q"]), scale=L.ptr(dq["scale"]), zero=L.ptr(dq["zero"]))
            w.group, w.q4_round_bf16 = group, rbf
        else:
            Wf = torch.randn(E, Rw, Cw, generator=g) * 0.05
            W, Wd = Wf.double(), Wf.to(DEV)
            w = F._ws(Rw, Cw, 1 << L.KIND_BF16, wf=L.ptr(Wd))
        tl, _ = F.count_tiles(counts, L.KIND_INT4 if kind == "int4" else L.KIND_BF16, DEV)
        A = torch.randn(rows, K + pad, generator=g)
        A[:, K:] = float("nan")   # never read
        Ad = A.to(DEV)
        for beta in (0.0, 1.0):
            for extra in (2, 3):
                C0 = torch.randn(rows + 1, N + extra, generator=g)
                Cd = C0.to(DEV)
                F.gmm(w, trans, tl, Ad, K + pad, Cd, N + extra, alpha=0.5, beta=beta)
                ref = C0.double().clone()
                ref[:rows, :N] *= beta
                r = 0
                for e, c in enumerate(counts):
                    ref[r:r + c, :N] += 0.5 * (A[r:r + c, :K].double() @ (W[e] if trans else W[e].t()))
                    r += c
                got = Cd.cpu()
                _check(got[:rows, :N], ref[:rows, :N], "C", tol=1e-6)
                assert torch.equal(got[:, N:], C0[:, N:]) and torch.equal(got[rows], C0[rows])


# (output columns, K, int4 group) of the tiles whose fp32 products run as bf16 parts: K of one step of 32 to more than a
# round of four waves, columns over an edge of 128, one to many groups; counts over every number of 16-row slices of a pass
SPLIT_COUNTS = [1, 16, 17, 33, 48, 49, 64, 65, 97, 128, 130, 0] * 6


@pytest.mark.parametrize("kind", ["int4", "int4_bf16"])
@pytest.mark.parametrize("trans,N,K,group", [(0, 901, 32, 32), (0, 901, 192, 96), (0, 1024, 320, 64), (1, 960, 32, 32),
                                             (1, 960, 160, 96), (1, 1088, 288, 64)])
def test_gmm_f32_split_int4_tiles(trans, N, K, group, kind):
    """Rows of very different sizes, and rows with values that do not split into bf16 parts (infinities, NaN, the largest
    finite number), against the fp64 product. Bound of a finite row: at most 6 K / 32 + 5 <= 65 roundings of 2^-24 of the
    running sum, adding as their square root (5e-7 of the result's typical size |A row| std(W)), with a factor of 4 for
    the largest of a million results; a row that is not finite has the fp64 product's infinities and NaN."""
    from smel import _lib as L
    from smel import moe_f32 as F
    _say(f"gmm_f32 split N={N} K={K} g={group} trans={trans} kind={kind}")
    torch.manual_seed(N + K)
    counts, Rw, Cw = SPLIT_COUNTS, (K if trans else N), (N if trans else K)
    E, rows = len(counts), sum(counts)
    q = _int4_bank(E, Rw, Cw, group, 3)
    W = R.dequant_int4(q["q"], q["scale"], q["zero"],
                       torch.bfloat16 if kind == "int4_bf16" else torch.float32).double()
    dq = {k: v.to(DEV) for k, v in q.items()}
    w = F._ws(Rw, Cw, 1 << L.KIND_INT4, q4=L.ptr(dq["q"]), scale=L.ptr(dq["scale"]), zero=L.ptr(dq["zero"]))
    w.group, w.q4_round_bf16 = group, int(kind == "int4_bf16")
    tl, _ = F.count_tiles(counts, L.KIND_INT4, DEV)
    A = torch.randn(rows, K) * torch.exp2(torch.randint(-60, 60, (rows, 1)).float())
    for i, v in enumerate((float("inf"), float("-inf"), float("nan"), 3.4028234e38)):
        A[torch.arange(100 + i, rows, 997), i] = v
    Ad, Cd = A.to(DEV), torch.full((rows, N), 7.0, device=DEV)
    F.gmm(w, trans, tl, Ad, K, Cd, N, alpha=0.5, beta=0.0)
    got = Cd.cpu().double()
    off = 0
    for e, c in enumerate(counts):
        ref = 0.5 * (A[off:off + c].double() @ (W[e] if trans else W[e].t()))
        g = got[off:off + c]
        fin = ref.isfinite()
        assert torch.equal(fin, g.isfinite()), f"expert {e}"
        assert torch.equal(torch.nan_to_num(ref[~fin], nan=1.5, posinf=2.5, neginf=3.5),
                           torch.nan_to_num(g[~fin], nan=1.5, posinf=2.5, neginf=3.5)), f"expert {e}"
        size = (A[off:off + c].double() ** 2).sum(1, keepdim=True).sqrt() * W[e].std()
        ok = fin.all(1)
        assert ((g - ref).abs() <= 2e-6 * size)[ok].all(), f"expert {e}: {((g - ref).abs() / size)[ok].max():.2e}"
        off += c


def _split_case(trans, kind, N=1024, K=256, group=64, seed=11, bank=None):
    """(weight set, tile list, rows, expert of each row, dequantized fp64 weights as [E][K][N]) of a bank whose tiles run as
    bf16 parts; ``bank`` changes the quantized bank first."""
    from smel import _lib as L
    from smel import moe_f32 as F
    counts, Rw, Cw = SPLIT_COUNTS, (K if trans else N), (N if trans else K)
    q = _int4_bank(len(counts), Rw, Cw, group, seed)
    if bank is not None:
        bank(q)
    W = R.dequant_int4(q["q"], q["scale"], q["zero"],
                       torch.bfloat16 if kind == "int4_bf16" else torch.float32).double()
    dq = {k: v.to(DEV) for k, v in q.items()}
    w = F._ws(Rw, Cw, 1 << L.KIND_INT4, q4=L.ptr(dq["q"]), scale=L.ptr(dq["scale"]), zero=L.ptr(dq["zero"]))
    w.group, w.q4_round_bf16, w._keep = group, int(kind == "int4_bf16"), dq
    tl, _ = F.count_tiles(counts, L.KIND_INT4, DEV)
    return w, tl, sum(counts), torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts)), \
        (W if trans else W.transpose(1, 2)).to(DEV)


def _split_run(w, trans, tl, A, N):
    from smel import moe_f32 as F
    C = torch.full((A.shape[0], N), 7.0, device=DEV)
    F.gmm(w, trans, tl, A, A.shape[1], C, N)
    return C


def _split_ref(A, W, expert):
    ref, size = (torch.empty(A.shape[0], W.shape[2], dtype=torch.float64, device=DEV) for _ in range(2))
    for e in expert.unique().tolist():
        r = (expert == e).to(DEV)
        ref[r] = A[r].double() @ W[e]
        size[r] = A[r].double().abs() @ W[e].abs()
    return ref, size


@pytest.mark.parametrize("kind", ["int4", "int4_bf16"])
@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("terms", [1, 2, 8])
def test_gmm_f32_split_few_terms(terms, trans, kind):
    """Results that one, two or eight products carry. A product's parts are exact; its largest and the sum of the others
    (2^-8 of it, a few roundings of 2^-24 each) meet in one fp32 addition: 2^-24 (1 + 2^-6) of a lone product. Two terms
    in one k-step: the instruction's sum of the largest parts loses up to 2^-23, the addition of the others 2^-24; terms in
    different steps round once each and once more per addition: n + 1 units of 2^-24 of sum |x w| for n terms."""
    N, K = 1024, 256
    w, tl, rows, expert, W = _split_case(trans, kind, N, K)
    g = torch.Generator(device=DEV).manual_seed(terms)
    A = torch.randn(rows, K, generator=g, device=DEV)
    keep = torch.rand(rows, K, generator=g, device=DEV).argsort(1)[:, :terms]
    A = A * torch.zeros_like(A).scatter_(1, keep, 1.0)
    ref, size = _split_ref(A, W, expert)
    err = ((_split_run(w, trans, tl, A, N).double() - ref).abs() / size)[size > 0].max().item()
    assert err <= 2.0 ** -24 * (1 + 2.0 ** -6) * (1 if terms == 1 else terms + 1), err


@pytest.mark.parametrize("kind", ["int4", "int4_bf16"])
@pytest.mark.parametrize("trans", [0, 1])
def test_gmm_f32_split_small_values(trans, kind):
    """Rows near the small end of the exponent range (whole rows, and single values in ordinary rows whose other weights'
    products cancel to nothing against them): no parts are lost. Bound as for ordinary rows: K = 256 roundings of 2^-24 at
    worst, adding as their square root, times 4 for the largest of a million results."""
    N, K = 1024, 256
    w, tl, rows, expert, W = _split_case(trans, kind, N, K)
    g = torch.Generator(device=DEV).manual_seed(3)
    A = torch.randn(rows, K, generator=g, device=DEV)
    A = torch.where(A.abs() < 2.0 ** -4, torch.full_like(A, 0.3), A)   # results stay above the subnormal numbers
    scale = torch.tensor([0, -60, -71, -73, -90, -100, -108, -112, -114], device=DEV)
    A = torch.ldexp(A, scale[torch.arange(rows, device=DEV) % len(scale)][:, None])
    A[::7, 5:] = 0.0                                                      # few terms, and rows that hold zeros
    ref, size = _split_ref(A, W, expert)
    err = ((_split_run(w, trans, tl, A, N).double() - ref).abs() / size)[size > 0]
    assert err.max().item() <= 4 * 16 * 2.0 ** -24, err.max().item()
    # one value at 2^-100 beside zeros: the product itself, to one rounding
    A = torch.zeros_like(A)
    A[:, 9] = torch.ldexp(torch.rand(rows, generator=g, device=DEV) + 1.0, torch.tensor(-100, device=DEV))
    ref, size = _split_ref(A, W, expert)
    err = ((_split_run(w, trans, tl, A, N).double() - ref).abs() / size)[size > 0].max().item()
    assert err <= 2.0 ** -24, err


@pytest.mark.parametrize("kind", ["int4", "int4_bf16"])
@pytest.mark.parametrize("trans", [0, 1])
def test_gmm_f32_split_rows_are_independent(trans, kind):
    """A row's bits do not depend on its tile's other rows, whatever those hold."""
    N, K = 1024, 256
    w, tl, rows, expert, W = _split_case(trans, kind, N, K)
    A = torch.randn(rows, K, generator=torch.Generator(device=DEV).manual_seed(5), device=DEV)
    base = _split_run(w, trans, tl, A, N)
    odd = torch.arange(0, rows, 5, device=DEV)
    rest = torch.ones(rows, dtype=torch.bool, device=DEV)
    rest[odd] = False
    for v in (float("inf"), float("nan"), 3.4028234e38, 1e-30):
        B = A.clone()
        B[odd, 17] = v
        assert torch.equal(_split_run(w, trans, tl, B, N)[rest], base[rest]), v


@pytest.mark.parametrize("kind", ["int4", "int4_bf16"])
@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("form", ["zero_bank", "no_zero", "no_scale", "small_zero", "large_zero", "tiny", "one_group"])
def test_gmm_f32_split_weights(form, trans, kind):
    """Banks with groups whose weights are a sum of two bf16 values in other ways (all zero, scale or zero missing) or are
    not (a zero far below or above the scale, values near the small end), everywhere or in one group: one product's
    rounding in rows of one term (2^-24 for the fp32 instruction, (1 + 2^-6) of it in parts), and ordinary rows."""
    def bank(q):
        s, z = q["scale"], q["zero"]
        if form == "zero_bank":
            s.fill_(1e-8), z.zero_()
        elif form == "no_zero":
            z.zero_()
        elif form == "no_scale":
            s.zero_()
        elif form == "small_zero":
            z.copy_(s.float() * 2.0 ** -9)
        elif form == "large_zero":
            z.copy_(s.float() * 1021.0)
        elif form == "tiny":
            s.copy_(s.float() * 2.0 ** -60), z.copy_(z.float() * 2.0 ** -60)
        else:
            z[3, 5, 0] = 1e-7

    N, K = 1024, 256
    w, tl, rows, expert, W = _split_case(trans, kind, N, K, bank=bank)
    g = torch.Generator(device=DEV).manual_seed(7)
    A = torch.randn(rows, K, generator=g, device=DEV)
    A[::2] *= torch.zeros_like(A[::2]).scatter_(1, torch.randint(0, K, (A[::2].shape[0], 1), generator=g, device=DEV), 1.0)
    ref, size = _split_ref(A, W, expert)
    err = (_split_run(w, trans, tl, A, N).double() - ref).abs() / size.clamp_min(1e-300)
    assert err[::2].max().item() <= 2.0 ** -24 * (1 + 2.0 ** -6)
    assert err[1::2].max().item() <= 4 * 16 * 2.0 ** -24


@pytest.mark.parametrize("M,N", [(16, 200), (200, 16), (8, 36), (36, 33), (1, 64), (17, 65)])
def test_wgrad_f32_shapes_against_fp64(M, N):
    """smel_wgrad_f32 with either side the narrower one, sides off the block sizes, and row counts around the waves'
    strides (one row to several rounds of 256)."""
    from smel import moe_f32 as F
    torch.manual_seed(M * N)
    counts = [1, 255, 257, 900, 0, 31]
    offs = torch.tensor([0] + list(itertools.accumulate(counts)), dtype=torch.int32)
    X, Y = torch.randn(sum(counts), M), torch.randn(sum(counts), N + 4)
    jobs = torch.arange(len(counts), dtype=torch.int32)
    out = torch.full((len(counts), M, N), float("nan"), device=DEV)
    Xd, Yd, od, jd = X.to(DEV), Y.to(DEV), offs.to(DEV), jobs.to(DEV)
    F.wgrad(Xd, M, Yd, N + 4, od, jd, len(counts), M, N, 2.0, out)
    for j in range(len(counts)):
        r0, r1 = int(offs[j]), int(offs[j + 1])
        ref = 2.0 * X[r0:r1].double().t() @ Y[r0:r1, :N].double()
        if r1 == r0:
            assert torch.equal(out[j].cpu(), torch.zeros(M, N))
        else:
            _check(out[j].cpu(), ref, f"job {j}", tol=1e-6)


def test_wgrad_f32_against_fp64():
    """smel_wgrad_f32: per job, alpha X^T Y over its group's rows (an empty group writes zeros; M, N not multiples of
    64; rows not multiples of 16), against fp64."""
    from smel import moe_f32 as F
    _say("wgrad_f32")
    torch.manual_seed(2)
    counts = [37, 0, 200, 5]
    offs = torch.tensor([0] + list(itertools.accumulate(counts)), dtype=torch.int32)
    rows, M, N = sum(counts), 40, 136
    X, Y = torch.randn(rows, M + 4), torch.randn(rows, N)
    jobs = torch.tensor([2, 1, 0, 3], dtype=torch.int32)
    out = torch.full((4, M, N), float("nan"), device=DEV)
    Xd, Yd, od, jd = X.to(DEV), Y.to(DEV), offs.to(DEV), jobs.to(DEV)
    F.wgrad(Xd, M + 4, Yd, N, od, jd, 4, M, N, 0.5, out)
    torch.cuda.synchronize()
    for j, g in enumerate(jobs.tolist()):
        r0, r1 = int(offs[g]), int(offs[g + 1])
        ref = 0.5 * X[r0:r1, :M].double().t() @ Y[r0:r1].double()
        if r1 == r0:
            assert torch.equal(out[j].cpu(), torch.zeros(M, N))
        else:
            _check(out[j].cpu(), ref, f"job {j} (group {g})", tol=1e-6)


# ------------------------------------------------------------------------------------------------ router


@pytest.mark.parametrize("E", [8, 64, 256, 300])
def test_route_select_f32_given_logits(E):
    """Selection from given fp32 logits against torch on the CPU (fp32 softmax, top-k, renorm): the ids exactly
    (lower id first among equal probabilities, planted ties included), probs and topv to an fp32 ulp or two."""
    from smel import _lib as L
    _say(f"route_select_f32 E={E}")
    torch.manual_seed(E)
    T, K = 300, min(8, E)
    lg = torch.randn(T, E) * 2
    lg[:20, 5] = lg[:20, 3]               # ties: equal logits give equal probabilities
    lg[20:40, :] = 0.25
    probs = torch.empty(T, E, device=DEV)
    topv = torch.empty(T, K, device=DEV)
    topi = torch.empty(T, K, dtype=torch.int64, device=DEV)
    topi32 = torch.empty(T, K, dtype=torch.int32, device=DEV)
    lgd = lg.to(DEV)
    L.call("smel_route_select_f32", L.ptr(lgd), E, T, E, K, None, L.ptr(probs), L.ptr(topv), L.ptr(topi),
           L.ptr(topi32), L.stream())
    torch.cuda.synchronize()
    p_ref = torch.softmax(lg, -1)
    _, i_ref = R.topk_lowest_index(probs.cpu(), K)   # the tie rule on the kernel's own probabilities
    assert torch.equal(topi.cpu(), i_ref) and torch.equal(topi32.cpu().long(), i_ref)
    assert torch.allclose(probs.cpu(), p_ref, rtol=1e-6, atol=1e-9)
    v_ref, i_cpu = R.topk_lowest_index(p_ref, K)
    assert torch.equal(i_cpu, i_ref)
    assert torch.allclose(topv.cpu(), v_ref / v_ref.sum(-1, keepdim=True), rtol=1e-6, atol=1e-9)


def test_route_f32_api_forward_backward():
    """route() on fp32 tensors: probs / topv against fp64, the ids equal to those of the fp64 router (no near-ties
    at this size), dX through topv against fp64 autograd of the reference formula."""
    from smel.moe import route
    _say("route fp32 API")
    torch.manual_seed(5)
    T, H, E, K = 512, 256, 64, 8
    x = torch.randn(T, H)
    w = torch.randn(E, H) * 0.05
    xd = x.to(DEV).requires_grad_(True)
    probs, topv, topi = route(xd, w.to(DEV), K)
    assert topv.dtype == torch.float32 and probs.dtype == torch.float32 and topi.dtype == torch.int64
    gy = torch.randn(T, K)
    (topv * gy.to(DEV)).sum().backward()
    x64 = x.double().requires_grad_(True)
    p64, v64, i64 = R.route(x64, w.double(), K)
    assert torch.equal(topi.cpu(), i64)
    _check(probs.cpu(), p64, "probs")
    _check(topv.cpu(), v64, "topv")
    (v64 * gy.double()).sum().backward()
    _check(xd.grad.cpu(), x64.grad, "dx")


def test_route_gemma4_f32_forward_backward(golden_c1):
    """route_gemma4 on fp32 tensors: the reference's golden fp32 probs / topv / ids on the C1 input, and dH through
    topv against fp64 autograd of the reference formula."""
    from smel.moe import route_gemma4
    _say("route_gemma4 fp32")
    t = golden_c1
    W = {k[len("gemma."):]: v for k, v in t.items() if k.startswith("gemma.router")}
    h = t["in.x"].to(DEV).requires_grad_(True)
    probs, topv, topi = route_gemma4(h, {k: v.to(DEV) for k, v in W.items()}, 2, 1e-6)
    assert torch.equal(topi.cpu(), t["gemma.topi"])
    _check(probs.cpu(), t["gemma.probs"], "probs vs golden")
    _check(topv.cpu(), t["gemma.topv"], "topv vs golden")
    gy = torch.randn(topv.shape, generator=torch.Generator().manual_seed(0))
    (topv * gy.to(DEV)).sum().backward()
    h64 = t["in.x"].double().requires_grad_(True)
    W64 = {k: v.double() for k, v in W.items()}
    _, v64, _ = R.route_gemma4(h64, W64, 2, 1e-6, forced_topi=topi.cpu())
    (v64 * gy.double()).sum().backward()
    _check(h.grad.cpu(), h64.grad, "dh")


# ------------------------------------------------------------------------------------------------ experts and layer


def _layer(T=384, H=256, E=16, I=128, K=4, n_sel=3, r=8, shared=128, int4=True, act="silu", seed=0, deq=torch.float32):
    x, ol = R.make_layer(T, H, E, I, K, n_sel=n_sel, r=r, shared_inter=shared, int4=int4, seed=seed, act_name=act,
                         dtype=torch.float32, lora_b_std=0.05)
    ol.deq_dtype = deq
    return x, ol


def test_frozen_experts_fn_f32():
    """FrozenExpertsFn on fp32 rows with the reference test's counts (an empty expert), forward and dX, against the
    oracle's restatement of the reference's per-group dequant / recompute backward in fp64."""
    from smel.moe import FrozenExpertsFn
    _say("FrozenExpertsFn fp32")
    x, ol = _layer(E=6, n_sel=0, shared=None)
    counts = [9, 0, 12, 7, 15, 7]
    rows = sum(counts)
    xs = torch.randn(rows, x.shape[1])
    gy = torch.randn(rows, x.shape[1])
    W, ex, _ = to_device_layer(ol, DEV, torch.float32)
    xd = xs.to(DEV).requires_grad_(True)
    out = FrozenExpertsFn.apply(xd, counts, ex.frozen, 32, "silu")
    out.backward(gy.to(DEV))
    x64 = xs.double().requires_grad_(True)
    ref = R._FrozenExperts.apply(x64, counts, ol, torch.float64)
    ref.backward(gy.double())
    _check(out.detach().cpu(), ref.detach(), "out")
    _check(xd.grad.cpu(), x64.grad, "dx")


@pytest.mark.parametrize("case", ["int4_sel_lora", "fp32bank_sel_lora", "int4_frozen_only", "gelu_r48",
                                  "int4_bf16_dtype", "shared_split"])
def test_moe_forward_f32_against_fp64(case):
    """moe_forward on fp32 tensors (router, routed experts with selected experts and LoRA, shared expert and its
    gate): y, dX and every LoRA gradient against the fp64 oracle with the kernel's routing forced (as the
    reference's tests force HF's routing). Ranks above 32 run here (r = 48)."""
    from smel.moe import moe_forward
    _say(f"moe_forward fp32 {case}")
    kw = dict(int4=case != "fp32bank_sel_lora", n_sel=0 if case == "int4_frozen_only" else 3,
              act="gelu_tanh" if case == "gelu_r48" else "silu", r=48 if case == "gelu_r48" else 8,
              deq=torch.bfloat16 if case == "int4_bf16_dtype" else torch.float32, seed=sum(map(ord, case)) % 97)
    x, ol = _layer(**kw)
    K = 4
    gy = torch.randn(x.shape, generator=torch.Generator().manual_seed(1))
    W, ex, lora = to_device_layer(ol, DEV, torch.float32)
    if case == "shared_split":   # gate and up as separate tensors of the W dict
        assert "mlp.shared_expert.gate_proj.weight" in W
    else:                        # the stacked view LayerWeights makes
        Is = W["mlp.shared_expert.down_proj.weight"].shape[1]
        gu = torch.cat((W.pop("mlp.shared_expert.gate_proj.weight"), W.pop("mlp.shared_expert.up_proj.weight")))
        W["mlp.shared_expert.gate_up_proj.weight"] = gu
        W["mlp.shared_expert.gate_proj.weight"], W["mlp.shared_expert.up_proj.weight"] = gu[:Is], gu[Is:]
    xd = x.to(DEV).requires_grad_(True)
    seen = {}
    y = moe_forward(xd, W, ex, K, lora, stats=lambda p, v, i: seen.update(p=p, v=v, i=i.clone()))
    assert y.dtype == torch.float32 and seen["p"].dtype == torch.float32 and seen["v"].dtype == torch.float32
    y.backward(gy.to(DEV))
    torch.cuda.synchronize()
    y64, dx64, g64 = R.moe_forward_backward(x, ol, K, gy, forced_topi=seen["i"].cpu(), dtype=torch.float64)
    _check(y.detach().cpu(), y64, "y")
    _check(xd.grad.cpu(), dx64, "dx")
    if lora is not None:
        for tag, mod in (("ex", lora.experts), ("sh", lora.shared)):
            if mod is None:
                continue
            for n in LORA_NAMES:
                _check(getattr(mod, n).grad.cpu(), g64[f"{tag}_{n}"], f"d_{tag}_{n}")


def test_mlp_lora_f32_gelu_nd():
    """mlp_lora on a 3-D fp32 input (GeGLU, separate gate / up weights, LoRA r=16): y, dX and the LoRA gradients
    against the fp64 plain formula (the reference's lora_linear / lora_gate_up)."""
    from smel.lora import MLPLoRA
    from smel.moe import mlp_lora
    _say("mlp_lora fp32 GeGLU 3-D")
    torch.manual_seed(7)
    B, S, H, I, r = 3, 50, 192, 160, 16
    x = torch.randn(B, S, H)
    wg, wu, wd = torch.randn(I, H) * 0.05, torch.randn(I, H) * 0.05, torch.randn(H, I) * 0.05
    lo = MLPLoRA(H, I, r, 32.0)
    with torch.no_grad():
        for n in ("B_gate", "B_up", "B_down"):
            getattr(lo, n).normal_(0, 0.05)
    lod = MLPLoRA(H, I, r, 32.0).to(DEV)
    with torch.no_grad():
        for n in LORA_NAMES:
            getattr(lod, n).copy_(getattr(lo, n))
    xd = x.to(DEV).requires_grad_(True)
    y = mlp_lora(xd, wg.to(DEV), wu.to(DEV), wd.to(DEV), lod, act_name="gelu_tanh")
    gy = torch.randn(B, S, H)
    y.backward(gy.to(DEV))
    x64 = x.double().reshape(-1, H).requires_grad_(True)
    L64 = {n: getattr(lo, n).detach().double().requires_grad_(True) for n in LORA_NAMES}
    y64 = R.mlp_lora(x64, torch.cat((wg, wu)).double(), wd.double(), L64, lo.scale, "gelu_tanh")
    y64.backward(gy.double().reshape(-1, H))
    _check(y.detach().cpu().reshape(-1, H), y64.detach(), "y")
    _check(xd.grad.cpu().reshape(-1, H), x64.grad, "dx")
    for n in LORA_NAMES:
        _check(getattr(lod, n).grad.cpu(), L64[n].grad, f"d_{n}")


def test_c1_golden_f32(golden_c1):
    """moe_forward on the reference's own C1 inputs in fp32 (the golden outputs were written by the reference's fp32
    path): the HIP router's ids equal the golden ones, and y, dX and all twelve LoRA gradients match the golden
    values at the reference's fp32 bar."""
    from smel.moe import moe_forward
    _say("C1 golden fp32")
    t = golden_c1
    W, ex, lora = to_device_layer(c1_layer(t), DEV, torch.float32)
    x = t["in.x"].to(DEV).requires_grad_(True)
    seen = {}
    y = moe_forward(x, W, ex, 2, lora, stats=lambda p, v, i: seen.update(p=p.clone(), v=v.clone(), i=i.clone()))
    y.backward(t["in.gy"].to(DEV))
    torch.cuda.synchronize()
    assert torch.equal(seen["i"].cpu(), t["out.topi"])
    _check(seen["p"].cpu(), t["out.probs"], "probs")
    _check(seen["v"].cpu(), t["out.topv"], "topv")
    _check(y.detach().cpu(), t["out.y"], "y")
    _check(x.grad.cpu(), t["out.dx"], "dx")
    for tag, mod in (("ex", lora.experts), ("sh", lora.shared)):
        for n in LORA_NAMES:
            _check(getattr(mod, n).grad.cpu(), t[f"out.d_{tag}_{n}"], f"d_{tag}_{n}")


def test_c1_golden_f32_frozen_only(golden_c1):
    """The golden frozen-only layer (no selected experts, no LoRA) in fp32: y and dX."""
    from smel.moe import moe_forward
    t = golden_c1
    W, ex, _ = to_device_layer(c1_layer(t, with_sel=False), DEV, torch.float32)
    x = t["in.x"].to(DEV).requires_grad_(True)
    y = moe_forward(x, W, ex, 2, None)
    y.backward(t["in.gy"].to(DEV))
    _check(y.detach().cpu(), t["out.y_frozen_only"], "y")
    _check(x.grad.cpu(), t["out.dx_frozen_only"], "dx")


def test_routed_experts_f32_bad_ids_reported():
    """fp32 routed_experts with an expert id outside [0, E): the slot is dropped (a zero row) and the error is
    reported without a host synchronisation, by check_routing_errors()."""
    from smel.moe import check_routing_errors, routed_experts
    x, ol = _layer(n_sel=0, shared=None)
    W, ex, _ = to_device_layer(ol, DEV, torch.float32)
    T = x.shape[0]
    topi = torch.randint(0, ol.E, (T, 4)).to(DEV)
    topi[3, 1] = ol.E + 2
    topv = torch.full((T, 4), 0.25, device=DEV)
    routed_experts(x.to(DEV), topv, topi, ex)
    with pytest.raises(IndexError):
        check_routing_errors()
    check_routing_errors()   # reported once


# ------------------------------------------------------------------------------------------------ bf16 beyond the bf16 kernels


@pytest.mark.parametrize("case", ["rank48", "hidden200_group8", "inter100"])
def test_bf16_layer_outside_bf16_kernel_limits(case):
    """bf16 activations of shapes the bf16 kernels do not take (LoRA rank above 32, a hidden size that is not a
    multiple of 64 with int4 groups of 8, an expert / shared intermediate size that is not a multiple of 32) run on
    the fp32 kernels with bf16 in and out: y, dX and every LoRA gradient against the fp32 oracle at the bf16 bar
    (the reference takes these shapes; its bf16 tests compare at 2e-2)."""
    from helpers import assert_close_bf16
    from smel.moe import moe_forward
    _say(f"bf16 layer beyond the bf16 kernels: {case}")
    H, I, group, r = {"rank48": (256, 128, 64, 48), "hidden200_group8": (200, 96, 8, 8),
                      "inter100": (256, 100, 4, 16)}[case]
    x, ol = R.make_layer(320, H, 16, I, 4, n_sel=3, r=r, shared_inter=I, group=group, seed=11, lora_b_std=0.05)
    W, ex, lora = to_device_layer(ol, DEV)
    gy = torch.randn(x.shape, generator=torch.Generator().manual_seed(2)).bfloat16()
    xd = x.to(DEV).requires_grad_(True)
    seen = {}
    y = moe_forward(xd, W, ex, 4, lora, stats=lambda p, v, i: seen.update(v=v, i=i.clone()))
    assert y.dtype == torch.bfloat16 and seen["v"].dtype == torch.bfloat16
    y.backward(gy.to(DEV))
    torch.cuda.synchronize()
    y32, dx32, g32 = R.moe_forward_backward(x.float(), ol, 4, gy.float(), forced_topi=seen["i"].cpu(),
                                            dtype=torch.float32)
    e, m, c = assert_close_bf16(y.detach().float().cpu(), y32, "y")
    _say(f"  y: rel {e:.2e} cos {c:.7f}")
    e, m, c = assert_close_bf16(xd.grad.float().cpu(), dx32, "dx")
    _say(f"  dx: rel {e:.2e} cos {c:.7f}")
    for tag, mod in (("ex", lora.experts), ("sh", lora.shared)):
        for n in LORA_NAMES:
            e, m, c = assert_close_bf16(getattr(mod, n).grad.float().cpu(), g32[f"{tag}_{n}"], f"d_{tag}_{n}")
            _say(f"  d_{tag}_{n}: rel {e:.2e}")


def test_bf16_frozen_experts_and_route_hidden_200():
    """FrozenExpertsFn and route() on bf16 rows whose hidden size (200) the bf16 kernels do not take: the fp32 kernels
    with bf16 in and out, against the fp32 oracle at the bf16 bar; the router's ids equal the oracle's on the same
    logits' ordering (no near-ties here)."""
    from helpers import assert_close_bf16
    from smel.moe import FrozenExpertsFn, route
    _say("bf16 FrozenExpertsFn / route, hidden 200")
    x, ol = R.make_layer(256, 200, 6, 96, 2, n_sel=0, group=8, seed=4)
    W, ex, _ = to_device_layer(ol, DEV)
    counts = [9, 0, 12, 7, 15, 7]
    xs = x[:sum(counts)].bfloat16()
    gy = torch.randn(xs.shape, generator=torch.Generator().manual_seed(3)).bfloat16()
    xd = xs.to(DEV).requires_grad_(True)
    out = FrozenExpertsFn.apply(xd, counts, ex.frozen, 32, "silu")
    assert out.dtype == torch.bfloat16
    out.backward(gy.to(DEV))
    x32 = xs.float().requires_grad_(True)
    ref = R._FrozenExperts.apply(x32, counts, ol, torch.float32)
    ref.backward(gy.float())
    assert_close_bf16(out.detach().float().cpu(), ref.detach(), "out")
    assert_close_bf16(xd.grad.float().cpu(), x32.grad, "dx")
    xr = x.bfloat16().to(DEV)
    probs, topv, topi = route(xr, W["mlp.gate.weight"], 2)
    assert topv.dtype == torch.bfloat16
    p32, _, i32 = R.route(x.bfloat16().float(), ol.gate_w.float(), 2)
    assert torch.equal(topi.cpu(), i32)
    assert_close_bf16(probs.cpu(), p32, "probs", rel=1e-5)
