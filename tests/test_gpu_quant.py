"""GPU int4 quantizer (smel_quantize_int4 through smel.quant.quantize_int4) against the reference's own bytes and
against the oracle's restatement of the reference's algorithm in torch ops (oracle/moe_ref.py, smel/quant.py:5-44).

Bar: the reference's golden bytes (tests/golden/quant_int4.safetensors, written by the reference's quantize_int4)
bit for bit. On larger random banks, every group's q equals clamp(rint((w - zero) / scale), 0, 15) for the scale
and zero it chose, and scale / zero equal those of the oracle's restatement in every group. The reference leaves
the order of the clip search's error sum to its library, so two candidates whose error sums agree to within fp32
rounding could be chosen differently; on these banks no group does (0 of 165 120 groups, the bound below), and the
fp64 check of such a tie stays in place for any bank that shows one."""
import os

import pytest
import torch

from oracle import moe_ref as R

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "quant_int4.safetensors")
CASES = ("normal", "outlier", "g32", "grid", "e20")
TIES_SEEN = 0   # groups of a random bank below whose clip choice differs from the restatement's (observed: none)


@pytest.fixture(scope="module")
def quant():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from smel import quant
    return quant


@pytest.mark.parametrize("case", CASES)
def test_golden_bytes(quant, case):
    from safetensors.torch import load_file
    g = load_file(GOLDEN)
    w = g[f"quant.{case}.w"].cuda()
    pk = quant.quantize_int4(w, 32 if case == "g32" else 64)
    assert torch.equal(pk["q"].cpu(), g[f"quant.{case}.q"])
    assert torch.equal(pk["scale"].cpu().view(torch.int16), g[f"quant.{case}.scale"].view(torch.int16))
    assert torch.equal(pk["zero"].cpu().view(torch.int16), g[f"quant.{case}.zero"].view(torch.int16))


def unpack(q):
    return torch.stack((q & 15, q >> 4), -1).reshape(*q.shape[:-1], q.shape[-1] * 2).float()


def group_err64(w, q, s, z, group):
    wg = w.double().reshape(*w.shape[:-1], -1, group)
    qg = q.double().reshape(wg.shape)
    return ((qg * s.double()[..., None] + z.double()[..., None] - wg) ** 2).sum(-1)


@pytest.mark.parametrize("dtype,group,shape", [(torch.bfloat16, 64, (8, 512, 2048)), (torch.float32, 32, (4, 256, 512)),
                                               (torch.bfloat16, 128, (4, 512, 1024)), (torch.float16, 64, (2, 64, 640))])
def test_random_banks(quant, dtype, group, shape):
    print(f"quant {dtype} g{group} {shape}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(group)
    w = (torch.randn(*shape, generator=g, device="cuda") * 0.02).to(dtype)
    w[0, 0, :group] = 0.0                                   # a constant group: scale clamps to 1e-8
    w[0, 1, :group] *= 50                                    # an outlier group
    got = quant.quantize_int4(w, group)
    ref = R.quantize_int4(w.cpu(), group)
    s, z = got["scale"].cpu().float(), got["zero"].cpu().float()
    # q is exactly the rounding of w for the chosen (scale, zero)
    wg = w.cpu().float().reshape(*shape[:-1], -1, group)
    qx = torch.round((wg - z[..., None]) / s[..., None]).clamp_(0, 15).reshape(*shape)
    assert torch.equal(unpack(got["q"].cpu()), qx)
    diff = (got["scale"].cpu().view(torch.int16) != ref["scale"].view(torch.int16)) | \
           (got["zero"].cpu().view(torch.int16) != ref["zero"].view(torch.int16))
    n = int(diff.sum())
    print(f"  {n} of {diff.numel()} groups chose another clip factor than the torch restatement", flush=True)
    assert n <= TIES_SEEN, f"{n} of {diff.numel()} groups chose another clip factor"
    if n:
        e_got = group_err64(w.cpu(), unpack(got["q"].cpu()), got["scale"].cpu().float(), got["zero"].cpu().float(),
                            group)[diff]
        e_ref = group_err64(w.cpu(), unpack(ref["q"]), ref["scale"].float(), ref["zero"].float(), group)[diff]
        assert torch.all((e_got - e_ref).abs() <= 2e-5 * torch.maximum(e_got, e_ref)), (e_got, e_ref)
    same = ~diff
    qa = got["q"].cpu().reshape(*shape[:-1], -1, group // 2)[same]
    qb = ref["q"].reshape(*shape[:-1], -1, group // 2)[same]
    assert torch.equal(qa, qb)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("group", [32, 64, 128])
def test_division_free_form_equals_the_division(quant, dtype, group):
    """The register kernels (no division) against the general kernel (the reference's division), which a start off the
    16-byte grid selects: the same bytes, on random values, on coarse grids where weights fall on the rounding ties,
    with tiny and huge ranges, infinities and NaN, and under odd clip factors."""
    g = torch.Generator(device="cuda").manual_seed(group)
    n = 64 * group
    rnd = torch.randn(48, n, generator=g, device="cuda")
    w = rnd * torch.logspace(-30, 4, 48, device="cuda")[:, None]
    w[8:16] = torch.round(rnd[8:16] * 8) / 16             # grids: many exact ties
    w[16:20] = torch.randint(-15, 16, (4, n), generator=g, device="cuda").float() * 0.03125
    w[20] = 0.25
    if dtype != torch.float16:
        w[21] = rnd[21] * 1e30                            # past the register form's range
        w[22] = rnd[22] * 1e-38
    w[23, ::group], w[24, 5::group], w[25, 7::3 * group] = float("inf"), float("-inf"), float("nan")
    w[26, :group] = float("nan")
    w = w.to(dtype)
    off = torch.empty(w.numel() + 8, dtype=dtype, device="cuda")
    off[1:1 + w.numel()] = w.reshape(-1)
    shifted = off[1:1 + w.numel()].view(w.shape)
    assert shifted.data_ptr() % 16 and w.data_ptr() % 16 == 0
    for clip in ((1.0, 0.95, 0.9, 0.85, 0.8), (0.0, 3.0, -1.0), (1e20, 1.0)):
        a, b = quant.quantize_int4(w, group, clip), quant.quantize_int4(shifted, group, clip)
        assert torch.equal(a["q"], b["q"])
        for k in ("scale", "zero"):
            assert torch.equal(a[k].view(torch.int16), b[k].view(torch.int16))


def test_bad_group_is_an_assertion(quant):
    with pytest.raises(AssertionError):
        quant.quantize_int4(torch.randn(2, 48, device="cuda"), 64)


def test_host_tensor_goes_through_the_gpu(quant):
    """A host tensor is quantized by the same kernel and comes back on the host, equal to the device result."""
    w = torch.randn(3, 8, 128) * 0.02
    a, b = quant.quantize_int4(w, 64), quant.quantize_int4(w.cuda(), 64)
    for k in ("q", "scale", "zero"):
        assert not a[k].is_cuda and torch.equal(a[k], b[k].cpu())
    e = quant.quantize_int4(torch.empty(0, 64, device="cuda"), 64)
    assert e["q"].shape == (0, 32) and e["scale"].shape == (0, 1)
