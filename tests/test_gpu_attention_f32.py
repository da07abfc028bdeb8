"""GPU parity: attention on the f32 matrix cores (float32, and bfloat16 head widths off 32 / 64 / 128)
at the edges of its 32-row tiles, its four-wave split and its padded widths."""
import numpy as np
import pytest
import torch

from oracle import scans
from tests.conftest import assert_close
from tests.gpu_util import TOL, announce, host, rounded, to_dev

pytestmark = pytest.mark.gpu


def _run(q, k, v, do, dtype, causal, cs=None):
    from edifice_amd import fused_scan as fs
    ts = [to_dev(a, dtype).requires_grad_() for a in (q, k, v)]
    if cs is not None:
        ts.append(to_dev(cs, dtype).requires_grad_())
        out = fs.fox_attention(*ts)
    else:
        out = fs.flash_attention(*ts, causal=causal)
    return [out] + list(torch.autograd.grad(out, ts, to_dev(do, dtype)))


# float32 sums of up to a few hundred terms differ from float64 by a few 1e-7 of the largest value
# (measured 5e-7); bfloat16 results by their rounding, half an ulp = 2^-9 of a value
REL = {torch.float32: 5e-6, torch.bfloat16: 2.0 ** -8}
# the bfloat16 gradients also take D = rowsum(dO o O) from the rounded O: an error of 2^-9 |dO| |O| in every
# dP - D, whose own size is the spread of dO . V over the keys, which the fewest keys leave smallest (two: a
# quarter of |dO| |V| is common), so 8 x 2^-9
REL_GRAD = {torch.float32: 5e-6, torch.bfloat16: 2.0 ** -6}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("shape", [(1, 1, 2, 5), (2, 1, 31, 24), (1, 3, 33, 36), (1, 2, 129, 96), (1, 1, 160, 33),
                                   (1, 2, 97, 104), (1, 1, 300, 80), (3, 1, 64, 128), (1, 2, 130, 72), (1, 1, 257, 120), (2, 1, 65, 8)])
def test_attention_tile_edges(shape, causal, dtype, rng):
    if dtype == torch.bfloat16 and shape[3] in (32, 64, 128):
        pytest.skip("bf16 at this width takes the bf16 kernels")
    announce("attention_tile_edges", shape=shape, causal=causal, dtype=dtype)
    q, k, v, do = (rng.normal(scale=shape[3] ** -0.25, size=shape) for _ in range(4))
    got = _run(q, k, v, do, dtype, causal)
    qr, kr, vr, dor = (rounded(a, dtype) for a in (q, k, v, do))
    want = [scans.flash_attention(qr, kr, vr, causal), *scans.flash_attention_backward(qr, kr, vr, dor, causal)]
    for name, g, w in zip(("o", "dq", "dk", "dv"), got, want):
        err = np.linalg.norm(host(g) - w) / np.linalg.norm(w)
        assert err <= (REL if name in ("o", "dv") else REL_GRAD)[dtype], f"{name}: {err:.2e}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", [(1, 2, 70, 48), (1, 1, 33, 128), (2, 1, 40, 7)])
def test_fox_tile_edges(shape, dtype, rng):
    if dtype == torch.bfloat16 and shape[3] == 128:
        pytest.skip("bf16 at this width takes the bf16 kernels")
    announce("fox_tile_edges", shape=shape, dtype=dtype)
    q, k, v, do = (rng.normal(scale=shape[3] ** -0.25, size=shape) for _ in range(4))
    cs = np.cumsum(-np.abs(rng.normal(scale=0.2, size=shape[:3])), axis=-1)
    got = _run(q, k, v, do, dtype, True, cs)
    qr, kr, vr, cr, dor = (rounded(a, dtype) for a in (q, k, v, cs, do))
    want = [scans.fox_attention(qr, kr, vr, cr), *scans.fox_attention_backward(qr, kr, vr, cr, dor)]
    for name, g, w in zip(("o", "dq", "dk", "dv", "dcs"), got, want):
        assert_close(host(g), w, TOL[dtype], name)


@pytest.mark.parametrize("d,dtype", [(64, torch.float32), (40, torch.float32), (33, torch.float32),
                                     (96, torch.bfloat16), (40, torch.bfloat16), (104, torch.bfloat16),
                                     (36, torch.bfloat16)], ids=str)
def test_masked_values_take_no_part(d, dtype, rng):
    """Causal rows before a position do not see it: with q, k, v (and the output gradient) infinite
    or NaN from row 70 on, the first 70 rows of the output and of dQ are those of the finite call (to
    float32 rounding: the tile holding row 70 sums its visible pairs one by one), and so are the later
    rows of dK and dV where the earlier rows' output gradient is infinite."""
    announce("masked_values", d=d, dtype=dtype)
    shape, cut = (1, 2, 90, d), 70
    q, k, v, do = (rng.normal(scale=d ** -0.25, size=shape) for _ in range(4))
    do[:, :, cut:] = 0
    near = dict(rtol=1e-4, atol=1e-6) if dtype == torch.float32 else dict(rtol=2.0 ** -7, atol=1e-4)
    base = _run(q, k, v, do, dtype, True)
    bad_k, bad_v = k.copy(), v.copy()
    bad_k[:, :, cut:] = np.inf
    bad_v[:, :, cut:] = np.nan
    bad_v[:, :, cut + 2:, ::3] = -np.inf
    got = _run(q, bad_k, bad_v, do, dtype, True)
    assert torch.allclose(got[0][:, :, :cut], base[0][:, :, :cut], **near)
    assert torch.allclose(got[1][:, :, :cut], base[1][:, :, :cut], **near)
    # keys from row 70 on see only later queries: the earlier ones, infinite, take no part
    do2 = do.copy()
    do2[:, :, cut:] = rng.normal(size=do2[:, :, cut:].shape)
    base = _run(q, k, v, do2, dtype, True)
    bad_do = do2.copy()
    bad_do[:, :, :cut] = np.inf
    got = _run(q, k, v, bad_do, dtype, True)
    for i in (2, 3):
        assert torch.allclose(got[i][:, :, cut:], base[i][:, :, cut:], **near)


@pytest.mark.parametrize("d,dtype", [(40, torch.float32), (64, torch.float32), (128, torch.float32),
                                     (36, torch.bfloat16), (96, torch.bfloat16)], ids=str)
@pytest.mark.parametrize("kind", ["plain", "causal", "fox"])
def test_only_visible_score_of_a_tile_is_minus_infinity(kind, d, dtype, rng):
    """A key whose score is -inf has probability 0, also where it is all that a query sees of a 32-key tile:
    causal, key 32 is all that query 32 sees of its last tile; otherwise it is the whole last tile of 33 keys."""
    announce("minus_infinity_tile", kind=kind, d=d, dtype=dtype)
    shape = (1, 2, 33 if kind == "plain" else 40, d)
    q, k, v, do = (rng.normal(scale=d ** -0.25, size=shape) for _ in range(4))
    q[..., 0] = -np.abs(q[..., 0]) - 0.1
    k[:, :, 32, 0] = np.inf
    cs = np.cumsum(-np.abs(rng.normal(scale=0.2, size=shape[:3])), axis=-1) if kind == "fox" else None
    got = _run(q, k, v, do, dtype, kind != "plain", cs)
    qr, kr, vr, dor = (rounded(a, dtype) for a in (q, k, v, do))
    kr[:, :, 32] = 0  # its score enters nothing: the reference leaves the key out by a bias
    s = np.einsum("bhid,bhjd->bhij", qr, kr) / np.sqrt(d)
    if kind == "fox":
        cr = rounded(cs, dtype)
        s += cr[..., :, None] - cr[..., None, :]
    if kind != "plain":
        s = np.where(np.tril(np.ones(s.shape[-2:], bool)), s, -np.inf)
    s[..., 32] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    assert_close(host(got[0]), np.einsum("bhij,bhjd->bhid", p, vr), TOL[dtype], "o")
    assert_close(host(got[3]), np.einsum("bhij,bhid->bhjd", p, dor), TOL[dtype], "dv")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("kind", ["plain", "causal", "fox"])
@pytest.mark.parametrize("d", [40, 72, 100, 130, 192, 256])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 24, 25, 32, 33])
def test_short_sequences_and_wide_heads(T, d, kind, dtype, rng):
    """Both sides of the lengths at which one wave per query gives way to tiles, and heads wider than 128, which
    keep it."""
    announce("short_and_wide", T=T, d=d, kind=kind, dtype=dtype)
    shape = (2, 3, T, d)
    q, k, v, do = (rng.normal(scale=d ** -0.25, size=shape) for _ in range(4))
    cs = np.cumsum(-np.abs(rng.normal(scale=0.2, size=shape[:3])), axis=-1) if kind == "fox" else None
    got = _run(q, k, v, do, dtype, kind == "causal", cs)
    qr, kr, vr, dor = (rounded(a, dtype) for a in (q, k, v, do))
    if kind == "fox":
        cr = rounded(cs, dtype)
        want = [scans.fox_attention(qr, kr, vr, cr), *scans.fox_attention_backward(qr, kr, vr, cr, dor)]
    else:
        want = [scans.flash_attention(qr, kr, vr, kind == "causal"),
                *scans.flash_attention_backward(qr, kr, vr, dor, kind == "causal")]
    for name, g, w in zip(("o", "dq", "dk", "dv", "dcs"), got, want):
        # one key: dq, dk and dcs are exactly 0, what is left of dP - D is the rounding of its two equal terms
        floor = 1.0 if T == 1 and name in ("dq", "dk", "dcs") else np.abs(w).max()
        assert np.abs(host(g) - w).max() <= TOL[dtype] * floor, name
