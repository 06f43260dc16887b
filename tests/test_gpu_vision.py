"""Vision tower on the gfx950 kernels against the CPU oracle (oracle/vision.py).

Tolerances (stated per op):
* bit-exact: pixel packing (the same fp32 quotient rounded once), the vision
  rotary (the same two fp32 products and sum, rounded once), the zero-padded
  V^T layout, the interpolated position embedding (fp32 products summed in tap
  order), graph replays against the eager step.
* LayerNorm: <= 1 bf16 ulp, exact for all but 2% (fp32 statistics summed in a
  different order than the oracle's).
* bf16 linear (+ GELU / residual): within 1 bf16 ulp + 2^-16 * sum_k |a_k w_k|
  of the fp64 product before the epilogue's rounding, and equal to the oracle's
  bf16 output for >= 95% of the elements; after GELU / residual within 2 ulps
  + that bound (an absolute bound: outputs near zero after cancellation carry
  it), equal for >= 90%.
* attention: |gpu - oracle| <= 1/64 absolute and relative RMS <= 0.5% (P rounded
  to bf16 inside the online softmax; the oracle is exact fp64).
* whole tower (teacher-forced per block and end to end over 3 blocks):
  relative L2 <= 1% per block output, <= 2% for the merged and DeepStack
  features; the full 27-block 8B tower teacher-forced to the same bars per
  block and merger, and end to end within 3%.
"""
import numpy as np
import pytest
import torch

from oracle import vision as OV
from tests.helpers import assert_bf16_close, bf16_ulps

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16
F32 = torch.float32
DEV = "cuda"


def _g(seed):
    return torch.Generator().manual_seed(seed)


def _rel_l2(a, b):
    a, b = a.float().cpu(), b.float().cpu()
    return float((a - b).norm() / b.norm())


def test_pack_pixels_bit_exact(gpu):
    from fastforward_amd.vision import pack_rgb
    rng = np.random.default_rng(3)
    for h, w in ((64, 96), (32, 32), (128, 64)):
        rgb = rng.integers(0, 256, size=(h, w, 3), dtype=np.uint8)
        got = pack_rgb(torch.from_numpy(rgb).to(DEV)).cpu()
        assert torch.equal(got, OV.pack_pixels(rgb)), (h, w)


@pytest.mark.parametrize("rows,h", [(37, 1152), (5, 4608), (64, 1024), (3, 64)])
def test_layer_norm(gpu, rows, h):
    from fastforward_amd.vision import Norm, layer_norm
    x = (torch.randn(rows, h, generator=_g(h)) * 3 + 0.5).to(BF16)
    w = (1 + 0.2 * torch.randn(h, generator=_g(h + 1))).to(BF16)
    b = (0.3 * torch.randn(h, generator=_g(h + 2))).to(BF16)
    got = layer_norm(x.to(DEV), Norm(w.to(DEV), b.to(DEV)), 1e-6).cpu()
    assert_bf16_close(got, OV.layer_norm(x, w, b, 1e-6), max_ulps=1, max_frac=0.02, what="layer_norm")


def _ulp(x):
    return torch.from_numpy(2.0 ** (np.floor(np.log2(np.maximum(np.abs(x.numpy()), 2.0 ** -126))) - 7))


def _linear_bound(x, w, b):
    """(exact, |y - exact| allowed before the epilogue rounding): 1 bf16 ulp +
    2^-16 sum_k |a_k w_k| (fp32 accumulation of exact bf16 products)."""
    xd, wd = x.to(torch.float64), w.to(torch.float64)
    exact = xd @ wd.T + b.to(torch.float64)
    mag = xd.abs() @ wd.abs().T
    return exact, _ulp(exact) + mag * 2.0 ** -16


def _assert_within(got, want, slack, what):
    """|got - want| <= 2 bf16 ulps of want + slack (an absolute bound carried from
    the GEMM), and equal to the oracle's bf16 value for >= 90% of the elements."""
    g, w_ = got.to(torch.float64), want.to(torch.float64)
    d = (g - w_).abs()
    ok = d <= 2 * _ulp(w_) + slack
    assert bool(ok.all()), f"{what}: {int((~ok).sum())} elements outside the bound"
    eq = float((got.to(BF16) == want.to(BF16)).float().mean())
    assert eq >= 0.9, f"{what}: only {eq:.3f} of the elements equal the oracle's"


def _assert_epilogues(x, w, b, h, run):
    """The bf16 linear's outputs against references of their own: the plain product within
    the fp32-accumulation bound of the 64-bit one, and from its bf16 values v, bit for
    bit, the activations (torch's ops on v) and the residual add (bf16(h + v)).
    run(act, resid) -> the output; h None: no residual. All on the device."""
    exact, bound = _linear_bound(x.cpu(), w.cpu(), b.cpu())
    v = run(0, None)
    assert bool(((v.cpu().to(torch.float64) - exact).abs() <= bound).all())
    assert torch.equal(run(1, None), torch.nn.functional.gelu(v, approximate="tanh"))
    assert torch.equal(run(2, None), torch.nn.functional.gelu(v))
    if h is not None:
        assert torch.equal(run(0, h), (h.float() + v.float()).to(BF16))


@pytest.mark.parametrize("m,n,k", [(300, 256, 1152), (64, 3456, 1152), (513, 1152, 4352), (2048, 512, 1536)])
def test_gemm_bf16_plain(gpu, m, n, k):
    from fastforward_amd.vision import Lin, linear
    x = torch.randn(m, k, generator=_g(m + k)).to(BF16)
    w = (torch.randn(n, k, generator=_g(n)) * 0.03).to(BF16)
    b = (torch.randn(n, generator=_g(n + 1)) * 0.1).to(BF16)
    got = linear(x.to(DEV), Lin(w.to(DEV), b.to(DEV))).cpu().to(torch.float64)
    exact, bound = _linear_bound(x, w, b)
    assert bool(((got - exact).abs() <= bound).all()), "bf16 GEMM outside the fp32-accumulation bound"
    eq = float((got.to(BF16) == OV.linear(x, w, b)).float().mean())
    assert eq >= 0.95, f"only {eq:.3f} of the outputs equal the oracle's"


@pytest.mark.parametrize("act", [1, 2])
def test_gemm_bf16_gelu(gpu, act):
    from fastforward_amd.vision import Lin, linear
    m, n, k = 200, 4352, 1152
    x = torch.randn(m, k, generator=_g(5)).to(BF16)
    w = (torch.randn(n, k, generator=_g(6)) * 0.05).to(BF16)
    b = (torch.randn(n, generator=_g(7)) * 0.1).to(BF16)
    got = linear(x.to(DEV), Lin(w.to(DEV), b.to(DEV)), act=act).cpu()
    f = OV.gelu_tanh if act == 1 else OV.gelu_erf
    _, bound = _linear_bound(x, w, b)
    # |gelu'| <= 1.13: the pre-activation bound carries over
    _assert_within(got, f(OV.linear(x, w, b)), 1.13 * bound, f"gemm_bf16 act {act}")


def test_gemm_bf16_residual_in_place(gpu):
    from fastforward_amd.vision import Lin, linear
    m, n, k = 260, 1152, 1152
    x = torch.randn(m, k, generator=_g(8)).to(BF16)
    w = (torch.randn(n, k, generator=_g(9)) * 0.03).to(BF16)
    b = (torch.randn(n, generator=_g(10)) * 0.1).to(BF16)
    h = torch.randn(m, n, generator=_g(11)).to(BF16)
    hd = h.to(DEV)
    linear(x.to(DEV), Lin(w.to(DEV), b.to(DEV)), resid=hd, out=hd)
    want = (h.float() + OV.linear(x, w, b).float()).to(BF16)
    _, bound = _linear_bound(x, w, b)
    _assert_within(hd.cpu(), want, bound, "gemm_bf16 residual")


FF_TUNE_GEMM_BF16_TILE = 2
BF16_TILES = [12, 22, 23, 24, 25, 34, 44, 36, 56, 66]


# one row and one column group; ragged rows and columns around the tiles' edges
# (32, 64, 96, 160, 192), a row of outputs that is not 16-byte aligned (n % 8 ==
# 4); one 64-k stage, fewer stages than are in flight, as many, and many more
@pytest.mark.parametrize("m,n,k", [(1, 4, 64), (33, 100, 128), (191, 196, 384), (193, 320, 448), (385, 1160, 1152)])
def test_gemm_bf16_every_tile(gpu, m, n, k):
    """ff_gemm_bf16 with each tile forced: bit-equal to the first one (the same
    products in the same order), whose outputs are checked on their own; the same for
    each activation and for a residual added in place."""
    from fastforward_amd._lib import call
    from fastforward_amd.vision import Lin, linear
    x = torch.randn(m, k, generator=_g(m + 21)).to(BF16)
    w = (torch.randn(n, k, generator=_g(n + 22)) * 0.05).to(BF16)
    b = (torch.randn(n, generator=_g(k + 23)) * 0.1).to(BF16)
    h = torch.randn(m, n, generator=_g(24)).to(BF16).to(DEV)
    xd, lin = x.to(DEV), Lin(w.to(DEV), b.to(DEV))

    def run(tile):
        call("ff_set_tuning", FF_TUNE_GEMM_BF16_TILE, tile)
        try:
            y = h.clone()
            linear(xd, lin, resid=y, out=y)
            return [linear(xd, lin, act=act) for act in (0, 1, 2)] + [y]
        finally:
            call("ff_set_tuning", FF_TUNE_GEMM_BF16_TILE, 0)
    ref = run(BF16_TILES[0])
    _assert_epilogues(x, w, b, h, lambda act, resid: ref[3] if resid is not None else ref[act])
    for tile in BF16_TILES[1:] + [0]:
        for a, c in zip(run(tile), ref):
            assert torch.equal(a, c), tile


def test_gelu_tanh_every_bf16(gpu):
    """The GELU-tanh epilogue at every finite bf16 value (an identity weight
    carries x to the epilogue exactly): within one bf16 ulp of the 64-bit function,
    plus 2^-24 |x| where the result itself is below that (the fp32 evaluation's
    absolute floor), and infinities and NaN as torch's."""
    from fastforward_amd.vision import Lin, linear
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(BF16)
    vals = bits[torch.isfinite(bits.float())]
    vals = torch.cat([vals, torch.zeros((-vals.numel()) % 64)]).to(BF16).reshape(-1, 64)
    eye = torch.eye(64).to(BF16)
    got = linear(vals.to(DEV), Lin(eye.to(DEV), torch.zeros(64, dtype=BF16, device=DEV)), act=1).cpu()
    v = vals.to(torch.float64)
    u = (2 / np.pi) ** 0.5 * (v + 0.044715 * v ** 3)
    want = v / (1 + torch.exp(-2 * u))
    ok = (got.to(torch.float64) - want).abs() <= _ulp(want) + v.abs() * 2.0 ** -24
    assert bool(ok.all()), vals[~ok][:8]
    sp = torch.zeros(1, 64, dtype=BF16)
    for x, f in ((float("inf"), lambda t: t == float("inf")), (float("nan"), torch.isnan)):
        sp[0, 0] = x
        out = linear(sp.to(DEV), Lin(eye.to(DEV)[:, :64].contiguous(), torch.zeros(64, dtype=BF16, device=DEV)),
                     act=1).cpu()
        assert bool(f(out[0, 0].float()))


@pytest.mark.parametrize("tile", [0, 12, 25, 44, 66, "split"])
def test_gelu_tanh_equals_torch(gpu, tile):
    """GELU-tanh of every bf16 pattern (as the bias of a zero product): the bits of torch's
    op on the same device, NaN for NaN and -inf, from the GEMM's epilogue and from the
    launch that adds a k split's partials."""
    from fastforward_amd._lib import call
    from fastforward_amd.vision import Lin, linear, split_workspace
    vals = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(BF16).to(DEV)
    want = torch.nn.functional.gelu(vals, approximate="tanh")
    if tile == "split":
        n, k = 8192, 1152
        assert split_workspace(1, n, k) > 0
        ws = torch.empty(split_workspace(1, n, k), dtype=torch.uint8, device=DEV)
    else:
        n, k, ws = 65536, 64, None
    w, x = torch.zeros(n, k, dtype=BF16, device=DEV), torch.zeros(1, k, dtype=BF16, device=DEV)
    if tile != "split":
        call("ff_set_tuning", FF_TUNE_GEMM_BF16_TILE, tile)
    try:
        got = torch.cat([linear(x, Lin(w, b).pack(), act=1, ws=ws)[0] for b in vals.split(n)])
    finally:
        call("ff_set_tuning", FF_TUNE_GEMM_BF16_TILE, 0)
    assert torch.equal(got.isnan(), want.isnan())
    ok = ~want.isnan()
    assert torch.equal(got[ok], want[ok])


# (m, k, n, act, resid): proj / fc2 of the tower with the residual add in place, the
# patch embedding, the mergers' fc1 + GELU and fc2, row and column counts of the 2B
# tower, ragged row counts, an odd number of 128-k steps (k 1152), the tower's qkv and
# fc1 (GELU-tanh), and n = 1000, which no tile divides
PK_VISION = [(2048, 1152, 1152, 0, True), (2048, 4352, 1152, 0, True), (2048, 1536, 1152, 0, False),
             (512, 4608, 4608, 2, False), (512, 4608, 4096, 0, False), (1536, 1152, 3456, 0, False),
             (1024, 1152, 4096, 1, False), (2000, 4352, 1152, 0, True), (2048, 1152, 3456, 0, False),
             (2048, 1152, 4352, 1, False), (600, 1152, 1000, 0, False)]


@pytest.mark.parametrize("m,k,n,act,resid", PK_VISION)
def test_gemm_bf16_packed_equals_rowmajor(gpu, m, k, n, act, resid):
    """linear() at the tower's sizes with every epilogue (bias, GELU-tanh, GELU-erf,
    residual add in place), on a Lin that holds a packed copy and one that does not: the
    unsplit product reads the row-major weight either way and gives the outputs of
    ``_assert_epilogues``."""
    from fastforward_amd.vision import Lin, linear
    x = torch.randn(m, k, generator=_g(m + n)).to(BF16).to(DEV)
    w = (torch.randn(n, k, generator=_g(k)) * 0.03).to(BF16).to(DEV)
    b = (torch.randn(n, generator=_g(n + 2)) * 0.1).to(BF16).to(DEV)
    h = torch.randn(m, n, generator=_g(n + 3)).to(BF16).to(DEV) if resid else None

    def run(a, r):
        outs = []
        for lin in (Lin(w, b), Lin(w, b).pack()):
            y = None if r is None else r.clone()
            outs.append(linear(x, lin, act=a, resid=y, out=y))
        assert torch.equal(outs[0], outs[1])
        return outs[0]
    _assert_epilogues(x, w, b, h, run)
    assert not torch.isnan(run(act, h).float()).any()


@pytest.mark.parametrize("m,k,n", [(2048, 1152, 1152), (2000, 1536, 1152)])
@pytest.mark.parametrize("pad", [8, 4])
def test_gemm_bf16_packed_strided_residual(gpu, m, k, n, pad):
    """The residual add with the residual a strided view (row stride n + pad elements) and
    the output a separate array, on every tile that takes a residual: pad 8 keeps the
    residual rows 16-byte aligned (the epilogue reads the tile that was copied into LDS
    during the main loop), pad 4 does not (it reads global memory); both are bf16(h + v)
    of the product v without a residual, bit for bit, and the residual is unchanged."""
    from fastforward_amd._lib import call
    from fastforward_amd.vision import Lin, linear
    x = torch.randn(m, k, generator=_g(m + n + 11)).to(BF16).to(DEV)
    w = (torch.randn(n, k, generator=_g(k + 12)) * 0.03).to(BF16).to(DEV)
    b = (torch.randn(n, generator=_g(n + 13)) * 0.1).to(BF16).to(DEV)
    wide = torch.randn(m, n + pad, generator=_g(n + 14)).to(BF16).to(DEV)
    h = wide[:, pad: pad + n]
    assert h.stride(0) == n + pad and (h.data_ptr() % 16 == 0 and h.stride(0) % 8 == 0) == (pad == 8)
    before = wide.clone()
    want = (h.float() + linear(x, Lin(w, b)).float()).to(BF16)
    for tile in [0] + BF16_TILES[:8]:
        call("ff_set_tuning", FF_TUNE_GEMM_BF16_TILE, tile)
        try:
            outs = [linear(x, lin, resid=h) for lin in (Lin(w, b), Lin(w, b).pack())]
        finally:
            call("ff_set_tuning", FF_TUNE_GEMM_BF16_TILE, 0)
        assert torch.equal(outs[0], want) and torch.equal(outs[1], want), tile
    assert torch.equal(wide, before)


# (m, k, n, act, resid): grids with no one-round packed tile whose unsplit
# fallback fills less than half the GPU, which the workspace entry points split
# along k: the tower at 400 patches (proj and fc2 with the residual in place,
# the patch embedding) and at 128 patches (fc1 + GELU-tanh), the mergers at 100
# merged tokens (fc1 + GELU-erf, fc2)
SPLIT_VISION = [(400, 1152, 1152, 0, True), (400, 4352, 1152, 0, True), (400, 1536, 1152, 0, False),
                (128, 1152, 4352, 1, False), (100, 4608, 4608, 2, False), (100, 4608, 4096, 0, False)]
FF_TUNE_BF16_PK_SPLIT = 10


@pytest.mark.parametrize("m,k,n,act,resid", SPLIT_VISION)
def test_gemm_bf16_split_matches_unsplit(gpu, m, k, n, act, resid):
    """ff_gemm_bf16_pk_ws with its k split (the partials added in split order by
    the epilogue launch) against the unsplit packed kernel: the same products
    summed in fp32 in another order, so within twice the fp32-accumulation
    bound of the exact product (plus the bf16 roundings after it) and nearly
    all equal; inside that bound of the exact product itself; identical on
    repeated calls; with the split turned off, the unsplit bits."""
    from fastforward_amd._lib import call
    from fastforward_amd.vision import Lin, linear, split_workspace
    need = split_workspace(m, n, k)
    assert need > 0, "the shape must split"
    x = torch.randn(m, k, generator=_g(m + n + 5)).to(BF16)
    w = (torch.randn(n, k, generator=_g(k + 1)) * 0.03).to(BF16)
    b = (torch.randn(n, generator=_g(n + 4)) * 0.1).to(BF16)
    h = torch.randn(m, n, generator=_g(n + 6)).to(BF16).to(DEV) if resid else None
    lin = Lin(w.to(DEV), b.to(DEV)).pack()
    ws = torch.full((need // 4,), float("nan"), device=DEV)
    xd = x.to(DEV)

    def run(split):
        y = h.clone() if resid else torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
        linear(xd, lin, act=act, resid=y if resid else None, out=y, ws=ws if split else None)
        return y
    ref = run(False)
    got = [run(True) for _ in range(2)]
    assert torch.equal(got[0], got[1]) and not torch.isnan(got[0].float()).any()
    # both sums lie within the fp32-accumulation bound of the exact product, so
    # they differ by at most twice it (carried through the GELU, |gelu'| <=
    # 1.13) plus a bf16 rounding of the term and, with a residual, of y
    _, bound = _linear_bound(x, w, b)
    g64, r64 = got[0].cpu().to(torch.float64), ref.cpu().to(torch.float64)
    t64 = r64 - h.cpu().to(torch.float64) if resid else r64
    allowed = 2 * bound * (1.13 if act else 1.0) + _ulp(t64) + (_ulp(r64) if resid else 0)
    assert bool(((g64 - r64).abs() <= allowed).all()), "split result outside the bound of the unsplit one"
    d = bf16_ulps(got[0], ref)
    assert float((d > 0).float().mean()) < 0.02
    if not act and not resid:
        exact, bound = _linear_bound(x, w, b)
        assert bool(((g64 - exact).abs() <= bound).all())
    call("ff_set_tuning", FF_TUNE_BF16_PK_SPLIT, 1)
    try:
        assert torch.equal(run(True), ref)
    finally:
        call("ff_set_tuning", FF_TUNE_BF16_PK_SPLIT, 0)


@pytest.mark.parametrize("m,k,n,in_place", [(400, 1152, 1152, True), (400, 4352, 1152, True),
                                            (400, 1536, 1152, False), (2048, 1152, 1152, True)])
def test_gemm_bf16_pk_ln(gpu, m, k, n, in_place):
    """linear_ln (a residual linear and the LayerNorm of its output): unsplit
    (2048 rows) bit for bit the linear followed by layer_norm; split (400 rows)
    the stored output within the split bound of the unsplit one (twice the
    fp32-accumulation bound plus the roundings) and the LayerNorm bit
    for bit ff_layer_norm of the output it stored; without a LayerNorm only
    the output is written. The residual in place (proj, fc2) or separate (the
    patch embedding's position embedding)."""
    from fastforward_amd.vision import Lin, Norm, layer_norm, linear, linear_ln, split_workspace
    x = torch.randn(m, k, generator=_g(m + 11)).to(BF16).to(DEV)
    w = (torch.randn(n, k, generator=_g(k + 12)) * 0.03).to(BF16).to(DEV)
    b = (torch.randn(n, generator=_g(n + 13)) * 0.1).to(BF16).to(DEV)
    r = torch.randn(m, n, generator=_g(n + 14)).to(BF16).to(DEV)
    nw = (1 + 0.1 * torch.randn(n, generator=_g(15))).to(BF16).to(DEV)
    nb = (0.1 * torch.randn(n, generator=_g(16))).to(BF16).to(DEV)
    norm = Norm(nw, nb)
    lin = Lin(w, b).pack()
    ws = torch.full((max(split_workspace(m, n, k) // 4, 64),), float("nan"), device=DEV)
    # unsplit reference: the linear with its residual, then the LayerNorm
    y_ref = r.clone() if in_place else torch.empty(m, n, device=DEV, dtype=BF16)
    linear(x, lin, resid=y_ref if in_place else r, out=y_ref)
    ln_ref = layer_norm(y_ref, norm, 1e-6)
    y = r.clone() if in_place else torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
    ln = torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
    linear_ln(x, lin, y if in_place else r, y, ws, norm, 1e-6, ln)
    split = split_workspace(m, n, k) > 0
    assert split == (m == 400)
    if split:
        _, bound = _linear_bound(x.cpu(), w.cpu(), b.cpu())
        y64, ref64, r64 = (v.cpu().to(torch.float64) for v in (y, y_ref, r))
        assert bool(((y64 - ref64).abs() <= 2 * bound + _ulp(ref64 - r64) + _ulp(ref64)).all())
        assert float((bf16_ulps(y, y_ref) > 0).float().mean()) < 0.02
        assert torch.equal(ln, layer_norm(y, norm, 1e-6))
    else:
        assert torch.equal(y, y_ref) and torch.equal(ln, ln_ref)
    y2 = r.clone() if in_place else torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
    linear_ln(x, lin, y2 if in_place else r, y2, ws)
    assert torch.equal(y2, y)


def test_pack_weight_bf16_layout(gpu):
    """ff_pack_weight_bf16: fragment (f, kt) at (kt n/16 + f) 4 KB, sub-block s,
    lane 16 g + r: row 16 f + r, k 128 kt + 64 (s / 2) + 16 g + 8 (s % 2) .. + 8."""
    from fastforward_amd._lib import call, ptr, stream
    n, k = 48, 384
    w = torch.randint(-30000, 30000, (n, k), generator=_g(90), dtype=torch.int16)
    p = torch.empty(n * k, device=DEV, dtype=torch.int16)
    wd = w.to(DEV)
    call("ff_pack_weight_bf16", ptr(wd), ptr(p), n, k, stream())
    got = p.cpu().numpy().reshape(k // 128, n // 16, 4, 64, 8)
    wn = w.numpy()
    for kt in range(k // 128):
        for f in range(n // 16):
            for s in range(4):
                for lane in range(64):
                    r, g = lane % 16, lane // 16
                    k0 = 128 * kt + 64 * (s // 2) + 16 * g + 8 * (s % 2)
                    assert np.array_equal(got[kt, f, s, lane], wn[16 * f + r, k0:k0 + 8]), (kt, f, s, lane)


def test_vision_rope_bit_exact_and_padded_layout(gpu):
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.vision import VISION_PRESETS, rope_tables, vision_rope
    cfg = VISION_PRESETS["qwen3vl-8b"]
    gh, gw = 8, 12
    n, nh, hd = gh * gw, cfg.heads, cfg.head_dim
    cos, sin = rope_tables(cfg, gh, gw)
    qkv = torch.randn(n, 3, nh, hd, generator=_g(12)).to(BF16)
    q, k = qkv[:, 0], qkv[:, 1]
    want_q, want_k = OV.vision_rope(q, k, cos, sin)
    qd = qkv.to(DEV)
    yq, yk = vision_rope(qd[:, 0], qd[:, 1], cos.to(DEV), sin.to(DEV))
    assert torch.equal(yq.cpu(), want_q) and torch.equal(yk.cpu(), want_k)
    # head-major, zero-padded to 128 (the attention layout); every device input
    # is held in a variable until the kernel has run
    pq = torch.full((nh, n, 128), float("nan"), device=DEV).to(BF16)
    pk = torch.full((nh, n, 128), float("nan"), device=DEV).to(BF16)
    cd, sd = cos.to(DEV), sin.to(DEV)
    call("ff_vision_rope", ptr(qd[:, 0]), ptr(qd[:, 1]), 3 * nh * hd, hd, ptr(cd), ptr(sd),
         ptr(pq), ptr(pk), 128, n * 128, n, nh, hd, 128, stream())
    torch.cuda.synchronize()
    assert torch.equal(pq[:, :, :hd].cpu(), want_q.transpose(0, 1))
    assert torch.equal(pk[:, :, :hd].cpu(), want_k.transpose(0, 1))
    assert not bool(pq[:, :, hd:].float().abs().sum()) and not bool(pk[:, :, hd:].float().abs().sum())


def test_vision_qkv_equals_rope_and_vt(gpu):
    """The one-launch form equals ff_vision_rope (padded, head-major) + ff_vision_vt."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.vision import VISION_PRESETS, rope_tables
    cfg = VISION_PRESETS["qwen3vl-8b"]
    gh, gw = 10, 12
    n, nh, hd, n_pad = gh * gw, cfg.heads, cfg.head_dim, 128
    cd, sd = (t.to(DEV) for t in rope_tables(cfg, gh, gw))
    qkv = torch.randn(n, 3 * nh * hd, generator=_g(14)).to(BF16).to(DEV)
    outs = []
    for fused in (False, True):
        yq, yk = (torch.full((nh, n, 128), float("nan"), device=DEV).to(BF16) for _ in range(2))
        vt = torch.full((nh, 128, n_pad), float("nan"), device=DEV).to(BF16)
        if fused:
            call("ff_vision_qkv", ptr(qkv), ptr(cd), ptr(sd), ptr(yq), ptr(yk), ptr(vt), n, n_pad, nh, hd, stream())
        else:
            call("ff_vision_rope", ptr(qkv), ptr(qkv[:, nh * hd:]), 3 * nh * hd, hd, ptr(cd), ptr(sd), ptr(yq),
                 ptr(yk), 128, n * 128, n, nh, hd, 128, stream())
            call("ff_vision_vt", ptr(qkv[:, 2 * nh * hd:]), 3 * nh * hd, hd, ptr(vt), n, n_pad, nh, hd, stream())
        torch.cuda.synchronize()
        outs.append((yq, yk, vt))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


# one token, a last rotary workgroup that is partly empty, odd head counts; heads of one
# 8-column group, of 64 (no group pair past 64), of 72 and of the full 128
@pytest.mark.parametrize("n,nh,hd", [(1, 1, 8), (5, 3, 64), (63, 3, 72), (64, 2, 120), (130, 16, 128), (400, 16, 72)])
def test_vision_qkv_sizes(gpu, n, nh, hd):
    """q, k rotated by two fp32 products and their sum, rounded once; v transposed; zeros past
    the head width and the tokens. Bit for bit, in torch's fp32 on the CPU."""
    from fastforward_amd._lib import call, ptr, stream
    n_pad = (n + 63) // 64 * 64
    qkv = torch.randn(n, 3, nh, hd, generator=_g(15)).to(BF16)
    cos, sin = (torch.randn(n, hd, generator=_g(s)) for s in (16, 17))
    yq, yk = (torch.full((nh, n, 128), float("nan"), device=DEV).to(BF16) for _ in range(2))
    vt = torch.full((nh, 128, n_pad), float("nan"), device=DEV).to(BF16)
    qkv_d, cos_d, sin_d = qkv.to(DEV), cos.to(DEV), sin.to(DEV)
    call("ff_vision_qkv", ptr(qkv_d), ptr(cos_d), ptr(sin_d), ptr(yq), ptr(yk), ptr(vt), n, n_pad, nh, hd, stream())
    for part, got in ((0, yq), (1, yk)):
        x = qkv[:, part].float()
        rot = torch.cat((-x[..., hd // 2:], x[..., :hd // 2]), -1)
        want = torch.zeros(nh, n, 128, dtype=BF16)
        want[..., :hd] = (x * cos[:, None] + rot * sin[:, None]).to(BF16).transpose(0, 1)
        assert torch.equal(got.cpu(), want)
    want = torch.zeros(nh, 128, n_pad, dtype=BF16)
    want[:, :hd, :n] = qkv[:, 2].permute(1, 2, 0)
    assert torch.equal(vt.cpu(), want)


def test_vision_vt_layout(gpu):
    from fastforward_amd._lib import call, ptr, stream
    n, nh, hd, n_pad = 100, 4, 72, 128
    v = torch.randn(n, nh, hd, generator=_g(13)).to(BF16)
    vt = torch.full((nh, 128, n_pad), float("nan"), device=DEV).to(BF16)
    vd = v.to(DEV)
    call("ff_vision_vt", ptr(vd), nh * hd, hd, ptr(vt), n, n_pad, nh, hd, stream())
    torch.cuda.synchronize()
    want = torch.zeros(nh, 128, n_pad, dtype=BF16)
    want[:, :hd, :n] = v.permute(1, 2, 0)
    assert torch.equal(vt.cpu(), want)


@pytest.mark.parametrize("n,nh,hd", [(300, 4, 72), (2048, 2, 72), (130, 3, 64)])
def test_attention_full(gpu, n, nh, hd):
    from fastforward_amd._lib import call, ptr, stream
    q, k, v = (torch.randn(n, nh, hd, generator=_g(20 + i)).to(BF16) for i in range(3))
    n_pad = (n + 63) // 64 * 64
    def pad(x):
        out = torch.zeros(nh, n, 128, dtype=BF16)
        out[:, :, :hd] = x.transpose(0, 1)
        return out.to(DEV)
    vt = torch.zeros(nh, 128, n_pad, dtype=BF16)
    vt[:, :hd, :n] = v.permute(1, 2, 0)
    y = torch.empty(n, nh * hd, device=DEV, dtype=BF16)
    qd, kd, vtd = pad(q), pad(k), vt.to(DEV)
    call("ff_attention_full", ptr(qd), ptr(kd), ptr(vtd), ptr(y), n, n_pad, nh, hd, float(hd ** -0.5), stream())
    torch.cuda.synchronize()
    want = OV.attention(q, k, v, hd ** -0.5).float()
    got = y.cpu().float()
    assert float((got - want).abs().max()) <= 1 / 64
    assert float(((got - want).norm() / want.norm())) <= 5e-3
    # one and two query tiles per wave (the built-in choice depends on the grid) give the same bits
    y2 = torch.empty_like(y)
    call("ff_set_tuning", 5, 2)  # FF_TUNE_ATTN_QT
    try:
        call("ff_attention_full", ptr(qd), ptr(kd), ptr(vtd), ptr(y2), n, n_pad, nh, hd, float(hd ** -0.5),
             stream())
    finally:
        call("ff_set_tuning", 5, 0)
    assert torch.equal(y2, y)


# 16 heads at one workgroup per CU (1000 tokens) and past that: an odd and an even
# number of 64-key blocks, ragged and full last blocks, each head width
@pytest.mark.parametrize("n,hd", [(1000, 72), (1025, 72), (1088, 64), (1100, 128), (1152, 72)])
@pytest.mark.parametrize("ramp", [0.0, 40.0, float("-inf")])
def test_attention_full_key_split(gpu, n, hd, ramp):
    """ff_attention_full against the oracle over many key blocks; with ``ramp`` the
    scores grow along the keys (by about 4 ramp in natural units), so that the running
    maximum moves in every block; with -inf the first two key blocks' scores are -inf
    (weight 0)."""
    from fastforward_amd._lib import call, ptr, stream
    nh = 16
    q, k, v = (torch.randn(n, nh, hd, generator=_g(50 + i)) for i in range(3))
    q[:, :, 0] = 4.0
    k[:, :, 0] = 0
    if ramp > 0:
        k[:, :, 0] = torch.linspace(0, ramp, n)[:, None] * hd ** 0.5 / 4
    elif ramp < 0:
        k[:128, :, 0] = ramp
    q, k, v = (t.to(BF16) for t in (q, k, v))
    n_pad = (n + 63) // 64 * 64
    qd, kd = (torch.zeros(nh, n, 128, dtype=BF16, device=DEV) for _ in range(2))
    qd[:, :, :hd], kd[:, :, :hd] = q.transpose(0, 1).to(DEV), k.transpose(0, 1).to(DEV)
    vt = torch.zeros(nh, 128, n_pad, dtype=BF16, device=DEV)
    vt[:, :hd, :n] = v.permute(1, 2, 0).to(DEV)
    y = torch.full((n, nh * hd), float("nan"), device=DEV, dtype=BF16)
    call("ff_attention_full", ptr(qd), ptr(kd), ptr(vt), ptr(y), n, n_pad, nh, hd, float(hd ** -0.5), stream())
    got, want = y.cpu().float(), OV.attention(q, k, v, hd ** -0.5).float()
    # bf16(p) and the bf16 output: 2^-9 each relative to the weights' mean of |v|
    assert float((got - want).norm() / want.norm()) <= 5e-3
    assert float((got - want).abs().max()) <= (1 / 16 if ramp > 0 else 1 / 64)   # |v| up to 4 with one key dominating


def _attention_full(q, k, v):
    """ff_attention_full of (n, heads, hd) bf16 q, k, v on the host; the output on the host."""
    from fastforward_amd._lib import call, ptr, stream
    n, nh, hd = q.shape
    n_pad = (n + 63) // 64 * 64
    qd, kd = (torch.zeros(nh, n, 128, dtype=BF16, device=DEV) for _ in range(2))
    qd[:, :, :hd], kd[:, :, :hd] = q.transpose(0, 1).to(DEV), k.transpose(0, 1).to(DEV)
    vt = torch.zeros(nh, 128, n_pad, dtype=BF16, device=DEV)
    vt[:, :hd, :n] = v.permute(1, 2, 0).to(DEV)
    y = torch.full((n, nh * hd), float("nan"), device=DEV, dtype=BF16)
    call("ff_attention_full", ptr(qd), ptr(kd), ptr(vt), ptr(y), n, n_pad, nh, hd, float(hd ** -0.5), stream())
    return y.cpu()


# 4 x 16, and past one workgroup per CU, queries of 16 heads; two heads of many patches
@pytest.mark.parametrize("n,nh,hd", [(130, 3, 72), (1000, 16, 64), (1100, 16, 72), (2300, 2, 128)])
def test_attention_full_peaked_precision(gpu, n, nh, hd):
    """Scores of standard deviation 4, where one weight of most queries is near 1: taken
    against the running maximum, that weight is exactly 1 in bf16. The distance from the
    64-bit result is then the bf16 rounding of the output and of the lesser weights, which
    the host computes; 1.1 of it leaves room for the fp32 sums, and a weight that is not
    1 (any other reference) makes it 1.4 of it."""
    q, k, v = (torch.randn(n, nh, hd, generator=_g(50 + i)) for i in range(3))
    q, k, v = (q * 4).to(BF16), k.to(BF16), v.to(BF16)
    got = _attention_full(q, k, v).double().reshape(n, nh, hd)
    err = floor = 0.0
    for h in range(nh):
        s = q[:, h].double() @ k[:, h].double().T * hd ** -0.5
        p = torch.exp(s - s.amax(1, keepdim=True))
        den, vh = p.sum(1, keepdim=True), v[:, h].double()
        exact = p @ vh / den
        err += float((got[:, h] - exact).square().sum())
        floor += float((exact.to(BF16).double() - exact).square().sum())
        floor += float((p.to(BF16).double() @ vh / den - exact).square().sum())
    assert err <= 1.1 ** 2 * floor


# one, two and more workgroups of 64 queries per CU
@pytest.mark.parametrize("n,nh,hd", [(400, 16, 72), (1100, 16, 72), (1100, 16, 128), (2300, 16, 64)])
def test_attention_full_bits_whatever_the_tile(gpu, n, nh, hd):
    """The key blocks are summed in order for every query, so the built-in choice, one and
    two query tiles per wave give the same bits at every grid size."""
    from fastforward_amd._lib import call
    q, k, v = (torch.randn(n, nh, hd, generator=_g(70 + i)).to(BF16) for i in range(3))
    ref = _attention_full(q, k, v)
    for qt in (1, 2):
        call("ff_set_tuning", 5, qt)  # FF_TUNE_ATTN_QT
        try:
            assert torch.equal(_attention_full(q, k, v), ref), qt
        finally:
            call("ff_set_tuning", 5, 0)


def test_attention_full_rows_stand_alone(gpu):
    """A query's output is the same bits whatever the other queries of its tile are; and
    where half of a tile's queries score -inf (a dot product past fp32's range) on the
    first two key blocks, those get weights of the keys after them and the other half
    the attention over all keys."""
    n, nh, hd = 300, 2, 72
    q, k, v = (torch.randn(n, nh, hd, generator=_g(60 + i)) for i in range(3))
    q[:, :, 0] = 0
    k[:128, :, 0] = -3e38
    q, k, v = (t.to(BF16) for t in (q, k, v))
    plain = _attention_full(q, k, v)
    mixed = q.clone()
    mixed[1::2] *= 5
    mixed[1::2, :, 0] = 4.0          # 4 x -3e38 is past the fp32 range
    got = _attention_full(mixed, k, v)
    assert torch.equal(got[::2], plain[::2])
    assert bool(torch.isfinite(got.float()).all())
    k0 = k.clone()
    k0[:, :, 0] = 0
    want = OV.attention(q, k0, v, hd ** -0.5).float()
    assert float((plain.float() - want).norm() / want.norm()) <= 5e-3
    s = torch.einsum("qhd,khd->hqk", mixed[1::2].double(), k[128:].double()) * hd ** -0.5
    want = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), v[128:].double()).reshape(-1, nh * hd)
    assert float((got[1::2].double() - want).norm() / want.norm()) <= 5e-3


def test_tower_packs_only_what_its_splits_read(gpu):
    """A tower holds packed copies of the linears whose k is split at its patch count and
    of no others; another geometry on the same weights adds its own."""
    import dataclasses
    from fastforward_amd.vision import VISION_PRESETS, VisionRuntime, make_vision
    cfg = dataclasses.replace(VISION_PRESETS["qwen3vl-8b"], depth=1, deepstack=())
    w = make_vision(cfg, seed=5)
    blk = w.blocks[0]
    names = dict(patch=w.patch, qkv=blk.qkv, proj=blk.proj, fc1=blk.fc1, fc2=blk.fc2, m1=w.merger.fc1, m2=w.merger.fc2)
    rgb = torch.randint(0, 256, (512, 1024, 3), dtype=torch.uint8, generator=_g(80))

    def run(gh, gw):
        rt = VisionRuntime(cfg, w, gh, gw)
        rt.set_image(rgb[:16 * gh, :16 * gw].contiguous())
        return rt.step()[0].clone()
    tall = run(32, 64)
    assert [k for k, lin in names.items() if lin.p is not None] == []
    run(20, 20)
    assert [k for k, lin in names.items() if lin.p is not None] == ["patch", "proj", "fc2", "m1", "m2"]
    assert torch.equal(run(32, 64), tall)


def test_pos_interp_bit_exact(gpu):
    from fastforward_amd.vision import VisionConfig, interp_taps
    from fastforward_amd._lib import call, ptr, stream
    cfg = VisionConfig("t", 1, 64, 2, 96, 32, (), pos_side=6)
    table = (torch.randn(36, 64, generator=_g(30)) * 0.1).to(BF16)
    shape = OV.VisionShape(depth=1, hidden=64, heads=2, inter=96, out_hidden=32, deepstack=(), pos_side=6)
    for gh, gw in ((4, 8), (6, 6), (2, 10)):
        idx, wt = interp_taps(cfg, gh, gw)
        out = torch.empty(gh * gw, 64, device=DEV, dtype=BF16)
        td, idd, wd = table.to(DEV), idx.to(DEV), wt.to(DEV)
        call("ff_pos_interp", ptr(td), ptr(idd), ptr(wd), ptr(out), gh * gw, 4, 64, 36, stream())
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), OV.pos_embeds(shape, table, gh, gw)), (gh, gw)


def _small_tower(seed=0):
    """A 3-block tower with the 8B head width (8 heads of 72), padded MLP
    (200 -> 256) and DeepStack after blocks 0 and 2."""
    from fastforward_amd.vision import VisionConfig, make_vision
    cfg = VisionConfig("small", 3, 576, 8, 200, 96, (0, 2), pos_side=6)
    return cfg, make_vision(cfg, seed=seed, std=0.05)


def _to_oracle(cfg, w):
    shape = OV.VisionShape(depth=cfg.depth, hidden=cfg.hidden, heads=cfg.heads, inter=cfg.inter,
                           out_hidden=cfg.out_hidden, deepstack=tuple(cfg.deepstack), pos_side=cfg.pos_side)
    c = lambda t: t.cpu()  # noqa: E731
    blocks = [OV.VisionBlock(c(b.norm1.w), c(b.norm1.b), c(b.qkv.w), c(b.qkv.b), c(b.proj.w), c(b.proj.b),
                             c(b.norm2.w), c(b.norm2.b), c(b.fc1.w[:cfg.inter]), c(b.fc1.b[:cfg.inter]),
                             c(b.fc2.w[:, :cfg.inter]), c(b.fc2.b)) for b in w.blocks]
    mg = lambda m: OV.Merger(c(m.norm.w), c(m.norm.b), c(m.fc1.w), c(m.fc1.b), c(m.fc2.w), c(m.fc2.b),  # noqa: E731
                             m.postshuffle)
    return shape, OV.VisionWeights(c(w.patch.w), c(w.patch.b), c(w.pos_embed), blocks, mg(w.merger),
                                   [mg(m) for m in w.deep])


def test_vision_tower_matches_oracle(gpu):
    from fastforward_amd.vision import VisionRuntime
    cfg, w = _small_tower()
    gh, gw = 8, 12
    rt = VisionRuntime(cfg, w, gh, gw)
    rng = np.random.default_rng(4)
    rgb = rng.integers(0, 256, size=(16 * gh, 16 * gw, 3), dtype=np.uint8)
    rt.set_image(torch.from_numpy(rgb))
    trace = []
    merged, deep = rt.step(trace)
    torch.cuda.synchronize()
    shape, ow = _to_oracle(cfg, w)
    otrace = []
    omerged, odeep = OV.tower(shape, ow, OV.pack_pixels(rgb), gh, gw, otrace)
    for j, (a, b) in enumerate(zip(trace, otrace)):
        assert _rel_l2(a, b) <= 1e-2, f"block {j}: {_rel_l2(a, b):.3e}"
    assert _rel_l2(merged, omerged) <= 2e-2
    for a, b in zip(deep, odeep):
        assert _rel_l2(a, b) <= 2e-2
    # teacher-forced: blocks 1.. from the oracle's input to them
    cos, sin = OV.rope_cos_sin(shape, gh, gw)
    for j in range(1, cfg.depth):
        rt.h.copy_(otrace[j - 1].to(DEV))
        _run_block(rt, j)
        want = OV.block(shape, ow.blocks[j], otrace[j - 1], cos, sin)
        assert _rel_l2(rt.h, want) <= 5e-3, f"teacher-forced block {j}: {_rel_l2(rt.h, want):.3e}"


def _run_block(rt, j):
    """Block j of the runtime's weights on rt.h in place (the step's calls)."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.vision import ACT_GELU_TANH, layer_norm, linear
    cfg, blk, s = rt.cfg, rt.w.blocks[j], stream()
    n, H, HD, NH = rt.n, cfg.hidden, cfg.head_dim, cfg.heads
    layer_norm(rt.h, blk.norm1, cfg.eps, out=rt.x)
    linear(rt.x, blk.qkv, out=rt.qkv)
    call("ff_vision_qkv", ptr(rt.qkv), ptr(rt.cos), ptr(rt.sin), ptr(rt.q), ptr(rt.k), ptr(rt.vt), n, rt.n_pad,
         NH, HD, s)
    call("ff_attention_full", ptr(rt.q), ptr(rt.k), ptr(rt.vt), ptr(rt.z), n, rt.n_pad, NH, HD, float(HD ** -0.5), s)
    linear(rt.z, blk.proj, resid=rt.h, out=rt.h)
    layer_norm(rt.h, blk.norm2, cfg.eps, out=rt.x)
    linear(rt.x, blk.fc1, ACT_GELU_TANH, out=rt.u)
    linear(rt.u, blk.fc2, resid=rt.h, out=rt.h)
    torch.cuda.synchronize()


def test_vision_graph_replays_equal_eager(gpu):
    from fastforward_amd.vision import VisionRuntime
    cfg, w = _small_tower(seed=1)
    rt = VisionRuntime(cfg, w, 8, 12)
    rng = np.random.default_rng(5)
    images = [rng.integers(0, 256, size=(128, 192, 3), dtype=np.uint8) for _ in range(2)]
    eager = []
    for img in images:
        rt.set_image(torch.from_numpy(img))
        m, d = rt.step()
        eager.append((m.clone(), [x.clone() for x in d]))
    rt.capture()
    for _ in range(2):
        for img, (em, ed) in zip(images, eager):
            rt.set_image(torch.from_numpy(img))
            torch.cuda.synchronize()
            m, d = rt.replay()
            torch.cuda.synchronize()
            assert torch.equal(m, em) and all(torch.equal(a, b) for a, b in zip(d, ed))


@pytest.mark.timeout(600)
def test_vision_8b_full_depth(gpu):
    """The whole 8B tower (27 blocks, 1152 hidden, 16 heads of 72, MLP 4304 padded
    to 4352, 4608-wide mergers, DeepStack after blocks 8, 16 and 24) on a 16 x 32
    patch grid. Teacher-forced: every block, given the GPU's own input to it,
    within 1% relative L2 of the oracle's block; every DeepStack merger and the
    final merger, given the GPU's block output, within 2%. End to end (the
    oracle's own tower from the same pixels): printed per block, and the merged
    and DeepStack features within 3%: the 27 residual updates each differ by
    <= 0.3% (the teacher-forced figures of this shape), as independent roundings
    that add in quadrature, sqrt(27) x 0.3% ~ 1.6%, and the bar is twice that."""
    from fastforward_amd.vision import VISION_PRESETS, VisionRuntime, make_vision
    cfg = VISION_PRESETS["qwen3vl-8b"]
    w = make_vision(cfg, seed=2)
    gh, gw = 16, 32
    rt = VisionRuntime(cfg, w, gh, gw)
    rng = np.random.default_rng(6)
    rgb = rng.integers(0, 256, size=(16 * gh, 16 * gw, 3), dtype=np.uint8)
    rt.set_image(torch.from_numpy(rgb))
    trace = []
    merged, deep = rt.step(trace)
    torch.cuda.synchronize()
    trace = [t.cpu() for t in trace]
    merged, deep = merged.cpu(), [d.cpu() for d in deep]
    del rt
    shape, ow = _to_oracle(cfg, w)
    del w
    torch.cuda.empty_cache()
    cos, sin = OV.rope_cos_sin(shape, gh, gw)
    pixels = OV.pack_pixels(rgb)
    h0 = OV.linear(pixels, ow.patch_w, ow.patch_b)
    h0 = OV.bf16(h0.to(F32) + OV.pos_embeds(shape, ow.pos_embed, gh, gw).to(F32)).to(BF16)
    hin = [h0] + trace
    for j in range(cfg.depth):
        got = _rel_l2(trace[j], OV.block(shape, ow.blocks[j], hin[j], cos, sin))
        print(f"8b vision block {j}: teacher-forced rel L2 {got:.2e}", flush=True)
        assert got <= 1e-2, f"teacher-forced block {j}: {got:.3e}"
    for k, j in enumerate(cfg.deepstack):
        got = _rel_l2(deep[k], OV.merge(shape, ow.deep[k], trace[j]))
        print(f"8b vision deepstack merger {k} (block {j}): teacher-forced rel L2 {got:.2e}", flush=True)
        assert got <= 2e-2
    got = _rel_l2(merged, OV.merge(shape, ow.merger, trace[-1]))
    print(f"8b vision merger: teacher-forced rel L2 {got:.2e}", flush=True)
    assert got <= 2e-2
    otrace = []
    omerged, odeep = OV.tower(shape, ow, pixels, gh, gw, otrace)
    print("8b vision end to end per block: " + " ".join(f"{_rel_l2(a, b):.1e}" for a, b in zip(trace, otrace)),
          flush=True)
    ends = [_rel_l2(merged, omerged)] + [_rel_l2(a, b) for a, b in zip(deep, odeep)]
    print(f"8b vision end to end merged / deepstack: {ends}", flush=True)
    assert max(ends) <= 3e-2
