"""Per-op parity of the gfx950 kernels against the CPU oracle on seeded inputs.

Tolerances (stated per op):
* bit-exact: add_rms residual, e4m3 activation / weight quantization codes and
  scales given the same bf16 input, int4 codes and scale indexing, embedding
  gather, fused-vs-unfused producers, V^T transposition.
* <= 1 bf16 ulp, exact for all but a small fraction: SwiGLU, readout, M-RoPE
  tables.
* FP8 GEMM: within the fp32-accumulation bound of the exact (fp64) product of
  the codes -- 1 bf16 ulp + 2^-16 * sum_k |a_k w_k| * sa * sw -- and equal to the
  oracle's bf16 result for >= 98% of elements up to K = 16384 and >= 97% beyond
  (cancellation-dominated outputs near zero are where the two summation orders
  round differently; the matrix unit sums each 32-product block with ~13 bits,
  so the share grows with the number of blocks).
* <= 2 bf16 ulps, exact for all but 0.2%: RMSNorm outputs and q/k norm + rotary.
  The fp32 sum of squares differs from the oracle's only in summation order;
  when that flips the intermediate bf16(x*rsqrt) by one ulp, the following
  multiply by the weight can carry it to two ulps of the output if the product
  lands in a lower binade.
* attention: |gpu - oracle| <= 1/64 absolute (values are O(1)) and relative RMS
  <= 0.5% (the block-online softmax rounds P to bf16 at different running maxima).
* W4A16 GEMM: relative RMS <= 0.5% vs the fp32-dequant product (the reference's own
  operator bar is 1%), bit-exact dequantized weights through one-hot rows.
"""
import numpy as np
import pytest
import torch

from oracle import ops as O
from tests.helpers import assert_bf16_close, bf16_ulps

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16
DEV = "cuda"


def _g(seed):
    return torch.Generator().manual_seed(seed)


def _norm_module(h, seed, jitter=0.1):
    from fastforward_amd.ops import RMSNorm
    w = (1 + jitter * torch.randn(h, generator=_g(seed))).to(BF16)
    return RMSNorm(w.to(DEV), 1e-6), w


# ------------------------------------------------------------------ norms

@pytest.mark.parametrize("t,h", [(320, 2048), (576, 4096), (37, 5120)])
def test_fast_norm(gpu, t, h):
    from fastforward_amd import ops
    x = (torch.randn(1, t, h, generator=_g(1)) * 3).to(BF16)
    mod, w = _norm_module(h, 2)
    got = ops.fast_norm(x.to(DEV), mod).cpu()
    want = O.fast_norm(x, w, 1e-6)
    assert_bf16_close(got, want, 2, 2e-3, "fast_norm")


@pytest.mark.parametrize("deep", [False, True])
@pytest.mark.parametrize("t,h", [(576, 4096), (320, 2048), (17, 5120)])
def test_add_rms(gpu, t, h, deep):
    from fastforward_amd import ops
    a = torch.randn(1, t, h, generator=_g(3)).to(BF16)
    b = torch.randn(1, t, h, generator=_g(4)).to(BF16)
    mod, w = _norm_module(h, 5)
    start, nv = (2, min(10, t - 2)) if deep else (0, 0)
    dp = torch.randn(nv, h, generator=_g(6)).to(BF16) if deep else None
    res, out = ops.add_rms(a.to(DEV), b.to(DEV), dp.to(DEV) if deep else None, mod, start, nv)
    rw, ow = O.add_rms(a, b, dp, w, 1e-6, start, nv)
    assert torch.equal(res.cpu(), rw), "residual must be bit-exact"
    assert_bf16_close(out.cpu(), ow, 2, 2e-3, "add_rms out")


def test_add_rms_quant_equals_unfused(gpu):
    from fastforward_amd import ops, _lib
    from fastforward_amd._lib import call, ptr, stream
    t, h = 576, 4096
    a = torch.randn(t, h, generator=_g(7)).to(BF16).to(DEV)
    b = torch.randn(t, h, generator=_g(8)).to(BF16).to(DEV)
    b[3] *= 50                                                   # an outlier row
    mod, _ = _norm_module(h, 9)
    dp = torch.randn(20, h, generator=_g(10)).to(BF16).to(DEV)
    res0, out0 = ops.add_rms(a, b, dp, mod, 5, 20)
    res = torch.empty_like(a)
    out = torch.empty_like(a)
    q = torch.empty(t, h, device=DEV, dtype=torch.float8_e4m3fn)
    s = torch.empty(t, device=DEV)
    call("ff_add_rms_quant", ptr(a), ptr(b), ptr(dp), ptr(mod.weight), ptr(res), ptr(out), ptr(q), ptr(s),
         t, h, 1e-6, 5, 20, stream())
    assert torch.equal(res, res0) and torch.equal(out, out0)
    qw, sw = O.quant_rows_dynamic(out0.cpu())
    assert torch.equal(q.view(torch.uint8).cpu(), qw.view(torch.uint8))
    assert torch.equal(s.cpu(), sw)
    # fast_norm_quant without the bf16 output
    q2 = torch.empty_like(q)
    s2 = torch.empty_like(s)
    call("ff_fast_norm_quant", ptr(res0), ptr(mod.weight), None, ptr(q2), ptr(s2), t, h, 1e-6, stream())
    qn, sn = O.quant_rows_dynamic(ops.fast_norm(res0, mod).cpu())
    assert torch.equal(q2.view(torch.uint8).cpu(), qn.view(torch.uint8)) and torch.equal(s2.cpu(), sn)
    _ = _lib


# ------------------------------------------------------------------ rotary

def _packed_qkv(t, hq, hk, d, seed):
    return (torch.randn(1, t, (hq + 2 * hk) * d, generator=_g(seed)) * 2).to(BF16)


@pytest.mark.parametrize("t,hq,hk", [(576, 32, 8), (320, 16, 8), (33, 64, 8)])
def test_qk_pair(gpu, t, hq, hk):
    from fastforward_amd import ops
    d = 128
    packed = _packed_qkv(t, hq, hk, d, 11)
    qn, wq = _norm_module(d, 12, 0.3)
    kn, wk = _norm_module(d, 13, 0.3)
    pos = O.mrope_positions(4, 4, 6, t) if t >= 28 else torch.arange(t).expand(3, t).clone()
    cos, sin = O.mrope_cos_sin(pos, 5e6, d)
    pg = packed.to(DEV)
    q = pg[..., : hq * d].view(1, t, hq, d)
    k = pg[..., hq * d:(hq + hk) * d].view(1, t, hk, d)
    yq, yk = ops.qk_pair(q, k, qn, kn, cos.to(DEV), sin.to(DEV))
    wq_, wk_ = O.qk_pair(packed[..., : hq * d].view(1, t, hq, d), packed[..., hq * d:(hq + hk) * d].view(1, t, hk, d),
                         wq, wk, 1e-6, 1e-6, cos, sin)
    assert_bf16_close(yq.cpu(), wq_, 2, 2e-3, "qk_pair q")
    assert_bf16_close(yk.cpu(), wk_, 2, 2e-3, "qk_pair k")


def test_qkv_post_matches_qk_pair_and_transposes_v(gpu):
    from fastforward_amd import ops
    from fastforward_amd._lib import call, ptr, stream
    t, hq, hk, d = 300, 32, 8, 128
    tp = 320
    packed = _packed_qkv(t, hq, hk, d, 14).to(DEV)[0]
    qn, _ = _norm_module(d, 15, 0.3)
    kn, _ = _norm_module(d, 16, 0.3)
    cos, sin = O.mrope_cos_sin(O.mrope_positions(4, 8, 8, t), 5e6, d)
    cos, sin = cos[0].to(DEV), sin[0].to(DEV)
    yq = torch.empty(hq, t, d, device=DEV, dtype=BF16)
    yk = torch.empty(hk, t, d, device=DEV, dtype=BF16)
    vt = torch.full((hk, d, tp), float("nan"), device=DEV, dtype=BF16)
    base, n3 = packed.data_ptr(), (hq + 2 * hk) * d
    call("ff_qkv_post", base, base + hq * d * 2, base + (hq + hk) * d * 2, n3, ptr(qn.weight), ptr(kn.weight),
         1e-6, 1e-6, ptr(cos), ptr(sin), ptr(yq), ptr(yk), ptr(vt), t, tp, hq, hk, d, stream())
    q = packed[:, : hq * d].view(1, t, hq, d)
    k = packed[:, hq * d:(hq + hk) * d].view(1, t, hk, d)
    rq, rk = ops.qk_pair(q, k, qn, kn, cos[None], sin[None])
    assert torch.equal(yq, rq[0]) and torch.equal(yk, rk[0])
    v = packed[:, (hq + hk) * d:].view(t, hk, d)
    assert torch.equal(vt[:, :, :t], v.permute(1, 2, 0))
    assert torch.all(vt[:, :, t:] == 0)


# ------------------------------------------------------------------ swiglu

@pytest.mark.parametrize("t,i", [(576, 12288), (1, 12288), (320, 6144)])
def test_swiglu(gpu, t, i):
    from fastforward_amd import ops
    gu = (torch.randn(t, 2 * i, generator=_g(17)) * 3).to(BF16)
    g, u = gu.to(DEV).chunk(2, -1)
    got = ops.swiglu(g, u).cpu()
    want = O.swiglu(*gu.chunk(2, -1))
    assert_bf16_close(got, want, 1, 5e-3, "swiglu")


def test_swiglu_quant_equals_unfused(gpu):
    from fastforward_amd import ops
    from fastforward_amd._lib import call, ptr, stream
    t, i = 200, 12288
    gu = (torch.randn(t, 2 * i, generator=_g(18)) * 3).to(BF16).to(DEV)
    g, u = gu.chunk(2, -1)
    y0 = ops.swiglu(g, u)
    y = torch.empty_like(y0)
    q = torch.empty(t, i, device=DEV, dtype=torch.float8_e4m3fn)
    s = torch.empty(t, device=DEV)
    call("ff_swiglu_quant", ptr(g), ptr(u), 2 * i, ptr(y), ptr(q), ptr(s), t, i, stream())
    assert torch.equal(y, y0)
    qw, sw = O.quant_rows_dynamic(y0.cpu())
    assert torch.equal(q.view(torch.uint8).cpu(), qw.view(torch.uint8)) and torch.equal(s.cpu(), sw)


# ------------------------------------------------------------------ quantization

@pytest.mark.parametrize("m,k", [(576, 4096), (576, 12288), (33, 25600), (5, 40960), (1, 2048)])
def test_quant_rows_fp8_bit_exact(gpu, m, k):
    from fastforward_amd.linear import FP8Linear
    x = torch.randn(m, k, generator=_g(19))
    x[torch.rand(m, k, generator=_g(20)) < 0.001] *= 20
    if m > 3:
        x[2] = 0
    x = x.to(BF16)
    op = FP8Linear.__new__(FP8Linear)
    q, s = op.quantize(x.to(DEV))
    qw, sw = O.quant_rows_dynamic(x)
    assert torch.equal(q.view(torch.uint8).cpu(), qw.view(torch.uint8))
    assert torch.equal(s.cpu(), sw)


def test_quant_static_bit_exact(gpu):
    from fastforward_amd._lib import call, ptr, stream
    m, k = 300, 4096
    x = (torch.randn(m, k, generator=_g(21)) * 40).to(BF16)
    inv = 448 / 37.5
    q = torch.full((304, k), 7, device=DEV, dtype=torch.uint8)
    x_d = x.to(DEV)
    call("ff_quant_static_fp8", ptr(x_d), ptr(q), m, 304, k, inv, stream())
    qw = O.quant_static(x, inv)
    assert torch.equal(q[:m].cpu(), qw.view(torch.uint8))
    assert torch.all(q[m:] == 0)


@pytest.mark.parametrize("per_channel", [True, False])
def test_weight_quant_fp8_bit_exact(gpu, per_channel):
    from fastforward_amd.linear import FP8Linear, StaticFP8Linear
    w = (torch.randn(6144, 4096, generator=_g(22)) * 0.02).to(BF16)
    w[5, 7] = 0.5                                               # a channel outlier
    qw, sw = O.fp8_weight_quant(w, per_channel)
    if per_channel:
        op = FP8Linear(w.to(DEV))
        assert torch.equal(op.scale.reshape(-1).cpu(), sw)
    else:
        op = StaticFP8Linear(w.to(DEV), 448 / 8.0)
        assert torch.equal(op.weight_scale.cpu(), sw)
    assert torch.equal(op.weight.view(torch.uint8).cpu(), qw.view(torch.uint8))


@pytest.mark.parametrize("sym,group", [(True, 128), (False, 32), (False, 128)])
def test_int4_quant_bit_exact(gpu, sym, group):
    from fastforward_amd.linear import Int4
    w = (torch.randn(512, 1024, generator=_g(23)) * 0.02).to(BF16)
    quant = O.int4_quantize_sym if sym else O.int4_quantize_asym
    _, packed, scales = quant(w, group)
    op = Int4(w.to(DEV), group=group, symmetric=sym)
    assert torch.equal(op.packed.cpu(), packed)
    assert torch.equal(op.scales.cpu(), scales)


# ------------------------------------------------------------------ GEMMs

# the microbench shapes, the 8B step's row-major tiles (qkv: 128 x 128 four-stage; o: 64 x 128;
# gate/up width: 128 x 128 two-stage), a tail row and ragged edges
FP8_SHAPES = [(320, 2048, 6144), (320, 6144, 2048), (576, 4096, 12288), (576, 12288, 4096),
              (1024, 5120, 25600), (576, 4096, 6144), (576, 4096, 4096), (576, 4096, 24576), (1, 4096, 24576),
              (17, 256, 384), (130, 1024, 200), (33, 25600, 1024)]


def _assert_fp8_gemm(y, qa, sa, qw, sw, oracle, what):
    """Against the exact product: sums of e4m3 x e4m3 products span < 53 bits, so
    the fp64 GEMM of the decoded codes is exact. The kernel accumulates in fp32,
    one addition per 128-deep MFMA step, so its accumulated error is at most
    (K/128) * 2^-24 * sum_k |a_k w_k| <= 2^-16 * sum_k |a_k w_k| for K <= 25600,
    plus one bf16 rounding of the result (<= 1 ulp of the exact value)."""
    import numpy as np
    from tests.numerics import ulp_bf16
    a, w = qa.double(), qw.double()
    sa_, sw_ = sa.double().reshape(-1, 1), sw.double().reshape(1, -1)
    exact = (a @ w.T) * sa_ * sw_
    abs_sum = (a.abs() @ w.abs().T) * sa_.abs() * sw_.abs()
    got = y.double()
    bound = torch.from_numpy(ulp_bf16(exact.numpy())) + abs_sum * 2.0 ** -16
    excess = (got - exact).abs() - bound
    assert float(excess.max()) <= 0, f"{what}: exceeds the accumulation bound by {float(excess.max())}"
    # and almost every element rounds to the same bf16 as the oracle's fp32 GEMM:
    # <= 2% up to K = 16384, 3% beyond (more 32-product blocks summed with ~13 bits)
    frac = float((y != oracle).float().mean())
    limit = 0.02 if a.shape[1] <= 16384 else 0.03
    assert frac <= limit, f"{what}: {frac:.4f} of elements differ from the oracle"
    _ = np


@pytest.mark.parametrize("m,k,n", FP8_SHAPES)
def test_gemm_fp8_dynamic(gpu, m, k, n):
    """Codes and scales come from the oracle's quantizers (pinned bit-exact above)."""
    from fastforward_amd._lib import call, ptr, stream
    x = torch.randn(m, k, generator=_g(24))
    x[torch.rand(m, k, generator=_g(25)) < 0.001] *= 20
    x = x.to(BF16)
    w = (torch.randn(n, k, generator=_g(26)) * 0.02).to(BF16)
    qa, sa = O.quant_rows_dynamic(x)
    qw, sw = O.fp8_weight_quant(w)
    want = O.fp8_gemm(qa, sa, qw, sw)
    y = torch.empty(m, n, device=DEV, dtype=BF16)
    # device copies are held in locals: a temporary's memory could be reused before the launch
    qa_d, sa_d, qw_d, sw_d = qa.to(DEV), sa.to(DEV), qw.to(DEV), sw.to(DEV)
    call("ff_gemm_fp8", ptr(qa_d), ptr(sa_d), 1, ptr(qw_d), ptr(sw_d), 1, ptr(y), n, m, n, k, stream())
    _assert_fp8_gemm(y.cpu(), qa, sa, qw, sw, want, f"gemm_fp8 {m}x{k}x{n}")


@pytest.mark.parametrize("m,i,k", [(576, 12288, 4096), (1, 12288, 4096), (130, 6144, 2048), (33, 640, 256)])
def test_gemm_fp8_swiglu_equals_unfused(gpu, m, i, k):
    """The gate/up GEMM with the SwiGLU epilogue equals ff_gemm_fp8 on the packed
    weight followed by swiglu, bit for bit; its row maxima equal max |h|; the
    quantisation from them equals ff_quant_rows_fp8 on h."""
    from fastforward_amd import ops
    from fastforward_amd._lib import call, ptr, stream
    x = (torch.randn(m, k, generator=_g(34)) * 2).to(BF16)
    w = (torch.randn(2 * i, k, generator=_g(35)) * 0.05).to(BF16)
    qa, sa = O.quant_rows_dynamic(x)
    qw, sw = O.fp8_weight_quant(w)
    qa_d, sa_d, qw_d, sw_d = qa.to(DEV), sa.to(DEV), qw.to(DEV), sw.to(DEV)
    gu = torch.empty(m, 2 * i, device=DEV, dtype=BF16)
    call("ff_gemm_fp8", ptr(qa_d), ptr(sa_d), 1, ptr(qw_d), ptr(sw_d), 1, ptr(gu), 2 * i, m, 2 * i, k, stream())
    want = ops.swiglu(*gu.chunk(2, -1))
    h = torch.full((m, i), float("nan"), device=DEV, dtype=BF16)
    pmax = torch.full((m, i // 64), float("nan"), device=DEV)
    call("ff_gemm_fp8_swiglu", ptr(qa_d), ptr(sa_d), ptr(qw_d), ptr(sw_d), ptr(h), i, ptr(pmax), m, i, k, stream())
    assert torch.equal(h, want)
    assert torch.equal(pmax, h.float().abs().view(m, i // 64, 64).amax(-1))
    q1, s1 = torch.empty(m, i, device=DEV, dtype=torch.uint8), torch.empty(m, device=DEV)
    q2, s2 = torch.empty_like(q1), torch.empty_like(s1)
    call("ff_quant_rows_pmax", ptr(h), i, ptr(pmax), i // 64, ptr(q1), ptr(s1), m, i, stream())
    call("ff_quant_rows_fp8", ptr(h), i, ptr(q2), ptr(s2), m, i, stream())
    assert torch.equal(q1, q2) and torch.equal(s1, s2)


def test_pack_weight_fp8_layout(gpu):
    """ff_pack_weight_fp8 stores fragment (f, kt) at (kt * n/16 + f) * 2048 with
    lane l = 16 g + r holding row 16 f + r, k bytes [128 kt + 32 g, +16) at 16 l
    and the next 16 at 1024 + 16 l."""
    from fastforward_amd._lib import call, ptr, stream
    n, k = 48, 384
    w = torch.randint(0, 256, (n, k), generator=_g(50), dtype=torch.uint8)
    p = torch.empty(n * k, device=DEV, dtype=torch.uint8)
    w_d = w.to(DEV)
    call("ff_pack_weight_fp8", ptr(w_d), ptr(p), n, k, stream())
    got = p.cpu().numpy().reshape(k // 128, n // 16, 2, 64, 16).transpose(1, 0, 2, 3, 4)
    wn = w.numpy()
    for f in range(n // 16):
        for kt in range(k // 128):
            for lane in range(64):
                r, g = lane % 16, lane // 16
                row = wn[16 * f + r, 128 * kt + 32 * g: 128 * kt + 32 * g + 32]
                assert np.array_equal(got[f, kt, 0, lane], row[:16]) and np.array_equal(got[f, kt, 1, lane], row[16:])


# 12288 channels (64 column tiles) take row tiles of 144 (576 tokens), 112
# (400), 96 (700) and 128 (1000); MLP widths that 192 does not divide take
# 128-channel tiles (4096; the 32B shape's 25600 at 1024 tokens; the 4B shape's
# 9728); up to 176 tokens, 64-channel tiles of one row tile (176, 100, 150, 17
# tokens: 176, 112, 144 and 64 rows)
@pytest.mark.parametrize("m,i,k", [(576, 12288, 4096), (300, 12288, 2048), (433, 6144, 4096), (3, 12288, 4096),
                                   (576, 4096, 4096), (176, 12288, 4096), (400, 12288, 4096), (700, 12288, 4096),
                                   (1000, 12288, 4096), (1024, 25600, 5120), (576, 9728, 2560), (300, 4160, 2048),
                                   (100, 12288, 4096), (150, 12288, 2048), (17, 12288, 4096)])
def test_gemm_fp8_swiglu_packed_equals_rowmajor(gpu, m, i, k):
    """The gate/up GEMM on the packed weight copy (BM x 384 tiles, or BM x 256 where
    192 does not divide the MLP width, BM = 80..144 by grid, weights straight into
    the MFMA operands) gives the same bits as ff_gemm_fp8_swiglu on the row-major
    weight, SwiGLU output and row maxima, including a ragged last token tile;
    shapes it does not take (3 rows, i % 128 != 0, too few tiles) go to the
    row-major kernels."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import FP8Linear
    x = (torch.randn(m, k, generator=_g(51)) * 2).to(BF16).to(DEV)
    op = FP8Linear((torch.randn(2 * i, k, generator=_g(52)) * 0.05).to(BF16).to(DEV), keep_rowmajor=True)
    qa, sa = op.quantize(x)
    outs = []
    for entry in ("ff_gemm_fp8_swiglu", "ff_gemm_fp8_swiglu_pk"):
        h = torch.full((m, i), float("nan"), device=DEV, dtype=BF16)
        pmax = torch.full((m, i // 64), float("nan"), device=DEV)
        args = [ptr(qa), ptr(sa), ptr(op.weight)] + ([ptr(op.packed)] if entry.endswith("pk") else [])
        call(entry, *args, ptr(op.scale), ptr(h), i, ptr(pmax), m, i, k, stream())
        outs.append((h, pmax))
    (h0, p0), (h1, p1) = outs
    assert not torch.isnan(h0.float()).any()
    assert torch.equal(h0, h1) and torch.equal(p0, p1)


# (m, n, k, row tile, splits the packed path takes); 0 = unsplit on the small
# packed tiles (576 x 4096 x 4096: 80 x 128, 256 workgroups; 500 x 4096 x 4096:
# 80 x 128, the last tile ragged; 576 / 500 x 6144 x 4096: 64 x 256,
# the last tile ragged; 300 x 4096 x 2048: 64 x 128, the candidate with the most
# workgroups on a short grid; k = 8192 wherever a small tile fills the GPU:
# 1000 x 6144 and the 32B o projection, 1024 x 5120, on 64 x 256) or the
# row-major kernels (3 rows, n % 128); short m (176 tokens, 2B widths at 64)
# takes 64-row tiles with a k split (8, 4 or 2 ways where they divide k, 6 or 5
# ways with uneven k ranges: 176 tokens of the 8B shape 5, the 2B down at 250
# tokens 6, the 4B down at 176 tokens 6); 576 x 2560 x 9728 (4B down) splits 76 k
# steps into 20, 20, 20 and 16
PK_SHAPES = [(576, 4096, 12288, 144, 4), (300, 2048, 8192, 144, 8), (1000, 6144, 8192, 0, 0),
             (1024, 5120, 8192, 0, 0), (576, 2560, 9728, 144, 4),
             (576, 12288, 4096, 144, 1), (640, 4096, 12288, 144, 3), (1152, 4096, 12288, 144, 2),
             (176, 4096, 12288, 64, 5), (176, 4096, 4096, 64, 5), (64, 2048, 2048, 64, 4), (250, 2048, 6144, 64, 6),
             (176, 2560, 9728, 64, 6),
             (576, 4096, 4096, 0, 0), (500, 4096, 4096, 0, 0), (576, 6144, 4096, 0, 0), (500, 6144, 4096, 0, 0),
             (300, 4096, 2048, 0, 0),
             (3, 4096, 4096, 0, 0), (576, 4160, 12288, 0, 0)]


@pytest.mark.parametrize("m,n,k,bm,splits", PK_SHAPES)
def test_gemm_fp8_pk_matches_rowmajor(gpu, m, n, k, bm, splits):
    """ff_gemm_fp8_pk on the packed weight: the same bits as ff_gemm_fp8 unsplit
    or where it falls back; with a k split, at most 1 bf16 ulp from it (only the
    fp32 order of adding the partials differs), identical bits on repeated calls
    and within the exact-product bound."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import FP8Linear, gemm_pk_workspace
    x = (torch.randn(m, k, generator=_g(60)) * 2).to(BF16).to(DEV)
    op = FP8Linear((torch.randn(n, k, generator=_g(61)) * 0.03).to(BF16).to(DEV), keep_rowmajor=True)
    qa, sa = op.quantize(x)
    need = gemm_pk_workspace(m, n, k)
    # the split count itself: fp32 partials of bm x 256 tiles over the rows padded to whole tiles
    assert need == ((m + bm - 1) // bm * (n // 256) * splits * bm * 256 * 4 if splits > 1 else 0)
    ws = torch.full((max(need, 256),), 0xFF, device=DEV, dtype=torch.uint8)  # no zeroing needed
    ref = torch.empty(m, n, device=DEV, dtype=BF16)
    call("ff_gemm_fp8", ptr(qa), ptr(sa), 1, ptr(op.weight), ptr(op.scale), 1, ptr(ref), n, m, n, k, stream())
    outs = []
    for _ in range(3):
        y = torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
        call("ff_gemm_fp8_pk", ptr(qa), ptr(sa), 1, ptr(op.weight), ptr(op.packed), ptr(op.scale), 1, ptr(y), n,
             m, n, k, ptr(ws), ws.numel(), stream())
        outs.append(y)
    assert all(torch.equal(outs[0], o) for o in outs[1:])
    if splits <= 1:
        assert torch.equal(outs[0], ref)
    else:
        d = bf16_ulps(outs[0], ref)
        assert int(d.max()) <= 1 and float((d > 0).float().mean()) < 0.01
    if (m, n, k) == (300, 2048, 8192):
        qa_c, sa_c, qw_c, sw_c = qa.cpu(), sa.cpu(), op.weight.cpu(), op.scale.cpu().reshape(-1)
        _assert_fp8_gemm(outs[0].cpu(), qa_c, sa_c, qw_c, sw_c, O.fp8_gemm(qa_c, sa_c, qw_c, sw_c),
                         "gemm_fp8_pk split 4")


# unsplit 256-column row tiles, by rounds of 256 workgroups x (rows + 16): 112, 128, 144,
# 176 and 208 rows, each with whole and ragged last row tiles and the shortest k
@pytest.mark.parametrize("m,n,k", [(1000, 12800, 512), (1120, 12800, 512), (576, 12288, 512), (640, 12288, 1024),
                                   (140, 49152, 512), (144, 49152, 1024), (1024, 10240, 1536), (1050, 10240, 512),
                                   (1024, 25600, 512), (1040, 12288, 1536)])
def test_gemm_fp8_pk_unsplit_row_tiles(gpu, m, n, k):
    """The unsplit row tiles: bit for bit ff_gemm_fp8 on the row-major codes, nothing
    written past the last row, and no workspace."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import FP8Linear, gemm_pk_workspace
    x = (torch.randn(m, k, generator=_g(62)) * 2).to(BF16).to(DEV)
    op = FP8Linear((torch.randn(n, k, generator=_g(63)) * 0.03).to(BF16).to(DEV), keep_rowmajor=True)
    qa, sa = op.quantize(x)
    assert gemm_pk_workspace(m, n, k) == 0
    ref = torch.empty(m, n, device=DEV, dtype=BF16)
    call("ff_gemm_fp8", ptr(qa), ptr(sa), 1, ptr(op.weight), ptr(op.scale), 1, ptr(ref), n, m, n, k, stream())
    y = torch.full((m + 1, n), float("nan"), device=DEV, dtype=BF16)
    call("ff_gemm_fp8_pk", ptr(qa), ptr(sa), 1, ptr(op.weight), ptr(op.packed), ptr(op.scale), 1, ptr(y), n,
         m, n, k, 0, 0, stream())
    assert torch.equal(y[:m], ref) and bool(y[m].isnan().all())


# grids of 64 x 128 tiles short of the GPU: 32 x 64 tiles (5 .. 65 rows, one row tile
# and its edges; the smallest n and k), 64 x 64 tiles from 128 of them up (ragged last
# row tile; an odd number of unrolled k blocks) and, past 256 of those, 64 x 128 tiles
# (a whole number per XCD: 64 x 19456, 576 x 2048, 176 x 6144) or 64 x 64 (400 x 2560)
@pytest.mark.parametrize("m,n,k", [(5, 128, 512), (31, 128, 1536), (32, 2048, 2048), (33, 2048, 512), (65, 1024, 1024),
                                   (300, 1024, 512), (320, 2048, 6144), (257, 2048, 1536), (576, 2048, 2048),
                                   (320, 2560, 4096), (176, 6144, 4096), (64, 19456, 512), (400, 2560, 1536),
                                   (512, 2048, 512)])
@pytest.mark.parametrize("rows", [True, False])
def test_gemm_fp8_pk_narrow_tiles(gpu, m, n, k, rows):
    """The narrow packed tiles: bit for bit ff_gemm_fp8 on the row-major codes, with
    per-token / per-channel and with scalar scales, with and without the row-major
    weight given, and no workspace."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import FP8Linear, gemm_pk_workspace
    x = (torch.randn(m, k, generator=_g(160)) * 2).to(BF16).to(DEV)
    op = FP8Linear((torch.randn(n, k, generator=_g(161)) * 0.03).to(BF16).to(DEV), keep_rowmajor=True)
    qa, sa = op.quantize(x)
    sw = op.scale
    if not rows:
        sa, sw = sa[:1].clone(), sw.reshape(-1)[:1].clone()
    if m > 256 or (m, n) == (176, 6144):
        assert gemm_pk_workspace(m, n, k) == 0
    r = 1 if rows else 0
    ref = torch.empty(m, n, device=DEV, dtype=BF16)
    call("ff_gemm_fp8", ptr(qa), ptr(sa), r, ptr(op.weight), ptr(sw), r, ptr(ref), n, m, n, k, stream())
    ws = torch.empty(max(gemm_pk_workspace(m, n, k), 256), device=DEV, dtype=torch.uint8)
    for w in (op.weight, None):
        y = torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
        call("ff_gemm_fp8_pk", ptr(qa), ptr(sa), r, ptr(w), ptr(op.packed), ptr(sw), r, ptr(y), n, m, n, k, ptr(ws),
             ws.numel(), stream())
        if gemm_pk_workspace(m, n, k) == 0:
            assert torch.equal(y, ref)
        else:   # short m, k split: only the fp32 order of the partials differs
            assert int(bf16_ulps(y, ref).max()) <= 1


@pytest.mark.parametrize("m,n,k,static,deep", [(576, 4096, 12288, False, True), (576, 4096, 12288, True, False),
                                               (500, 4096, 12288, False, False), (300, 2048, 8192, True, True),
                                               (576, 4096, 4096, False, False), (1, 4096, 12288, False, False),
                                               (1, 4096, 12288, True, False), (640, 4096, 12288, False, True),
                                               (1152, 4096, 12288, True, False), (176, 4096, 12288, False, True),
                                               (176, 4096, 12288, True, False), (576, 2560, 9728, False, True)])
def test_gemm_fp8_pk_add_rms_equals_unfused(gpu, m, n, k, static, deep):
    """ff_gemm_fp8_pk_add_rms_quant(_static) == ff_gemm_fp8_pk followed by
    ff_add_rms_quant(_static), bit for bit in y, the residual, the e4m3 codes
    and the scales: on the split shapes the add_rms launch adds the split-K
    partials itself (500 rows: the last 144-row tile ragged; DeepStack rows
    inside the range), elsewhere (k = 4096, one row) the two entry points
    run."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import FP8Linear, gemm_pk_workspace
    x = (torch.randn(m, k, generator=_g(64)) * 2).to(BF16).to(DEV)
    op = FP8Linear((torch.randn(n, k, generator=_g(65)) * 0.03).to(BF16).to(DEV))
    qa, sa = op.quantize(x)
    a = (torch.randn(m, n, generator=_g(66)) * 4).to(BF16).to(DEV)
    w = (1 + 0.1 * torch.randn(n, generator=_g(67))).to(BF16).to(DEV)
    dp = (torch.randn(40, n, generator=_g(68))).to(BF16).to(DEV) if deep else None
    start, nv = (min(10, m - 1), min(40, m - min(10, m - 1))) if deep else (0, 0)
    ws = torch.full((max(gemm_pk_workspace(m, n, k), 256),), 0xFF, device=DEV, dtype=torch.uint8)
    inv = 448 / 30.0
    outs = []
    for fused in (False, True):
        y = torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
        res = torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
        q = torch.full((m, n), 0x7F, device=DEV, dtype=torch.uint8)
        sc = torch.full((m,), float("nan"), device=DEV)
        gemm = [ptr(qa), ptr(sa), 1, ptr(op.weight), ptr(op.packed), ptr(op.scale), 1, ptr(y)]
        if fused:
            tail = [ptr(a), ptr(dp), ptr(w), ptr(res), ptr(q)] + ([inv] if static else [ptr(sc)])
            call("ff_gemm_fp8_pk_add_rms_quant" + ("_static" if static else ""), *gemm, m, n, k, ptr(ws), ws.numel(),
                 *tail, 1e-6, start, nv, stream())
        else:
            call("ff_gemm_fp8_pk", *gemm, n, m, n, k, ptr(ws), ws.numel(), stream())
            if static:
                call("ff_add_rms_quant_static", ptr(a), ptr(y), ptr(dp), ptr(w), ptr(res), None, ptr(q), inv, m, n,
                     1e-6, start, nv, stream())
            else:
                call("ff_add_rms_quant", ptr(a), ptr(y), ptr(dp), ptr(w), ptr(res), None, ptr(q), ptr(sc), m, n,
                     1e-6, start, nv, stream())
        outs.append((y, res, q, sc))
    (y0, r0, q0, s0), (y1, r1, q1, s1) = outs
    assert not torch.isnan(y0.float()).any() and not torch.isnan(r0.float()).any()
    assert torch.equal(y0, y1) and torch.equal(r0, r1) and torch.equal(q0, q1)
    if not static:
        assert torch.equal(s0, s1)


def test_gemm_fp8_pk_scalar_scales(gpu):
    """Per-tensor scales (sa_rows = sw_cols = 0) on the split path agree with ff_gemm_fp8."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import FP8Linear, gemm_pk_workspace
    m, n, k = 576, 4096, 12288
    x = (torch.randn(m, k, generator=_g(62))).to(BF16).to(DEV)
    op = FP8Linear((torch.randn(n, k, generator=_g(63)) * 0.03).to(BF16).to(DEV), keep_rowmajor=True)
    qa, _ = op.quantize(x)
    sa, sw = torch.tensor([0.01], device=DEV), torch.tensor([0.002], device=DEV)
    ws = torch.zeros(gemm_pk_workspace(m, n, k), device=DEV, dtype=torch.uint8)
    ref, y = (torch.empty(m, n, device=DEV, dtype=BF16) for _ in range(2))
    call("ff_gemm_fp8", ptr(qa), ptr(sa), 0, ptr(op.weight), ptr(sw), 0, ptr(ref), n, m, n, k, stream())
    call("ff_gemm_fp8_pk", ptr(qa), ptr(sa), 0, ptr(op.weight), ptr(op.packed), ptr(sw), 0, ptr(y), n, m, n, k,
         ptr(ws), ws.numel(), stream())
    assert int(bf16_ulps(y, ref).max()) <= 1


def test_gemm_fp8_static_scalars(gpu):
    from fastforward_amd.linear import StaticFP8Linear
    m, k, n = 576, 4096, 4096
    x = (torch.randn(m, k, generator=_g(27)) * 3).to(BF16)
    w = (torch.randn(n, k, generator=_g(28)) * 0.02).to(BF16)
    op = StaticFP8Linear(w.to(DEV), 448 / 12.0)
    y = op(x.to(DEV)).cpu()
    want = O.fp8_linear_static(x, op.weight.cpu(), op.weight_scale.cpu(), op.inverse_scale, op.input_scale.cpu())
    qa = O.quant_static(x, op.inverse_scale)
    _assert_fp8_gemm(y, qa, op.input_scale.cpu(), op.weight.cpu(), op.weight_scale.cpu(), want, "static fp8")


@pytest.mark.parametrize("sym,group", [(True, 128), (False, 32)])
@pytest.mark.parametrize("m,k,n", [(576, 4096, 6144), (1, 12288, 4096), (100, 1024, 384)])
def test_gemm_w4a16(gpu, m, k, n, sym, group):
    from fastforward_amd.linear import Int4
    x = torch.randn(m, k, generator=_g(29)).to(BF16)
    w = (torch.randn(n, k, generator=_g(30)) * 0.02).to(BF16)
    op = Int4(w.to(DEV), group=group, symmetric=sym)
    y = op(x.to(DEV)).cpu().double()
    want = O.w4a16_linear(x, op.packed.cpu(), op.scales.cpu(), group).double()
    exact = x.double() @ O.int4_dequant(op.packed.cpu(), op.scales.cpu(), group).double().T
    rel = float((y - exact).pow(2).mean().sqrt() / exact.pow(2).mean().sqrt())
    assert rel <= 5e-3, rel
    assert float((want - exact).pow(2).mean().sqrt() / exact.pow(2).mean().sqrt()) <= 5e-3


W4_TILES = {"64x256": 1, "192x192": 2}


@pytest.fixture
def tuning(gpu):
    """ff_set_tuning(knob, value) for one test; every knob is reset afterwards."""
    from fastforward_amd._lib import call
    used = []

    def set_(knob, value):
        used.append(knob)
        call("ff_set_tuning", knob, value)
    yield set_
    for knob in used:
        call("ff_set_tuning", knob, 0)


FF_TUNE_W4A16_TILE, FF_TUNE_W4A16_SPLITS = 3, 4


@pytest.mark.parametrize("tile,splits", [("64x256", None), ("64x256", 1), ("64x256", 3), ("192x192", None)])
@pytest.mark.parametrize("m,k,n", [(576, 4096, 6144), (200, 1024, 392), (1, 12288, 4096)])
def test_gemm_w4a16_both_tiles(gpu, tuning, m, k, n, tile, splits):
    """Each tile shape of the W4A16 GEMM (chosen by size in production) and the
    split-K form of the 64 x 256 tile (automatic, off, forced to 3) against the
    fp64 product with the exactly dequantised weight, asymmetric group 32 and
    ragged M / N edges included."""
    from fastforward_amd.linear import Int4
    tuning(FF_TUNE_W4A16_TILE, W4_TILES[tile])
    if splits is not None:
        tuning(FF_TUNE_W4A16_SPLITS, splits)
    x = torch.randn(m, k, generator=_g(36)).to(BF16)
    w = (torch.randn(n, k, generator=_g(37)) * 0.02).to(BF16)
    for sym, group in ((True, 128), (False, 32)):
        op = Int4(w.to(DEV), group=group, symmetric=sym)
        y = op(x.to(DEV)).cpu().double()
        exact = x.double() @ O.int4_dequant(op.packed.cpu(), op.scales.cpu(), group).double().T
        rel = float((y - exact).pow(2).mean().sqrt() / exact.pow(2).mean().sqrt())
        assert rel <= 5e-3, (tile, sym, rel)
        # worst element against the output scale: bf16 operand and output rounding only
        worst = float((y - exact).abs().max() / exact.pow(2).mean().sqrt())
        assert worst <= 0.05, (tile, sym, worst)


@pytest.mark.parametrize("tile", ["64x256", "192x192"])
def test_w4a16_dequant_bit_exact_via_one_hot(gpu, tuning, tile):
    """x = rows of the identity: y[r, n] = bf16((q-8)*s + z) for k = r exactly.
    Columns 0-39 hold a constant 64.0 in their first 32 k: the asymmetric
    quantizer then stores s = bf16(1e-6), z = 64, for which z - 8s is not exact
    in fp32, so those stages take the kernel's exact (q-8, then fma) form."""
    from fastforward_amd.linear import Int4
    tuning(FF_TUNE_W4A16_TILE, W4_TILES[tile])
    k, n = 256, 128
    w = (torch.randn(n, k, generator=_g(31)) * 0.02).to(BF16)
    w[:40, :32] = 64.0
    for sym, group in ((True, 128), (False, 32)):
        op = Int4(w.to(DEV), group=group, symmetric=sym)
        if not sym:
            s, z = op.scales[0, 0].double().cpu().tolist()          # exact in float64
            z8_f32 = float(torch.tensor(z - 8 * s, dtype=torch.float64).float())
            assert z == 64.0 and z8_f32 != z - 8 * s                  # z8 inexact in fp32
        eye = torch.eye(k, dtype=BF16, device=DEV)
        y = op(eye).cpu()
        dq = O.int4_dequant(op.packed.cpu(), op.scales.cpu(), group).to(BF16)
        assert torch.equal(y, dq.T.contiguous())


# ------------------------------------------------------------------ attention

@pytest.mark.parametrize("t,hq,hk", [(576, 32, 8), (320, 16, 8), (70, 64, 8), (640, 32, 8), (176, 32, 8), (641, 32, 8)])
def test_attention_causal(gpu, t, hq, hk):
    from fastforward_amd import ops
    d = 128
    q = torch.randn(1, hq, t, d, generator=_g(32)).to(BF16)
    k = torch.randn(1, hk, t, d, generator=_g(33)).to(BF16)
    v = torch.randn(1, hk, t, d, generator=_g(34)).to(BF16)
    v[:, 1] += 2                                                 # distinguishes kv heads
    got = ops.attention_direct(q.to(DEV), k.to(DEV), v.to(DEV), d ** -0.5).cpu().float()
    want = O.attention_direct(q, k, v, d ** -0.5).float()
    diff = (got - want).abs()
    assert float(diff.max()) <= 1 / 64, float(diff.max())
    assert float((got - want).pow(2).mean().sqrt() / want.pow(2).mean().sqrt()) <= 5e-3


@pytest.mark.parametrize("t,hq,hk", [(576, 32, 8), (1000, 64, 8), (129, 16, 4), (17, 8, 2), (320, 16, 8),
                                     (130, 8, 8), (1536, 32, 8), (1100, 16, 8), (2048, 32, 8)])
def test_attention_prefill_matches_per_head_kernel(gpu, t, hq, hk):
    """The grouped prefill kernel (1, 2 or a multiple of 4 query heads per kv
    head, K/V staged in LDS; one or two query tiles per wave) and the per-head
    kernel (taken when positions are given) run the same 64-key-block online
    softmax in the same order: results are bit-identical. With 2 or 1 heads
    per workgroup the waves hold different query rows and stop at different
    key blocks."""
    from fastforward_amd import ops
    d = 128
    q = torch.randn(1, hq, t, d, generator=_g(40)).to(BF16).to(DEV)
    k = torch.randn(1, hk, t, d, generator=_g(41)).to(BF16).to(DEV)
    v = (torch.randn(1, hk, t, d, generator=_g(42)) * 3).to(BF16).to(DEV)
    pos = torch.arange(t, device=DEV)
    grouped = ops.attention_direct(q, k, v, d ** -0.5)
    per_head = ops.attention_direct(q, k, v, d ** -0.5, positions=pos)
    assert torch.equal(grouped, per_head)


def test_attention_selected_positions_and_strided_v(gpu):
    from fastforward_amd import ops
    t, hq, hk, d = 576, 32, 8, 128
    packed = torch.randn(1, t, (hq + 2 * hk) * d, generator=_g(35)).to(BF16)
    q = torch.randn(1, hq, 3, d, generator=_g(36)).to(BF16)
    k = torch.randn(1, hk, t, d, generator=_g(37)).to(BF16)
    pick = torch.tensor([575, 100, 0])
    pg = packed.to(DEV)
    v = pg[..., (hq + hk) * d:].view(1, t, hk, d).transpose(1, 2)        # strided view, as the reference passes it
    got = ops.attention_direct(q.to(DEV), k.to(DEV), v, d ** -0.5, positions=pick.to(DEV)).cpu().float()
    want = O.attention_direct(q, k, packed[..., (hq + hk) * d:].view(1, t, hk, d).transpose(1, 2), d ** -0.5,
                              positions=pick).float()
    assert float((got - want).abs().max()) <= 1 / 64


@pytest.mark.parametrize("t,hq,hk", [(576, 32, 8), (2000, 16, 8)])
def test_attention_decode_follows_sequential_schedule(gpu, t, hq, hk):
    """Selected rows (<= 16 queries, the pick-only tail) run split over keys, but
    P is rounded against the running max the reference's sequential 64-key walk
    holds at each block (_legacy/limit_kernels.py:8-45): against the oracle the
    output is within relative RMS 2e-4 (a split walk whose waves keep their own
    maxima measured 2.7e-3, the size of P's bf16 rounding itself), and it equals
    the sequential per-head kernel (17 rows take that one) to 1 bf16 ulp for
    all but 0.1 % of values (only the fp32 order of the rescales differs)."""
    from fastforward_amd import ops
    d = 128
    q = torch.randn(1, hq, 17, d, generator=_g(40)).to(BF16)
    k = torch.randn(1, hk, t, d, generator=_g(41)).to(BF16)
    v = torch.randn(1, hk, t, d, generator=_g(42)).to(BF16)
    pos = torch.cat([torch.tensor([t - 1, 0, 63, 64]), torch.randint(0, t, (13,), generator=_g(43))])
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    seq = ops.attention_direct(qd, kd, vd, d ** -0.5, positions=pos.to(DEV)).cpu()            # per-head kernel
    dec = ops.attention_direct(qd[:, :, :16].contiguous(), kd, vd, d ** -0.5, positions=pos[:16].to(DEV)).cpu()
    want = O.attention_direct(q[:, :, :16], k, v, d ** -0.5, positions=pos[:16])
    rel = float((dec.float() - want.float()).norm() / want.float().norm())
    print(f"decode t={t}: rel RMS vs oracle {rel:.2e}", flush=True)
    assert rel <= 2e-4, rel
    assert_bf16_close(dec, seq[:, :16], 1, 1e-3, "decode vs sequential per-head kernel")


# ------------------------------------------------------------------ readout, gathers, rope

def test_lm_readout(gpu):
    from fastforward_amd import ops
    h = 4096
    x = (torch.randn(1, h, generator=_g(38)) * 4).to(BF16)
    mod, w = _norm_module(h, 39)
    head = (torch.randn(8, h, generator=_g(40)) * 0.02).to(BF16)
    got = ops.lm_readout(x.to(DEV), mod, head.to(DEV)).cpu()
    want = O.lm_readout(x, w, 1e-6, head)
    assert got.shape == (1, 8) and got.dtype == torch.float32
    assert_bf16_close(got.to(BF16), want.to(BF16), 1, 0.25, "lm_readout")


def test_embed_and_gather_exact(gpu):
    from fastforward_amd._lib import call, ptr, stream
    vocab, h, t = 1000, 4096, 100
    table = torch.randn(vocab, h, generator=_g(41)).to(BF16).to(DEV)
    ids = torch.randint(0, vocab, (t,), generator=_g(42))
    out = torch.empty(t, h, device=DEV, dtype=BF16)
    ids_d = ids.to(DEV)
    call("ff_embed", ptr(ids_d), ptr(table), ptr(out), t, h, vocab, stream())
    assert torch.equal(out.cpu(), table.cpu()[ids])
    idx = torch.tensor([99, 3], device=DEV)
    g = torch.empty(2, h, device=DEV, dtype=BF16)
    call("ff_gather_rows", ptr(out), h, ptr(idx), ptr(g), h, 2, h, t, stream())
    assert torch.equal(g, out[[99, 3]])


@pytest.mark.parametrize("s0,gh,gw,t", [(4, 16, 32, 576), (4, 30, 32, 1024), (4, 16, 16, 320)])
def test_mrope_cos_sin(gpu, s0, gh, gw, t):
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.runtime import mrope_positions, rope_inv_freq
    pos = torch.from_numpy(mrope_positions(s0, gh, gw, t))
    assert torch.equal(pos, O.mrope_positions(s0, gh, gw, t))
    cos = torch.empty(t, 128, device=DEV, dtype=BF16)
    sin = torch.empty(t, 128, device=DEV, dtype=BF16)
    pos_d, inv_d = pos.to(DEV), rope_inv_freq(5e6, 128).to(DEV)
    call("ff_mrope_cos_sin", ptr(pos_d), ptr(inv_d), ptr(cos), ptr(sin), t, 128, 20, 20, stream())
    wc, ws = O.mrope_cos_sin(pos, 5e6, 128)
    assert_bf16_close(cos.cpu(), wc[0], 1, 1e-2, "cos")
    assert_bf16_close(sin.cpu(), ws[0], 1, 1e-2, "sin")


def test_bad_arguments_raise(gpu):
    from fastforward_amd import ops
    from fastforward_amd._lib import call, ptr, stream
    x = torch.zeros(4, 4096, device=DEV, dtype=BF16)
    with pytest.raises(RuntimeError, match="multiple of"):
        call("ff_gemm_fp8", ptr(x), ptr(x), 1, ptr(x), ptr(x), 1, ptr(x), 4096, 4, 4096, 100, stream())
    with pytest.raises(AssertionError):
        ops.add_rms(x, x[:2], None, ops.RMSNorm(torch.ones(4096, device=DEV, dtype=BF16)))
    _ = np, bf16_ulps


@pytest.mark.parametrize("t,k,hq,hk", [(576, 4096, 32, 8), (300, 2048, 16, 8), (100, 1024, 8, 2), (1024, 5120, 64, 8)])
def test_gemm_fp8_qkv_equals_unfused(gpu, t, k, hq, hk):
    """The QKV GEMM with the norm + rotary + V^T epilogue equals ff_gemm_fp8 on the
    packed weight followed by ff_qkv_post, bit for bit (including the zero
    padding of V^T)."""
    from fastforward_amd._lib import call, ptr, stream
    d = 128
    tp = (t + 63) // 64 * 64
    n = (hq + 2 * hk) * d
    x = torch.randn(t, k, generator=_g(36)).to(BF16)
    w = (torch.randn(n, k, generator=_g(37)) * 0.03).to(BF16)
    qa, sa = O.quant_rows_dynamic(x)
    qw, sw = O.fp8_weight_quant(w)
    qa_d, sa_d, qw_d, sw_d = qa.to(DEV), sa.to(DEV), qw.to(DEV), sw.to(DEV)
    qn, _ = _norm_module(d, 38, 0.3)
    kn, _ = _norm_module(d, 39, 0.3)
    cos, sin = O.mrope_cos_sin(O.mrope_positions(4, 8, 8, t), 5e6, d)
    cos, sin = cos[0].to(DEV), sin[0].to(DEV)
    packed = torch.empty(t, n, device=DEV, dtype=BF16)
    call("ff_gemm_fp8", ptr(qa_d), ptr(sa_d), 1, ptr(qw_d), ptr(sw_d), 1, ptr(packed), n, t, n, k, stream())
    rq = torch.empty(hq, t, d, device=DEV, dtype=BF16)
    rk = torch.empty(hk, t, d, device=DEV, dtype=BF16)
    rv = torch.full((hk, d, tp), float("nan"), device=DEV, dtype=BF16)
    base = packed.data_ptr()
    call("ff_qkv_post", base, base + hq * d * 2, base + (hq + hk) * d * 2, n, ptr(qn.weight), ptr(kn.weight),
         1e-6, 1e-6, ptr(cos), ptr(sin), ptr(rq), ptr(rk), ptr(rv), t, tp, hq, hk, d, stream())
    yq = torch.full_like(rq, float("nan"))
    yk = torch.full_like(rk, float("nan"))
    vt = torch.full_like(rv, float("nan"))
    call("ff_gemm_fp8_qkv", ptr(qa_d), ptr(sa_d), 1, ptr(qw_d), ptr(sw_d), 1, t, k, hq, hk, ptr(qn.weight), ptr(kn.weight),
         1e-6, 1e-6, ptr(cos), ptr(sin), ptr(yq), ptr(yk), ptr(vt), tp, stream())
    assert torch.equal(yq, rq) and torch.equal(yk, rk)
    assert torch.equal(vt, rv)


@pytest.mark.parametrize("t,k,hq,hk,static", [(576, 4096, 32, 8, False), (500, 4096, 32, 8, False),
                                               (1024, 4096, 32, 8, False), (576, 4096, 32, 8, True),
                                               (300, 2048, 16, 8, False), (3, 4096, 32, 8, False),
                                               (176, 4096, 32, 8, False), (176, 4096, 32, 8, True),
                                               (400, 4096, 32, 8, False), (460, 4096, 32, 8, False),
                                               (640, 4096, 32, 8, False), (1200, 4096, 64, 8, False)])
def test_gemm_fp8_qkv_packed_equals_rowmajor(gpu, t, k, hq, hk, static):
    """ff_gemm_fp8_qkv_pk on the packed weight -- one-head tiles of the fewest
    rows among 64, 96 and 128 whose grid fits 256 workgroups and whose rows
    cover the V^T padding (176 and 300 tokens 64 rows; 400 tokens 96 rows; 460
    tokens 128 rows, since 96-row tiles would leave V^T columns 480..511
    unwritten; 576, 640 and ragged 500 tokens 128 rows), else 64-token x
    two-head tiles (1024 tokens at 32/8 heads) -- equals ff_gemm_fp8_qkv bit
    for bit, V^T zero padding included, per-token and per-tensor scales; shapes
    outside its plan (1200 tokens at 64/8 heads; 3 tokens) run ff_gemm_fp8_qkv
    itself."""
    from fastforward_amd._lib import call, ptr, stream
    d = 128
    tp, n = (t + 63) // 64 * 64, (hq + 2 * hk) * d
    qa = torch.randint(0, 126, (t, k), generator=_g(84), dtype=torch.uint8)
    qa[torch.rand(t, k, generator=_g(85)) < 0.5] |= 0x80
    qw = torch.randint(0, 126, (n, k), generator=_g(86), dtype=torch.uint8)
    qw[torch.rand(n, k, generator=_g(87)) < 0.5] |= 0x80
    qa_d, qw_d = qa.to(DEV), qw.to(DEV)
    packed = torch.empty_like(qw_d)
    call("ff_pack_weight_fp8", ptr(qw_d), ptr(packed), n, k, stream())
    if static:
        sa, sw = torch.tensor([0.011], device=DEV), torch.tensor([0.0007], device=DEV)
    else:
        sa = (torch.rand(t, generator=_g(88)) * 0.02 + 0.001).to(DEV)
        sw = (torch.rand(n, generator=_g(89)) * 0.001 + 1e-4).to(DEV)
    qn, _ = _norm_module(d, 90, 0.3)
    kn, _ = _norm_module(d, 91, 0.3)
    ang = torch.randn(t, d, generator=_g(92)) * 3
    cos, sin = ang.cos().to(BF16).to(DEV), ang.sin().to(BF16).to(DEV)
    outs = []
    for entry in ("ff_gemm_fp8_qkv", "ff_gemm_fp8_qkv_pk"):
        yq = torch.full((hq, t, d), float("nan"), device=DEV, dtype=BF16)
        yk = torch.full((hk, t, d), float("nan"), device=DEV, dtype=BF16)
        vt = torch.full((hk, d, tp), float("nan"), device=DEV, dtype=BF16)
        w = [ptr(qw_d)] + ([ptr(packed)] if entry.endswith("pk") else [])
        call(entry, ptr(qa_d), ptr(sa), 0 if static else 1, *w, ptr(sw), 0 if static else 1, t, k, hq, hk,
             ptr(qn.weight), ptr(kn.weight), 1e-6, 1e-6, ptr(cos), ptr(sin), ptr(yq), ptr(yk), ptr(vt), tp, stream())
        outs.append((yq, yk, vt))
    (q0, k0, v0), (q1, k1, v1) = outs
    assert not torch.isnan(q0.float()).any() and not torch.isnan(v0.float()).any()
    assert torch.equal(q1, q0) and torch.equal(k1, k0) and torch.equal(v1, v0)


# ------------------------------------------------------------------ static-scale (calibrated) producers

@pytest.mark.parametrize("deep", [False, True])
def test_norm_quant_static_equals_unfused(gpu, deep):
    """ff_add_rms_quant_static / ff_fast_norm_quant_static write the same
    residual and normalised row as ff_add_rms / ff_fast_norm and the codes
    ff_quant_static_fp8 gives on that row (the reference's quantize_runtime,
    _family/depth_fp8.py:8-19), bit for bit."""
    from fastforward_amd import ops
    from fastforward_amd._lib import call, ptr, stream
    t, h, inv = 576, 4096, 448.0 / 6.5
    a = torch.randn(1, t, h, generator=_g(70)).to(BF16).to(DEV)
    b = torch.randn(1, t, h, generator=_g(71)).to(BF16).to(DEV)
    mod, _ = _norm_module(h, 72)
    start, nv = (4, 512) if deep else (0, 0)
    dp = torch.randn(nv, h, generator=_g(73)).to(BF16).to(DEV) if deep else None
    res, out = ops.add_rms(a, b, dp, mod, start, nv)
    want = torch.empty(t, h, device=DEV, dtype=torch.uint8)
    call("ff_quant_static_fp8", ptr(out), ptr(want), t, t, h, inv, stream())
    r2 = torch.empty_like(res)
    q = torch.full((t, h), 0xAA, device=DEV, dtype=torch.uint8)
    call("ff_add_rms_quant_static", ptr(a), ptr(b), ptr(dp), ptr(mod.weight), ptr(r2), None, ptr(q), inv, t, h,
         1e-6, start, nv, stream())
    assert torch.equal(r2, res) and torch.equal(q, want)
    fn = ops.fast_norm(a, mod)
    call("ff_quant_static_fp8", ptr(fn), ptr(want), t, t, h, inv, stream())
    o2 = torch.empty_like(fn)
    call("ff_fast_norm_quant_static", ptr(a), ptr(mod.weight), ptr(o2), ptr(q), inv, t, h, 1e-6, stream())
    assert torch.equal(o2, fn) and torch.equal(q, want)


@pytest.mark.parametrize("t,hq,hk", [(576, 32, 8), (320, 16, 8), (1024, 64, 8)])
def test_attention_q_equals_unfused(gpu, t, hq, hk):
    """ff_attention_vt_q writes the codes of exactly the bf16 output
    ff_attention_vt gives (causal prefill), under the static multiplier."""
    from fastforward_amd._lib import call, ptr, stream
    d, inv = 128, 448.0 / 3.0
    tp = (t + 63) // 64 * 64
    q = torch.randn(hq, t, d, generator=_g(74)).to(BF16).to(DEV)
    k = torch.randn(hk, t, d, generator=_g(75)).to(BF16).to(DEV)
    vt = torch.zeros(hk, d, tp, dtype=BF16)
    vt[:, :, :t] = torch.randn(hk, d, t, generator=_g(76)).to(BF16)
    vt = vt.to(DEV)
    y = torch.empty(t, hq * d, device=DEV, dtype=BF16)
    call("ff_attention_vt", ptr(q), ptr(k), ptr(vt), None, 0, ptr(y), t, t, tp, hq, hk, d, d ** -0.5, stream())
    want = torch.empty(t, hq * d, device=DEV, dtype=torch.uint8)
    call("ff_quant_static_fp8", ptr(y), ptr(want), t, t, hq * d, inv, stream())
    got = torch.full((t, hq * d), 0xAA, device=DEV, dtype=torch.uint8)
    call("ff_attention_vt_q", ptr(q), ptr(k), ptr(vt), ptr(got), inv, t, t, tp, hq, hk, d, d ** -0.5, stream())
    assert torch.equal(got, want)
    with pytest.raises(RuntimeError, match="causal prefill"):
        call("ff_attention_vt_q", ptr(q), ptr(k), ptr(vt), ptr(got), inv, 1, t, tp, hq, hk, d, d ** -0.5, stream())


@pytest.mark.parametrize("m,i,k", [(576, 12288, 4096), (320, 6144, 2048), (1, 12288, 4096), (3, 640, 256),
                                   (640, 12288, 4096), (176, 12288, 4096)])
def test_gemm_swiglu_static_equals_unfused(gpu, m, i, k):
    """ff_gemm_fp8_swiglu_static (packed tile, row-major tile and GEMV by shape)
    equals ff_gemm_fp8 with per-tensor scales, then swiglu, then the static cast,
    bit for bit."""
    from fastforward_amd import ops
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import StaticFP8Linear
    op = StaticFP8Linear((torch.randn(2 * i, k, generator=_g(77)) * 0.03).to(BF16).to(DEV), 448.0 / 5.0,
                         keep_rowmajor=True)
    x = torch.randn(m, k, generator=_g(78)).to(BF16).to(DEV)
    qa = torch.empty(m, k, device=DEV, dtype=torch.uint8)
    call("ff_quant_static_fp8", ptr(x), ptr(qa), m, m, k, float(op.inverse_scale), stream())
    gu = torch.empty(m, 2 * i, device=DEV, dtype=BF16)
    call("ff_gemm_fp8", ptr(qa), ptr(op.input_scale), 0, ptr(op.weight), ptr(op.weight_scale), 0, ptr(gu), 2 * i, m,
         2 * i, k, stream())
    hh = ops.swiglu(*gu.chunk(2, -1)).contiguous()
    inv = 448.0 / 0.75
    want = torch.empty(m, i, device=DEV, dtype=torch.uint8)
    call("ff_quant_static_fp8", ptr(hh), ptr(want), m, m, i, inv, stream())
    got = torch.full((m, i), 0xAA, device=DEV, dtype=torch.uint8)
    call("ff_gemm_fp8_swiglu_static", ptr(qa), ptr(op.input_scale), ptr(op.weight), ptr(op.packed),
         ptr(op.weight_scale), ptr(got), i, inv, m, i, k, stream())
    assert torch.equal(got, want)


def test_gemm_qkv_static_scales_equal_unfused(gpu):
    """ff_gemm_fp8_qkv with per-tensor scales (sa_rows = sw_cols = 0) equals
    ff_gemm_fp8 with the same scalars followed by ff_qkv_post, bit for bit."""
    from fastforward_amd._lib import call, ptr, stream
    t, k, hq, hk, d = 576, 4096, 32, 8, 128
    tp, n = (t + 63) // 64 * 64, (hq + 2 * hk) * d
    qa = torch.randint(0, 126, (t, k), generator=_g(79), dtype=torch.uint8)
    qa[torch.rand(t, k, generator=_g(80)) < 0.5] |= 0x80
    qw = torch.randint(0, 126, (n, k), generator=_g(81), dtype=torch.uint8)
    qa_d, qw_d = qa.to(DEV), qw.to(DEV)
    sa, sw = torch.tensor([0.011], device=DEV), torch.tensor([0.0007], device=DEV)
    qn, _ = _norm_module(d, 82, 0.3)
    kn, _ = _norm_module(d, 83, 0.3)
    cos, sin = O.mrope_cos_sin(O.mrope_positions(4, 16, 32, t), 5e6, d)
    cos, sin = cos[0].to(DEV), sin[0].to(DEV)
    raw = torch.empty(t, n, device=DEV, dtype=BF16)
    call("ff_gemm_fp8", ptr(qa_d), ptr(sa), 0, ptr(qw_d), ptr(sw), 0, ptr(raw), n, t, n, k, stream())
    rq, rk = torch.empty(hq, t, d, device=DEV, dtype=BF16), torch.empty(hk, t, d, device=DEV, dtype=BF16)
    rv = torch.empty(hk, d, tp, device=DEV, dtype=BF16)
    base = raw.data_ptr()
    call("ff_qkv_post", base, base + hq * d * 2, base + (hq + hk) * d * 2, n, ptr(qn.weight), ptr(kn.weight), 1e-6,
         1e-6, ptr(cos), ptr(sin), ptr(rq), ptr(rk), ptr(rv), t, tp, hq, hk, d, stream())
    yq, yk, vt = torch.empty_like(rq), torch.empty_like(rk), torch.empty_like(rv)
    call("ff_gemm_fp8_qkv", ptr(qa_d), ptr(sa), 0, ptr(qw_d), ptr(sw), 0, t, k, hq, hk, ptr(qn.weight),
         ptr(kn.weight), 1e-6, 1e-6, ptr(cos), ptr(sin), ptr(yq), ptr(yk), ptr(vt), tp, stream())
    assert torch.equal(yq, rq) and torch.equal(yk, rk) and torch.equal(vt, rv)


# ------------------------------------------------------------------ one weight copy

@pytest.mark.parametrize("m,k,n", [(1, 4096, 4096), (3, 12288, 4096), (4, 4096, 6144), (5, 4096, 4096),
                                   (17, 4096, 6144), (176, 4096, 4096), (576, 12288, 4096)])
def test_fp8linear_keeps_one_copy(gpu, m, k, n):
    """FP8Linear keeps only the MFMA-fragment copy of its codes: ``weight`` is a
    stand-in with a NULL data pointer whose unpacked codes (ff_unpack_weight_fp8)
    equal the oracle's quantisation bit for bit, and op(x) runs on the packed
    copy alone: bit-identical to the op that also keeps the row-major codes for
    m > 4 (the same packed tiles), and within the exact-product bound for the
    single-row kernel (m <= 4; its fp32 sums are in another order than the
    row-major GEMV's)."""
    from fastforward_amd.linear import FP8Linear, PackedCodes
    x = torch.randn(m, k, generator=_g(90))
    x[torch.rand(m, k, generator=_g(91)) < 0.001] *= 20
    x = x.to(BF16)
    w = (torch.randn(n, k, generator=_g(92)) * 0.02).to(BF16)
    one = FP8Linear(w.to(DEV))
    two = FP8Linear(w.to(DEV), keep_rowmajor=True)
    assert isinstance(one.weight, PackedCodes) and one.weight.data_ptr() == 0 and tuple(one.weight.shape) == (n, k)
    qw, sw = O.fp8_weight_quant(w)
    assert torch.equal(one.weight.cpu().view(torch.uint8), qw.view(torch.uint8))
    xd = x.to(DEV)
    y1, y2 = one(xd), two(xd)
    if m > 4:
        assert torch.equal(y1, y2)
    qa, sa = O.quant_rows_dynamic(x)
    _assert_fp8_gemm(y1.cpu(), qa, sa, qw, sw, O.fp8_gemm(qa, sa, qw, sw), f"one-copy FP8Linear {m}x{k}x{n}")


# the smallest k and n of the packed layout, ragged numbers of k steps per wave, the
# limits of the codes' LDS (49152 bytes) and past it
@pytest.mark.parametrize("m,k,n", [(1, 512, 128), (4, 512, 128), (2, 2560, 256), (3, 9728, 128), (4, 12288, 256),
                                   (1, 25600, 128), (2, 25600, 128), (1, 49152, 128)])
@pytest.mark.parametrize("static", [False, True])
def test_linear_rows_equals_quantise_and_gemm(gpu, m, k, n, static):
    """A linear of at most four rows quantises inside the product's launch
    (ff_linear_fp8_rows, up to 49152 codes): bit for bit the quantiser and the GEMM
    as two calls, for rows of ordinary values, zeros, one infinity and one NaN, and
    for a strided view."""
    from fastforward_amd.linear import FP8Linear, StaticFP8Linear, _packed_gemm, rows_fit
    w = (torch.randn(n, k, generator=_g(190)) * 0.02).to(BF16).to(DEV)
    op = StaticFP8Linear(w, 56.0) if static else FP8Linear(w)
    assert rows_fit(op, m) == (m * k <= 49152)
    wide = torch.randn(m, k + 8, generator=_g(191)).to(BF16)
    special = wide.clone()
    special[0] = 0
    special[-1, 3] = float("inf")
    if m > 1:
        special[1, 5] = float("nan")
    for x in (wide[:, :k], wide[:, :k].contiguous(), special[:, :k].contiguous()):
        x = x.to(DEV) if x.is_contiguous() else wide.to(DEV)[:, :k]
        got = op(x)
        ref = torch.empty(m, n, device=DEV, dtype=BF16)
        if static:
            q = torch.empty(m, k, device=DEV, dtype=torch.float8_e4m3fn)
            from fastforward_amd._lib import call, ptr, stream
            xc = x.contiguous()
            call("ff_quant_static_fp8", ptr(xc), ptr(q), m, m, k, float(op.inverse_scale), stream())
            _packed_gemm(op, q, op.input_scale, 0, op.weight_scale, 0, ref)
        else:
            op.gemm(*op.quantize(x), out=ref)
        assert got.shape == (m, n)
        assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("m,i,k", [(1, 12288, 4096), (3, 6144, 2048), (4, 640, 512), (20, 6144, 2048)])
def test_swiglu_single_copy_rows(gpu, m, i, k):
    """The gate/up + SwiGLU launch on the packed copy alone (qw NULL): for m <= 4
    the single-row kernel adds g and u in the order of the plain single-row
    kernel, so h equals the oracle's swiglu of ff_gemm_fp8_pk's g and u on the
    same codes (<= 1 ulp from the SiLU rounding) with its row maxima, and the
    static form writes the runtime-scale cast of that h; m > 4 takes a packed
    tile whatever its grid (20 rows: fewer than 192 workgroups) and equals the
    launch that keeps the row-major weight."""
    from fastforward_amd import ops
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import FP8Linear, StaticFP8Linear
    w = (torch.randn(2 * i, k, generator=_g(93)) * 0.04).to(BF16).to(DEV)
    op = FP8Linear(w)
    x = torch.randn(m, k, generator=_g(94)).to(BF16).to(DEV)
    qa, sa = op.quantize(x)
    h = torch.full((m, i), float("nan"), device=DEV, dtype=BF16)
    pmax = torch.full((m, i // 64), float("nan"), device=DEV)
    call("ff_gemm_fp8_swiglu_pk", ptr(qa), ptr(sa), None, ptr(op.packed), ptr(op.scale), ptr(h), i, ptr(pmax), m, i,
         k, stream())
    if m > 4:
        two = FP8Linear(w, keep_rowmajor=True)
        h2 = torch.full((m, i), float("nan"), device=DEV, dtype=BF16)
        p2 = torch.full((m, i // 64), float("nan"), device=DEV)
        call("ff_gemm_fp8_swiglu_pk", ptr(qa), ptr(sa), ptr(two.weight), ptr(two.packed), ptr(two.scale), ptr(h2), i,
             ptr(p2), m, i, k, stream())
        assert torch.equal(h, h2) and torch.equal(pmax, p2)
        return
    raw = op.gemm(qa, sa)
    want = ops.swiglu(*raw.chunk(2, -1))
    assert_bf16_close(h.cpu(), want.cpu(), 1, 1e-3, "single-row swiglu vs swiglu(plain single-row product)")
    assert torch.equal(pmax.cpu(), h.cpu().float().abs().view(m, i // 64, 64).amax(-1))
    # the static form: per-tensor scales, h written as its runtime-scale cast
    st = StaticFP8Linear(w, 448.0 / 4.0)
    qs = torch.empty(m, k, device=DEV, dtype=torch.uint8)
    call("ff_quant_static_fp8", ptr(x), ptr(qs), m, m, k, float(st.inverse_scale), stream())
    inv = 448.0 / 0.5
    got = torch.full((m, i), 0xAA, device=DEV, dtype=torch.uint8)
    call("ff_gemm_fp8_swiglu_static", ptr(qs), ptr(st.input_scale), None, ptr(st.packed), ptr(st.weight_scale),
         ptr(got), i, inv, m, i, k, stream())
    raw_s = torch.empty(m, 2 * i, device=DEV, dtype=BF16)
    call("ff_gemm_fp8_pk", ptr(qs), ptr(st.input_scale), 0, None, ptr(st.packed), ptr(st.weight_scale), 0,
         ptr(raw_s), 2 * i, m, 2 * i, k, None, 0, stream())
    hs = ops.swiglu(*raw_s.chunk(2, -1)).contiguous()
    want_q = torch.empty(m, i, device=DEV, dtype=torch.uint8)
    call("ff_quant_static_fp8", ptr(hs), ptr(want_q), m, m, i, inv, stream())
    d = (got.cpu().view(torch.float8_e4m3fn).float() - want_q.cpu().view(torch.float8_e4m3fn).float()).abs()
    # codes of h values one bf16 ulp apart (the SiLU rounding) can differ by one e4m3 step
    assert float((d > 0).float().mean()) <= 2e-3


@pytest.mark.parametrize("t", [3, 33])
def test_qkv_single_copy_short(gpu, t):
    """The QKV launch on the packed copy alone (qw NULL) for prompts the packed
    tile's plan would leave to the row-major kernel (3 and 33 tokens) runs the
    packed tile and equals ff_gemm_fp8_qkv on the row-major codes bit for bit."""
    from fastforward_amd._lib import call, ptr, stream
    from fastforward_amd.linear import FP8Linear
    d, hq, hk, k = 128, 32, 8, 4096
    tp, n = (t + 63) // 64 * 64, (hq + 2 * hk) * d
    op = FP8Linear((torch.randn(n, k, generator=_g(95)) * 0.02).to(BF16).to(DEV), keep_rowmajor=True)
    x = torch.randn(t, k, generator=_g(96)).to(BF16).to(DEV)
    qa, sa = op.quantize(x)
    qn = (1 + 0.2 * torch.randn(d, generator=_g(97))).to(BF16).to(DEV)
    kn = (1 + 0.2 * torch.randn(d, generator=_g(98))).to(BF16).to(DEV)
    cos = torch.randn(t, d, generator=_g(99)).to(BF16).to(DEV)
    sin = torch.randn(t, d, generator=_g(100)).to(BF16).to(DEV)
    outs = []
    for qw in (ptr(op.weight), None):
        yq = torch.full((hq, t, d), float("nan"), device=DEV, dtype=BF16)
        yk = torch.full((hk, t, d), float("nan"), device=DEV, dtype=BF16)
        vt = torch.full((hk, d, tp), float("nan"), device=DEV, dtype=BF16)
        if qw is None:
            call("ff_gemm_fp8_qkv_pk", ptr(qa), ptr(sa), 1, None, ptr(op.packed), ptr(op.scale), 1, t, k, hq, hk,
                 ptr(qn), ptr(kn), 1e-6, 1e-6, ptr(cos), ptr(sin), ptr(yq), ptr(yk), ptr(vt), tp, stream())
        else:
            call("ff_gemm_fp8_qkv", ptr(qa), ptr(sa), 1, qw, ptr(op.scale), 1, t, k, hq, hk, ptr(qn), ptr(kn), 1e-6,
                 1e-6, ptr(cos), ptr(sin), ptr(yq), ptr(yk), ptr(vt), tp, stream())
        outs.append((yq, yk, vt))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
