"""CPU checks of the C ABI: the library loads without a GPU, exports every
function include/ff_amd.h declares, and the ctypes binding agrees with the
header on names and parameter counts. No compute call is made."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "ff_amd.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    decls = {}
    for m in re.finditer(r"(?:int64_t|int|const char\*)\s+(ff_\w+)\s*\(([^)]*)\)\s*;", text):
        params = m.group(2).strip()
        n = 0 if params in ("", "void") else len(params.split(","))
        decls[m.group(1)] = n
    return decls


@pytest.fixture(scope="module")
def lib_path():
    from fastforward_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        from fastforward_amd import build
        build.build(verbose=False)
    return _lib.LIB_PATH


def test_header_declares_entry_points():
    d = _declared()
    assert len(d) >= 24
    for name in ("ff_gemm_fp8", "ff_gemm_w4a16", "ff_attention_vt", "ff_add_rms", "ff_qk_pair",
                 "ff_swiglu", "ff_fast_norm", "ff_lm_readout"):
        assert name in d


def test_library_exports_every_declared_symbol(lib_path):
    lib = ctypes.CDLL(lib_path)
    for name in _declared():
        assert hasattr(lib, name), name


def test_binding_matches_header(lib_path):
    from fastforward_amd import _lib
    d = _declared()
    assert set(d) == set(_lib.SIGNATURES)
    for name, n in d.items():
        assert len(_lib.SIGNATURES[name]) == n, name
    lib = _lib.load()
    assert lib.ff_version() >= 100
    assert lib.ff_last_error() == b""


def test_tuning_knobs_validate_without_a_gpu(lib_path):
    """ff_set_tuning checks knob and value ranges on the host and never reads the
    environment; 0 restores the built-in choice."""
    from fastforward_amd import _lib
    _lib.load()
    _lib.call("ff_set_tuning", 3, 2)
    _lib.call("ff_set_tuning", 3, 0)
    with pytest.raises(RuntimeError, match="unknown knob"):
        _lib.call("ff_set_tuning", 99, 1)
    with pytest.raises(RuntimeError, match="out of range"):
        _lib.call("ff_set_tuning", 4, 9)
    for tile in (1, 2, 3, 12, 22, 23, 24, 25, 34, 44, 36, 56, 66, 0):   # ff_gemm_bf16's tiles
        _lib.call("ff_set_tuning", 2, tile)
    for tile in (4, 11, 13, 33, 55, 65, 67):
        with pytest.raises(RuntimeError, match="out of range"):
            _lib.call("ff_set_tuning", 2, tile)
    text = "".join(open(os.path.join(ROOT, "fastforward_amd", "csrc", f)).read()
                   for f in os.listdir(os.path.join(ROOT, "fastforward_amd", "csrc")))
    assert "getenv" not in text


def test_linear_fp8_rows_takes_what_the_two_calls_take(lib_path):
    """Sizes are checked on the host before anything is launched: weights of 2^31 codes
    and more are refused, as ff_gemm_fp8_pk refuses them without the row-major copy."""
    from fastforward_amd import _lib
    _lib.load()
    buf = (ctypes.c_char * 4096)()
    p = (ctypes.addressof(buf) + 15) // 16 * 16
    for m, n, k in ((1, 151936, 16384), (1, 1 << 22, 512), (5, 128, 512), (1, 128, 384), (4, 128, 12288 + 128),
                    (1, 120, 512), (1, 128, 520)):
        with pytest.raises(RuntimeError, match="ff_linear_fp8_rows: bad sizes"):
            _lib.call("ff_linear_fp8_rows", p, k, None, 0.0, p, p, 1, p, n, m, n, k, None)
    with pytest.raises(RuntimeError, match="ff_gemm_fp8_pk"):
        _lib.call("ff_gemm_fp8_pk", p, p, 1, None, p, p, 1, p, 151936, 1, 151936, 16384, None, 0, None)


def test_w4a16_swiglu_shape_query_without_a_gpu(lib_path):
    """ff_gemm_w4a16_swiglu_fits answers on the host: m > 4 with i % 128 and k % 256,
    or m <= 4 with i % 16 and k % 128; a power-of-two group >= 32 dividing k."""
    import ctypes
    from fastforward_amd import _lib
    _lib.load()

    def fits(m, i, k, group):
        ok = ctypes.c_int(-1)
        _lib.call("ff_gemm_w4a16_swiglu_fits", m, i, k, group, ctypes.byref(ok))
        return ok.value

    assert fits(576, 12288, 4096, 128) == 1 and fits(320, 6144, 2048, 32) == 1 and fits(100, 640, 1024, 64) == 1
    assert fits(4, 12288, 4096, 128) == 1 and fits(1, 16, 128, 32) == 1  # the tail's rows: the packed GEMV
    assert fits(1, 8, 128, 32) == 0                # the GEMV takes 16-row blocks
    assert fits(576, 12288 + 64, 4096, 128) == 0   # i % 128
    assert fits(576, 12288, 4096 + 128, 128) == 0  # k % 256
    assert fits(576, 12288, 4096, 96) == 0         # group not a power of two


# (m, n, k, row tile, splits) the packed FP8 plain GEMM takes: the 8B down
# projection at the bucket sizes that pick 5 (64-row tiles, short m), 4, 3 and 2
# splits (k = 12288), the 176-token o projection on 64-row tiles split 5 ways
# (short m: 6 or 5 splits with uneven k ranges where 8, 4 or 2 do not fit: the
# 2B down at 250 tokens 6, the 4B o at 176 tokens 5; the 2B o at 176 tokens, 16
# k steps, keeps 4),
# splits of unequal length where k is not a multiple of 4 x splits x 128 (the
# 4B and 32B down projections, k = 9728 and 25600),
# unsplit grids and shapes left to the small tiles or the row-major kernels (0):
# at k = 8192 a split only where no small tile fills the GPU (the 32B o
# projection at 1024 and 576 tokens runs unsplit on small tiles).
# The plan is host code, so the workspace query pins it without a GPU.
PLAN_SHAPES = [(176, 4096, 12288, 64, 5), (576, 4096, 12288, 144, 4), (640, 4096, 12288, 144, 3),
               (1152, 4096, 12288, 144, 2), (300, 2048, 8192, 144, 8), (1000, 6144, 8192, 0, 0),
               (1024, 5120, 8192, 0, 0), (576, 5120, 8192, 0, 0),
               (576, 12288, 4096, 144, 1), (576, 4096, 4096, 0, 0), (176, 4096, 4096, 64, 5), (64, 2048, 2048, 64, 4),
               (250, 2048, 6144, 64, 6), (176, 2560, 2560, 64, 5), (176, 2048, 2048, 64, 4),
               (300, 4096, 2048, 0, 0), (3, 4096, 4096, 0, 0), (1024, 5120, 25600, 144, 3),
               (576, 2560, 9728, 144, 4), (576, 5120, 25600, 144, 3)]


@pytest.mark.parametrize("m,n,k,bm,splits", PLAN_SHAPES)
def test_fp8_pk_split_plan(lib_path, m, n, k, bm, splits):
    from fastforward_amd.linear import gemm_pk_workspace
    need = gemm_pk_workspace(m, n, k)
    assert need == ((m + bm - 1) // bm * (n // 256) * splits * bm * 256 * 4 if splits > 1 else 0)


def test_rows_in_one_launch_where_they_gain():
    """``rows_fit``: one row always, two to four per-token rows up to 32768 columns among
    them, static-scale rows whatever the columns; never past the kernel's LDS nor where
    the row-major codes are kept."""
    import torch
    from fastforward_amd.linear import FP8Linear, PackedCodes, StaticFP8Linear, rows_fit

    def op(cls, n, k, packed=True):
        o = object.__new__(cls)
        o.weight = PackedCodes(torch.empty(0), (n, k)) if packed else torch.empty((n, k), device="meta")
        return o
    for m, n, k, dynamic, static in ((1, 51200, 5120, True, True), (4, 8192, 4096, True, True),
                                     (4, 8208, 4096, False, True), (2, 19456, 2560, False, True),
                                     (2, 12288, 4096, True, True), (2, 5120, 25600, False, False),
                                     (5, 128, 512, False, False), (0, 128, 512, False, False)):
        assert rows_fit(op(FP8Linear, n, k), m) is dynamic, (m, n, k)
        assert rows_fit(op(StaticFP8Linear, n, k), m) is static, (m, n, k)
        assert not rows_fit(op(FP8Linear, n, k, False), m)


# (m, n, k, row tile, splits): 144 rows where a lower tile would take another round or more
# k steps (130 x 5120 x 25600, 400 x 4096 x 12288), 96 where it does not and where a second
# row tile only fills the GPU (100 and 130 x 4096 x 2048), unsplit grids (0)
@pytest.mark.parametrize("m,n,k,bm,splits", [(130, 5120, 25600, 144, 8), (400, 4096, 12288, 144, 5),
                                             (500, 4096, 4096, 128, 4), (100, 4096, 2048, 96, 8),
                                             (130, 4096, 2048, 96, 8), (700, 4096, 2048, 96, 2),
                                             (576, 4096, 12288, 144, 4), (1024, 10240, 5120, 96, 0)])
def test_w4a16_pk_plan(lib_path, m, n, k, bm, splits):
    """Row tile and k splits of the packed W4A16 product, from the workspace it asks for."""
    from fastforward_amd import _lib
    _lib.load()
    need = ctypes.c_int64(-1)
    _lib.call("ff_gemm_w4a16_pk_workspace", m, n, k, 128, ctypes.byref(need))
    assert need.value == -(-m // bm) * bm * n * splits * 4
