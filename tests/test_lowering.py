"""Lowering of user mask / score callables (CPU): the traced expression
evaluates like the callable itself, Python's integer semantics survive,
derivatives with respect to the score match finite differences, untraceable
callables are refused with a reason, and the generated policy compiles for
gfx950 through the C ABI (fa_mods_compile needs no GPU)."""
import re
import shutil
import subprocess

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import pallas_flexattn as pf  # noqa: E402
from pallas_flexattn import lowering as L  # noqa: E402

Q = np.arange(-5, 40)[:, None]
K = np.arange(0, 37)[None, :]

MASKS = {
    "prefix_lm": lambda q, kv: (kv < 8) | (q >= kv),
    "parity": lambda q, kv: (q - kv) % 2 == 0,
    "floordiv_blocks": lambda q, kv: (q // 16) == (kv // 16),
    "where_window": lambda q, kv: torch.where(q > 20, (q - kv) < 4, kv <= q),
    "not_and": lambda q, kv: ~(kv > q) & (torch.abs(q - kv) <= 9),
    "numpy_ops": lambda q, kv: np.logical_and(q >= kv, np.remainder(q + kv, 3) != 1),
}


@pytest.mark.parametrize("name", list(MASKS))
def test_traced_mask_evaluates_like_the_callable(name):
    fn = MASKS[name]
    low = L.lower_mask(fn)
    want = fn(torch.from_numpy(Q), torch.from_numpy(K)) if name != "numpy_ops" else fn(Q, K)
    want = np.broadcast_to(np.asarray(want), (Q.shape[0], K.shape[1]))
    np.testing.assert_array_equal(low(Q, K), want)


def test_integer_semantics_follow_python():
    # floor division and modulo take the divisor's sign, as in Python / torch
    low = L.lower_mask(lambda q, kv: ((q - kv) // 7 == -2) | ((q - kv) % -5 == -3))
    d = Q - K
    np.testing.assert_array_equal(low(Q, K), ((d // 7) == -2) | ((d % -5) == -3))
    src = L.policy_source(low.expr, None)
    assert "um_ifloordiv" in src and "um_imod" in src
    # the smallest int32 stays an int literal in C++ (a bare -2147483648 is
    # the negation of a long)
    assert L.emit(L.const(-2 ** 31)) == "(-2147483647 - 1)"
    low = L.lower_mask(lambda q, kv: (q - kv) > -2 ** 31)
    np.testing.assert_array_equal(low(Q, K), np.broadcast_to(True, (Q.shape[0], K.shape[1])))


def test_captured_tensor_reads_and_batch_head_dependence():
    allowed = torch.rand(2, 3, 45, 37) > 0.5
    low = L.lower_mask(lambda b, h, q, kv: allowed[b, h, q, kv] | (q == kv))
    assert low.batch_dependent and low.head_dependent and len(low.tensors) == 1
    for b in range(2):
        for h in range(3):
            got = low(b, h, np.arange(45)[:, None], np.arange(37)[None, :])
            want = allowed[b, h].numpy() | (np.arange(45)[:, None] == np.arange(37)[None, :])
            np.testing.assert_array_equal(got, want)
    # reads are clamped into the tensor (no out-of-bounds access)
    np.testing.assert_array_equal(low(0, 0, np.array([[100]]), np.array([[-3]])),
                                  allowed[0, 0, 44, 0].numpy() | False)


SCORES = {
    "softcap": (lambda s, b, h, q, kv: 20.0 * torch.tanh(s / 20.0)),
    "alibi_like": (lambda s, b, h, q, kv: s - 0.25 * (h + 1) * torch.abs(q - kv)),
    "quadratic_exp": (lambda s, b, h, q, kv: 0.1 * s * s + torch.exp(s / 8.0) + (q % 3)),
    "clamp_where": (lambda s, b, h, q, kv: torch.where(s > 2.0, 2.0 + 0.5 * (s - 2.0), torch.clamp(s, min=-3.0))),
    "sigmoid_log": (lambda s, b, h, q, kv: torch.log(torch.sigmoid(s) + 1.0) + torch.sqrt(s * s + 1.0)),
    # quotients: the divisor depends on the score, on the position only, or is a constant
    "softsign": (lambda s, b, h, q, kv: s / (1.0 + torch.abs(s))),
    "rational": (lambda s, b, h, q, kv: 3.0 * s / (1.0 + s * s)),
    "logistic": (lambda s, b, h, q, kv: 1.0 / (1.0 + torch.exp(-s))),
    "algebraic": (lambda s, b, h, q, kv: s / torch.sqrt(1.0 + s * s)),
    "reciprocal": (lambda s, b, h, q, kv: 5.0 / (20.0 + s)),
    "by_position": (lambda s, b, h, q, kv: s / (1 + torch.abs(q - kv))),
    "by_constant": (lambda s, b, h, q, kv: (s * s + s) / 3.7),
}


@pytest.mark.parametrize("name", list(SCORES))
def test_score_derivative_matches_finite_differences(name):
    fn = SCORES[name]
    low = L.lower_score(fn)
    rng = np.random.default_rng(1)
    s = rng.standard_normal((45, 37)).astype(np.float64) * 4
    h = 2
    val = low(s.astype(np.float32), 0, h, Q, K)
    want = fn(torch.from_numpy(s), 0, h, torch.from_numpy(Q), torch.from_numpy(K)).numpy()
    np.testing.assert_allclose(val, want, rtol=2e-5, atol=2e-5)
    eps = 1e-3
    fd = (fn(torch.from_numpy(s + eps), 0, h, torch.from_numpy(Q), torch.from_numpy(K)).numpy()
          - fn(torch.from_numpy(s - eps), 0, h, torch.from_numpy(Q), torch.from_numpy(K)).numpy()) / (2 * eps)
    g = low.grad(s.astype(np.float32), 0, h, Q, K)
    near_kink = np.abs(s - 2.0) < 2 * eps if name == "clamp_where" else np.zeros_like(s, bool)
    near_kink |= np.abs(s + 3.0) < 2 * eps if name == "clamp_where" else False
    np.testing.assert_allclose(np.where(near_kink, fd, g), fd, rtol=1e-3, atol=1e-3)


def test_descriptors_trace_to_their_own_predicates():
    """MaskSpec / ScoreSpec inside a traced callable lower to the same values."""
    dm = pf.document_mask([[10, 20, 15], [30, 15]])
    both = L.lower_mask(lambda b, h, q, kv: dm(b, h, q, kv) & pf.causal_mask(q, kv) &
                        pf.sliding_window_mask(12, -1)(q, kv))
    q, k = np.arange(45)[:, None], np.arange(45)[None, :]
    for b in range(2):
        want = dm(b, 0, q, k) & (q >= k) & (q - k <= 12)
        np.testing.assert_array_equal(both(b, 0, q, k), want)
    sc = pf.compose_score_mods(pf.alibi_score_mod(4), pf.softcap_score_mod(30.0))
    low = L.lower_score(lambda s, b, h, qi, ki: sc(s, b, h, qi, ki))
    s = np.random.default_rng(2).standard_normal((45, 45)).astype(np.float32) * 20
    for h in range(4):
        np.testing.assert_allclose(low(s, 0, h, q, k), sc(s, 0, h, q, k), rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("fn,why", [
    (lambda q, kv: q >= kv if q > 3 else q < kv, "control flow"),
    (lambda q, kv: [1, 2, 3][q] > 0, "concrete integer"),
    (lambda q, kv: np.arange(10)[q] > kv, "tracing the callable raised IndexError"),
    (lambda q, kv: torch.erf(q) > 0, "cannot be lowered"),
])
def test_untraceable_callables_are_refused(fn, why):
    with pytest.raises(L.LoweringError, match=why):
        L.lower_mask(fn)


def test_policy_compiles_for_gfx950_without_a_gpu():
    from pallas_flexattn import _lib
    bias = torch.randn(4, 8)
    mods = L.UserMods(L.lower_mask(MASKS["prefix_lm"]),
                      L.lower_score(lambda s, b, h, q, kv: 30.0 * torch.tanh((s + bias[h, kv % 8]) / 30.0)))
    assert len(mods.tensors) == 1 and mods.flags(False) == 3
    for dtype in (_lib.DTYPE_BF16, _lib.DTYPE_F32):
        blob = _lib.compile_mods(mods.source, dtype, 128, mods.flags(False))
        assert len(blob) > 1000
    with pytest.raises(_lib.FlexAttnError, match="compiling the user mods failed"):
        _lib.compile_mods("struct UserMod { this is not C++ };", _lib.DTYPE_BF16, 64, 1)


def test_policy_must_match_its_flags():
    """fa_mods_compile refuses a policy whose kMask / kScore disagree with the
    flags it is compiled under (the launches set up the mask walk and the
    score epilogue from the flags), and a user score together with the
    built-in ALiBi / soft-cap (which only run without a user score)."""
    from pallas_flexattn import _lib
    mods = L.UserMods(L.lower_mask(MASKS["parity"]), None)
    assert mods.flags(False) == _lib.MODS_MASK
    with pytest.raises(_lib.FlexAttnError, match="kMask disagrees"):
        _lib.compile_mods(mods.source, _lib.DTYPE_BF16, 64, 0)
    with pytest.raises(_lib.FlexAttnError, match="kScore disagrees"):
        _lib.compile_mods(mods.source, _lib.DTYPE_BF16, 64, _lib.MODS_MASK | _lib.MODS_SCORE)
    smods = L.UserMods(None, L.lower_score(lambda s, b, h, q, kv: s * 0.5))
    with pytest.raises(_lib.FlexAttnError, match="exit 3"):
        _lib.compile_mods(smods.source, _lib.DTYPE_BF16, 64, _lib.MODS_SCORE | _lib.MODS_BUILTIN_SCORE)


def test_blob_from_other_kernel_headers_is_refused():
    """A code blob records the ABI version, the hash of the kernel headers it
    was compiled from and the kernel argument sizes; fa_mods_load refuses a
    blob that differs in any of them (FA_ERR_VERSION) before any GPU call,
    so a stale cached or stored blob is never launched with another argument
    layout.  Header layout: magic u32, abi_version u32, header hash u64,
    sizeof(FwdArgs) u32, sizeof(BwdArgs) u32."""
    import ctypes
    from pallas_flexattn import _lib
    lib = _lib.load()
    mods = L.UserMods(L.lower_mask(MASKS["parity"]), None)
    blob = _lib.compile_mods(mods.source, _lib.DTYPE_BF16, 64, mods.flags(False))
    assert int.from_bytes(blob[4:8], "little") == _lib.ABI_VERSION
    assert int.from_bytes(blob[8:16], "little") == lib.fa_mods_source_hash()
    fwd_bytes, bwd_bytes = int.from_bytes(blob[16:20], "little"), int.from_bytes(blob[20:24], "little")
    assert 0 < fwd_bytes < 4096 and bwd_bytes > fwd_bytes - 512

    def load(b):
        h = ctypes.c_void_p()
        return lib.fa_mods_load(bytes(b), len(b), ctypes.byref(h))

    FA_ERR_SHAPE, FA_ERR_VERSION = -2, -8
    for lo, hi, delta in ((4, 8, 1), (8, 16, 1), (16, 20, 8), (20, 24, 8)):
        bad = bytearray(blob)
        bad[lo:hi] = ((int.from_bytes(blob[lo:hi], "little") + delta) % (1 << (8 * (hi - lo)))).to_bytes(
            hi - lo, "little")
        assert load(bad) == FA_ERR_VERSION, (lo, hi)
    bad = bytearray(blob)
    bad[0] ^= 1  # not a blob
    assert load(bad) == FA_ERR_SHAPE
    assert load(blob[:-1]) == FA_ERR_SHAPE  # truncated code object
    assert load(blob[:20]) == FA_ERR_SHAPE  # shorter than the header


def test_shared_functions_and_constant_factors_are_emitted_once():
    """A soft-cap's tanh serves the score and its derivative, whose constant factors cancel."""
    low = L.lower_score(lambda s, b, h, q, kv: 30.0 * torch.tanh(s / 30.0))
    src = L.policy_source(None, low.expr)
    body = src[src.index("struct UserMod"):]
    assert body.count("um_tanh(") == 1 and " / " not in body
    assert "*dsds = ((1.0f) - (t1 * t1));" in body
    # a divisor without a reciprocal in the normal range keeps its division
    assert "/ (0.0f)" in L.policy_source(None, L.lower_score(lambda s, b, h, q, kv: s / 0.0).expr)


@pytest.mark.parametrize("name,fn", [
    ("tiny_divisor", lambda s, b, h, q, kv: s / 1e-50),
    ("huge_divisor", lambda s, b, h, q, kv: s / 1e300),
    ("nested", lambda s, b, h, q, kv: torch.tanh(torch.tanh(s * 1e-30) * 1e-30) * 1e20 * 1e20 * 1e20),
    ("growing", lambda s, b, h, q, kv: torch.tanh(torch.tanh(s * 1e30) * 1e30) * 1e-20),
    ("subnormal", lambda s, b, h, q, kv: torch.sin(torch.sin(s * 1e-20) * 1e-20) + s),
    ("divisors", lambda s, b, h, q, kv: torch.tanh(s / 1e30) / 1e-30 / 1e-30)])
def test_folded_constants_stay_in_float32(name, fn):
    """Constant factors of a derivative are folded only where their product is a normal float32: the emitted
    code holds no literal that the program did not write and that is 0, subnormal or infinite in float32."""
    expr = L.lower_score(fn).expr
    src = L.policy_source(None, expr)
    body = src[src.index("struct UserMod"):]
    written = {float(x) for x in re.findall(r"(?<![\w.])(\d+\.?\d*(?:e[-+]?\d+)?)f", L.emit(expr))}
    for text in re.findall(r"(?<![\w.])(\d+\.?\d*(?:e[-+]?\d+)?)f", body):
        v = float(text)
        with np.errstate(over="ignore", under="ignore"):
            f = np.float32(v)
        assert v == 0 or v in written or (np.isfinite(f) and abs(f) >= np.finfo(np.float32).tiny), (text, body)


def test_derivative_of_integer_factors_is_a_float_product():
    for fn in (lambda s, b, h, q, kv: s * (kv * 0.5) * 2.0 * q, lambda s, b, h, q, kv: s * kv * q):
        low = L.lower_score(fn)
        n = np.array([[70000]], dtype=np.int32)
        np.testing.assert_allclose(low.grad(np.ones((1, 1), np.float32), 0, 0, n, n), 70000.0 ** 2, rtol=1e-6)
        body = L.policy_source(None, low.expr)
        assert "*dsds = (((float)(kv)) * ((float)(q)));" in body, body


@pytest.mark.parametrize("name", ["tables", "functions", "sine-and-tables"])
def test_float32_policies_with_many_registers_compile(name):
    """float32 at D = 128, where the kernels leave a policy the fewest registers: table reads with a tanh, and a
    sum of several functions (the compiler crashed on both next to a dK/dV kernel that fills the register file);
    a sine with table reads crashes it next to dQ too and gets the general kernels."""
    from pallas_flexattn import _lib
    t, near = torch.rand(2, 4, 64, 64), torch.rand(4, 128)

    def sine(s, b, h, q, kv):
        x = torch.clamp(s + 0.1 * torch.sin(s), min=-30.0, max=30.0) + t[b, h, q % 64, kv % 64]
        return x + near[h, torch.clamp(q - kv, min=0, max=127)] + t[b, h, q % 64, kv % 64]

    mask, score = {
        "sine-and-tables": (lambda b, h, q, kv: t[b, h, q % 64, kv % 64] > 0.3, sine),
        "tables": (lambda b, h, q, kv: t[b, h, q % 64, kv % 64] > 0.3,
                   lambda s, b, h, q, kv: s * t[b, h, kv % 64, q % 64] + t[b, h, q % 64, kv % 64] + 10 * torch.tanh(s / 10)),
        "functions": (lambda q, kv: ((q // 3) % 5 != (kv // 7) % 5) | (q == kv),
                      lambda s, b, h, q, kv: torch.log(torch.sigmoid(s) + 1.0)
                      + torch.sqrt(s * s + 1.0) * torch.exp(-torch.abs(q - kv) / 64.0) + torch.sin(s)),
    }[name]
    mods = L.UserMods(L.lower_mask(mask), L.lower_score(score))
    assert len(_lib.compile_mods(mods.source, _lib.DTYPE_F32, 128, mods.flags(False))) > 1000


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_generated_tanh_is_as_exact_as_a_float32_library_function(tmp_path):
    """um_tanh compiled for the host (exact exponential and reciprocal, as the GPU's to half a unit): every 128th
    float of [2^-10, 16] within 2.5 * 2^-24 of the value, the largest error of the GPU library's tanhf (2.4 on
    the GPU itself), odd, and right at 0, the infinities and NaN."""
    (tmp_path / "t.cpp").write_text("""
#include <math.h>
#include <stdio.h>
#include <string.h>
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_exp2f(x) exp2f(x)
""" + L._PRELUDE + """
int main() {
  double worst = 0;
  for (unsigned u = 0x3a800000u; u <= 0x41800000u; u += 128) {
    float x;
    memcpy(&x, &u, 4);
    const double t = tanh((double)x), e = fabs(um::um_tanh(x) - t) / t;
    worst = e > worst ? e : worst;
    if (um::um_tanh(-x) != -um::um_tanh(x)) return 1;
  }
  if (um::um_tanh(0.f) != 0.f || um::um_tanh(INFINITY) != 1.f || !isnan(um::um_tanh(NAN))) return 2;
  if (um::um_tanh(1e-40f) != 1e-40f) return 3;
  printf("%.3f\\n", worst * 16777216.0);
}
""")
    subprocess.run(["g++", "-O1", "-ffp-contract=off", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0, r.returncode
    assert float(r.stdout) <= 2.5, r.stdout


def test_general_float32_kernels_flag():
    """FA_MODS_GENERAL: the general kernels by name, the same flags in the blob; float32 only; what compiling falls
    back to when the compiler is ended by a signal."""
    from pallas_flexattn import _lib
    mods = L.UserMods(None, L.lower_score(lambda s, b, h, q, kv: s * 0.5))
    f = mods.flags(False)
    for flags, name in ((f, b"fwd_f32_kernel"), (f | _lib.MODS_GENERAL, b"10fwd_kernelIfLi64")):
        blob = _lib.compile_mods(mods.source, _lib.DTYPE_F32, 64, flags)
        assert int.from_bytes(blob[32:36], "little") == f and name in blob
    with pytest.raises(_lib.FlexAttnError, match="exit 3"):
        _lib.compile_mods(mods.source, _lib.DTYPE_BF16, 64, f | _lib.MODS_GENERAL)
