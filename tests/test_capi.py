"""The C-ABI library loads and exports every symbol include/sfl.h declares (no GPU calls)."""

import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
INVALID, UNSUPPORTED = -1, -2  # SFL_ERR_*


def declared_symbols():
    text = (ROOT / "include" / "sfl.h").read_text()
    return sorted(set(re.findall(r"\b(sfl_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_entry_points():
    names = declared_symbols()
    assert "sfl_decode_attention" in names and "sfl_last_error" in names


def test_library_exports_every_declared_symbol():
    from systems_for_llms_amd import _lib

    if not _lib.LIB_PATH.exists():
        pytest.skip("libsfl.so not built (run __graft_entry__.build())")
    handle = _lib.lib()
    missing = [name for name in declared_symbols() if not hasattr(handle, name)]
    assert not missing
    assert handle.sfl_version().decode().startswith("sfl")
    assert set(_lib.SIGNATURES) <= set(declared_symbols())


def test_argument_errors_are_reported_without_a_launch():
    import ctypes

    from systems_for_llms_amd import _lib

    if not _lib.LIB_PATH.exists():
        pytest.skip("libsfl.so not built")
    with pytest.raises(RuntimeError, match="null pointer"):
        _lib.call("sfl_decode_attention", None, None, None, None, None, None, None, None,
                  1, 1, 1, 1, 64, 1, 0.125, 1, 1, 1, None)
    buf = ctypes.create_string_buffer(64)
    p = ctypes.addressof(buf)
    with pytest.raises(RuntimeError, match="divisible"):
        _lib.call("sfl_decode_attention", p, p, p, p, p, p, p, p, 1, 3, 2, 16, 64, 1, 0.125, 1, 1, 1, None)
    with pytest.raises(RuntimeError, match="head dim"):
        _lib.call("sfl_decode_attention", p, p, p, p, p, p, p, p, 1, 2, 2, 16, 48, 1, 0.125, 1, 1, 1, None)


def test_folded_norm_entry_points_reject_bad_arguments_without_a_launch():
    """Every call here fails an argument check before anything reaches HIP."""
    import ctypes

    from systems_for_llms_amd import _lib

    if not _lib.LIB_PATH.exists():
        pytest.skip("libsfl.so not built")
    buf = ctypes.create_string_buffer(256)
    p = (ctypes.addressof(buf) + 15) // 16 * 16  # 16-byte aligned host address (never dereferenced)
    with pytest.raises(RuntimeError, match="null pointer"):
        _lib.call("sfl_gemm_residual_norm", p, p, p, 64, 128, 64, None, p, p, 1, None)
    with pytest.raises(RuntimeError, match="multiple of 4"):
        _lib.call("sfl_gemm_residual_norm", p, p, p, 64, 130, 64, p, p, p, 1, None)
    with pytest.raises(RuntimeError, match="multiple of 64"):
        _lib.call("sfl_gemm_residual_norm", p, p, p, 64, 128, 72, p, p, p, 1, None)
    with pytest.raises(RuntimeError, match="16-byte"):
        _lib.call("sfl_gemm_residual_norm", p, p, p + 4, 64, 128, 64, p, p, p, 1, None)
    with pytest.raises(RuntimeError, match="sizes must be positive"):
        _lib.call("sfl_norm_scale", p, 0, 64, 128, p, None)
    with pytest.raises(RuntimeError, match="dtype must be BF16 or F16"):
        _lib.call("sfl_rmsnorm_rows_scaled", p, p, p, p, 4, 128, 0, None)
    with pytest.raises(RuntimeError, match="dtype must be F32, BF16 or F16"):
        _lib.call("sfl_gemm", p, p, p, 64, 128, 64, 5, 0, 0, None)
    with pytest.raises(RuntimeError, match="F32 inputs need an F32 output"):
        _lib.call("sfl_gemm", p, p, p, 64, 128, 64, 0, 1, 0, None)
    with pytest.raises(RuntimeError, match="head dim must be 16, 32, 64 or 128"):
        s3 = (ctypes.c_long * 3)(0, 0, 64)
        _lib.call("sfl_causal_attention_f32", p, p, p, p, 1, 1, 8, 48, s3, s3, s3, s3, 0.1, None)
    with pytest.raises(RuntimeError, match="output dtype must be F32 or the input dtype"):
        _lib.call("sfl_gemm", p, p, p, 64, 128, 64, 2, 1, 0, None)
    with pytest.raises(RuntimeError, match="at most 2048"):
        _lib.call("sfl_rmsnorm_rows_scaled", p, p, p, p, 4, 4096, 1, None)
    with pytest.raises(RuntimeError, match="null pointer"):
        _lib.call("sfl_gemm_qkv_rope_scaled", p, p, None, 64, 64, 128, 2, p, p, p, p, p, 64, 1, None)
    with pytest.raises(RuntimeError, match="multiple of 64"):
        _lib.call("sfl_gemm_qkv_rope_scaled", p, p, p, 64, 64, 96, 2, p, p, p, p, p, 64, 1, None)
    with pytest.raises(RuntimeError, match="batch \\* seq"):
        _lib.call("sfl_gemm_qkv_rope_scaled", p, p, p, 65, 64, 128, 2, p, p, p, p, p, 64, 1, None)
    with pytest.raises(RuntimeError, match="multiple of 8"):
        _lib.call("sfl_gemm_swiglu_scaled", p, p, p, p, 64, 100, 128, 1, None)
    with pytest.raises(RuntimeError, match="multiple of 64"):
        _lib.call("sfl_gemm_swiglu_scaled", p, p, p, p, 64, 128, 72, 1, None)


def test_prefill_layers_rejects_before_any_launch():
    import ctypes

    from systems_for_llms_amd import _lib

    one = (_lib.P * 1)(16)
    sizes = dict(dtype=2, layers=1, batch=1, seq=4, given_len=4, d_model=64, heads=2, d_ff=64, capacity=4, fold=0, scale=1.0)
    pointers = {name: one if kind is not _lib.P else 16 for name, kind in _lib.PrefillArgs._fields_
                if name not in sizes}
    assert _lib.lib().sfl_prefill_layers(None, None) != 0
    for change in ({"x": None}, {"w_qkv": None}, {"layers": 0}, {"heads": 3}, {"seq": 1 << 30, "batch": 8},
                   {"fold": 1, "ss": None},
                   {"given_len": 3}, {"given_len": 5}, {"d_model": 66}, {"x_last": 24}, {"dtype": 7}):
        args = _lib.PrefillArgs(**{**sizes, **pointers, **change})
        assert _lib.lib().sfl_prefill_layers(ctypes.addressof(args), None) != 0, change
        assert "prefill_layers" in _lib.lib().sfl_last_error().decode()


def test_prefill_layers_refuses_what_its_layers_would_before_any_launch():
    """Argument errors (-1, -2), not the failed launch (-3) a call without a GPU ends with."""
    import ctypes

    from systems_for_llms_amd import _lib

    sizes = dict(dtype=2, layers=2, batch=1, seq=4, given_len=4, d_model=64, heads=2, d_ff=64, capacity=4, fold=0,
                 scale=1.0)
    pointers = {name: 16 if kind is _lib.P else (_lib.P * 2)(16, 16) for name, kind in _lib.PrefillArgs._fields_
                if name not in sizes}
    second, odd = (lambda: (_lib.P * 2)(16, None)), (lambda: (_lib.P * 2)(16, 20))
    fold, f32 = dict(fold=1), dict(dtype=0)
    for change, code in ((dict(fold, dtype=0), UNSUPPORTED), (dict(fold, d_ff=96), UNSUPPORTED),
                         (dict(fold, d_model=96, heads=3), UNSUPPORTED),
                         (dict(fold, d_model=4096, heads=32), UNSUPPORTED), (dict(fold, ffn_norm=odd()), INVALID),
                         (dict(fold, attn_norm=odd()), INVALID), (dict(fold, act=20), INVALID),
                         (dict(d_model=96), UNSUPPORTED), (dict(heads=4), UNSUPPORTED), (dict(d_ff=60), UNSUPPORTED),
                         (dict(cos_t=None), INVALID), (dict(sin_t=None), INVALID), (dict(scale=0.0), INVALID),
                         (dict(scale=float("nan")), INVALID), (dict(f32, act=24), INVALID),
                         (dict(f32, w2=odd()), INVALID),
                         (dict(f32, batch=1 << 22, seq=2, d_model=48, heads=3), UNSUPPORTED),
                         *((dict({name: second()}), INVALID) for name in ("attn_norm", "w_qkv", "w_out", "ffn_norm",
                                                                         "w13", "w2", "k_cache", "v_cache"))):
        args = _lib.PrefillArgs(**{**sizes, **pointers, **change})
        assert _lib.lib().sfl_prefill_layers(ctypes.addressof(args), None) == code, change


def test_output_projection_is_shared_only_while_the_rows_stay_cached():
    """Workgroups per head by (batch, heads, capacity, head dim, dtype): every head's K and V is
    read by each, so long caches, and heads whose workgroups sit on several XCDs, keep one."""
    from systems_for_llms_amd import _lib

    count = _lib.lib().sfl_decode_out_proj_workgroups
    bf16, f32 = 1, 0
    for args, want in (((1, 16, 4096, 64, bf16), 4), ((4, 16, 4096, 64, bf16), 4), ((4, 16, 8192, 64, bf16), 2),
                       ((4, 16, 16384, 64, bf16), 1), ((4, 16, 65536, 64, bf16), 1), ((8, 16, 4096, 64, bf16), 2),
                       ((8, 16, 4096, 64, f32), 1), ((8, 16, 16384, 64, bf16), 1), ((16, 16, 256, 64, bf16), 1),
                       ((1, 12, 1024, 64, bf16), 4), ((1, 12, 4096, 64, bf16), 4), ((1, 12, 8192, 64, bf16), 1),
                       ((10, 12, 1024, 64, bf16), 2), ((9, 12, 1024, 64, bf16), 1), ((1, 6, 1024, 64, bf16), 1),
                       ((1, 4, 64, 16, f32), 1), ((0, 4, 64, 64, bf16), 0), ((1, 4, 64, 64, 7), 0)):
        assert count(*args) == want, args
