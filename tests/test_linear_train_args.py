"""Argument checks of the entry points of include/tg_fp8_train.h and tg_fp8_prefill.h (no GPU): the headers
and the ctypes tables agree, and bad calls are answered before any launch."""
import re
import os

import _tglib as L

N = None
BIG = 1 << 40


def test_header_and_signatures_agree():
    for header, table in (("tg_fp8_train.h", L.TRAIN_SIGNATURES), ("tg_fp8_prefill.h", L.PREFILL_SIGNATURES)):
        text = open(os.path.join(os.path.dirname(L.HEADER_PATH), header)).read()
        names = set(re.findall(r"\b(tg_[a-z0-9_]+)\s*\(", re.sub(r"/\*.*?\*/", "", text, flags=re.S)))
        assert names == set(table)


def _einval(rc, what):
    assert rc == L.TG_EINVAL and what in L.lib().tg_last_error().decode()


def test_bad_calls():
    lib = L.lib()
    _einval(lib.tg_linear_fwd(N, 0, N, 0, N, 4, 4, 128, 0, N, N, BIG, N), "null pointer")
    _einval(lib.tg_linear_fwd(N, 0, N, 0, N, -4, 4, 128, 0, N, N, BIG, N), "bad GEMM shape")
    _einval(lib.tg_linear_fwd(N, 0, N, 0, N, 4, 4, 100, 0, N, N, BIG, N), "not divisible")
    _einval(lib.tg_linear_fwd(N, 2, N, 0, N, 4, 4, 128, 0, N, N, BIG, N), "bf16 or f32")
    _einval(lib.tg_linear_fwd(N, 0, N, 0, N, 4, 128, 128, 1, N, N, BIG, N), "whole blocks")
    assert lib.tg_linear_fwd(N, 0, N, 0, N, 0, 4, 128, 0, N, N, 0, N) == L.TG_OK
    _einval(lib.tg_linear_bwd_kept(N, 3, N, 0, 256, 0, 256, 0, 128, 128, 128, N, BIG, N), "null pointer")
    _einval(lib.tg_linear_bwd_kept(N, 1, N, 0, 256, 0, N, 0, 128, 128, 128, N, BIG, N), "not kept")
    _einval(lib.tg_linear_bwd_kept(N, 3, N, 0, 256, 0, 256, 0, 100, 128, 128, N, BIG, N), "multiples of 128")
    _einval(lib.tg_linear_bwd(N, 0, N, 0, N, 0, 256, 256, 4, 4, 128, N, BIG, N), "null pointer")
    _einval(lib.tg_linear_bwd(N, 0, N, 0, N, 3, 256, 256, 4, 4, 128, N, BIG, N), "bf16 or f32")
    _einval(lib.tg_linear_bwd(256, 0, 256, 0, 256, 0, 256, 256, 4, 4, 128, 256, 0, N), "workspace too small")
    assert lib.tg_linear_bwd(N, 0, N, 0, N, 0, N, N, 4, 4, 128, N, 0, N) == L.TG_OK


def test_negative_extents_and_empty_problems():
    """Negative extents are refused before the pointers are looked at; an empty problem without a wanted gradient
    is a no-op (test_gpu_empty_extents.py has the wanted ones)."""
    lib = L.lib()
    for m, n in ((-128, 128), (128, -128)):
        _einval(lib.tg_linear_fwd(N, 0, N, 0, N, m, n, 128, 0, N, N, BIG, N), "bad GEMM shape")
        _einval(lib.tg_linear_bwd_kept(N, 3, N, 0, 256, 0, 256, 0, m, n, 128, N, BIG, N), "bad GEMM shape")
        _einval(lib.tg_linear_bwd(N, 0, N, 0, N, 0, 256, 256, m, n, 128, N, BIG, N), "bad GEMM shape")
    for m, n in ((0, 128), (128, 0), (0, 0)):
        assert lib.tg_linear_fwd(N, 0, N, 0, N, m, n, 128, 0, N, N, 0, N) == L.TG_OK
        assert lib.tg_linear_bwd_kept(N, 3, N, 0, N, 0, N, 0, m, n, 128, N, 0, N) == L.TG_OK
        assert lib.tg_linear_bwd(N, 0, N, 0, N, 0, N, N, m, n, 128, N, 0, N) == L.TG_OK
    # the gradient of an operand that was not kept stays refused
    _einval(lib.tg_linear_bwd_kept(N, 1, N, 0, 256, 0, N, 0, 128, 0, 128, N, 0, N), "not kept")


def test_operand_alignment():
    """b at an odd element is refused beside a bf16 a, except where only a.T is kept; g, except where only dW is
    asked for."""
    lib = L.lib()
    fwd = lambda ac, b, bc, keep: lib.tg_linear_fwd(256, ac, b, bc, 256, 128, 128, 128, keep, 256, 256, BIG, N)
    for ac, b, bc, keep in ((0, 258, 0, 0), (0, 258, 0, 2), (0, 258, 0, 3), (1, 257, 0, 0), (0, 257, 0, 1)):
        _einval(fwd(ac, b, bc, keep), "16-byte")
    _einval(lib.tg_linear_bwd_kept(256, 3, 258, 0, 256, 0, 256, 0, 128, 128, 128, 256, BIG, N), "16-byte")
    _einval(lib.tg_linear_bwd_kept(256, 1, 257, 0, N, 0, 256, 0, 128, 128, 128, 256, BIG, N), "16-byte")


def test_prefill_kv_bad_calls():
    lib = L.lib()
    _einval(lib.tg_prefill_kv(N, N, N, 1, 4, 2, 8, 128, N), "null pointer")
    _einval(lib.tg_prefill_kv(N, N, N, 1, 9, 2, 8, 128, N), "more rows")
    _einval(lib.tg_prefill_kv(N, N, N, 1, 4, 2, 8, 100, N), "multiple of 8")
    _einval(lib.tg_prefill_kv(N, N, N, -1, 4, 2, 8, 128, N), "bad shape")
    assert lib.tg_prefill_kv(N, N, N, 0, 4, 2, 8, 128, N) == L.TG_OK
