"""Argument checks of include/tg_fp8_train.h's entry points (no GPU): the header
and the ctypes table agree, and bad calls are answered before any launch."""
import re
import os

import _tglib as L

N = None
BIG = 1 << 40


def test_header_and_signatures_agree():
    text = open(os.path.join(os.path.dirname(L.HEADER_PATH), "tg_fp8_train.h")).read()
    names = set(re.findall(r"\b(tg_[a-z0-9_]+)\s*\(", re.sub(r"/\*.*?\*/", "", text, flags=re.S)))
    assert names == set(L.TRAIN_SIGNATURES)


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
