"""Shapes that take each tile of the FP8 GEMM on 256 compute units, for the GPU tests of those tiles and the CPU
test that they still do (test_gemm_tile_choice.py)."""
import ctypes

import _tglib as L

CUS = 256


def tile_of(M, N, K, km, f32=False, cus=CUS):
    r, c = ctypes.c_int(), ctypes.c_int()
    L.check(L.lib().tg_gemm_fp8_tile(M, N, K, int(km), L.TG_DTYPE_F32 if f32 else L.TG_DTYPE_BF16, cus, ctypes.byref(r),
                                     ctypes.byref(c)))
    return r.value, c.value


# tile -> (M, N, K, scales K-block-major): M and N that end inside a tile and on its edge, widths of whole 16-byte rows,
# of 8 bytes and odd ones, one K block, and more than the stages in flight
GEMM = {
    (256, 256): [(4097, 2304, 128, True), (4096, 4096, 640, False), (1025, 8191, 9216, False), (2049, 4404, 9216, False),
                 # several tiles per workgroup, N % 8 != 0 and N % 8 == 0
                 (5000, 5001, 9216, False), (5000, 5000, 384, True)],
    (128, 256): [(385, 14336, 128, True), (4097, 1500, 896, False), (513, 12301, 128, False), (512, 14336, 512, False),
                 (2049, 3080, 640, True)],
    (128, 192): [(257, 14336, 128, True), (4097, 1001, 640, False), (640, 8191, 256, True), (640, 6912, 640, False),
                 (300, 14336, 4096, False)],
    (128, 128): [(200, 12300, 2304, False), (257, 10240, 2304, False), (3000, 1001, 2304, False), (129, 12304, 4096, False)],
    (64, 128): [(65, 12304, 128, True), (1025, 1501, 640, False), (257, 10240, 384, False), (5000, 384, 640, True)],
    (64, 96): [(4097, 200, 128, True), (257, 4404, 640, False), (300, 8191, 384, True), (640, 2304, 640, True)],
    (64, 64): [(33, 10240, 128, True), (4097, 97, 128, False), (385, 1500, 640, True), (2049, 384, 384, False)],
    (32, 64): [(1, 8, 128, True), (31, 384, 1152, False), (63, 577, 384, True), (513, 200, 128, False)],
}

# (M, K, N) of a float32 linear and the tiles of its gradients dX (M, K) over N and dW (K, N) over M
LINEAR_F32 = {
    (1000, 640, 520): ((64, 64), (32, 64)),
    (640, 2304, 896): ((64, 96), (64, 128)),
    (1025, 2304, 2304): ((64, 96), (128, 192)),
    (300, 2304, 9216): ((64, 64), (256, 256)),
    (513, 8192, 136): ((128, 192), (64, 96)),
    (2049, 4352, 200): ((256, 256), (64, 96)),
    (1000, 6912, 390): ((128, 256), (64, 128)),
}


def up128(n):
    return -(-n // 128) * 128
