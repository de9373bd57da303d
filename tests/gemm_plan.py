"""The library's own choice of GEMM kernel, asked without a launch: gemm_plan
and split_tag of gemm_dispatch.hip (C++ functions, so by their mangled names).
"""

import ctypes


class Plan(ctypes.Structure):
    """bm = 0: 256x256 tiles (Stream-K when workers > 0), else a bm x bn block
    over `splits` K ranges."""
    _fields_ = [("bm", ctypes.c_int), ("bn", ctypes.c_int), ("splits", ctypes.c_int),
                ("workers", ctypes.c_int)]

    def __repr__(self):
        return f"Plan(bm={self.bm}, bn={self.bn}, splits={self.splits}, workers={self.workers})"


class _Limits(ctypes.Structure):
    _fields_ = [("slot_bytes", ctypes.c_size_t), ("counter_words", ctypes.c_size_t)]


def split_tag(lib):
    fn = lib._ZN4wave4gemm9split_tagEv
    fn.restype, fn.argtypes = ctypes.c_uint64, []
    return fn()


def plan(lib, M, N, K, cus=256, vec4=None, workers=0, slot_bytes=0, counter_words=0,
         c_vec=None):
    """What wave_gemm_launch runs (no workspace limits given); c_vec: by default
    that of a 16-bit row-major C."""
    fn = lib._ZN4wave4gemm9gemm_planEiiiibbiRKNS0_11SplitLimitsE
    fn.restype = Plan
    fn.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool] * 2 + [ctypes.c_int,
                                                              ctypes.POINTER(_Limits)]
    limits = _Limits(slot_bytes, counter_words)
    return fn(M, N, K, cus, K % 4 == 0 if vec4 is None else vec4,
              N % 8 == 0 if c_vec is None else c_vec, workers, ctypes.byref(limits))


def auto_plan(lib, M, N, K, short_m, workers, cus=256):
    """What wave_gemm_auto_launch runs with its whole workspace: short_m is
    (column block, splits) of the workspace for M <= 128 ((0, 0): none), workers
    Stream-K's (0: none)."""
    bn, s = short_m
    if s:
        tiles = -(-N // bn)
        return plan(lib, M, N, K, cus, slot_bytes=tiles * s * 128 * bn * 4,
                    counter_words=2 * tiles)
    if workers:
        return plan(lib, M, N, K, cus, workers=workers,
                    slot_bytes=workers * 2 * 256 * 256 * 4 - 4096 * 8, counter_words=4096)
    return plan(lib, M, N, K, cus)
