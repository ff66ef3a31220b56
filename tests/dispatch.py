"""The launchers' choices, from the headers that the launchers themselves use
(tests/cpp/dispatch.cpp)."""
import ctypes
import os
import subprocess

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
CUS = 256   # an MI355X
FP8_FORMS = ("wide 256x256", "wide 256x128", "wide 128x160", "wide 128x128", "wide 64x64", "wide mixed", "rows 256x256",
             "rows 256x128", "rows 128x128", "rows 64x64")
W8A16_FORMS = ("256x256", "128x256", "128x160", "128x128", "64x128", "64x64", "64 rows", "stream-K")   # -2 and -1 last
_lib = None


def lib():
    global _lib
    if _lib is None:
        subprocess.run(["make", "-C", CPP, "build/libdispatch.so"], check=True, capture_output=True)
        _lib = ctypes.CDLL(os.path.join(CPP, "build", "libdispatch.so"))
        _lib.attention_stream_plan.argtypes = [ctypes.c_size_t] * 3 + [ctypes.c_int, ctypes.c_size_t, ctypes.c_void_p]
        _lib.fp8_form.argtypes = [ctypes.c_uint32] * 3 + [ctypes.c_int, ctypes.c_uint64]
        _lib.w8a16_form.argtypes = [ctypes.c_uint32] * 3 + [ctypes.c_uint64]
        _lib.attention_splits.argtypes = [ctypes.c_size_t]
    return _lib


def attention_stream_plan(nh, nkv, length, split=True, cus=CUS):
    out = (ctypes.c_uint32 * 8)()
    lib().attention_stream_plan(nh, nkv, length, int(split), cus, out)
    return dict(zip(("splits", "tiles", "more", "gb", "hgw", "waves", "gx", "gy"), out))


def fp8_form(M, N, K, aligned=True, cus=CUS):
    """The form of an fp8 x fp8 product; aligned: its output starts on 16 bytes."""
    return FP8_FORMS[lib().fp8_form(M, N, K, int(aligned), cus)]


def w8a16_form(M, N, K, cus=CUS):
    """The form of a w8a16 product of more than 64 rows."""
    return W8A16_FORMS[lib().w8a16_form(M, N, K, cus)]
