"""ctypes view of the GPU tests' device-side comparisons (tests/native/checks.hip, built with
the library)."""
import ctypes as C
import os

from mbirtem import capi

PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libmbir_checks.so")


def load():
    capi.lib()  # the library whose functions the checks call
    lib = C.CDLL(PATH)
    lib.checks_selector.argtypes = [C.c_int, C.c_uint64, C.c_int, C.POINTER(C.c_ulonglong)]
    lib.checks_project_wide.argtypes = [C.c_void_p, C.POINTER(C.c_float), C.POINTER(C.c_double)]
    return lib
