"""The C-ABI library loads and exports every entry point ``include/t2w.h`` declares (no GPU calls)."""

import ctypes
import os
import re

import pytest

import t2w_amd  # noqa: F401
from t2w_amd import _lib

HEADER = os.path.join(os.path.dirname(os.path.dirname(__file__)), "include", "t2w.h")


def declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(t2w_\w+)\s*\(", text)))


def test_header_declares_the_bound_symbols():
    assert set(declared()) == set(_lib.exported_symbols())


def test_library_exports_every_declared_symbol():
    L = _lib.lib()
    missing = [n for n in declared() if not hasattr(L, n)]
    assert not missing, missing
    assert L.t2w_abi_version() == 1


def ring_args(**kw):
    """t2w_gemm_ring arguments that name no memory (every call here is refused before a launch)."""
    a = _lib.RingArgs(M=256, N=1024, K=1024, lda=1024, ldc=1024, splits=1, H=1024, eps_qk=1e-6)
    for k in ("A", "W", "bias", "gate", "C", "q_out", "k_pool", "v_pool", "slots", "qn_w", "qn_b", "kn_w", "kn_b"):
        setattr(a, k, 1 << 20)
    for k, v in kw.items():
        setattr(a, k, v)
    return a


def ring_refuses(**kw):
    assert _lib.lib().t2w_gemm_ring(ctypes.byref(ring_args(**kw)), None) == 1
    assert _lib.lib().t2w_last_error().decode() == "ring gemm: invalid argument"


@pytest.mark.parametrize("tile", [2, 3, 4])
def test_ring_qkv_needs_whole_tiles(tile):
    """A 128-column tile over 3 H columns that are not a multiple of 128 would store the overhang as a head of v."""
    ring_refuses(epi=5, tile=tile, H=960, N=2880, K=960, lda=960)


@pytest.mark.parametrize("kw", [{"M": (1 << 21) - 65536}, {"M": (1 << 31) - 1}, {"N": 1 << 21}, {"M": (1 << 21) - 65536, "epi": 6, "splits": 2}], ids=str)
def test_ring_refuses_operands_beyond_32_bit_offsets(kw):
    """The ring's copies name their rows by 32-bit byte offsets: operands of 4 GiB are refused by the ring itself, whoever
    calls it."""
    ring_refuses(tile=0, **kw)
