"""No kernel takes more scratch memory than a few bytes a lane.

Scratch memory (registers that spill, arrays indexed at run time) is not allocated by the library:
the runtime takes it from the device at the launch, 64 lanes x 8192 waves x the bytes below, and with
the card nearly full it cannot, and ends the process's queue where an allocation of the library
would fail with an error.  The figures are those that the compiler wrote into the built library.
"""
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIMIT = 32  # bytes a lane: 16 MiB


def _text(b, at):
    """The MessagePack string at `at`."""
    t = b[at]
    if 0xA0 <= t <= 0xBF:
        return b[at + 1:at + 1 + t - 0xA0]
    n = {0xD9: 1, 0xDA: 2}[t]
    size = int.from_bytes(b[at + 1:at + 1 + n], "big")
    return b[at + 1 + n:at + 1 + n + size]


def _number(b, at):
    t = b[at]
    return t if t < 0x80 else int.from_bytes(b[at + 1:at + 1 + {0xCC: 1, 0xCD: 2, 0xCE: 4}[t]], "big")


def scratch_of_kernels(path):
    """{kernel symbol: scratch bytes a lane} of the device code in a built library."""
    b = open(path, "rb").read()
    key, sym, res, at = b".private_segment_fixed_size", b".symbol", {}, 0
    while (at := b.find(key, at)) >= 0:
        at += len(key)
        res[_text(b, b.index(sym, at) + len(sym)).decode()] = _number(b, at)
    return res


def test_scratch_of_every_kernel():
    from mrchem_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("libmwgreen.so not built")
    res = scratch_of_kernels(_lib.LIB_PATH)
    assert len(res) > 50 and any("k_contract_slices64" in k for k in res)
    assert {k: v for k, v in res.items() if v > LIMIT} == {}
