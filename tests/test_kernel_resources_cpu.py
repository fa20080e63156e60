"""Scratch memory of the built kernels, from the metadata the compiler wrote into
the library: none in the steps of states up to d = 16 with a selection basis,
their pairs, the reference-mode steps without one (their updates spill when the
covariance is updated by columns), the d = 12 batch of up to 5 joints and the
four-lane d = 24 steps."""
import re
import struct

import msgpack
import pytest

from mkfbodytracker_pdaf_amd import _build

NO_SCRATCH = (
    r"k_stepILi(8|12|16)ELi[01]ELi[1-8]ELb[01]E",        # k_step<D, MODE, SELJ, REC>
    r"k_step_pairILi(8|12|16)ELi0ELi3E",                 # k_step_pair<D, MODE, SELJ>
    r"k_stepILi(8|12|16)ELi0ELi0ELb[01]E",
    r"k_batch_stepILi12ELi[1-5]ELi[12]E",                # k_batch_step<D, SELJ, PPL>
    r"k_batch_step_q24ILi[35]ELb[01]E",                  # k_batch_step_q24<SELJ, MFMA>
)


def _kernels(path):
    """Kernel metadata by mangled name: the AMDGPU notes (type 32) of every
    device ELF embedded in the library."""
    with open(path, "rb") as f:
        data = f.read()
    out, pos = {}, data.find(b"\x7fELF", 4)
    while pos >= 0:
        if data[pos + 4] == 2 and struct.unpack_from("<H", data, pos + 18)[0] == 224:   # ELF64, EM_AMDGPU
            shoff, = struct.unpack_from("<Q", data, pos + 40)
            shsize, shnum = struct.unpack_from("<HH", data, pos + 58)
            for k in range(shnum):
                sh = pos + shoff + k * shsize
                kind, = struct.unpack_from("<I", data, sh + 4)
                off, = struct.unpack_from("<Q", data, sh + 24)
                if kind != 7:                                                           # SHT_NOTE
                    continue
                name, desc, note = struct.unpack_from("<III", data, pos + off)
                start = pos + off + 12 + ((name + 3) & ~3)
                if note == 32:
                    meta = msgpack.unpackb(data[start:start + desc], raw=False)
                    out.update({q[".name"]: q for q in meta["amdhsa.kernels"]})
        pos = data.find(b"\x7fELF", pos + 4)
    return out


@pytest.fixture(scope="module")
def kernels():
    from mkfbodytracker_pdaf_amd import capi
    capi.lib()
    return _kernels(_build.LIB)


@pytest.mark.parametrize("pattern", NO_SCRATCH)
def test_no_scratch(kernels, pattern):
    found = {n: q for n, q in kernels.items() if re.search(pattern, n)}
    assert found, pattern
    assert not [n for n, q in found.items() if q[".private_segment_fixed_size"]]
