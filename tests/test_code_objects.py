"""What the compiler made of the fused kernels, read from the built library: the kernels of models with a row tile and those
whose private regions are in LDS hold every function inlined.

A function left out of line takes the model, the state view and the LDS pointers by reference: LDS is then reached by flat
accesses and every model array through an address loaded per lane (five boxes in a row, 30 dofs, x1024: 2685 us a step
instead of 1894)."""

from __future__ import annotations

import struct

from genesis_amd import runtime

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
STT_FUNC = 2


def _code_objects(data):
    """The gfx950 ELF images of every offload bundle in the library."""
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24 : p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield data[at + off : at + off + size]
        at = data.find(MAGIC, at + 1)


def _symbols(elf):
    """(name, type) of every symbol of a 64-bit little-endian ELF image."""
    (shoff,) = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    sections = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shentsize) for i in range(shnum)]
    for _, kind, _, _, off, size, link, _, _, entsize in sections:
        if kind not in (2, 11):  # SHT_SYMTAB, SHT_DYNSYM
            continue
        strings = sections[link][4]
        for k in range(size // entsize):
            name, info = struct.unpack_from("<IB", elf, off + k * entsize)
            text = elf[strings + name : elf.index(b"\0", strings + name)].decode()
            yield text, info & 15


def _fused_units():
    with open(runtime.LIB_PATH, "rb") as f:
        data = f.read()
    for elf in _code_objects(data):
        functions = {n for n, kind in _symbols(elf) if kind == STT_FUNC}
        kernels = {n for n in functions if "k_fused_" in n}
        if kernels:
            yield kernels, functions


def test_row_tile_and_lds_kernels_hold_their_functions_inlined():
    runtime.load_library()
    units = [(k, f) for k, f in _fused_units() if any("k_fused_wave" in n or "k_fused_largeILb1E" in n for n in k)]
    assert len(units) == 3  # two row-tile classes, the larger models with their region in LDS
    for kernels, functions in units:
        called = sorted(functions - kernels)
        print(sorted(kernels), called)
        for n in called:
            if "k_sched_flip" not in n:
                assert not any(t in n for t in ("DModel", "DState", "LState", "FusedArgs", "WorkRows")), n


def test_no_kernel_calls_its_solver():
    runtime.load_library()
    units = list(_fused_units())
    assert len(units) == 6
    for kernels, functions in units:
        solver = [n for n in functions if "wave_solve" in n or "wave_linesearch" in n or "cholesky" in n]
        assert not solver, (sorted(kernels), solver)
