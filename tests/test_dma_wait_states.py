"""Wait states of the LDS DMA loads in the built library.

A buffer load that reads scalar registers written by a VALU instruction (a
``v_readfirstlane`` that forms its resource, a ``v_readlane`` that reloads a spilled one)
needs five wait states in between.  The compiler inserts them for its own loads, but not for
a load written in inline asm, as the 32x32x16 tile kernels' are: a resource read too early
makes the load take another operand's range.  These tests disassemble the gfx950 code of
``libkohakutt_amd.so`` and count them, and feed the count a planted listing."""

from __future__ import annotations

import re
import struct
import subprocess

import pytest

from kohakutt_amd import _build

OBJDUMP = _build.ROCM / "llvm" / "bin" / "llvm-objdump"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
NEEDED = 5


def _scalars(arg):
    """The scalar registers of one operand."""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", arg)
    if m:
        return range(int(m.group(1)), int(m.group(2)) + 1)
    m = re.fullmatch(r"s(\d+)", arg)
    return [int(m.group(1))] if m else []


def short_waits(listing):
    """(LDS DMA loads of a listing, [(kernel, wait states, load)] with too few)."""
    kernel, written, at, loads, short = None, {}, 0, 0, []
    for line in listing.splitlines():
        m = re.match(r"[0-9a-f]+ <(.+)>:", line)
        if m:
            kernel, written, at = m.group(1), {}, 0
            continue
        m = re.match(r"\s+(\S+)\s*(.*?)\s*(//.*)?$", line)
        if not m or line[0] not in " \t":
            continue
        op, args = m.group(1), m.group(2)
        if op == "s_nop":
            at += int(args, 0) + 1
            continue
        if op.startswith("buffer_load") and re.search(r"\blds\b", args):
            loads += 1
            wait = min((at - written[r] - 1 for a in args.split(", ") for r in _scalars(a) if r in written), default=NEEDED)
            if wait < NEEDED:
                short.append((kernel, wait, f"{op} {args}"))
        dst = _scalars(args.split(", ")[0])
        for r in dst:
            if op.startswith("v_"):
                written[r] = at
            else:
                written.pop(r, None)
        at += 1
    return loads, short


def _device_images(data):
    """The gfx950 code objects of a host library's offload bundles."""
    at = data.find(BUNDLE)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24 : p + 24 + length] and size:
                yield data[at + offset : at + offset + size]
            p += 24 + length
        at = data.find(BUNDLE, at + 1)


@pytest.mark.parametrize("between,ok", [
    ("s_mov_b32 m0, s5\n\ts_nop 0", False),
    ("s_mov_b32 m0, s5\n\ts_nop 3", True),
    ("s_nop 4", True),
    ("s_nop 3", False),
])  # fmt: skip
def test_planted_listing(between, ok):
    text = ("0000000000001000 <kernel>:\n\ts_mov_b32 s6, s2\n\tv_readfirstlane_b32 s6, v3 // 0: 1\n\t" + between +
            "\n\tbuffer_load_dwordx4 v1, s[4:7], 0 offen lds // 4: 2\n\tbuffer_load_dword v1, v2, s[8:11], 0 offen\n")
    loads, short = short_waits(text)
    assert loads == 1 and (not short) == ok, short


def test_built_kernels_wait_for_their_resources(tmp_path):
    total, bad = 0, []
    for i, image in enumerate(_device_images(_build.CAPI_LIB.read_bytes())):
        if b"attn_tile_kernel" not in image and b"attn_bwd_tile_kernel" not in image:
            continue
        path = tmp_path / f"{i}.co"
        path.write_bytes(image)
        out = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", str(path)], stdout=subprocess.PIPE, text=True, check=True)
        loads, short = short_waits(out.stdout)
        total += loads
        bad += short
    assert total > 0
    assert not bad, f"{len(bad)} loads, the first: {bad[:3]}"
