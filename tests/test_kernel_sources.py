"""Rules of the kernels' sources that no run shows to be broken."""

import glob
import os
import re

import mlx_lm_amd

CSRC = os.path.join(os.path.dirname(os.path.abspath(mlx_lm_amd.__file__)), "csrc")


def _kernels(text):
    """``(name, body)`` of every ``__global__`` function that has a body."""
    for m in re.finditer(r"__global__", text):
        start = text.index("{", m.end())
        name = re.findall(r"(\w+)\s*\([^()]*\)\s*$", text[m.end() : start])[-1]
        depth, at = 0, start
        while True:
            depth += {"{": 1, "}": -1}.get(text[at], 0)
            at += 1
            if depth == 0:
                break
        yield name, text[start:at]


def _asks_without_wait(body):
    """The places in a kernel's body that ask for copies into LDS without a wait for all of them ahead of the next way out."""
    outs = [m.start() for m in re.finditer(r"\breturn\b", body)] + [len(body)]
    asks = [m.start() for m in re.finditer(r"\bask\(", body)]
    return [at for at in asks if "copies_arrived<0>()" not in body[at : next(o for o in outs if o > at)]]


def test_copies_into_lds_are_waited_for_before_a_wave_ends():
    """A kernel that asks for copies beyond the end of its ring (``lds_copy.h``) waits for all of them behind its loop, on each
    way out (waves that only copy have one of their own): LDS that another block has by then must not be written."""
    seen = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip"))):
        with open(path) as f:
            text = f.read()
        for name, body in _kernels(text):
            if "copy16_to_lds(" in body:
                seen.append(name)
                assert not _asks_without_wait(body), (os.path.basename(path), name)
                # each of the waits is needed
                for m in re.finditer(r"copies_arrived<0>\(\);", body):
                    assert _asks_without_wait(body[: m.start()] + body[m.end() :]), (name, m.start())
    assert {"gemm_bf16_tile_kernel", "gemm_f32_tile_kernel", "gemm_f32_cut_kernel"} <= set(seen)
