"""The host side of include/wkv7_segments.h: which calls ask for a workspace,
and what the two entry points refuse (they run no HIP call for it)."""

import ctypes

import pytest

from conftest import load_pkg

F32, BF16 = 0, 1
FAKE = 0x100000   # aligned addresses that are never dereferenced


@pytest.fixture(scope="module")
def native():
    return load_pkg()._native


def _bytes(native, which, B, T, H, chunk, dtype, options=None):
    return getattr(native.lib(), f"wkv7_{which}_workspace_bytes")(
        B, T, H, 64, chunk, dtype, native.options_ref(options))


@pytest.mark.parametrize("which", ["forward", "backward"])
def test_workspace_is_asked_for_where_the_gpu_would_idle(native, which):
    assert _bytes(native, which, 1, 4096, 32, 16, BF16) > 0
    # shapes that fill the GPU, are too short, or run on the step kernels
    for args in ((8, 4096, 32, 16, BF16), (1, 65536, 256, 16, BF16), (1, 16, 1, 16, BF16),
                 (1, 0, 1, 16, BF16), (0, 4096, 4, 16, BF16), (1, 4096, 0, 16, BF16),
                 (1, 4096, 1, 8, BF16)):
        assert _bytes(native, which, *args) == 0, args
    step = native.Wkv7Options(native.KERNELS_STEP, 0)
    assert _bytes(native, which, 1, 4096, 32, 16, BF16, step) == 0
    # invalid arguments
    for args in ((1, 100, 1, 16, BF16), (1, 64, 1, 16, 7), (-1, 64, 1, 16, BF16)):
        assert _bytes(native, which, *args) == -1, args
    assert _bytes(native, which, 1, 4096, 32, 16, BF16, native.Wkv7Options(9, 0)) == -1


@pytest.mark.parametrize("which", ["forward", "backward"])
def test_more_segments_than_the_gpu_runs_at_once_are_not_cut(native, which):
    for pairs in (1, 2, 3, 7, 31, 85, 127, 128, 129, 255, 256):
        for chunks in (1, 2, 5, 16, 31, 64, 257):
            n = _bytes(native, which, 1, 16 * chunks, pairs, 16, BF16)
            segments, rest = divmod(n, pairs * (2 * 4096 * 4 + 4))
            assert rest == 0 and segments != 1 and segments <= min(256 // pairs, chunks), (pairs, chunks)


def test_workspace_checks(native):
    lib, n = native.lib(), _bytes(native, "forward", 1, 4096, 32, 16, BF16)
    toks = [FAKE + (i << 32) for i in range(6)]
    outs = [FAKE + (i << 34) for i in range(2, 5)]

    def fwd(ws, nbytes):
        return lib.wkv7_forward_ws(*toks, None, 1, 4096, 32, 64, 16, BF16, 0, 0, *outs, None, None,
                                   ws, nbytes, None)
    assert fwd(FAKE + 8 + (1 << 40), n) == 6           # WKV7_ERR_ALIGNMENT
    assert fwd(toks[2], n) == 7                        # WKV7_ERR_OVERLAP (an input)
    assert fwd(outs[1] + 4096, n) == 7                 # (an output)
    assert fwd(FAKE + (1 << 40), -1) == 2              # WKV7_ERR_SHAPE
    grads = [FAKE + (i << 36) for i in range(1, 7)]

    def bwd(ws, nbytes):
        return lib.wkv7_backward_ws(*toks, *outs[:2], outs[2], None, 1, 4096, 32, 64, 16, BF16, 0, 0,
                                    *grads, None, None, ws, nbytes, None)
    n = _bytes(native, "backward", 1, 4096, 32, 16, BF16)
    assert bwd(FAKE + 8 + (1 << 40), n) == 6
    assert bwd(outs[0], n) == 7 and bwd(grads[3], n) == 7
    assert ctypes.sizeof(native.Wkv7Options) == 8
