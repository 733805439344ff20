"""The fp32 linear entry points on the CPU: rejected arguments, and the M0
invariant of their inline LDS-DMA copies in the compiled kernels."""

from __future__ import annotations

import pytest

from test_isa_invariants import CSRC, _assembly
from transformer_opt import _native


def _linear(lib, **over):
    args = dict(x=1 << 20, w=2 << 20, wp=3 << 20, b=None, y=4 << 20, M=64, N=64, K=64, ldx=64, ldw=64, ldy=64,
                act=_native.TTK_ACT_NONE, stream=None)
    args.update(over)
    return lib.ttk_linear_f32_fwd(args["x"], args["w"], args["wp"], args["b"], args["y"], args["M"], args["N"],
                                  args["K"], args["ldx"], args["ldw"], args["ldy"], args["act"], args["stream"])


@pytest.mark.parametrize("over,status,message", [
    (dict(act=7), _native.TTK_EINVAL, "activation"),
    (dict(M=-1), _native.TTK_EINVAL, "M must be"),
    (dict(N=0), _native.TTK_EINVAL, "positive"),
    (dict(x=None), _native.TTK_EINVAL, "NULL"),
    (dict(wp=None), _native.TTK_EINVAL, "NULL"),
    (dict(K=48, ldx=48, ldw=48), _native.TTK_EUNSUPPORTED, "multiple of 32"),
    (dict(N=62), _native.TTK_EUNSUPPORTED, "multiple of 4"),
    (dict(x=(1 << 20) + 4), _native.TTK_EUNSUPPORTED, "16-byte aligned"),
    (dict(b=(5 << 20) + 8), _native.TTK_EUNSUPPORTED, "16-byte aligned"),
    (dict(ldx=62), _native.TTK_EUNSUPPORTED, "multiples of 4"),
    (dict(ldw=60), _native.TTK_EUNSUPPORTED, "ldw"),
    (dict(ldy=1 << 22), _native.TTK_EUNSUPPORTED, "below 2^22"),
    (dict(y=(3 << 20) + 64 * 64 * 6 - 16), _native.TTK_EINVAL, "overlaps"),
    (dict(y=1 << 20), _native.TTK_EINVAL, "overlaps"),
    (dict(M=0), _native.TTK_OK, ""),
])
def test_fp32_linear_argument_errors_are_reported_without_launching(over, status, message):
    lib = _native.load()
    assert _linear(lib, **over) == status
    assert message in _native.last_error()


def test_split_weight_arguments_and_sizes():
    lib = _native.load()
    size, split = lib.ttk_linear_f32_split_bytes, lib.ttk_linear_f32_split_weight
    assert size(64, 64) == 64 * 64 * 6 and size(33, 32) == 64 * 32 * 6
    assert size(0, 64) == size(64, 0) == size(-1, 64) == size(64, 1 << 22) == 0
    assert split(None, 1 << 20, 64, 64, 64, None) == _native.TTK_EINVAL
    assert split(1 << 20, 2 << 20, 64, 40, 40, None) == _native.TTK_EUNSUPPORTED
    assert split(1 << 20, (1 << 20) + 16, 64, 64, 64, None) == _native.TTK_EINVAL
    assert split(1 << 20, 2 << 20, 64, 64, 32, None) == _native.TTK_EUNSUPPORTED


def test_workspace_arguments():
    lib = _native.load()
    size, split_bytes = lib.ttk_linear_f32_workspace_size, lib.ttk_linear_f32_split_bytes
    assert size(32, 64, 64) == size(256, 1024, 256) == 0  # small products read W alone
    assert size(8192, 4096, 1024) == split_bytes(4096, 1024)
    assert size(0, 64, 64) == size(-1, 64, 64) == size(1 << 31, 64, 64) == size(64, 64, 1 << 22) == 0

    # Few tiles of long K: sums of 2 to 32 workgroups a tile, 4096 bytes to 32 x 32 results.
    for m, n, k in ((16, 2048, 8192), (1, 4, 1024), (128, 2048, 8192), (64, 1024, 4096)):
        need = size(m, n, k)
        tiles32, tiles64 = -(-m // 32) * -(-n // 32), -(-m // 64) * -(-n // 64)
        assert any(need % t == 0 and 2 <= need // t <= 32 for t in (tiles32 * 4096, tiles64 * 16384))

    # One tile more than a launch takes workgroups goes to the persistent grid,
    # however little work a tile has (the rule alone: nothing is launched).
    last = (2 ** 32 - 1) // 512 - 8
    for rows in (32 * last + 1, 64 * last + 1, (1 << 31) - 1):
        assert size(rows, 4, 32) == split_bytes(4, 32)

    def call(**over):
        m, n, k = 8192, 4096, 1024
        a = dict(x=1 << 30, w=2 << 30, b=None, y=3 << 30, M=m, N=n, K=k, ws=4 << 30, bytes=split_bytes(n, k))
        a.update(over)
        return lib.ttk_linear_f32_fwd_ws(a["x"], a["w"], a["b"], a["y"], a["M"], a["N"], a["K"], a["K"], a["K"], a["N"],
                                         _native.TTK_ACT_NONE, a["ws"], a["bytes"], None)

    for over, status, message in (
        (dict(ws=None), _native.TTK_EINVAL, "NULL"),
        (dict(bytes=split_bytes(4096, 1024) - 1), _native.TTK_EINVAL, "must hold"),
        (dict(ws=(4 << 30) + 8), _native.TTK_EUNSUPPORTED, "16-byte aligned"),
        (dict(ws=(2 << 30) + 16), _native.TTK_EINVAL, "overlaps w"),
        (dict(ws=(1 << 30) + 16), _native.TTK_EINVAL, "overlaps an input"),
        (dict(b=(4 << 30) + 32), _native.TTK_EINVAL, "overlaps an input"),
        (dict(y=(4 << 30) + 32), _native.TTK_EINVAL, "y overlaps"),
        (dict(M=16, N=2048, K=8192, ws=None, bytes=1 << 24), _native.TTK_EINVAL, "NULL"),
        (dict(M=16, N=2048, K=8192, bytes=size(16, 2048, 8192) - 1), _native.TTK_EINVAL, "must hold"),
        (dict(M=16, N=2048, K=8192, ws=(3 << 30) + 16), _native.TTK_EINVAL, "y overlaps"),
        (dict(M=0), _native.TTK_OK, ""),
    ):
        assert call(**over) == status
        assert message in _native.last_error()


def test_m0_is_only_written_by_the_inline_copies(tmp_path):
    in_asm, inside, outside = False, 0, 0
    for line in _assembly(CSRC / "linear_f32_fwd.hip", tmp_path).splitlines():
        text = line.strip()
        if text.startswith(";;#ASM"):
            in_asm = text.startswith(";;#ASMSTART")
        elif not text.startswith(";") and "m0" in text.replace(",", " ").split():
            inside, outside = inside + in_asm, outside + (not in_asm)
    assert inside > 0 and outside == 0
