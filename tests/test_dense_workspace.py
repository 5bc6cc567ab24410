"""Workspace of the dense panels' K split."""
import ctypes as ct


def test_workspace_covers_every_narrower_product(srt):
    """Fewer columns are split further, so the workspace for n columns is the
    most that any width up to n takes, at most 256 tiles of 128 x 128 floats:
    without it a narrower product runs unsplit (1024 x 4096 x 512 in a plan made
    for 1600 columns: 63 us, 49 in one of its own)."""
    need = srt._lib.lib()._ZN3srt28dense_panels_workspace_bytesEiii
    need.restype, need.argtypes = ct.c_size_t, [ct.c_int] * 3
    for panels in (1, 7, 8, 9, 64, 100, 256, 1024, 3000):
        for groups in (1, 4, 5, 16, 31, 64, 256, 4096):
            last = 0
            for n in (1, 64, 128, 129, 256, 300, 512, 1000, 1024, 1600, 2048, 4096, 16384, 1 << 20):
                tiles, stages = -(-panels // 8) * -(-n // 128), -(-groups // 4)
                ranges = max(1, min(32, 256 // tiles, stages))
                ranges = -(-stages // -(-stages // ranges))  # none of them empty
                here = need(panels, groups, n)
                assert here >= last and here <= 256 * 65536
                assert ranges == 1 or here >= ranges * tiles * 65536
                last = here
