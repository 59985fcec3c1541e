"""Where the experts' product of many rows reads its weights (csrc/grouped.hip), worked out on the host: every read lies inside
the expert and on the row and piece it stands for, also where columns or k end inside a workgroup's, and past the columns
nothing is read at all."""
import ctypes

import pytest

from dinfer_amd.kernels import lib


def byte():
    fn = lib.load_library("grouped").dinfer_experts_weights_byte
    fn.argtypes, fn.restype = [ctypes.c_int, ctypes.c_int, ctypes.c_int64] + [ctypes.c_int] * 6, ctypes.c_int64
    return fn


# columns: one past a workgroup's, waves wholly past the end, whole workgroups; k: one piece, a step and a piece, part of a step
@pytest.mark.parametrize("gated,N", [(0, 1), (0, 40), (0, 257), (0, 1409), (0, 256), (1, 24), (1, 129), (1, 128), (1, 1409)])
@pytest.mark.parametrize("K,ldw", [(8, 8), (72, 72), (200, 208), (128, 128)])
def test_reads_stay_inside_the_expert(gated, N, K, ldw):
    fn, rows = byte(), 2 * N if gated else N
    cols = 32 if gated else 64                                  # of a wave; a workgroup has four
    for c0 in range(max(0, N // (4 * cols) - 1) * 4 * cols, -(-N // (4 * cols)) * 4 * cols, cols):
        for k0 in range(0, K + 64, 64):                         # (the last: what is asked for ahead of a step that is not there)
            for j in range(2):
                for r in range(4):
                    for lane in range(64):
                        at = fn(gated, N, ldw, K, c0, j, r, lane, k0)
                        n = c0 + (0 if gated else 32 * j) + 16 * (lane >> 2 & 1) + 4 * (lane >> 3 & 3) + r
                        k = min(k0 + 8 * (4 * (lane >> 5) + (lane & 3)), K - 8)
                        if n >= N:
                            assert at == -1
                        else:
                            row = n + N * j if gated else n
                            assert row < rows and at == 2 * (row * ldw + k) and at + 16 <= 2 * rows * ldw
