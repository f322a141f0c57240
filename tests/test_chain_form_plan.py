"""Workspace of the segmented chain form (CPU): what gdn_chunk_fwd_noalloc refuses is still
decided by the buffers without segments, and the backward's workspace covers the forward's."""
import re

import pytest

from avelang_amd import _native

LIMIT = 32 << 20


def _plain(T, Hqk, Hv, K, l2, N=0):
    """Bytes without segments: per (chunk, v-head) G and the Tb, P fragments; with l2norm the
    fp16 K, Q copies per (chunk, qk-head); each buffer rounded up to 256, the two tables too."""
    n = (T + 63 * N) // 64 if N else -(-T // 64)   # (N packed sequences)
    up = lambda x: -(-x // 256) * 256  # noqa: E731
    return (up(4 * N + 4) + 256 + up(n * Hv * 256) + 2 * up(n * Hv * 6144) +
            (2 * up(n * Hqk * 64 * K * 2) if l2 else 0))


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("l2", [0, 1])
@pytest.mark.parametrize("Hqk,Hv", [(1, 2), (2, 4), (4, 8), (16, 16), (16, 32)])
def test_workspace_with_segments(Hqk, Hv, K, l2):
    lib = _native.lib()
    fake = [i << 40 for i in range(1, 6)] + [None, None, 6 << 40, None]
    grown = 0
    for chunks in list(range(1, 200, 7)) + [256, 300, 500, 700, 1000, 2000, 6000]:
        T = 64 * chunks - 3
        plain = _plain(T, Hqk, Hv, K, l2)
        got = lib.gdn_chunk_workspace_bytes(1, T, Hqk, Hv, K, K, 1, 0, l2)
        assert got >= plain
        grown += got > plain
        assert lib.gdn_chunk_bwd_workspace_bytes(1, T, Hqk, Hv, K, K, 1, 0, l2) > got
        if plain > LIMIT:   # (refused before any launch; what is accepted would launch)
            assert lib.gdn_chunk_fwd_noalloc(*fake, 1, T, Hqk, Hv, K, K, 1, 0.1, l2, None) == -4
            assert str(plain) in lib.gdn_last_error().decode()
    assert grown > 0   # some of them do run in segments


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("N", [16, 64, 256, 1024, 4096])
def test_packed_workspace_has_no_room_for_uncut_sequences(N, K):
    """Buffers for the segments that another follows, not for every sequence's last one, and about
    one per compute unit and v-head at most (a segment is its load): many short prompts do not pay
    for a few long ones that they might hold."""
    lib = _native.lib()
    for T in (16384, 262144):
        plain = _plain(T, 16, 32, K, 0, N)
        got = lib.gdn_chunk_workspace_bytes(1, T, 16, 32, K, K, N, 1, 0)
        assert plain <= got <= plain + 2 * 256 * (8 * K * K + 4) + 8 * (N + 1) + 5 * 256


@pytest.mark.parametrize("Hv", list(range(2, 129, 2)))
def test_segments_fill_the_gpu_once(Hv):
    """The first pass over the segments has a workgroup for each one's own contribution and, but
    for a chain's first, its transfer matrix, the last segment apart: no more of them than compute
    units (256 where no GPU is seen), beside which a few more would run alone."""
    T = 64 * 1024
    buffers = (_native.lib().gdn_chunk_workspace_bytes(1, T, Hv, Hv, 128, 128, 1, 0, 0) -
               _plain(T, Hv, Hv, 128, 0)) // (Hv * 8 * 128 * 128)   # segments that another follows
    assert buffers >= 1
    assert Hv * (2 * buffers - 1) <= 256


def _least(lib, entry, B, T, Hqk, Hv, K, N, cu, l2):
    """Bytes that a forward of these sizes cannot do without (from its refusal of none)."""
    fake = [i << 40 for i in range(1, 6)] + [None, None, 6 << 40, (7 << 40) if cu else None]
    assert entry(*fake, B, T, Hqk, Hv, K, K, N, 0.1, l2, None, 0, None) == -4
    return int(re.search(r"workspace needs (\d+) bytes", lib.gdn_last_error().decode()).group(1))


@pytest.mark.parametrize("cu", [0, 1])
@pytest.mark.parametrize("l2", [0, 1])
@pytest.mark.parametrize("save", [0, 1])
@pytest.mark.parametrize("Hqk,Hv,K", [(2, 4, 128), (16, 32, 128), (4, 8, 64)])
def test_a_buffer_for_the_largest_problem_holds_every_smaller_one(Hqk, Hv, K, save, l2, cu):
    """The form that a call takes, and with it the workspace it takes at its best, changes with the
    sizes; what it needs grows with B, T and N, up to what any larger problem's query gave."""
    lib = _native.lib()
    entry, query = ((lib.gdn_chunk_fwd_save, lib.gdn_chunk_bwd_workspace_bytes) if save else
                    (lib.gdn_chunk_fwd, lib.gdn_chunk_workspace_bytes))
    Ts = [1, 64, 500, 2048, 4352, 5184, 5248, 8192, 16384, 40000]
    Ns = [1, 2, 3, 4, 8, 13, 64, 300]
    seen = 0   # problems whose best is over a larger one's
    for i, T in enumerate(Ts):
        for j, N in enumerate(Ns):
            dims = (1, T, Hqk, Hv, K, N) if cu else (N, T, Hqk, Hv, K, N)
            least = _least(lib, entry, *dims, cu, l2)
            best = query(dims[0], T, Hqk, Hv, K, K, N, cu, l2)
            assert least <= best
            for T2, N2 in ((T, Ns[j:]), (Ts[min(i + 1, len(Ts) - 1)], Ns[j:])):
                for n in N2:
                    size = query(1 if cu else n, T2, Hqk, Hv, K, K, n, cu, l2)
                    assert least <= size, (T, N, T2, n)
                    seen += best > size
    assert seen or K == 64 or save or l2
