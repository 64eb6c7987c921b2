"""The choice of a kernel path and the workspace queries, on the host (no GPU needed): whatever
path a call takes, with or without adapters that ask for their down-projection, the workspace
that the query returned for its sizes is enough."""

import ctypes

import pytest


@pytest.fixture(scope="module")
def lib():
    from solution import _lib

    return _lib.load()


def _weights(shapes, blocksize=64):
    """Descriptors of stacked [rows, cols] weights; the addresses are aligned, and not read."""
    from solution._lib import NF4Weight

    at = 1 << 12
    return (NF4Weight * len(shapes))(*[
        NF4Weight(packed=at, absmax=at, absmax2=at, code2=at, code=at, nested=1, rows=r, cols=c,
                  blocksize=blocksize, blocksize2=256) for r, c in shapes])


FWD, DX, DX_NOALLOC = 0, 1, 2
STATIC_SCRATCH = 64 << 20  # NF4_STATIC_SCRATCH_BYTES
TILED, SMALL, DECODE, ROWS, SKINNY, SKINNY32, DENSE = range(7)


def path(lib, shapes, m, op=FWD, rank=0):
    """(path, bytes of scratch it uses, bytes the query returns)."""
    ws = _weights(shapes)
    scratch = ctypes.c_size_t(0)
    p = lib.nf4_linear_path(m, ws, len(shapes), op, rank, ctypes.byref(scratch))
    query = lib.nf4_linear_dx_workspace if op == DX else lib.nf4_linear_fwd_workspace
    return p, scratch.value, query(m, ws, len(shapes), 0)


@pytest.mark.parametrize("rank", [0, 5, 16, 17, 64])
def test_the_workspace_query_covers_every_forward_path(lib, rank):
    seen = set()
    for rows in [256, 1536, 4608, 16384, 29952, 33792, 35072, 37888, 41024, 52032, 65664, 81920]:
        for k in [256, 1536, 3584, 4992, 8192, 8960, 16384, 18944]:
            for m in [1, 2, 3, 8, 9, 16, 17, 24, 32, 33, 48, 64, 65, 512, 1300]:
                for shapes in ([(rows, k)], [(rows // 2, k)] * 2):
                    p, used, query = path(lib, shapes, m, rank=rank)
                    assert p >= 0 and used <= query, (shapes, m, rank, p, used, query)
                    seen.add(p)
    assert seen == {TILED, DECODE, ROWS, SKINNY, SKINNY32, DENSE}


@pytest.mark.parametrize("op", [FWD, DX])
def test_dense_tiles_are_counted_in_32_bits(lib, op):
    """The dense kernel finds its tile in 32-bit arithmetic (band_tile in nf4_dense.hip: products of
    up to tile rows x bands of about five): no call whose products could wrap takes it."""
    dense = 0
    for n in (12, 16, 18, 20, 22, 23, 24, 25, 26, 28, 30):
        for m in ((1 << n) - 1, 1 << n, 38_000_000):
            for shapes in ([(896, 896), (128, 896), (128, 896)], [(1536, 1536)], [(4864, 896)] * 2,
                           [(896, 4864)], [(3584, 3584), (512, 3584), (512, 3584)]):
                if path(lib, shapes, m, op)[0] != DENSE:
                    continue
                dense += 1
                for tile in (128, 256):
                    mt = -(-m // tile)
                    bands = 1 if mt < 8 else (mt + 2) // 5
                    assert (mt + 1) * bands < 1 << 32, (shapes, m)
    assert dense > 20


def test_noalloc_shares_its_array_only_where_its_fused_plan_would(lib):
    """nf4_linear_dx_noalloc dequantizes into its array only where its fused plan is split and
    uses the array in any case: elsewhere a call has no scratch, so calls may overlap."""
    shapes = ([(1536, 1536), (256, 1536), (256, 1536)], [(3584, 3584), (512, 3584), (512, 3584)],
              [(3584, 3584)], [(1536, 8960)], [(3008, 1536), (64, 1536)], [(8960, 1536)] * 2,
              [(18944, 3584)] * 2)
    seen = set()
    for s in shapes:
        for m in (64, 300, 700, 1025, 1243, 1300, 2048, 2500, 3000, 4096, 6000, 8192):
            p, used, query = path(lib, s, m, DX)
            q, noalloc, _ = path(lib, s, m, DX_NOALLOC)
            assert noalloc <= STATIC_SCRATCH, (s, m)
            if q == DENSE:  # as nf4_linear_dx
                assert p == DENSE and noalloc == used, (s, m)
            elif p == DENSE:
                assert noalloc == 0 or used > STATIC_SCRATCH, (s, m, noalloc)
            elif query <= STATIC_SCRATCH:
                assert noalloc == used, (s, m)
            seen.add((p, q, noalloc > 0))
    assert {(DENSE, TILED, False), (DENSE, DENSE, True), (TILED, TILED, False),
            (TILED, TILED, True)} <= seen


@pytest.mark.parametrize("k", [0, 64, 192, 256, 4096])
@pytest.mark.parametrize("rows", [(0,), (0, 0), (0, 96)])
def test_queries_answer_for_empty_weights(lib, rows, k):
    """No rows or no columns: nothing to launch, and nothing to divide by either."""
    shapes = [(r, k) for r in rows]
    ws = _weights(shapes)
    for m in (1, 2, 3, 16, 17, 20, 32, 33, 64, 65, 600, 3000):
        empty = sum(rows) == 0 or k == 0
        for op in (FWD, DX, DX_NOALLOC):
            p, used, query = path(lib, shapes, m, op)
            assert used <= max(query, STATIC_SCRATCH if op == DX_NOALLOC else 0)
            if empty:
                assert p == -1 and (op == DX or query == 0)


def test_an_empty_reduction_of_few_tokens_is_refused(lib):
    """K = 0 with rows to write: refused before any launch."""
    from solution._lib import NF4_ERR_UNSUPPORTED

    buf = (ctypes.c_uint16 * 4096)()
    at = ctypes.addressof(buf) + 255 & ~255
    for m in (1, 3, 20, 64):
        assert lib.nf4_linear_fwd(at, m, 8, _weights([(32, 0)]), 1, None, None, 0, at, 32, 0, None,
                                  0, None) == NF4_ERR_UNSUPPORTED
