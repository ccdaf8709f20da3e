"""GPU parity of kg_life_u8 (gameoflife on uint8 cells, X mode) against the
oracle's oracle_life_u8, which is itself pinned to a brute-force Conway rule
and to the glider/blinker known answers in test_oracle.py.  Integer work:
tolerance 0 (every byte equal, border bytes of the output untouched)."""
import ctypes as C

import numpy as np
import pytest

import kgspec as K

pytestmark = pytest.mark.gpu

SIZES = [(3, 3), (4, 5), (16, 3), (17, 12), (18, 18), (33, 5), (48, 40), (100, 37),
         (4096, 19), (4113, 9), (8192, 33), (1040, 70),
         # band and segment edges of the vector kernel: 16-row bands, 1024-cell
         # wave segments, 4096-cell workgroups, a last band of one row
         (32, 66), (2064, 100), (1024, 35), (5120, 34), (4112, 67),
         # 150 workgroups: rounds of 8 chunks of 8 bands (128) plus a tail
         (8192, 300), (4096, 600)]


def _oracle_steps(oracle, board, nt, fill=0xAB):
    ny, nx = board.shape
    cur = board.copy()
    for _ in range(nt):
        nxt = np.full_like(cur, fill) if nt == 1 else cur.copy()
        oracle.lib.oracle_life_u8(C.c_int(nx), C.c_int(ny), C.c_void_p(cur.ctypes.data),
                                  C.c_void_p(nxt.ctypes.data))
        cur = nxt
    return cur


def _gpu_steps(ctx, board, nt, fill=0xAB):
    ny, nx = board.shape
    a = ctx.array(board)
    b = ctx.array(np.full_like(board, fill) if nt == 1 else board)
    for _ in range(nt):
        ctx.call("life_u8", nx, ny, a, b)
        a, b = b, a
    ctx.sync()
    out = a.download()
    a.free()
    b.free()
    return out


@pytest.mark.parametrize("dims", SIZES)
def test_life_u8_matches_oracle_ragged(gpu_ctx, oracle, dims):
    nx, ny = dims
    rng = np.random.default_rng(nx * 7 + ny)
    board = (rng.random((ny, nx)) < 0.3).astype(np.uint8)
    # one step into a buffer prefilled with 0xAB: the border must stay 0xAB
    np.testing.assert_array_equal(_gpu_steps(gpu_ctx, board, 1), _oracle_steps(oracle, board, 1),
                                  err_msg=f"life_u8 {dims} one step")
    np.testing.assert_array_equal(_gpu_steps(gpu_ctx, board, 5), _oracle_steps(oracle, board, 5),
                                  err_msg=f"life_u8 {dims} five steps")


def test_life_u8_nonbinary_cells(gpu_ctx, oracle):
    """Any nonzero byte counts as alive (values up to 0xff, including 0x80)."""
    rng = np.random.default_rng(11)
    nx, ny = 4096 + 64, 40
    board = rng.integers(0, 256, (ny, nx), dtype=np.uint8)
    board[rng.random((ny, nx)) < 0.6] = 0
    board[0, :16] = 0x80
    np.testing.assert_array_equal(_gpu_steps(gpu_ctx, board, 1), _oracle_steps(oracle, board, 1))


def test_life_u8_full_size_bernoulli(gpu_ctx, oracle):
    """The X-mode configuration: 8192x8192 cells, Bernoulli p = 0.3, 3 steps."""
    rng = np.random.default_rng(2024)
    board = (rng.random((8192, 8192)) < 0.3).astype(np.uint8)
    np.testing.assert_array_equal(_gpu_steps(gpu_ctx, board, 3), _oracle_steps(oracle, board, 3))


def test_life_u8_glider_translates(gpu_ctx):
    """A glider moves one cell diagonally every 4 generations."""
    nx, ny = 64, 48
    board = np.zeros((ny, nx), np.uint8)
    for (y, x) in [(1, 2), (2, 3), (3, 1), (3, 2), (3, 3)]:
        board[10 + y, 20 + x] = 1
    out = _gpu_steps(gpu_ctx, board, 8)
    np.testing.assert_array_equal(out, np.roll(board, (2, 2), axis=(0, 1)))


def test_life_u8_rejects_bad_arguments(gpu_ctx, kgmod):
    a = gpu_ctx.empty((64,), np.uint8)
    with pytest.raises(kgmod.KGError):
        gpu_ctx.call("life_u8", 8, 8, a, a)
    with pytest.raises(kgmod.KGError):
        gpu_ctx.call("life_u8", 8, 8, None, a)
    b = gpu_ctx.empty((80,), np.uint8)
    with pytest.raises(kgmod.KGError):
        gpu_ctx.call("life_u8", 8, 8, a.ptr + 1, b)


@pytest.mark.parametrize("nx", [20, 21, 31, 33, 47, 1001, 1023, 1025, 1039, 1041, 2047, 4095, 4097, 4101, 5000])
def test_life_u8_row_ends(gpu_ctx, oracle, nx):
    """Rows that end in the middle of a lane's 16 cells: in a wave's first
    lane, its last one and between, one to fifteen cells in, on whole and
    partial bands, the last of which ends with the buffer."""
    for ny in (3, 6, 9, 23):
        cells = np.random.default_rng(nx * ny).integers(0, 2, (ny, nx)).astype(np.uint8)
        for steps in (1, 3):
            np.testing.assert_array_equal(_gpu_steps(gpu_ctx, cells, steps),
                                          _oracle_steps(oracle, cells, steps), err_msg=f"{nx} x {ny}")


@pytest.mark.parametrize("nx,ny", [(20, 6147), (20, 6151), (100, 9001), (257, 7003), (258, 6300), (259, 7003), (20, 1538)])
def test_life_u8_narrow_rows(gpu_ctx, oracle, nx, ny):
    """Ragged rows on either side of the kernels' dividing line: 258 cells and
    6 bands of 4 rows per compute unit (6144 rows on 256 of them)."""
    cells = np.random.default_rng(nx + ny).integers(0, 2, (ny, nx)).astype(np.uint8)
    for steps in (1, 2):
        np.testing.assert_array_equal(_gpu_steps(gpu_ctx, cells, steps), _oracle_steps(oracle, cells, steps))


@pytest.mark.parametrize("nx", [20, 259])
def test_life_u8_rows_past_a_vector_launch(gpu_ctx, oracle, nx):
    """More rows than the vector kernel's work-items in one launch can hold."""
    period, ny = 1024, 2 ** 26 + 1029
    cells = np.random.default_rng(nx).integers(0, 2, (period, nx)).astype(np.uint8)
    a, b = gpu_ctx.empty((ny, nx), np.uint8), gpu_ctx.empty((ny, nx), np.uint8)
    copy = lambda dst, src, n: gpu_ctx.lib.kg_d2d(gpu_ctx.ptr, dst, src, n)  # noqa: E731
    first = gpu_ctx.array(cells)
    assert copy(a.ptr, first.ptr, period * nx) == 0
    rows = period
    while rows < ny:                       # the board repeats every `period` rows
        n = min(rows, ny - rows)
        assert copy(a.ptr + rows * nx, a.ptr, n * nx) == 0
        rows += n
    gpu_ctx.call("life_u8", nx, ny, a, b)
    for y in (1, 2 ** 25 + 7, 2 ** 26 - 40, ny - 81):
        got = np.empty((80, nx), np.uint8)
        assert gpu_ctx.lib.kg_d2h(gpu_ctx.ptr, got.ctypes.data, b.ptr + y * nx, got.nbytes) == 0
        src = cells[np.arange(y - 1, y + 81) % period]
        np.testing.assert_array_equal(got[:, 1:-1], _oracle_steps(oracle, src, 1)[1:-1, 1:-1], err_msg=f"row {y}")
    for t in (a, b, first):
        t.free()


@pytest.mark.parametrize("nx,ny", [(16384, 8200), (11585, 11586)])
def test_life_u8_levels_past_the_caches(gpu_ctx, oracle, nx, ny):
    """Two levels of more than 256 MiB, whole and ragged rows."""
    cells = np.random.default_rng(nx).integers(0, 2, (ny, nx)).astype(np.uint8)
    np.testing.assert_array_equal(_gpu_steps(gpu_ctx, cells, 1), _oracle_steps(oracle, cells, 1))


def test_life_u8_rows_past_the_vector_kernels_offsets(gpu_ctx, oracle):
    """More than 2^24 cells a row: cell by cell, over many tiles side by side."""
    nx, ny = 2 ** 24 + 37, 5
    cells = np.random.default_rng(3).integers(0, 2, (ny, nx)).astype(np.uint8)
    np.testing.assert_array_equal(_gpu_steps(gpu_ctx, cells, 1), _oracle_steps(oracle, cells, 1))
