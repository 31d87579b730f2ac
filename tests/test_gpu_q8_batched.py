"""GPU parity: fkv_gemm_q8_0_batched (Q8_0 GEMM of a token batch on the matrix cores).

The bar is the reference's own one between its backends, bit-identity
(crates/kernels/src/tests.rs:770-830, bits_eq on Q8_0 gemm): every output equals the
oracle's fo_q8_gemm (dot_q8_row_q8_act, q8_dot.rs:72-109, pinned in
test_cpu_oracle_q8_gemm.py) and fkv_gemm_q8_0's GEMV result, bit for bit, on:
- token counts on and off the 16-token MFMA tile and the 64-token workgroup, row counts
  off the 16-row tile, the Llama-3-8B projection shapes of a 64-sequence decode batch;
- several matrices sharing the activation in one launch;
- non-finite and extreme activations and weight scales;
- the calls the matrix-core path does not take (fewer than 8 tokens, columns off a
  multiple of 64, weights not 4-byte aligned, launches that the GEMV runs at once), which
  run the GEMV; which of the two a call took is seen by its workspace, which the GEMV
  leaves alone;
and a workspace that is too small is rejected before anything runs, or, for widths off a
multiple of 1024 and weights off 16 bytes, makes the call a GEMV.
"""
import numpy as np
import pytest

from oracle import ref
from tests.test_gpu_q8_gemm import _dev, _same, _weights

pytestmark = pytest.mark.gpu


def _batched(ws, rows, cols, x, offset=0, workspace=None):
    """fkv_gemm_q8_0_batched through ferrum_amd; each weight placed `offset` bytes into
    its device buffer."""
    import torch
    import ferrum_amd as fa
    n_tokens = x.shape[0]
    wd = []
    for w in ws:
        buf = torch.zeros(w.size + offset + 16, dtype=torch.uint8, device="cuda")
        buf[offset:offset + w.size] = _dev(w)
        wd.append(buf[offset:offset + w.size])
    ys = [torch.full((n_tokens, r), 3.0, dtype=torch.float32, device="cuda") for r in rows]
    fa.gemm_q8_0_batched(wd, rows, cols, _dev(x.astype(np.float32)), n_tokens, ys,
                         workspace=workspace)
    torch.cuda.synchronize()
    return [y.cpu().numpy() for y in ys]


def _gemv(w, rows, cols, x):
    import torch
    import ferrum_amd as fa
    y = torch.full((x.shape[0], rows), 5.0, dtype=torch.float32, device="cuda")
    fa.gemm_q8_0(_dev(w), rows, cols, _dev(x), x.shape[0], y)
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("rows,cols,n_tokens", [
    (16, 1024, 8), (16, 1024, 16), (33, 1024, 17), (48, 2048, 63), (40, 1024, 64),
    (17, 3072, 65), (64, 2048, 200), (1, 1024, 8), (40, 4096, 37), (4100, 2048, 50),
    (16400, 2048, 40),
    # on the matrix cores, off and on their tiles of rows and tokens
    (3073, 1024, 8), (3088, 2048, 9), (1569, 1024, 16), (1456, 3072, 17), (801, 1024, 31),
    (784, 1024, 32), (736, 4096, 33), (513, 1024, 48), (399, 2048, 63), (385, 1024, 64),
    (400, 3072, 65), (129, 2048, 200), (4097, 1024, 8), (17, 1024, 770),
    # one to four token tiles a workgroup with 8 groups loaded ahead, an odd number of runs
    (3100, 8704, 16), (1600, 8704, 32), (3090, 8704, 40), (3090, 8704, 64),
    (16400, 1024, 8), (20500, 1024, 20), (16400, 1024, 40),  # with spare LDS
])
def test_matches_oracle_and_gemv(rows, cols, n_tokens):
    rng = np.random.default_rng(rows * 131 + cols + n_tokens)
    w = _weights(rng, rows, cols)
    x = (rng.standard_normal((n_tokens, cols)) *
         rng.choice([1e-4, 1.0, 300.0], (n_tokens, 1))).astype(np.float32)
    got, = _batched([w], [rows], cols, x)
    _same(got, ref.q8_gemm(w, rows, cols, x))
    _same(got, _gemv(w, rows, cols, x))


@pytest.mark.parametrize("rows,cols", [(4096, 4096), (1024, 4096), (14336, 4096),
                                       (4096, 14336)])
def test_llama3_8b_shapes_decode_batch(rows, cols):
    """attn_q/attn_output, attn_k/attn_v, ffn_gate/up and ffn_down of a 64-sequence
    decode step (C2's batch), against the GEMV bit for bit."""
    rng = np.random.default_rng(rows ^ cols)
    w = _weights(rng, rows, cols)
    x = rng.standard_normal((64, cols)).astype(np.float32)
    got, = _batched([w], [rows], cols, x)
    _same(got, _gemv(w, rows, cols, x))
    sel = rng.choice(rows, 24, replace=False)  # and a sample of rows against the oracle
    wr = w.reshape(rows, -1)[sel].reshape(-1)
    _same(got[:, sel], ref.q8_gemm(wr, sel.size, cols, x))


@pytest.mark.parametrize("shapes", [[64, 16, 0, 33], [640, 160, 0, 33]])  # GEMV, matrix cores
def test_several_matrices_one_launch(shapes):
    """q/k/v of one activation: each output is its own call's, with an empty matrix in
    the middle of the batch."""
    rng = np.random.default_rng(77)
    cols, n_tokens = 2048, 40
    ws = [_weights(rng, r, cols) if r else np.zeros(0, np.uint8) for r in shapes]
    x = rng.standard_normal((n_tokens, cols)).astype(np.float32)
    ys = _batched(ws, shapes, cols, x)
    for r, w, y in zip(shapes, ws, ys):
        if r:
            _same(y, ref.q8_gemm(w, r, cols, x))


@pytest.mark.parametrize("rows", [40, 1301])  # GEMV, matrix cores
def test_non_finite_and_extreme_inputs(rows):
    rng = np.random.default_rng(12)
    cols = 1024
    w = _weights(rng, rows, cols, special=True)
    x = rng.standard_normal((20, cols)).astype(np.float32)
    x[0, 3] = np.nan
    x[1, 70] = np.inf
    x[2, 64:96] = 0.0
    x[2, 100] = -np.inf
    x[3, :32] = np.float32(1e-40)
    x[3, 32:64] = np.float32(3e38)
    x[19, 1000] = np.nan
    want = ref.q8_gemm(w, rows, cols, x)
    assert np.isnan(want).any() and np.isfinite(want).any()
    got, = _batched([w], [rows], cols, x)
    _same(got, want)


@pytest.mark.parametrize("rows,cols,n_tokens", [
    ([16385], 1024, 48),              # 257 workgroups: 16 x 16 tiles
    ([28673], 1024, 48),              # 449, one row past the last row tile: 32 x 32
    ([28673], 1024, 33),              # the fewest tokens
    ([28673], 1024, 32),              # and one fewer: 16 x 16 tiles
    ([12289], 1024, 33),              # up to 256, past 192
    ([8200], 2048, 65),               # one token past a tile: 16 x 16 tiles,
    ([14400], 1024, 65),              # and of more rows 32 x 32
    ([4032, 64, 1], 1024, 256),       # three matrices, whole tiles and one row
    ([5056, 64, 1], 1024, 256),
    ([4100], 3072, 250), ([5200], 3072, 250),
])
def test_large_launches(rows, cols, n_tokens):
    """Launches of 256 workgroups of 64 x 64 outputs or more, on either side of the line
    between the two kernels, non-finite scales among the weights and activations: every
    output is the oracle's."""
    rng = np.random.default_rng(cols + n_tokens)
    ws = [_weights(rng, r, cols, special=True) for r in rows]
    x = (rng.standard_normal((n_tokens, cols)) *
         rng.choice([1e-4, 1.0, 300.0], (n_tokens, 1))).astype(np.float32)
    x[1, 70], x[2, 100], x[3, 3], x[4, 32:64] = np.inf, -np.inf, np.nan, 3e38
    for r, w, y in zip(rows, ws, _batched(ws, rows, cols, x)):
        _same(y, ref.q8_gemm(w, r, cols, x))


@pytest.mark.parametrize("rows,cols,n_tokens,offset", [
    (17, 64, 8, 0),        # one pair of blocks
    (33, 192, 16, 4),      # an odd number of pairs, weights 4 mod 16
    (16, 448, 17, 8),      # a partial last group of blocks
    (50, 576, 33, 12),     # one pair past 16 blocks
    (2048, 5632, 11, 0),
    (16400, 320, 70, 4),   # 32 x 32 tiles, an odd number of pairs
    # the same widths in launches large enough for the matrix cores
    (3080, 64, 8, 0), (1569, 192, 16, 4), (1456, 448, 17, 8), (752, 576, 33, 12),
    (2070, 5632, 11, 0), (3090, 8256, 16, 4), (3090, 8256, 40, 8), (16400, 320, 9, 4),
    (20500, 320, 20, 0),
    # 32 x 32 tiles of one and two chunks of blocks, whole and not
    (8200, 64, 70, 12), (8200, 128, 70, 8), (8200, 192, 70, 0), (8200, 256, 70, 4),
])
def test_columns_off_1024(rows, cols, n_tokens, offset):
    """Any multiple of 64 columns and 4-byte aligned weights, non-finite scales among them;
    the same bits through the GEMV when the workspace is too small."""
    import ferrum_amd as fa
    rng = np.random.default_rng(rows + cols + n_tokens)
    w = _weights(rng, rows, cols, special=True)
    x = (rng.standard_normal((n_tokens, cols)) *
         rng.choice([1e-4, 1.0, 300.0], (n_tokens, 1))).astype(np.float32)
    x[1, 40], x[2, cols - 1], x[3, 3] = np.inf, -np.inf, np.nan
    want = ref.q8_gemm(w, rows, cols, x)
    assert fa.gemm_q8_0_batched_workspace_bytes(cols, n_tokens) > 0
    _same(_batched([w], [rows], cols, x, offset=offset)[0], want)
    import torch
    small = torch.empty(16, dtype=torch.uint8, device="cuda")
    _same(_batched([w], [rows], cols, x, offset=offset, workspace=small)[0], want)


@pytest.mark.parametrize("rows,cols,n_tokens,offset,matrix_cores", [
    (20, 1024, 7, 0, False),       # too few tokens
    (20, 544, 30, 0, False),       # columns off a multiple of 64
    (1600, 544, 30, 0, False),
    (20, 1024, 30, 2, False),      # weights 2 mod 4
    (1600, 1024, 30, 2, False),
    (20, 1024, 30, 8, False),      # the GEMV's workgroups all at once
    (1600, 1024, 30, 8, True),
    (3072, 1024, 8, 0, False),     # 768 of them, three a CU
    (3073, 1024, 8, 0, True),      # and one more of rows
    (48, 576, 510, 4, False),      # 765 in 255 slices of tokens
    (48, 576, 513, 4, True),
    (256, 14336, 64, 0, False),    # two of them fill a CU's LDS: 512
    (256, 14336, 65, 0, True),
])
def test_which_calls_the_matrix_cores_take(rows, cols, n_tokens, offset, matrix_cores):
    import torch
    import ferrum_amd as fa
    rng = np.random.default_rng(rows + cols + n_tokens + offset)
    w = _weights(rng, rows, cols)
    x = rng.standard_normal((n_tokens, cols)).astype(np.float32)
    size = max(fa.gemm_q8_0_batched_workspace_bytes(cols, n_tokens), 1 << 20)
    ws = torch.full((size,), 0x5a, dtype=torch.uint8, device="cuda")
    got, = _batched([w], [rows], cols, x, offset=offset, workspace=ws)
    _same(got, ref.q8_gemm(w, rows, cols, x))
    assert bool((ws != 0x5a).any()) == matrix_cores


def test_workspace_size_and_rejection():
    import torch
    import ferrum_amd as fa
    assert fa.gemm_q8_0_batched_workspace_bytes(4096, 7) == 0
    assert fa.gemm_q8_0_batched_workspace_bytes(544, 64) == 0
    need = fa.gemm_q8_0_batched_workspace_bytes(4096, 64)
    assert need == 4 * 128 * 16 * 32 + 4 * 128 * 16 * 4
    rng = np.random.default_rng(1)
    w = _dev(_weights(rng, 16, 4096))
    x = _dev(rng.standard_normal((64, 4096)).astype(np.float32))
    y = torch.full((64, 16), 5.0, dtype=torch.float32, device="cuda")
    small = torch.empty(need - 16, dtype=torch.uint8, device="cuda")
    with pytest.raises(fa.InvalidRequest, match="^gemm workspace too small$"):
        fa.gemm_q8_0_batched([w], [16], 4096, x, 64, [y], workspace=small)
    torch.cuda.synchronize()
    assert np.all(y.cpu().numpy() == 5.0)


@pytest.mark.parametrize("cols,refused", [(576, False), (1024, True)])
def test_workspaces_through_the_c_abi(cols, refused):
    """NULL, too small and misaligned: refused where columns are a multiple of 1024, a GEMV
    elsewhere (the workspace untouched), and the matrix cores with one that does."""
    import ctypes
    import torch
    from ferrum_amd import _lib
    lib = _lib.load()
    rows, n_tokens = 1600, 30
    rng = np.random.default_rng(cols)
    w = _weights(rng, rows, cols)
    x = rng.standard_normal((n_tokens, cols)).astype(np.float32)
    want = ref.q8_gemm(w, rows, cols, x)
    wd, xd = _dev(w), _dev(x)
    need = ctypes.c_uint64()
    assert lib.fkv_gemm_q8_0_batched_workspace_size(cols, n_tokens, ctypes.byref(need)) == 0
    need = need.value
    ws = torch.full((need + 16,), 0x5a, dtype=torch.uint8, device="cuda")
    for ptr, size, error in [(None, 0, "too small"), (None, need, "too small"),
                             (ws.data_ptr(), need - 1, "too small"),
                             (ws.data_ptr() + 4, need, "must be 16-byte aligned"),
                             (ws.data_ptr(), need, None)]:
        y = torch.full((n_tokens, rows), 5.0, dtype=torch.float32, device="cuda")
        one = lambda t, v: (t * 1)(v)
        st = lib.fkv_gemm_q8_0_batched(
            1, one(ctypes.c_void_p, wd.data_ptr()), one(ctypes.c_uint64, wd.numel()),
            one(ctypes.c_uint64, rows), cols, xd.data_ptr(), xd.numel(), n_tokens,
            one(ctypes.c_void_p, y.data_ptr()), one(ctypes.c_uint64, y.numel()), ptr, size,
            torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        if error and refused:
            assert st == _lib.FKV_ERR_INVALID
            assert lib.fkv_last_error().decode() == "gemm workspace " + error
            assert bool((y == 5.0).all())
        else:
            assert st == 0
            _same(y.cpu().numpy(), want)
        assert bool((ws != 0x5a).any()) == (error is None)


@pytest.mark.parametrize("case", range(20))
def test_randomized_batches_against_oracle_and_gemv(case):
    """Seeded random launches: 1 to 4 matrices (an empty one possible) sharing an
    activation, row counts from 1 to ~5,000, columns 64 to 6,144 in multiples of 64, weights
    at 0, 4, 8 or 12 mod 16, 8 to 150 tokens with activation rows of widely different
    scales; every output against the GEMV bit for bit and a sample of rows against the
    oracle bit for bit."""
    rng = np.random.default_rng(4000 + case)
    cols = int(rng.choice([1024, 2048, 3072, 4096, 6144]) if case % 2 else 64 * rng.integers(1, 97))
    offset = int(rng.choice([0, 4, 8, 12]))
    n_tokens = int(rng.integers(8, 151))
    nm = int(rng.integers(1, 5))
    rows = [int(rng.choice([0, 1, 15, 16, 17, int(rng.integers(1, 300)), int(rng.integers(300, 5000))]))
            for _ in range(nm)]
    if not any(rows):
        rows[0] = 33
    if case % 4:  # three in four past the launches that run as a GEMV
        rows[-1] += 16 * (1664 // n_tokens)
    ws = [_weights(rng, r, cols) if r else np.zeros(0, np.uint8) for r in rows]
    x = (rng.standard_normal((n_tokens, cols)) *
         rng.choice([1e-3, 1.0, 50.0], (n_tokens, 1))).astype(np.float32)
    ys = _batched(ws, rows, cols, x, offset=offset)
    for r, w, y in zip(rows, ws, ys):
        if not r:
            continue
        _same(y, _gemv(w, r, cols, x))
        sel = np.unique(rng.integers(0, r, min(r, 24)))
        wr = w.reshape(r, -1)[sel].reshape(-1)
        _same(y[:, sel], ref.q8_gemm(wr, sel.size, cols, x))
