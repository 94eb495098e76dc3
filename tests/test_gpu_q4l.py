"""GPU o_proj over Q4_L weights (lnskv_q4l_gemv_accumulate) against the
float64 oracle: y_in + W x for every vector, within 2e-6 of
sum_c |W[r][c] x[c]| + |y_in| (f32 sums of exact f16 x f16 products: ~cols/32
f32 roundings of the sub-block partial sums, x split into two f16 parts
rounded toward zero, to 2^-20; measured at most 1.8e-7 at 4096 columns.
Dropping the lo part of x would give ~2^-11).  Shapes cover one vector, odd counts, row counts that
are not multiples of 16, padded strides, more than 64 vectors (the other kernel),
the Llama-3-8B o_proj shape at batch 32 and wider rows whose waves take two
blocks each (the next block's weights arriving during the products); every
call gives the same bits, and the padding of y is not written."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import say
from lnskv.device import Q4LMatrix, sync

pytestmark = pytest.mark.gpu


def _disk(rng, rows, cols):
    n = rows * (cols // 256)
    d = rng.integers(0, 256, (n, O.Q4L_DISK_BYTES), dtype=np.uint8)
    g = np.exp2(rng.uniform(-12, -2, n)).astype(np.float16)  # scale_global ~ max |w| of a block
    g[::13] = np.float16(3.0e-5)                             # f16 subnormal global scales
    d[:, 0:2] = g.view(np.uint8).reshape(n, 2)
    return d.reshape(-1)


@pytest.mark.parametrize("rows,cols,n_vec,xpad,ypad", [
    (16, 256, 1, 0, 0),
    (37, 512, 3, 4, 3),
    (64, 1024, 8, 0, 0),
    (100, 2048, 13, 8, 5),
    (48, 512, 70, 0, 0),
    (4096, 4096, 32, 0, 0),
    (2048, 8192, 3, 0, 0),    # split launch, two blocks per wave (one vector tile)
    (4096, 8192, 24, 4, 0),   # split launch, two blocks per wave (two vector tiles)
    (512, 4096, 70, 0, 3),    # more than 64 vectors, split over four workgroups per tile
])
def test_q4l_gemv_accumulate(gpu, rows, cols, n_vec, xpad, ypad):
    say("q4l gemv", rows, cols, n_vec, xpad, ypad)
    rng = np.random.default_rng(rows + cols + n_vec)
    disk = _disk(rng, rows, cols)
    W = Q4LMatrix(disk, rows, cols, gpu)
    x = rng.standard_normal((n_vec, cols + xpad)).astype(np.float32)
    y0 = rng.standard_normal((n_vec, rows + ypad)).astype(np.float32)
    xd = torch.from_numpy(x).to(gpu)[:, :cols] if xpad == 0 else torch.from_numpy(x).to(gpu)
    yd = torch.from_numpy(y0).to(gpu)
    W.gemv_accumulate(xd, yd)
    sync()
    got = yd.cpu().numpy()
    dev = W.blocks.cpu().numpy()
    assert np.array_equal(dev, O.q4l_prepare(disk))
    ref = O.q4l_gemv_f64(dev, x[:, :cols], y0[:, :rows], rows, cols)
    wabs = np.abs(O.q4l_decode_matrix(dev, rows, cols).astype(np.float64))
    bound = 2e-6 * (np.abs(x[:, :cols]).astype(np.float64) @ wabs.T + np.abs(y0[:, :rows])) + 1e-30
    err = np.abs(got[:, :rows] - ref)
    say("max err / bound", float((err / bound).max()))
    assert np.all(err <= bound)
    assert np.array_equal(got[:, rows:], y0[:, rows:])  # padding untouched
    # the same bits on a second call
    yd2 = torch.from_numpy(y0).to(gpu)
    W.gemv_accumulate(xd, yd2)
    sync()
    assert torch.equal(yd2, yd)


PART_BYTES = 64 * 128 * 4  # a workgroup's partial sums in a split launch of more than 64 vectors


def _split_parts(W, x, y, gpu):
    """y += W x with a caller's workspace whose partial area holds a NaN
    pattern: the PART_BYTES pieces that the call wrote (workgroups per tile
    times tiles; 0 when it did not split).  Its arrival counts are left zero."""
    from lnskv import _lib
    ws = torch.full((_lib.WORKSPACE_HEADER_BYTES + 256 * PART_BYTES,), 0xFF, dtype=torch.uint8, device=gpu)
    ws[:_lib.WORKSPACE_HEADER_BYTES] = 0
    assert W.workspace_size(x.shape[0]) <= ws.numel()
    W.gemv_accumulate(x, y, ws)
    sync()
    assert int(ws[:_lib.WORKSPACE_HEADER_BYTES].count_nonzero()) == 0
    return int((ws[_lib.WORKSPACE_HEADER_BYTES:].view(-1, PART_BYTES) != 0xFF).any(1).sum())


@pytest.mark.parametrize("rows,cols,n_vec,split", [
    (1, 256, 65, 1),        # one row, one block: a tile of 128 rows and one of 64 vectors nearly empty
    (127, 512, 128, 1),     # one row short of a tile, whole vector tiles
    (128, 768, 129, 1),     # a whole row tile, one vector in the last tile, an odd count of blocks
    (129, 2048, 100, 2),    # two workgroups of 4 blocks per tile
    (300, 5120, 191, 5),    # five workgroups of 4 blocks per tile
    (300, 5632, 191, 5),    # the last of five with 2 blocks, the others with 5
    (16, 4096, 65, 4),      # one row group: the blocks limit the split
    (2100, 1280, 257, 1),
    (4096, 4096, 100, 4),   # 64 tiles: one workgroup per CU limits the split
])
def test_q4l_many_vectors(gpu, rows, cols, n_vec, split):
    """More than 64 vectors (tiles of 64 vectors x 128 rows, a row's blocks
    split over `split` workgroups): every vector within the bound of
    test_q4l_gemv_accumulate at the tiles' edges, padded strides, the padding of
    y untouched, the vectors of one call as the calls of up to 64 give them,
    within both bounds, and a caller's workspace the bits of the library's
    buffer.  Vectors differ in scale by 2^10, the smallest ~2^-4: x in two f16
    parts is off by up to 2^-25 however small it is, 5e-7 of a vector of 2^-4."""
    say("q4l many vectors", rows, cols, n_vec)
    rng = np.random.default_rng(rows + cols + n_vec)
    disk = _disk(rng, rows, cols)
    W = Q4LMatrix(disk, rows, cols, gpu)
    x = (rng.standard_normal((n_vec, cols + 4)) * np.exp2(rng.uniform(-4, 6, (n_vec, 1)))).astype(np.float32)
    y0 = rng.standard_normal((n_vec, rows + 3)).astype(np.float32)
    xd, yd = torch.from_numpy(x).to(gpu), torch.from_numpy(y0).to(gpu)
    W.gemv_accumulate(xd, yd)
    few = torch.from_numpy(y0).to(gpu)
    for v in range(0, n_vec, 64):
        W.gemv_accumulate(xd[v:v + 64], few[v:v + 64])
    sync()
    got = yd.cpu().numpy()
    dev = W.blocks.cpu().numpy()
    ref = O.q4l_gemv_f64(dev, x[:, :cols], y0[:, :rows], rows, cols)
    wabs = np.abs(O.q4l_decode_matrix(dev, rows, cols).astype(np.float64))
    bound = 2e-6 * (np.abs(x[:, :cols]).astype(np.float64) @ wabs.T + np.abs(y0[:, :rows])) + 1e-30
    err = np.abs(got[:, :rows] - ref)
    say("max err / bound", float((err / bound).max()))
    assert np.all(err <= bound)
    assert np.all(np.abs(got[:, :rows] - few.cpu().numpy()[:, :rows]) <= 2 * bound)
    assert np.array_equal(got[:, rows:], y0[:, rows:])
    own = torch.from_numpy(y0).to(gpu)
    tiles = ((rows + 127) // 128) * ((n_vec + 63) // 64)
    assert _split_parts(W, xd, own, gpu) == (split * tiles if split > 1 else 0)
    assert torch.equal(own, yd)


def test_q4l_many_vectors_small_workspace(gpu):
    """A workspace below lnskv_q4l_workspace_size that holds what launches of 64
    vectors at a time would use (4096 x 4096: 4 workgroups for each of 64 row
    groups of 64 rows, 16 KiB each) is taken, with fewer workgroups per tile;
    so is a library buffer of that size under capture.  One below is refused
    and leaves y as it was."""
    from lnskv import _lib
    from lnskv._lib import check, lib
    say("q4l many vectors, small workspace")
    rng = np.random.default_rng(31)
    rows, cols, n_vec = 4096, 4096, 100
    W = Q4LMatrix(_disk(rng, rows, cols), rows, cols, gpu)
    x = torch.from_numpy(rng.standard_normal((n_vec, cols)).astype(np.float32)).to(gpu)
    y0 = torch.from_numpy(rng.standard_normal((n_vec, rows)).astype(np.float32)).to(gpu)
    least = _lib.WORKSPACE_HEADER_BYTES + 4 * 64 * 16384
    assert least < W.workspace_size(n_vec)
    ws = torch.zeros(least, dtype=torch.uint8, device=gpu)
    want = y0.clone()
    W.gemv_accumulate(x, want, ws)
    y = y0.clone()
    with pytest.raises(RuntimeError, match="workspace"):
        W.gemv_accumulate(x, y, ws[:least - 16])
    sync()
    assert torch.equal(y, y0)
    ref = y0.double() + x.double() @ torch.from_numpy(
        O.q4l_decode_matrix(W.blocks.cpu().numpy(), rows, cols)).to(gpu).double().t().contiguous()
    assert float((want.double() - ref).norm() / ref.norm()) < 6e-7
    check(lib().lnskv_workspace_release())
    check(lib().lnskv_workspace_reserve(0, 0, least))
    sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        W.gemv_accumulate(x, y)
    for rep in range(3):
        y.copy_(y0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), rep
    del g
    torch.cuda.synchronize()
    check(lib().lnskv_workspace_release())


@pytest.mark.parametrize("n_vec", [64, 65])
def test_q4l_x_past_f16_range(gpu, n_vec):
    """|x| above 65504, which a nearest-even hi part would make infinite: hi is
    65504 and lo the rest, both exact here (multiples of 32), so the bound of
    test_q4l_gemv_accumulate holds on both sides of the kernels' dividing line."""
    say("q4l large x", n_vec)
    rng = np.random.default_rng(n_vec)
    rows, cols = 130, 512
    disk = _disk(rng, rows, cols)
    W = Q4LMatrix(disk, rows, cols, gpu)
    x = rng.choice(np.array([65536.0, -65536.0, 98304.0, -131008.0, 1.0], np.float32), (n_vec, cols))
    yd = torch.zeros((n_vec, rows), device=gpu)
    W.gemv_accumulate(torch.from_numpy(x).to(gpu), yd)
    sync()
    dev = W.blocks.cpu().numpy()
    ref = O.q4l_gemv_f64(dev, x, np.zeros((n_vec, rows), np.float32), rows, cols)
    wabs = np.abs(O.q4l_decode_matrix(dev, rows, cols).astype(np.float64))
    assert np.all(np.abs(yd.cpu().numpy() - ref) <= 2e-6 * (np.abs(x).astype(np.float64) @ wabs.T) + 1e-30)


@pytest.mark.parametrize("n_vec", [64, 65])
def test_q4l_scale_past_f16_range(gpu, n_vec):
    """Effective scales that overflow f16 (a global scale of 65504 with a local
    scale above 7) are infinite: where x and the weights of a row are positive
    its sum is +inf, and -inf with the global scale's sign turned, zero codes,
    finite sub-blocks of the same row and x that is one f16 (no lo part)
    notwithstanding, on both sides of the kernels' dividing line; a NaN scale
    gives NaN; the other rows stay within the bound of
    test_q4l_gemv_accumulate."""
    say("q4l infinite scales", n_vec)
    rng = np.random.default_rng(n_vec)
    rows, cols = 130, 512
    disk = _disk(rng, rows, cols).reshape(rows, cols // 256, O.Q4L_DISK_BYTES)
    disk[:, :, 6:] &= 0x77                                            # positive weights, zero codes among them
    local = np.array([0x3F, 0x00, 0x70, 0x08], np.uint8)              # sub-blocks 0 and 6 infinite, the others finite
    for at, g in ((0, 65504.0), (2, -65504.0)):
        disk[at::9, 1, 0:2] = np.array([g], np.float16).view(np.uint8)
        disk[at::9, 1, 2:6] = local
    disk[4::9, 0, 0:2] = np.array([np.nan], np.float16).view(np.uint8)
    W = Q4LMatrix(disk, rows, cols, gpu)
    x = rng.uniform(0.5, 2.0, (n_vec, cols)).astype(np.float32)
    x[::2] = x[::2].astype(np.float16)
    yd = torch.zeros((n_vec, rows), device=gpu)
    W.gemv_accumulate(torch.from_numpy(x).to(gpu), yd)
    sync()
    got, dev = yd.cpu().numpy(), W.blocks.cpu().numpy()
    assert int(np.isposinf(got[:, 0::9]).sum()) == got[:, 0::9].size
    assert int(np.isneginf(got[:, 2::9]).sum()) == got[:, 2::9].size
    assert int(np.isnan(got[:, 4::9]).sum()) == got[:, 4::9].size
    rest = np.setdiff1d(np.arange(rows), np.r_[0:rows:9, 2:rows:9, 4:rows:9])
    with np.errstate(invalid="ignore"):
        ref = O.q4l_gemv_f64(dev, x, np.zeros((n_vec, rows), np.float32), rows, cols)[:, rest]
    assert np.all(np.abs(got[:, rest] - ref) <= 2e-6 * ref + 1e-30)


def test_q4l_caller_workspace(gpu):
    """A caller's workspace (arrival counts zeroed once) gives the bits of the
    library's buffer, call after call and across shapes that share it (every
    call leaves the counts zero); one too small is refused before any
    launch, leaving y untouched."""
    from lnskv import _lib
    say("q4l caller workspace")
    rng = np.random.default_rng(11)
    shapes = [(4096, 4096, 32), (1000, 2048, 5), (4096, 4096, 64), (300, 5632, 191), (4096, 4096, 100)]
    mats = {}
    need = 0
    for rows, cols, n_vec in shapes:
        mats[(rows, cols)] = Q4LMatrix(_disk(rng, rows, cols), rows, cols, gpu)
        need = max(need, mats[(rows, cols)].workspace_size(n_vec))
    assert need > _lib.WORKSPACE_HEADER_BYTES
    ws = torch.zeros(need, dtype=torch.uint8, device=gpu)
    for rep in range(2):
        for rows, cols, n_vec in shapes:
            W = mats[(rows, cols)]
            x = torch.from_numpy(rng.standard_normal((n_vec, cols)).astype(np.float32)).to(gpu)
            y0 = torch.from_numpy(rng.standard_normal((n_vec, rows)).astype(np.float32)).to(gpu)
            ya, yb = y0.clone(), y0.clone()
            W.gemv_accumulate(x, ya, ws)
            W.gemv_accumulate(x, yb)
            sync()
            assert torch.equal(ya, yb), (rep, rows, cols, n_vec)
    assert int(ws[:_lib.WORKSPACE_HEADER_BYTES].count_nonzero()) == 0
    W = mats[(4096, 4096)]
    # the call's own need (its launch plan) is at most the query's bound; the
    # count header alone holds none of its partial sums
    small = torch.zeros(_lib.WORKSPACE_HEADER_BYTES + 16, dtype=torch.uint8, device=gpu)
    x = torch.ones((32, 4096), device=gpu)
    y = torch.zeros((32, 4096), device=gpu)
    with pytest.raises(RuntimeError, match="workspace"):
        W.gemv_accumulate(x, y, small)
    sync()
    assert int(y.count_nonzero()) == 0


@pytest.mark.parametrize("n_vec", [32, 100])
def test_q4l_graph_replay_library_buffer(gpu, n_vec):
    """lnskv_workspace_reserve grows the library's Q4L buffer (its arrival
    counts zeroed) before a capture; the captured y = y0; y += W x (a split
    launch, 4096 x 4096, of either kernel) then replays with unrelated eager
    work between the replays, each replay equal to the eager call bit for
    bit, so the counts are back at zero after every replay."""
    from lnskv._lib import check, lib
    say("q4l graph replay")
    rng = np.random.default_rng(21)
    rows, cols = 4096, 4096
    W = Q4LMatrix(_disk(rng, rows, cols), rows, cols, gpu)
    check(lib().lnskv_workspace_reserve(0, 0, W.workspace_size(n_vec)))
    x = torch.from_numpy(rng.standard_normal((n_vec, cols)).astype(np.float32)).to(gpu)
    y0 = torch.from_numpy(rng.standard_normal((n_vec, rows)).astype(np.float32)).to(gpu)
    want = y0.clone()
    W.gemv_accumulate(x, want)
    y = torch.empty_like(y0)
    sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y.copy_(y0)
        W.gemv_accumulate(x, y)
    torch.cuda.synchronize()
    scratch = torch.randn(1 << 20, device=gpu)
    for rep in range(4):
        y.zero_()
        g.replay()
        got = y.clone()
        scratch.mul_(1.0001)  # unrelated eager work between replays
        torch.cuda.synchronize()
        assert torch.equal(got, want), rep
