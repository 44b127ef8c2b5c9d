"""Preparing, packing and expanding at the sizes where their kernels change
hands: a row more or less than a wavefront, than a workgroup's turn, row
lengths that are all alike or that fill more bins than a workgroup has threads.
The symbols a form was made from are the reference: they come back whole."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def gpu():
    from qmoe_amd import sub1, sub1_hip
    assert torch.cuda.is_available() and sub1.DEC
    return sub1, sub1_hip


def symbols_of(height, width, shares, seed):
    """uint8 [height, width] on the GPU; row r has a share of about
    shares[r % len(shares)] non-zero symbols."""
    g = torch.Generator().manual_seed(seed)
    share = torch.tensor(shares)[torch.arange(height) % len(shares)][:, None]
    drawn = torch.rand((height, width), generator=g) < share
    return (drawn * torch.randint(1, 3, (height, width), generator=g)).to(torch.uint8).cuda()


def packed(gpu, symbols):
    """(w_comp, row_off) of symbols by the library's encoder."""
    sub1, op = gpu
    row_off = torch.zeros(symbols.shape[0] + 1, dtype=torch.int32, device='cuda')
    return op.sub1pack(sub1.TRIE, symbols.to(torch.int32), row_off), row_off


@pytest.mark.parametrize('height,width,shares', [
    (1, 700, [0.1]), (63, 40, [0.0]), (64, 40, [1.0]), (65, 40, [0.5]),       # equal counts, ties
    (512, 33, [0.0, 1.0]), (513, 33, [0.3]), (1025, 16, [0.1, 0.1, 0.9]),     # a turn of 512 rows, and one more
    (130, 9000, [0.0, 0.01, 0.3, 0.99]),                                      # more bins than threads
    (65534, 3, [0.4])])                                                       # the most rows of a matrix
def test_prepared_rows_come_back_whole(gpu, height, width, shares):
    sub1, op = gpu
    symbols = symbols_of(height, width, shares, seed=height + width)
    w_comp, row_off = packed(gpu, symbols)
    minmax = torch.randn(2 * height, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    prepared = op.PreparedMatrix(sub1.DEC[0], w_comp, row_off, minmax, width)
    assert torch.equal(prepared.decode(), symbols)
    # every row with its own minimum and maximum: the row order took the pairs along.  One
    # activation of 1.0: y is the weight in that column, exactly
    column = width // 2
    x = torch.zeros((1, width), dtype=torch.bfloat16, device='cuda')
    x[0, column] = 1.0
    y = torch.zeros((1, height), dtype=torch.bfloat16, device='cuda')
    prepared.matvec_tokens(x, y)
    values = torch.cat((torch.zeros((height, 1), dtype=torch.bfloat16, device='cuda'), minmax.view(-1, 2)), 1)
    assert torch.equal(y[0], values.gather(1, symbols[:, column:column + 1].long())[:, 0])


def test_preparing_names_a_bad_pointer(gpu):
    """The pointer tables are looked over on the GPU before any of them is
    followed; the message names the matrix."""
    import ctypes
    from qmoe_amd import _lib
    sub1, op = gpu
    lib = _lib.load()
    symbols = symbols_of(64, 64, [0.1], seed=3)
    w_comp, row_off = packed(gpu, symbols)
    minmax = torch.ones(128, dtype=torch.bfloat16, device='cuda')

    def table(pointers):
        return torch.tensor(pointers, dtype=torch.int64, device='cuda')

    good = [table([t.data_ptr()] * 3) for t in (w_comp, row_off, minmax)]
    meta = torch.empty(lib.sub1_moe_prepared_meta_bytes(3, 64, 64), dtype=torch.uint8, device='cuda')
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for at, pointers, status, words in (
            (0, [w_comp.data_ptr(), 0, w_comp.data_ptr()], -1, 'w_comp of matrix 1 is NULL'),
            (1, [row_off.data_ptr()] * 2 + [row_off.data_ptr() + 2], -3, 'row_off of matrix 2')):
        bad = list(good)
        bad[at] = table(pointers)
        layers = _lib.MoeLayers(sub1.DEC[0].data_ptr(), good[0].data_ptr(), bad[0].data_ptr(),
                                good[1].data_ptr(), bad[1].data_ptr(), good[2].data_ptr(),
                                bad[2].data_ptr(), 3, 64, 64)
        out = _lib.MoePrepared()
        assert lib.sub1_moe_prepare_layout_from_layers(ctypes.byref(layers), meta.data_ptr(), meta.numel(),
                                                       ctypes.byref(out), stream) == status
        assert words in lib.sub1_last_error().decode()
