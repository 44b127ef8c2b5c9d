"""Preparing and packing at the sizes where their kernels change
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


@pytest.mark.parametrize('height,width,count,shares', [
    (700, 2000, 3, [1.0, 0.1, 0.1]),                 # a few of them to a workgroup
    (65534, 300, 34, [1.0, 0.0, 0.0, 0.0])])         # more than it keeps a list of
def test_many_long_rows_come_back_whole(gpu, height, width, count, shares):
    sub1, op = gpu
    symbols = symbols_of(height, width, shares, seed=height + width)
    w_comp, row_off = packed(gpu, symbols)
    minmax = torch.randn(2 * height, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    prepared = op.PreparedMatrix(sub1.DEC[0], w_comp, row_off.repeat(count), minmax.repeat(count), width,
                                 torch.zeros(count, dtype=torch.int64, device='cuda'))
    for matrix in (0, count // 2, count - 1):
        assert torch.equal(prepared.decode(matrix), symbols), matrix


@pytest.mark.parametrize('d_model,d_ff', [(303, 250), (64, 1400), (1024, 65), (229, 3001)])
def test_long_gaps_and_dropped_digits_are_counted_as_they_are_written(gpu, oracle, d_model, d_ff):
    """Gaps about the longest step (59 to 64 columns, at every column of sixteen and with
    either symbol at both ends), gaps of many steps, rows of one code, of eight and of nine,
    and digits past an odd width: as many entries as the oracle has, and the symbols back."""
    sub1, op = gpu
    triples, want, entries = [], [], 0
    for kind, (height, width) in enumerate(((d_ff, d_model), (d_model, d_ff))):
        even = (width + 1) // 2 * 2
        g = torch.Generator().manual_seed(height * width)
        symbols = torch.zeros((height, even), dtype=torch.uint8)
        for r in range(height):
            at = int(torch.randint(0, 70, (1,), generator=g))
            while at < even:
                symbols[r, at] = 1 + int(torch.randint(0, 2, (1,), generator=g))
                near = int(torch.randint(58, 66, (1,), generator=g))
                at += [near, near, 1, 2, 14, near + 60, 28 * 7, 400][int(torch.randint(0, 8, (1,), generator=g))]
        symbols[:, even - 1] = torch.randint(0, 3, (height,), generator=g)   # past the width, where that is odd
        symbols[0], symbols[1] = 0, 1
        w_comp, row_off = packed(gpu, symbols.cuda())
        codes, offsets = w_comp.cpu().numpy().view('uint16'), row_off.tolist()
        for r in range(height):
            # (the oracle's last entry goes from the last non-zero onto a zero column: not counted)
            entries += max(len(oracle.gap_entries(codes[offsets[r]:offsets[r + 1]], width)) - 1, 0)
        triples.append([(w_comp, row_off, torch.ones(2 * height, dtype=torch.bfloat16, device='cuda'))])
        want.append(symbols[:, :width].cuda())
    prepared = op.PreparedStack.from_layers(sub1.DEC[0], *triples)
    assert prepared.entry_counts()[1] == entries
    for kind in (0, 1):
        assert torch.equal(prepared.decode(0, kind), want[kind])


@pytest.mark.parametrize('width,codes', [
    (141, [27, 64, 65, 71]), (1601, [511, 512, 513, 801]), (8193, [1024, 1025, 1537, 4097])])
def test_rows_of_many_codes_come_back_whole(gpu, oracle, width, codes):
    """Rows of more than twice the average of codes: about a lane's eight and a turn's 512 of
    them, alone and side by side, with gaps of many steps between and digits past an odd
    width; and rows of this kind that are bad."""
    sub1, op = gpu
    even = (width + 1) // 2 * 2
    g = torch.Generator().manual_seed(width)
    symbols = torch.zeros((200, even), dtype=torch.uint8)
    symbols[::3, 0] = 1
    for i, n in enumerate(codes * 3):
        r = [0, 70, 71, 72, 73, 74, 150, 151, 152, 190, 191, 199][i]
        pairs = min(n, even // 2)       # (a code to a pair without zeros)
        first = 2 * int(torch.randint(0, even // 2 - pairs + 1, (1,), generator=g))
        symbols[r, first:first + 2 * pairs] = torch.randint(1, 3, (2 * pairs,), generator=g).to(torch.uint8)
        if i % 3 == 2:
            symbols[r, -1] = 2
            symbols[r, first + pairs // 2:first + pairs // 2 + even // 5] = 0
    w_comp, row_off = packed(gpu, symbols.cuda())
    sizes = row_off[1:] - row_off[:-1]
    longs = [r for r in range(200) if (int(sizes[r]) - 16) * 200 > 2 * int(row_off[-1])]
    assert len(longs) >= 9
    pairs = torch.ones(400, dtype=torch.bfloat16, device='cuda')
    other = packed(gpu, torch.zeros((width, 200), dtype=torch.uint8, device='cuda'))
    prepared = op.PreparedStack.from_layers(
        sub1.DEC[0], [(w_comp, row_off, pairs)],
        [other + (torch.ones(2 * width, dtype=torch.bfloat16, device='cuda'),)])
    assert torch.equal(prepared.decode(0, 0), symbols[:, :width].cuda())
    want, offsets = w_comp.cpu().numpy().view('uint16'), row_off.tolist()
    entries = sum(max(len(oracle.gap_entries(want[offsets[r]:offsets[r + 1]], width)) - 1, 0) for r in range(200))
    assert prepared.entry_counts()[1] == entries
    # walked from the checkpoints by many wavefronts, and from the front: the same sums
    matrix = op.PreparedMatrix(sub1.DEC[0], w_comp, row_off, pairs, width)
    x = torch.randn((1, width), generator=torch.Generator().manual_seed(3)).bfloat16().cuda()
    few, many = (matrix.product_tokens(x.expand(t, width).contiguous()) for t in (1, 600))
    assert torch.equal(few[0], many[599])
    exact = (symbols[:, :width] > 0).double() @ x[0].double().cpu()
    # bf16 of a sum of up to 8193 terms of 2 or so in fp32
    assert ((few[0].double().cpu() - exact).abs() <= 2 ** -8 * exact.abs() + 8193 * 2 ** -24 * 200).all()
    # the last code of two long rows missing: they are counted, and the rows behind them, with one too many
    a = longs[1]
    b = next(r for r in longs if r > a + 1)
    short = row_off.clone()
    short[a + 1] -= 1
    short[b + 1] -= 1
    with pytest.raises(op._lib.Sub1Error, match='codes of 4 rows'):
        op.PreparedMatrix(sub1.DEC[0], w_comp, short, pairs, width)


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


def symbols_by_torch(w):
    """The rule of reference sub1.py:146-155 in torch: (symbols, ter_minmax)."""
    minmax = torch.column_stack((w.min(1)[0], w.max(1)[0])).flatten()
    symbols = torch.zeros(w.shape, dtype=torch.uint8, device=w.device)
    symbols[w == minmax[0::2].reshape(-1, 1)] = 1
    symbols[w == minmax[1::2].reshape(-1, 1)] = 2
    return symbols, minmax


@pytest.mark.parametrize('height,width,share', [
    (5, 1, 0.5), (3, 2, 1.0), (9, 27, 0.1), (9, 29, 0.1),          # shorter than an entry, one symbol more
    (70, 127, 0.15), (66, 513, 0.02), (64, 1040, 0.35),            # bytes of a plane, a lane's turn
    (6, 8191, 0.1), (6, 8194, 0.1), (3, 16400, 0.12)])             # one window of a row, two, three
def test_weights_pack_like_their_symbols(gpu, oracle, height, width, share):
    sub1, op = gpu
    symbols = symbols_of(height, width, [share, share / 3, 0.0, 0.7], seed=height * width)
    scale = torch.rand(height, 1, generator=torch.Generator().manual_seed(2)).cuda() + 0.5
    w = (torch.tensor([0.0, -1.0, 1.0], device='cuda')[symbols.long()] * scale).bfloat16()
    if height > 8:   # rows of one value, of zeros of both signs, with an infinity, with a NaN
        w[0], w[1], w[2, 0], w[3, -1] = 0.25, -0.0, float('inf'), float('nan')
        w[4], w[4, ::2] = 0.0, 3.0
    want, minmax = symbols_by_torch(w)
    before = w.clone()
    w_comp, row_off, got_minmax = op.sub1pack_weights(w)
    assert torch.equal(w.view(torch.int16), before.view(torch.int16))
    assert torch.equal(torch.nan_to_num(got_minmax.float()), torch.nan_to_num(minmax.float()))
    codes, offsets = oracle.encode(want.cpu().numpy())
    assert (row_off.cpu().numpy() == offsets).all()
    assert (w_comp.cpu().numpy().view('uint16') == codes).all()
    # and from the symbols themselves
    p_comp, p_off = packed(gpu, want)
    assert torch.equal(p_comp, w_comp) and torch.equal(p_off, row_off)


@pytest.mark.parametrize('width', [2047, 2048, 2300, 4096, 8194, 16400])   # a form for narrow rows; one window and several
def test_rows_pack_alike_alone_and_by_a_workgroup(gpu, width):
    """Few wide rows are packed by a workgroup each, many by a wavefront each: the same codes."""
    sub1, op = gpu
    rows, cus = 40, torch.cuda.get_device_properties(0).multi_processor_count
    symbols = symbols_of(rows, width, [0.1, 0.05, 0.0, 1.0, 0.3], seed=width)
    symbols[7, :width // 2] = 0                                   # entries of many and of few pairs, and where they meet
    symbols[8, width // 3:] = 0
    w = torch.tensor([0.0, -1.0, 1.0], device='cuda')[symbols.long()].bfloat16()
    few = op.sub1pack_weights(w)
    many = op.sub1pack_weights(w.repeat(10 * cus // rows + 1, 1))
    codes = few[0].numel()
    assert torch.equal(many[1][:rows + 1], few[1]) and torch.equal(many[0][:codes], few[0])
    assert torch.equal(many[0][-codes:], few[0])
    symbols, _ = symbols_by_torch(w)
    s_comp, s_off = packed(gpu, symbols)
    assert torch.equal(s_comp, few[0]) and torch.equal(s_off, few[1])
    m_comp, _ = packed(gpu, symbols.repeat(10 * cus // rows + 1, 1))
    assert torch.equal(m_comp, many[0])


def test_packing_with_a_trie_of_ones_own(gpu):
    """A trie that is not the fixed dictionary's (here: cut off below three
    pairs, and with the symbols' order of a few entries changed) is walked as it
    is."""
    sub1, op = gpu
    trie = sub1.trie.clone()
    depth3 = set()
    level = [int(c) for c in trie[65536]]
    for _ in range(2):
        level = [int(c) for n in level for c in trie[n] if c >= 0]
    depth3.update(level)
    trie[sorted(depth3)] = -1
    trie[65536, 1], trie[65536, 2] = trie[65536, 2].clone(), trie[65536, 1].clone()
    symbols = symbols_of(70, 201, [0.1, 0.5, 0.0], seed=11)
    row_off = torch.zeros(71, dtype=torch.int32, device='cuda')
    w_comp = op.sub1pack(trie.cuda(), symbols.to(torch.int32), row_off)
    want, offsets = [], [0]
    for row in symbols.cpu().tolist():
        row.append(0)
        node = 65536
        for i in range(0, 201, 2):
            child = int(trie[node, row[i] + 3 * row[i + 1]])
            if child < 0:
                want.append(node)
                child = int(trie[65536, row[i] + 3 * row[i + 1]])
            node = child
        want.append(node)
        offsets.append(len(want))
    assert row_off.tolist() == offsets
    assert w_comp.cpu().numpy().view('uint16').tolist() == want


@pytest.mark.parametrize('height,width,shares', [
    (1, 1, [1.0]), (7, 3, [0.5]), (66, 31, [0.2]), (5, 1023, [0.1, 0.0]),      # rows that begin at any byte of a word
    (4, 1024, [0.1]), (3, 9001, [0.0, 0.05, 0.99])])                          # runs of 64 codes, and many of them
def test_expanding_gives_the_symbols_and_their_weights(gpu, height, width, shares):
    sub1, op = gpu
    symbols = symbols_of(height, width, shares, seed=width)
    w_comp, row_off = packed(gpu, symbols)
    minmax = torch.randn(2 * height, generator=torch.Generator().manual_seed(4)).bfloat16().cuda()
    values = torch.cat((torch.zeros((height, 1), dtype=torch.bfloat16, device='cuda'), minmax.view(-1, 2)), 1)
    want = values.gather(1, symbols.long())
    tern, w, bad = op.sub1decode(sub1.DEC[0], w_comp, row_off, minmax, width)
    assert bad == 0 and torch.equal(tern, symbols) and torch.equal(w, want)
    # either alone, and both into buffers that begin within a word, with what lies around them
    import ctypes
    lib, stream = op._lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    n = height * width
    for at_t, at_w in ((0, None), (None, 0), (1, 1), (3, 2), (2, 0)):
        t_buf = torch.full((n + 8,), 77, dtype=torch.uint8, device='cuda')
        w_buf = torch.full((n + 8,), 77.0, dtype=torch.bfloat16, device='cuda')
        assert lib.sub1_decode(sub1.DEC[0].data_ptr(), w_comp.data_ptr(), row_off.data_ptr(), minmax.data_ptr(),
                               None if at_t is None else t_buf[at_t:].data_ptr(),
                               None if at_w is None else w_buf[at_w:].data_ptr(), None, height, width, stream) == 0
        for buf, at, ref in ((t_buf, at_t, symbols), (w_buf, at_w, want)):
            if at is not None:
                assert torch.equal(buf[at:at + n].view(height, width), ref)
                assert bool((buf[:at] == 77).all()) and bool((buf[at + n:] == 77).all())


def test_expanding_codes_that_do_not_fit_the_width(gpu):
    """Rows whose codes end before the row does are filled with zeros and counted,
    rows with codes to spare are cut off and counted."""
    sub1, op = gpu
    symbols = symbols_of(3, 4000, [0.3], seed=9)
    w_comp, row_off = packed(gpu, symbols)
    minmax = torch.ones(6, dtype=torch.bfloat16, device='cuda')
    moved = row_off.clone()
    moved[1] -= 200
    tern, _, bad = op.sub1decode(sub1.DEC[0], w_comp, moved, minmax, 4000)
    assert bad == 2
    whole, _, _ = op.sub1decode(sub1.DEC[0], w_comp, row_off, minmax, 4000)
    assert torch.equal(tern[2], whole[2])
    kept = int((tern[0] != whole[0]).nonzero()[0])           # the first symbol lost
    assert 0 < kept < 4000 and torch.equal(tern[0, :kept], whole[0, :kept]) and not tern[0, kept:].any()


def test_calls_that_wait_for_the_gpu_come_from_any_thread_and_stream(gpu):
    """More calls at once than the library has places to answer in, each with a count of its
    own; and a stream that is being captured is refused without spoiling the capture."""
    import threading
    sub1, op = gpu
    symbols = symbols_of(40, 300, [0.3], seed=2)
    w_comp, row_off = packed(gpu, symbols)
    minmax = torch.tensor([-1.0, 1.0] * 40, device='cuda').bfloat16()
    weights = torch.tensor([0.0, -1.0, 1.0], device='cuda')[symbols.long()].bfloat16()
    weights[:, 0], weights[:, 1] = -1.0, 1.0
    whole = op.sub1pack_weights(weights)
    torch.cuda.synchronize()
    wrong = []

    def calls(n):
        with torch.cuda.stream(torch.cuda.Stream()):
            for i in range(6):
                rows = 1 + (n + 5 * i) % 39
                moved = row_off[:rows + 1].clone()
                moved[rows] -= n % 2                    # the last row lacks a code, or not
                bad = op.sub1decode(sub1.DEC[0], w_comp, moved, minmax[:2 * rows], 300)[2]
                packs = op.sub1pack_weights(weights[:rows].contiguous())
                if bad != n % 2 or not torch.equal(packs[0], whole[0][:int(whole[1][rows])]):
                    wrong.append((n, i, bad))

    threads = [threading.Thread(target=calls, args=(n,)) for n in range(80)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    graph, y = torch.cuda.CUDAGraph(), torch.zeros(8, device='cuda')
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        with pytest.raises(op._lib.Sub1Error, match='captured'):
            op.sub1decode(sub1.DEC[0], w_comp, row_off, minmax, 300)
        y += 1
    graph.replay()
    graph.replay()
    assert y.tolist() == [2.0] * 8


def test_a_count_starts_from_zero_on_whichever_stream_the_next_call_is(gpu):
    """Calls that take turns on two streams get one place to answer in after another: what
    one has counted is gone before the next, on the other stream, adds to it."""
    sub1, op = gpu
    rows = 700
    symbols = symbols_of(rows, 64, [0.3], seed=6)
    w_comp, row_off = packed(gpu, symbols)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    short = [row_off.clone() for _ in range(4)]
    for n in range(4):                              # n rows lack their last code, n have one too many
        short[n][1:2 * n + 1:2] -= 1
    torch.cuda.synchronize()
    for i in range(200):
        with torch.cuda.stream(streams[i % 2]):
            n = i * 7 % 4
            assert op.sub1decode(sub1.DEC[0], w_comp, short[n], None, 64, want_w=False)[2] == 2 * n, i


@pytest.mark.parametrize('at_t,at_w', [(0, 0), (1, 0)])      # one launch, and one for each output
def test_what_a_counted_expansion_wrote_may_be_read_anywhere_once_it_returns(gpu, at_t, at_w):
    import ctypes
    sub1, op = gpu
    height, width = 3072, 2080
    symbols = symbols_of(height, width, [0.1], seed=3)
    w_comp, row_off = packed(gpu, symbols)
    minmax = torch.tensor([-1.0, 1.0] * height, device='cuda').bfloat16()
    want = torch.tensor([0.0, -1.0, 1.0], device='cuda')[symbols.long()].bfloat16()
    n = height * width
    t_buf, w_buf = torch.zeros(n + 8, dtype=torch.uint8, device='cuda'), torch.zeros(n + 8, dtype=torch.bfloat16, device='cuda')
    lib, here, there, bad = op._lib.load(), torch.cuda.Stream(), torch.cuda.Stream(), ctypes.c_int32(-1)
    torch.cuda.synchronize()
    for i in range(20):
        with torch.cuda.stream(here):
            t_buf.fill_(77)
            w_buf.fill_(77)
        assert lib.sub1_decode_counted(sub1.DEC[0].data_ptr(), w_comp.data_ptr(), row_off.data_ptr(), minmax.data_ptr(),
                                       t_buf[at_t:].data_ptr(), w_buf[at_w:].data_ptr(), ctypes.byref(bad), height, width,
                                       here.cuda_stream) == 0
        with torch.cuda.stream(there):      # (the last first: they are the last to be written)
            got_w, got_t = w_buf.flip(0)[8 - at_w:][:n], t_buf.flip(0)[8 - at_t:][:n]
        there.synchronize()
        assert bad.value == 0
        assert torch.equal(got_w.flip(0).view(height, width), want), i
        assert torch.equal(got_t.flip(0).view(height, width), symbols), i


def test_what_a_compression_counted_may_be_read_anywhere_once_it_returns(gpu):
    import ctypes
    _, op = gpu
    height, width = 6144, 96
    weights = torch.randn((height, 3), generator=torch.Generator().manual_seed(5)).cuda().bfloat16()
    weights[:, 0] = 0
    weights = weights.gather(1, symbols_of(height, width, [0.1, 0.5], seed=7).long()).contiguous()
    _, want, minmax = op.sub1pack_weights(weights)
    codes = torch.empty((height, width // 2), dtype=torch.int16, device='cuda')
    row_off, pairs = torch.empty_like(want), torch.empty_like(minmax)
    lib, here, there, total = op._lib.load(), torch.cuda.Stream(), torch.cuda.Stream(), ctypes.c_int32(-1)
    torch.cuda.synchronize()
    for i in range(20):
        with torch.cuda.stream(here):
            row_off.fill_(-1)
            pairs.zero_()
        assert lib.sub1_pack_weights_total(weights.data_ptr(), codes.data_ptr(), pairs.data_ptr(), row_off.data_ptr(),
                                           ctypes.byref(total), height, width, here.cuda_stream) == 0
        with torch.cuda.stream(there):
            got, got_pairs = row_off.flip(0), pairs.clone()
        there.synchronize()
        assert total.value == int(want[-1]) and torch.equal(got.flip(0), want) and torch.equal(got_pairs, minmax), i


def test_calls_that_end_by_an_error_leave_their_places_as_they_were(gpu):
    """More of them than there are places, each behind launches that count and store."""
    from qmoe_amd import synthetic
    sub1, op = gpu
    lib = op._lib.load()
    symbols = symbols_of(40, 300, [0.3], seed=2)
    w_comp, row_off = packed(gpu, symbols)
    short = row_off.clone()
    short[1:7:2] -= 1                       # six bad rows
    weights = torch.tensor([0.0, -1.0, 1.0], device='cuda')[symbols.long()].bfloat16()
    whole = op.sub1pack_weights(weights)
    stack = synthetic.build_stack(2, 96, 160, 0.9, seed=5)
    calls = (lambda: op.sub1decode(sub1.DEC[0], w_comp, short, None, 300, want_w=False)[2],
             lambda: op.sub1pack_weights(weights), stack.prepare)
    try:
        for call in calls:
            op._lib.check(lib.sub1_test_fail_answers(70))
            for _ in range(70):
                with pytest.raises(op._lib.Sub1Error, match='made to fail'):
                    call()
    finally:
        op._lib.check(lib.sub1_test_fail_answers(0))
    assert lib.sub1_test_fail_answers(-1) != 0
    for _ in range(70):
        assert calls[0]() == 6
    assert all(torch.equal(a, b) for a, b in zip(calls[1](), whole))
    x, route = synthetic.activations(4, 96, 6), torch.arange(4, dtype=torch.int32, device='cuda') % 2
    assert calls[2]().forward(x, route).isfinite().all()


@pytest.mark.parametrize('height,width', [(1, 1), (70, 200), (1025, 31), (4100, 16)])
def test_counting_without_waiting_gives_what_counting_with_it_does(gpu, height, width):
    import ctypes
    _, op = gpu
    lib, stream = op._lib.load(), torch.cuda.current_stream().cuda_stream
    weights = torch.tensor([0.0, -1.5, 2.0], device='cuda')[symbols_of(height, width, [0.2, 0.9], seed=4).long()].bfloat16()
    results, total = [], ctypes.c_int32(-1)
    for function, extra in ((lib.sub1_pack_weights_count, ()), (lib.sub1_pack_weights_total, (ctypes.byref(total),))):
        codes = torch.zeros((height, (width + 1) // 2), dtype=torch.int16, device='cuda')
        minmax, row_off = torch.zeros(2 * height, dtype=torch.bfloat16, device='cuda'), torch.zeros(height + 1, dtype=torch.int32, device='cuda')
        assert function(weights.data_ptr(), codes.data_ptr(), minmax.data_ptr(), row_off.data_ptr(), *extra, height, width, stream) == 0
        w_comp = torch.zeros(int(row_off[height]), dtype=torch.int16, device='cuda')
        assert lib.sub1_pack_weights_emit(codes.data_ptr(), row_off.data_ptr(), w_comp.data_ptr(), height, width, stream) == 0
        results.append((row_off, minmax, w_comp))
    assert total.value == results[0][2].numel() > 0
    assert all(torch.equal(a, b) for a, b in zip(*results))
    w_comp, row_off, minmax = op.sub1pack_weights(weights)
    assert all(torch.equal(a, b) for a, b in zip(results[0], (row_off, minmax, w_comp)))


FIRST_PACK_IN_A_CAPTURE = r'''
import ctypes, sys
sys.path.insert(0, sys.argv[1])
import torch
from qmoe_amd import _lib, sub1, sub1_hip

lib = _lib.load()
_lib.check_faults()
g = torch.Generator().manual_seed(1)
symbols = ((torch.rand((70, 200), generator=g) < 0.2) * torch.randint(1, 3, (70, 200), generator=g)).to(torch.int32).cuda()
t = torch.empty_like(symbols)
off = torch.zeros(71, dtype=torch.int32, device='cuda')
stream = torch.cuda.Stream()
c_stream = ctypes.c_void_p(stream.cuda_stream)
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph, stream=stream):
    t.copy_(symbols)
    _lib.check(lib.sub1_pack_count(sub1.TRIE.data_ptr(), t.data_ptr(), off.data_ptr(), 70, 200, c_stream))
counted = []
for _ in range(3):
    off.fill_(-5)
    graph.replay()
    torch.cuda.synchronize()
    counted.append(off.tolist())
want = torch.zeros_like(off)
sub1_hip.sub1pack(sub1.TRIE, symbols.clone(), want)
assert counted == [want.tolist()] * 3, counted
print('first call in a capture: fine')
'''


def test_the_first_pack_of_a_process_may_be_captured():
    """The first call fills the tables that the encoder keeps on a GPU, also where its
    stream is being captured.  (A process of its own: in this one they are there.)"""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, '-c', FIRST_PACK_IN_A_CAPTURE, root], stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, timeout=110)
    assert res.returncode == 0 and 'first call in a capture: fine' in res.stdout, res.stdout


@pytest.mark.parametrize('height,width,shares', [
    (1088, 900, [0.0, 0.1, 0.9]), (1023, 1100, [0.02, 1.0]),                  # a part per wavefront, some without rows
    (2000, 3100, [0.0, 0.5, 0.99]), (700, 6000, [0.0, 0.9]), (8200, 40, [0.1, 0.5])])   # fewer parts; a turn of a part and more
def test_rows_that_are_ordered_in_parts_come_back_whole(gpu, height, width, shares):
    test_prepared_rows_come_back_whole(gpu, height, width, shares)


UNEVEN_SPLIT, UNEVEN_SHARED = 'moe_prepared_uneven_split_kernel<%s>', 'moe_prepared_shared_kernel<%s, %s>'
UNEVEN_FUSED = 'moe_prepared_fused_kernel<false, false, true>'


@pytest.mark.parametrize('d_model,d_ff,long_rows,shared', [
    (300, 4467, 5, ['Few Few', 'Differ Few']),          # wo: one slice of 62 groups of entries and four of a few
    (2080, 1100, 70, ['Few Few', 'Differ Differ']),     # wi: one and a bit of 29 groups, wo of 33 slices
    (900, 900, 1, ['Few Few']),                         # a single long row
    (130, 12000, 64, ['Differ Few', 'Differ Differ']),  # partial sums for which LDS has no room
    (650, 3000, 750, ['Few Few', 'Differ Few']),        # more long slices than are shared
    (600, 9000, 150, ['Few Few', 'Differ Few', 'Differ Differ'])])   # three, with room for two
def test_a_few_tokens_share_long_rows(oracle, d_model, d_ff, long_rows, shared):
    """The longest slices of a matrix are shared by wavefronts according to their lengths, to the bit:
    all the slices that a workgroup has, if they are few, or those that their lengths say."""
    import numpy as np
    from oracle import sub1_oracle as so
    from qmoe_amd import sub1, sub1_hip
    rng = np.random.default_rng(d_model)

    def layer(height, width):
        share = rng.uniform(0.0, 0.3, (height, 1))
        share[rng.permutation(height)[:min(long_rows, height // 4)]] = 1.0
        t = ((rng.random((height, width)) < share) * rng.integers(1, 3, (height, width))).astype(np.int32)
        minmax = np.abs(rng.standard_normal((height, 2))) * (-1.0, 1.0)
        return oracle.encode(t) + (so.f32_to_bf16_bits(minmax.ravel().astype(np.float32)),)

    def dev(l):
        return torch.from_numpy(l[0].view(np.int16)).cuda(), torch.from_numpy(l[1]).cuda(), \
            torch.from_numpy(l[2].view(np.int16)).cuda().view(torch.bfloat16)

    wi, wo = [layer(d_ff, d_model) for _ in range(2)], [layer(d_model, d_ff) for _ in range(2)]
    stack = sub1_hip.PreparedStack.from_layers(sub1.DEC[0], [dev(l) for l in wi], [dev(l) for l in wo])
    xs = np.stack([so.synthetic_activation(d_model, 30 + i) for i in range(4)])
    want = [oracle.expert_ffn(wi[i % 2], wo[i % 2], xs[i], order=2)[0] for i in range(4)]
    x = torch.from_numpy(xs.view(np.int16)).cuda().view(torch.bfloat16)
    kernels = set()
    for tokens in (1, 2, 3, 9, 33, 64, 128, 255, 600):
        ids = torch.arange(tokens) % 4
        for _ in range(2):                  # the control words are left as they were found
            y = stack.forward(x[ids.cuda()].contiguous(), (ids % 2).to(torch.int32).cuda(), None, False)
            got = y.view(torch.int16).cpu().numpy().view(np.uint16)
            assert stack.launch_faults(tokens) == (0, 0)
            assert (got == np.stack(want)[ids]).all(), tokens
            kernels.add(sub1_hip._lib.load().sub1_last_kernel().decode())
    assert kernels == {UNEVEN_SPLIT % 'kFew', UNEVEN_FUSED} | {
        UNEVEN_SHARED % tuple('k' + kind for kind in kinds.split()) for kinds in shared}


@pytest.mark.parametrize('d_model,d_ff,tokens,kernel', [
    (6144, 12000, 1, UNEVEN_SPLIT % 'kDiffer'),        # several slices of wi to a workgroup, and little room
    (7000, 700, 1, 'moe_prepared_tagged_kernel<kFew>'), (7000, 12000, 1, 'moe_prepared_tagged_kernel<kDiffer>')])
def test_a_token_or_two_through_large_uneven_rows(oracle, d_model, d_ff, tokens, kernel):
    import numpy as np
    from qmoe_amd import _lib, synthetic
    stack = synthetic.build_stack(1, d_model, d_ff, synthetic.ROWS, seed=d_model)
    prepared = stack.prepare()
    x = synthetic.activations(tokens, d_model, seed=3)
    y = prepared.forward(x, torch.zeros(tokens, dtype=torch.int32, device='cuda'))
    assert _lib.load().sub1_last_kernel().decode() == kernel

    def bits(t):
        return t.view(torch.int16).cpu().numpy().view(np.uint16) if t.dtype != torch.int32 else t.cpu().numpy()

    wi, wo = [tuple(bits(t) for t in layer) for layer in synthetic.expert_layers(stack, 0)]
    for got, token in zip(bits(y), bits(x)):
        assert (got == oracle.expert_ffn(wi, wo, token, order=2)[0]).all()
    assert prepared.launch_faults(tokens) == (0, 0)


@pytest.mark.parametrize('height,width,long_rows', [(3000, 1100, 40), (1100, 4467, 70), (64 * 33, 700, 3)])
def test_matrices_of_long_rows(oracle, height, width, long_rows):
    """Single matrices, a token through its own of them: tiles whose longest slices are shared by length, to the bit."""
    import numpy as np
    from oracle import sub1_oracle as so
    from qmoe_amd import _lib, sub1, sub1_hip
    rng = np.random.default_rng(height)

    def one():
        share = rng.uniform(0.0, 0.3, (height, 1))
        share[rng.permutation(height)[:long_rows]] = 1.0
        t = ((rng.random((height, width)) < share) * rng.integers(1, 3, (height, width))).astype(np.int32)
        minmax = np.abs(rng.standard_normal((height, 2))) * (-1.0, 1.0)
        return oracle.encode(t) + (so.f32_to_bf16_bits(minmax.ravel().astype(np.float32)),)

    def dev(bits):
        return torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)

    made = [one() for _ in range(2)]
    pm = sub1_hip.PreparedMatrix(sub1.DEC[0], [torch.from_numpy(m[0].view(np.int16)).cuda() for m in made],
                                 [torch.from_numpy(m[1]).cuda() for m in made], [dev(m[2]) for m in made], width)
    xs = np.stack([so.synthetic_activation(width, 30 + i) for i in range(4)])
    zero = np.zeros(height, np.uint16)
    want = np.stack([oracle.matvec_gap(*made[i % 2], xs[i], y=zero) for i in range(4)])
    kernels = set()
    for tokens in (1, 7, 100, 300):
        ids = np.arange(tokens) % 4
        y = torch.zeros((tokens, height), dtype=torch.bfloat16, device='cuda')
        pm.matvec_tokens(dev(xs)[torch.from_numpy(ids).cuda()].contiguous(), y,
                         torch.from_numpy((ids % 2).astype(np.int32)).cuda())
        kernels.add(_lib.load().sub1_last_kernel())
        assert (y.view(torch.int16).cpu().numpy().view(np.uint16) == want[ids]).all(), tokens
    assert b'moe_prepared_kernel<kDiffer>' in kernels
