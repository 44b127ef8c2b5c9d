"""The expert layer on the matrix cores (forward_batch).

The first test's numbers are small integers times powers of two, with few enough
terms that every fp32 sum of them is exact whatever its order: the results must be
the oracle's to the bit.  |x| <= 2 and |weights| <= 2 give |h| <= 4 width and, h
rounded to bf16, sums of multiples of 1/4 below 8 d_model d_ff < 2^22 (at these shapes):
24 bits hold them.  The others compare with the walking kernels; where sums are
not exact, the two orders differ by bf16 roundings here and there: 2e-4 of the norm
(4.5e-5 at most between any two of this library's orders)."""
import numpy as np
import pytest
import torch

from oracle import sub1_oracle as so
from test_gpu_parity import bf16_dev, bits_host


def layers(oracle, height, width, p0, seed):
    rng = np.random.default_rng(seed)
    share = 1 - p0 if np.isscalar(p0) else 1 - np.asarray(p0)[np.arange(height) % len(p0)][:, None]
    t = ((rng.random((height, width)) < share) * rng.integers(1, 3, (height, width))).astype(np.int32)
    minmax = rng.choice([0.5, 1.0, 2.0], (height, 2)) * (-1.0, 1.0)
    return oracle.encode(t) + (so.f32_to_bf16_bits(minmax.ravel().astype(np.float32)),)


def prepared(wi, wo):
    from qmoe_amd import sub1, sub1_hip

    def dev(layer):
        codes, row_off, minmax = layer
        return torch.from_numpy(codes.view(np.int16)).cuda(), torch.from_numpy(row_off).cuda(), bf16_dev(minmax)

    return sub1_hip.PreparedStack.from_layers(sub1.DEC[0], [dev(l) for l in wi], [dev(l) for l in wo])


@pytest.mark.gpu
@pytest.mark.parametrize('d_model,d_ff,p0,counts', [
    (1, 1, 0.0, [1, 0, 33]),                              # one step, a row alone in its slice
    (15, 65, 0.5, [31, 32, 33, 64]), (16, 64, 0.5, [65, 1, 96]), (17, 63, 0.5, [2, 129, 0]),
    (33, 130, [0.0, 1.0, 0.5], [40, 40]),                 # whole rows and empty ones
    (768, 400, 0.9, [33, 5]), (400, 768, 0.9, [5, 64]),
    (1100, 470, [0.9] * 63 + [0.02], [70, 3]),            # a row of many groups in every slice
    (130, 3500, 0.98, [34]), (130, 3500, 0.8, [65]),      # eight wavefronts to a slice of wo,
    (66, 6200, 0.985, [65]), (66, 6200, 0.85, [34])])     # twelve and codes that fill LDS: most of
                                                          # them without a group of chunks, and none
def test_exact_sums_equal_the_oracle(oracle, d_model, d_ff, p0, counts):
    experts = len(counts)
    wi = [layers(oracle, d_ff, d_model, p0, 10 + e) for e in range(experts)]
    wo = [layers(oracle, d_model, d_ff, p0, 20 + e) for e in range(experts)]
    prep = prepared(wi, wo)
    if d_ff > 3000:
        assert batch_plan(prep._c, 1)[1] == (8 if d_ff == 3500 else 12)
    rng = np.random.default_rng(1)
    route = np.concatenate([np.full(n, e) for e, n in enumerate(counts)] + [[-1, experts, -7]]).astype(np.int32)
    rng.shuffle(route)
    xs = so.f32_to_bf16_bits(rng.integers(-2, 3, (route.size, d_model)).astype(np.float32))
    x, te = bf16_dev(xs), torch.from_numpy(route).cuda()
    y = prep.forward_batch(x, te)
    assert prep.launch_faults(route.size) == (0, 1)
    got = bits_host(y)
    for i in range(route.size):
        e = route[i]
        if e < 0 or e >= experts:
            assert np.array_equal(got[i], xs[i])
        elif i % 7 == 0 or route.size < 50:
            assert np.array_equal(got[i], oracle.expert_ffn(wi[e], wo[e], xs[i], order=2)[0]), (i, e)
    # every token, and into its own input
    assert torch.equal(prep.forward(x, te), y)
    own = x.clone()
    assert prep.forward_batch(own, te, y=own) is own and torch.equal(own, y)


@pytest.mark.gpu
@pytest.mark.parametrize('d_model,d_ff', [(20, 9700), (9700, 70), (51, 128), (52, 64 * 3 + 1)])
def test_wherever_the_table_of_columns_lies(oracle, d_model, d_ff):
    """Rows of 9700 columns: their codes fill LDS, the table of where they go is kept in
    global memory (either projection); and steps that are no whole turns.  Exact sums, as above."""
    wi = [layers(oracle, d_ff, d_model, 0.97, 30 + e) for e in range(2)]
    wo = [layers(oracle, d_model, d_ff, 0.97, 40 + e) for e in range(2)]
    prep = prepared(wi, wo)
    route = np.repeat(np.int32([1, 0, -1]), [37, 33, 2])
    xs = so.f32_to_bf16_bits(np.random.default_rng(5).integers(-2, 3, (route.size, d_model)).astype(np.float32))
    x, te = bf16_dev(xs), torch.from_numpy(route).cuda()
    y = prep.forward_batch(x, te)
    assert torch.equal(prep.forward(x, te), y)
    got = bits_host(y)
    for i in (0, 36, 37, 69):
        assert np.array_equal(got[i], oracle.expert_ffn(wi[route[i]], wo[route[i]], xs[i], order=2)[0]), i
    x[3, d_model - 1] = float('nan')       # walked, in its own place
    want = prep.forward(x, te)
    assert prep.forward_batch(x, te, y=x) is x
    assert torch.equal(x.view(torch.int16), want.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize('d_model,d_ff,copies,plan', [
    (100, 4600, 1, (2, 8)), (113, 4530, 1, (2, 8)),       # both slices in one workgroup of sixteen wavefronts
    (50, 4600, 1, (1, 12)),                               # one slice alone
    (130, 4700, 1, (2, 8)),                               # three slices: the second workgroup has one
    (66, 4800, 128, (1, 8)), (66, 4800, 127, (1, 12)),    # a table in global memory; slices too few for that
    (66, 5040, 128, (1, 8)), (66, 5060, 128, (1, 12)),
    (150, 3072, 1, (3, 4)), (250, 3072, 1, (1, 8)),       # three slices fill a workgroup, four do not
    (300, 3150, 1, (1, 8))])
def test_two_slices_and_a_table_that_do_not_fit_twice(oracle, d_model, d_ff, copies, plan):
    """Exact sums, as above (at 93 % zeros the wider ones have few enough weights for that)."""
    wi = [layers(oracle, d_ff, d_model, 0.93, 50 + e) for e in range(2)]
    wo = [layers(oracle, d_model, d_ff, 0.93, 60 + e) for e in range(2)]
    prep = prepared(wi * copies, wo * copies)
    assert batch_plan(prep._c, 1)[:2] == plan
    last = 2 * copies - 1
    route = np.repeat(np.int32([last, 0, -1, last // 2]), [70, 33, 2, 3])
    xs = so.f32_to_bf16_bits(np.random.default_rng(6).integers(-2, 3, (route.size, d_model)).astype(np.float32))
    x, te = bf16_dev(xs), torch.from_numpy(route).cuda()
    y = prep.forward_batch(x, te)
    assert torch.equal(prep.forward(x, te), y)
    got = bits_host(y)
    for i in (0, 69, 70, 102, 105, 107):
        e = route[i] % 2
        assert np.array_equal(got[i], oracle.expert_ffn(wi[e], wo[e], xs[i], order=2)[0]), i


@pytest.mark.gpu
def test_a_token_without_finite_activations_spoils_no_other(oracle):
    """x with an infinity or a NaN, and x whose h overflows: what the walking kernel
    gives for the token alone; the tokens of its block are as without it."""
    wi = [layers(oracle, 200, 96, 0.9, 1)]
    wo = [layers(oracle, 96, 200, 0.9, 2)]
    prep = prepared(wi, wo)
    x = torch.randn((70, 96), generator=torch.Generator().manual_seed(3)).bfloat16().cuda()
    te = torch.zeros(70, dtype=torch.int32, device='cuda')
    plain = prep.forward_batch(x, te)
    x[3, 5] = float('inf')
    x[40, 95] = float('nan')
    x[41] = -float('inf')
    x[69] = 3e38
    y = prep.forward_batch(x, te)
    spoiled = [3, 40, 41, 69]
    for t in spoiled:
        alone = prep.forward(x[t:t + 1].contiguous(), te[:1])
        assert torch.equal(y[t].view(torch.int16), alone[0].view(torch.int16)), t
    others = [t for t in range(70) if t not in spoiled]
    assert torch.equal(y[others], plain[others])
    assert torch.isfinite(y[others].float()).all()


@pytest.mark.gpu
@pytest.mark.parametrize('projection', [0, 1])
@pytest.mark.parametrize('value', [np.inf, -np.inf, np.nan])
def test_a_weight_that_is_not_finite_gives_what_walking_gives(oracle, projection, value):
    """An infinite or NaN min or max, also one that no weight of its row has; the other
    experts' tokens are as without it."""
    layer = [[layers(oracle, 200, 96, 0.9, 1 + e) for e in range(3)], [layers(oracle, 96, 200, 0.9, 11 + e) for e in range(3)]]
    x = torch.randn((200, 96), generator=torch.Generator().manual_seed(5)).bfloat16().cuda()
    te = (torch.arange(200, dtype=torch.int32) % 3).cuda()
    plain = prepared(*layer).forward_batch(x, te)
    height, width = (200, 96) if projection == 0 else (96, 200)
    t = np.zeros((height, width), dtype=np.int32)
    t[:, ::7] = 1
    t[5, ::7], t[70, 3], t[90] = 2, 2, 0          # row 5: no min; row 70: one max; row 90: nothing
    minmax = np.tile(np.float32([-1.0, 1.0]), (height, 1))
    minmax[5, 0] = minmax[70, 1] = minmax[90, 0] = value
    layer[projection][1] = oracle.encode(t) + (so.f32_to_bf16_bits(minmax.ravel()),)
    prep = prepared(*layer)
    y, walked = prep.forward_batch(x, te), prep.forward(x, te)
    assert torch.equal(y[1::3].view(torch.int16), walked[1::3].view(torch.int16))
    assert torch.equal(y[::3], plain[::3]) and torch.equal(y[2::3], plain[2::3])


@pytest.mark.gpu
def test_large_batches_through_the_layer():
    """What Sub1Experts sends where: equal to rounding either way, a token's bits the
    same in any batch that goes through the matrix cores, batches of several pieces,
    views that are not aligned."""
    from qmoe_amd import sub1, sub1_hip, synthetic
    experts, d_model, d_ff = 12, 512, 1030
    stack = synthetic.build_stack(experts, d_model, d_ff, 0.9, seed=4)
    pairs = [synthetic.expert_layers(stack, e) for e in range(experts)]

    def linear(buffers):
        layer = sub1.Sub1Linear(buffers[1].numel() - 1, buffers[0].numel())
        layer.w_comp, layer.row_off, layer.ter_minmax = buffers
        return layer

    layer = sub1.Sub1Experts([linear(p[0]) for p in pairs], [linear(p[1]) for p in pairs])
    prep = layer._launcher()
    last = lambda: sub1_hip._lib.load().sub1_last_kernel().decode()
    tokens = 20000
    x = synthetic.activations(tokens, d_model, seed=5)
    route = synthetic.softmax_router(tokens, experts, seed=6)
    y = layer(x, route)
    assert last() == 'batch_product_kernel'
    layer.matrix_cores = False
    walked = layer(x, route)
    assert last() != 'batch_product_kernel'
    assert (y.float() - walked.float()).norm() <= 2e-4 * walked.float().norm()
    assert torch.equal(prep.forward_batch(x[700:1500], route[700:1500]), y[700:1500])
    shifted = torch.empty(1000 * d_model + 1, dtype=torch.bfloat16, device='cuda')[1:].view(1000, d_model)
    shifted.copy_(x[:1000])
    assert torch.equal(prep.forward_batch(shifted, route[:1000]), y[:1000])
    one = torch.full((300,), 7, dtype=torch.int32, device='cuda')       # all to one expert
    assert torch.equal(prep.forward_batch(x[:300], one)[route[:300] == 7], y[:300][route[:300] == 7])
    layer.matrix_cores = True
    layer(x[:64], route[:64])
    assert last() != 'batch_product_kernel'


@pytest.mark.gpu
def test_a_small_batch_is_not_priced(monkeypatch):
    """The calls that last as long as the host takes to make them: no estimate is asked for."""
    from qmoe_amd import sub1, sub1_hip, synthetic
    stack = synthetic.build_stack(4, 64, 96, 0.9, seed=14)
    layers_of = [[sub1.Sub1Linear(1, 1) for _ in range(4)] for _ in range(2)]
    for e in range(4):
        for linear, buffers in zip((layers_of[0][e], layers_of[1][e]), synthetic.expert_layers(stack, e)):
            linear.w_comp, linear.row_off, linear.ter_minmax = buffers
    layer = sub1.Sub1Experts(*layers_of)
    x, route = synthetic.activations(200, 64, seed=15), synthetic.softmax_router(200, 4, seed=16)
    asked = []
    monkeypatch.setattr(sub1_hip.PreparedStack, 'batch_pays', lambda self, tokens: bool(asked.append(tokens)))
    for tokens in (1, 13, 127, 128, 200):
        layer(x[:tokens], route[:tokens])
    assert asked == [128, 200]


@pytest.mark.gpu
@pytest.mark.parametrize('d_model,d_ff,experts,each,pays', [
    # us measured, walking and on the matrix cores, with 90 % zeros
    (768, 3072, 128, 32, True),        # 270, 131
    (2080, 6144, 40, 16, True),        # 313, 169
    (1024, 4096, 64, 64, True),        # 419, 157
    (768, 3072, 512, 16, True),        # 460, 365
    (768, 3072, 1, 2048, True),        # 172, 77
    (768, 3072, 32, 8, False),         # 35, 57
    (768, 3072, 512, 8, False),        # 280, 363
    # batches of several pieces: a piece has 8 tokens an expert, or fewer
    (768, 3072, 1024, 8, False),       # 513, 742
    (768, 3072, 1024, 16, False),      # 883, 1473
    (768, 3072, 1024, 64, False),      # 3134, 5854
    (768, 3072, 2048, 16, False),      # 1735, 5862
    (512, 2000, 1024, 32, False),      # 833, 1443
    (2080, 6144, 2048, 16, False)])    # four pieces with 4 tokens an expert
def test_the_matrix_cores_are_taken_where_they_are_faster(d_model, d_ff, experts, each, pays):
    import ctypes
    from qmoe_amd import _lib
    p = _lib.MoePrepared()
    p.meta = p.codes = 256
    p.experts, p.d_model, p.d_ff, p.meta_bytes = experts, d_model, d_ff, 1 << 40
    p.total_chunks = int(experts * 2 * d_model * d_ff * 0.1045 / 576)
    lib = _lib.load()
    assert bool(lib.sub1_moe_batch_pays(ctypes.byref(p), experts * each)) == pays
    for tokens in (100, 5000, 8192, 8193, 16385, 100000, 1 << 20):
        piece = tokens / -(-tokens // 8192)
        if lib.sub1_moe_batch_pays(ctypes.byref(p), tokens):
            assert piece >= 8 * experts, tokens


@pytest.mark.gpu
def test_pieces_of_a_batch_through_many_experts():
    from qmoe_amd import synthetic
    prep = synthetic.build_stack(700, 96, 130, 0.9, seed=11).prepare()
    x = synthetic.activations(17000, 96, seed=12)
    route = synthetic.softmax_router(17000, 700, seed=13)
    route[::50] = -1
    y, walked = prep.forward_batch(x, route), prep.forward(x, route)
    assert torch.equal(y[::50], x[::50])
    assert (y.float() - walked.float()).norm() <= 2e-4 * walked.float().norm()


@pytest.mark.gpu
def test_two_threads_with_stacks_of_other_shapes():
    """Each on a stream of its own: their launches take different amounts of LDS."""
    import threading
    from qmoe_amd import synthetic
    work = []
    for d_model, d_ff in ((96, 5000), (700, 130)):
        prep = synthetic.build_stack(3, d_model, d_ff, 0.9, seed=17).prepare()
        x, route = synthetic.activations(160, d_model, seed=18), synthetic.softmax_router(160, 3, seed=19)
        x[7, 0] = float('inf')
        work.append((prep, x, route, prep.forward_batch(x, route), []))
    torch.cuda.synchronize()

    def run(prep, x, route, want, differ):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(40):
                y = prep.forward_batch(x, route)
                differ.append(not torch.equal(y.view(torch.int16), want.view(torch.int16)))

    threads = [threading.Thread(target=run, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert [w[4] for w in work] == [[False] * 40] * 2


@pytest.mark.gpu
@pytest.mark.parametrize('tokens', [1, 40, 300])
def test_two_threads_with_uneven_stacks_of_other_shapes(tokens):
    """As above, the forms that share long slices, and the packed launch."""
    import threading
    from qmoe_amd import synthetic
    work = []
    for d_model, d_ff in ((587, 4467), (700, 330)):
        stack = synthetic.build_stack(3, d_model, d_ff, synthetic.ROWS, seed=21)
        x, route = synthetic.activations(tokens, d_model, seed=18), synthetic.softmax_router(tokens, 3, seed=19)
        work += [(s, x, route, s.forward(x, route), []) for s in (stack.prepare(), stack)]
    torch.cuda.synchronize()

    def run(stack, x, route, want, differ):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(40):
                y = stack.forward(x, route)
                differ.append(not torch.equal(y.view(torch.int16), want.view(torch.int16)))

    threads = [threading.Thread(target=run, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert [w[4] for w in work] == [[False] * 40] * 4


@pytest.mark.gpu
def test_replays_from_a_graph():
    from qmoe_amd import synthetic
    stack = synthetic.build_stack(4, 200, 300, 0.9, seed=7)
    prep = stack.prepare()
    x = synthetic.activations(150, 200, seed=8)
    route = synthetic.softmax_router(150, 4, seed=9)
    y = torch.empty_like(x)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        prep.forward_batch(x, route, y=y)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        prep.forward_batch(x, route, y=y)
    for rep in range(3):
        x.copy_(synthetic.activations(150, 200, seed=20 + rep))
        route.copy_(synthetic.softmax_router(150, 4, seed=30 + rep))
        want = prep.forward_batch(x, route)
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), rep


def batch_plan(prep, projection):
    import ctypes
    from qmoe_amd import _lib
    plan = (ctypes.c_int32 * 3)()
    _lib.check(_lib.load().sub1_test_batch_plan(ctypes.byref(prep), projection, plan))
    return tuple(plan)


@pytest.mark.parametrize('d_model,d_ff', [(768, 3072), (1024, 4096), (2080, 6144), (1100, 3500), (512, 2000)])
@pytest.mark.parametrize('entries', [0.06, 0.11, 0.21])      # of a weight, at 95, 90 and 80 % zeros
def test_a_compute_unit_holds_twelve_wavefronts_of_a_product(d_model, d_ff, entries):
    """Whatever the share of zeros: a slice of few entries takes as much LDS as any."""
    from qmoe_amd import _lib
    p = _lib.MoePrepared()
    p.meta = p.codes = 256
    p.experts, p.d_model, p.d_ff, p.meta_bytes = 64, d_model, d_ff, 1 << 40
    p.total_chunks = int(64 * 2 * d_model * d_ff * entries / 576)
    for projection in (0, 1):
        slices, shared_by, lds = batch_plan(p, projection)
        assert (160 * 1024 - 64) // lds * slices * shared_by >= 12, (projection, slices, shared_by, lds)


def test_bad_arguments_are_refused_on_the_host():
    import ctypes
    from qmoe_amd import _lib
    lib = _lib.load()
    one, odd = ctypes.c_void_p(256), ctypes.c_void_p(257)
    p = _lib.MoePrepared()
    p.meta = p.codes = 256
    p.experts, p.d_model, p.d_ff, p.total_chunks, p.meta_bytes = 4, 64, 128, 100, 1 << 30
    ref = ctypes.byref(p)
    scratch = lib.sub1_moe_batch_scratch_bytes(ref, 100)
    ws = lib.sub1_moe_workspace_bytes(100, 128)
    assert scratch > 0

    def call(te=one, x=one, tokens=100, ws=ws, scratch=scratch, at=one):
        return lib.sub1_moe_batch_prepared(ref, te, x, one, tokens, one, ws, at, scratch, None)

    assert lib.sub1_moe_batch_prepared(None, one, one, one, 1, one, ws, one, scratch, None) == -1
    assert call(te=None) == -1 and call(at=None) == -1
    assert call(tokens=-1) == -2 and call(tokens=(1 << 20) + 1) == -2
    assert call(scratch=scratch - 1) == -2 and call(ws=ws - 1) == -2
    assert call(at=odd) < 0 and call(x=odd) < 0
    assert call(tokens=0, te=None) == 0
    # no growth past a piece; no form where a row's codes do not fit LDS, or of too many experts
    assert lib.sub1_moe_batch_scratch_bytes(ref, 1 << 20) <= lib.sub1_moe_batch_scratch_bytes(ref, 8192)
    p.d_ff = 12288
    assert lib.sub1_moe_batch_scratch_bytes(ref, 100) == 0 and call() == -2
    p.d_ff, p.experts = 128, 4097
    assert lib.sub1_moe_batch_scratch_bytes(ref, 100) == 0
    assert lib.sub1_moe_batch_scratch_bytes(None, 100) == 0 and lib.sub1_moe_batch_pays(None, 100) == 0


@pytest.mark.gpu
@pytest.mark.parametrize('experts,tokens,kept', [
    (3, 1, 1), (3, 1023, 3), (3, 1024, 1), (3, 1025, 2),     # a token a thread and more; all of one expert
    (1030, 2049, 1030), (40, 8192, 40), (40, 8193, 1),      # more experts than threads; a piece, and pieces of one expert
    (2, 100, 0)])                                           # no token with an expert
def test_every_token_has_a_slot(oracle, experts, tokens, kept):
    """Tokens in blocks of their expert's, whatever their number: exact sums, so that the walking kernels'
    bits are the answer; dropped ones keep their input."""
    made = [(layers(oracle, 20, 24, 0.5, 10 + e), layers(oracle, 24, 20, 0.5, 20 + e)) for e in range(3)]
    prep = prepared([made[e % 3][0] for e in range(experts)], [made[e % 3][1] for e in range(experts)])
    rng = np.random.default_rng(tokens)
    route = rng.integers(0, kept, tokens) if kept else np.full(tokens, -1)
    drop = rng.random(tokens) < 0.1
    route[drop] = rng.choice([-1, experts], int(drop.sum()))
    xs = rng.integers(-2, 3, (tokens, 24)).astype(np.float32)
    x, te = bf16_dev(so.f32_to_bf16_bits(xs)), torch.from_numpy(route.astype(np.int32)).cuda()
    for _ in range(2):
        got = bits_host(prep.forward_batch(x, te))
        assert prep.launch_faults(tokens) == (0, int((route == experts).sum()))
    assert np.array_equal(got, bits_host(prep.forward(x, te)))
