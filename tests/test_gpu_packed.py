"""The expert launch on the packed layout where rows differ in length: groups of
32 codes share out a row between lanes, a row may take more than a wavefront's 64
groups, or fewer codes than one load.  To the bit against the oracle's sums in the
same order."""
import numpy as np
import pytest
import torch

from oracle import sub1_oracle as so
from test_gpu_parity import bf16_dev, bits_host

pytestmark = pytest.mark.gpu


def uneven_layer(oracle, height, width, shares, seed):
    rng = np.random.default_rng(seed)
    share = np.asarray(shares)[np.arange(height) % len(shares)][:, None]
    t = ((rng.random((height, width)) < share) * rng.integers(1, 3, (height, width))).astype(np.int32)
    minmax = np.abs(rng.standard_normal((height, 2))) * (-1.0, 1.0)
    minmax = so.f32_to_bf16_bits(minmax.ravel().astype(np.float32))
    return oracle.encode(t) + (minmax,)


@pytest.mark.parametrize('d_model,d_ff,shares', [
    (12, 70, [0.2, 1.0, 0.0]),               # rows of one to six codes, and of up to 47
    (100, 200, [0.0]), (64, 66, [1.0]),      # all alike: one code after another, none without a weight
    (700, 130, [0.1] * 63 + [0.95]),         # one long row among 64
    (900, 2100, [0.05, 0.25, 0.5, 0.9, 0.0]),   # cut into parts, a wavefront's rows into turns
    (311, 1037, [0.1]),                      # runs of rows that do not divide a tile's
    (12288, 40, [0.02, 0.9, 0.0, 0.3])])     # rows of up to 150 groups
def test_rows_of_different_lengths_on_the_packed_layout(oracle, d_model, d_ff, shares):
    from qmoe_amd import sub1, sub1_hip
    experts = 2
    wi = [uneven_layer(oracle, d_ff, d_model, shares, 10 + e) for e in range(experts)]
    wo = [uneven_layer(oracle, d_model, d_ff, shares, 20 + e) for e in range(experts)]

    def dev(layer):
        codes, row_off, minmax = layer
        return torch.from_numpy(codes.view(np.int16)).cuda(), torch.from_numpy(row_off).cuda(), bf16_dev(minmax)

    stack = sub1_hip.ExpertStack.from_layers(sub1.DEC[0], [dev(l) for l in wi], [dev(l) for l in wo])
    kernels = set()
    for tokens in (1, 3, 24, 257):
        xs = np.stack([so.synthetic_activation(d_model, 30 + i) for i in range(tokens)])
        route = (torch.arange(tokens, dtype=torch.int32) * 5 % experts).cuda()
        got = bits_host(stack.forward(bf16_dev(xs), route))
        kernels.add(sub1_hip._lib.load().sub1_last_kernel().decode())
        assert stack.launch_faults(tokens) == (0, 0)
        for i in sorted({0, tokens // 2, tokens - 1}):
            want, _ = oracle.expert_ffn(wi[int(route[i])], wo[int(route[i])], xs[i], order=1)
            assert np.array_equal(got[i], want), (tokens, i)
    assert kernels == {'moe_kernel<256>', 'moe_kernel<1024>'}


@pytest.mark.parametrize('d_model,d_ff,experts,tokens', [
    (3, 5, 2, 1), (64, 3, 3, 255), (5, 300, 2, 96),        # fewer rows than wavefronts; a tile or two a token
    (1200, 2100, 3, 9), (768, 3072, 4, 38), (768, 3072, 4, 39)])   # a turn a wavefront; the last before the other form
def test_a_workgroup_for_every_tile(oracle, d_model, d_ff, experts, tokens):
    from qmoe_amd import sub1, sub1_hip
    wi = [uneven_layer(oracle, d_ff, d_model, [0.1, 0.3], 10 + e) for e in range(experts)]
    wo = [uneven_layer(oracle, d_model, d_ff, [0.1, 0.02, 1.0], 20 + e) for e in range(experts)]

    def dev(layer):
        codes, row_off, minmax = layer
        return torch.from_numpy(codes.view(np.int16)).cuda(), torch.from_numpy(row_off).cuda(), bf16_dev(minmax)

    stack = sub1_hip.ExpertStack.from_layers(sub1.DEC[0], [dev(l) for l in wi], [dev(l) for l in wo])
    xs = np.stack([so.synthetic_activation(d_model, 30 + i) for i in range(tokens)])
    route = [i * 7 % experts for i in range(tokens)]
    bad = [i for i in (3, 8) if i < tokens]
    for i, e in zip(bad, (-1, experts)):
        route[i] = e
    x, te = bf16_dev(xs), torch.tensor(route, dtype=torch.int32).cuda()
    for _ in range(3):                  # the control words are left as they were found
        got = bits_host(stack.forward(x, te))
        assert stack.launch_faults(tokens) == (0, len(bad) // 2)
        for i in sorted({0, tokens // 2, tokens - 1} | set(bad)):
            want = xs[i] if i in bad else oracle.expert_ffn(wi[route[i]], wo[route[i]], xs[i], order=1)[0]
            assert np.array_equal(got[i], want), i
    weights = tokens * d_model * d_ff
    assert sub1_hip._lib.load().sub1_last_kernel().decode() == (
        'moe_kernel<1024>' if tokens >= 10 and weights >= 90000000 else 'moe_kernel<256>')


TOKEN_WORDS = 4 * (64 + 2 * 2 * 12288)     # where in a workspace the words begin that launches count with, 64 bytes a token


@pytest.mark.parametrize('late', [0, 200])
@pytest.mark.parametrize('d_model,d_ff', [(768, 3072), (64, 3), (2080, 1100)])
def test_tiles_whose_workgroups_start_late_are_done_by_others(oracle, d_model, d_ff, late):
    """A workgroup of wo that waits for a tile of wi that nobody has begun does it itself, and the one that
    comes for it later finds that; on several streams, that all overlap, too."""
    from qmoe_amd import sub1, sub1_hip
    lib = sub1_hip._lib.load()
    wi = [uneven_layer(oracle, d_ff, d_model, [0.1, 0.3], 10 + e) for e in range(2)]
    wo = [uneven_layer(oracle, d_model, d_ff, [0.1, 0.02, 1.0], 20 + e) for e in range(2)]

    def dev(layer):
        codes, row_off, minmax = layer
        return torch.from_numpy(codes.view(np.int16)).cuda(), torch.from_numpy(row_off).cuda(), bf16_dev(minmax)

    stack = sub1_hip.ExpertStack.from_layers(sub1.DEC[0], [dev(l) for l in wi], [dev(l) for l in wo])
    xs = np.stack([so.synthetic_activation(d_model, 30 + i) for i in range(4)])
    want = np.stack([oracle.expert_ffn(wi[i % 2], wo[i % 2], xs[i], order=1)[0] for i in range(4)])
    calls = [np.arange(t) % 4 for t in (38, 1, 14, 9)]
    inputs = [(bf16_dev(xs[i]), torch.from_numpy((i % 2).astype(np.int32)).cuda()) for i in calls]
    streams = [torch.cuda.Stream() for _ in calls]
    assert lib.sub1_test_late_tiles(-1) != 0 and lib.sub1_test_late_tiles(10001) != 0
    torch.cuda.synchronize()
    try:
        sub1_hip._lib.check(lib.sub1_test_late_tiles(late))
        outs = []
        for _ in range(5):
            for k, stream in enumerate(streams):
                with torch.cuda.stream(stream):
                    outs.append((k, stack.forward(*inputs[k])))
                assert lib.sub1_last_kernel() == b'moe_kernel<256>'
        torch.cuda.synchronize()
    finally:
        sub1_hip._lib.check(lib.sub1_test_late_tiles(0))
    assert all(np.array_equal(bits_host(y), want[calls[k]]) for k, y in outs)
    for k, stream in enumerate(streams):
        with torch.cuda.stream(stream):
            tokens = len(calls[k])
            assert stack.launch_faults(tokens) == (0, 0)
            assert not bool(stack.workspace(tokens)[TOKEN_WORDS:TOKEN_WORDS + 64 * tokens].any())
