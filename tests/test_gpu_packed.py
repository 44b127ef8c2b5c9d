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
