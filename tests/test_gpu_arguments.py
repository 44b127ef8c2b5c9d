"""How calls look their tensors over: what is plainly in order goes by its address,
everything else gets the answer that the slow way gives."""
import pytest
import torch

from qmoe_amd import _lib, sub1_hip

SPEC = ((torch.bfloat16, 'a', 2), (torch.int32, 'b', -1))


class Wrapped(torch.Tensor):
    pass


def test_nothing_but_plain_gpu_tensors_goes_by_its_address():
    look = _lib.tensor_args().addresses
    cpu = (torch.zeros(2, 4, dtype=torch.bfloat16), torch.zeros(3, dtype=torch.int32))
    for spec, tensors, numels, device in (
            (SPEC, cpu, (-1, -1), 0), (SPEC, (1, None), (-1, -1), 0), (SPEC, cpu, (-1,), 0), (SPEC, cpu[:1], (-1, -1), 0),
            (SPEC, cpu, (-1, -1), None), (((1, 'a', -1),) * 2, cpu, (-1, -1), 0), (SPEC, cpu, (None, 1 << 70), 0)):
        assert look(spec, tensors, numels, device) is None
    table = torch.zeros(2, 1, dtype=torch.int64)
    fill = _lib.tensor_args().layer_addresses
    for args in ((table, 0, [cpu], SPEC, (-1, -1), 0), (table, 1, [cpu], SPEC, (-1, -1), 0), (table, -1, [cpu], SPEC, (-1, -1), 0),
                 (table, 0, cpu, SPEC, (-1, -1), 0), (table.int(), 0, [cpu], SPEC, (-1, -1), 0), (None, 0, [cpu], SPEC, (-1, -1), 0)):
        assert fill(*args) is False


@pytest.mark.gpu
def test_addresses_and_refusals_are_those_of_the_slow_way():
    dev = torch.device('cuda:0')
    a, b = torch.zeros(4, 6, dtype=torch.bfloat16, device=dev), torch.zeros(9, dtype=torch.int32, device=dev)
    for good in ((a, b), (torch.nn.Parameter(a, requires_grad=False), b[2:]), (a[1:3], b.view(3, 3)), (a.as_subclass(Wrapped), b),
                 (a[:0], b[:0])):
        assert list(sub1_hip._addresses(SPEC, good, (-1, good[1].numel()), dev)) == [t.data_ptr() for t in good]
    for bad, numels, error in (
            ((a.float(), b), (-1, -1), TypeError), ((a, b.long()), (-1, -1), TypeError), ((a, 'b'), (-1, -1), TypeError),
            ((a, b.cpu()), (-1, -1), ValueError), ((a.t(), b), (-1, -1), ValueError), ((a, b[::2]), (-1, -1), ValueError),
            ((a, b), (-1, 8), ValueError), ((a, b), (23, 9), ValueError), ((a.view(-1), b), (-1, -1), ValueError)):
        with pytest.raises(error):
            sub1_hip._addresses(SPEC, bad, numels, dev)


@pytest.mark.gpu
@pytest.mark.parametrize('form', ['tuples', 'lists', 'wrapped'])
def test_a_layer_may_come_in_any_form(form):
    from qmoe_amd import sub1, synthetic
    stack = synthetic.build_stack(3, 96, 160, 0.9, seed=5)
    pairs = [synthetic.expert_layers(stack, e) for e in range(3)]
    x = synthetic.activations(7, 96, 6)
    route = torch.arange(7, dtype=torch.int32, device=x.device) % 3
    want = stack.prepare().forward(x, route)
    wi, wo = [p[0] for p in pairs], [p[1] for p in pairs]
    if form == 'lists':
        wi, wo = tuple(list(t) for t in wi), [list(t) for t in wo]
    if form == 'wrapped':
        wo[1] = (wo[1][0].as_subclass(Wrapped),) + tuple(wo[1][1:])
    made = sub1_hip.PreparedStack.from_layers(sub1.DEC[0], wi, wo)
    assert torch.equal(made.forward(x, route).view(torch.int16), want.view(torch.int16))
    for broken, error in (((wo[1][0].int(),) + tuple(wo[1][1:]), TypeError), (tuple(wo[1][:1]) + (wo[1][1][:-1], wo[1][2]), ValueError),
                          ((wo[1][0], None, wo[1][2]), TypeError)):
        with pytest.raises(error):
            sub1_hip.PreparedStack.from_layers(sub1.DEC[0], wi, [wo[0], broken, wo[2]])


@pytest.mark.gpu
def test_a_layer_is_prepared_the_same_under_another_default_device():
    from qmoe_amd import sub1, synthetic
    stack = synthetic.build_stack(2, 96, 160, 0.9, seed=5)
    wi, wo = zip(*[synthetic.expert_layers(stack, e) for e in range(2)])
    wo = (wo[0], (wo[1][0].as_subclass(Wrapped),) + tuple(wo[1][1:]))     # one half of the table each way
    x, route = synthetic.activations(4, 96, 6), torch.arange(4, dtype=torch.int32, device='cuda') % 2
    want = stack.prepare().forward(x, route)
    with torch.device('cuda'):
        made = sub1_hip.PreparedStack.from_layers(sub1.DEC[0], wi, wo)
    assert torch.equal(made.forward(x, route).view(torch.int16), want.view(torch.int16))
