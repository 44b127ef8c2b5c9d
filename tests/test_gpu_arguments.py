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


def with_one_changed(args, changes):
    for at, values in changes.items():
        for value in values:
            yield args[:at] + (value,) + args[at + 1:]


@pytest.mark.gpu
def test_each_argument_is_looked_at_where_the_tensors_are_in_order():
    """What is refused here is refused for the one thing that is wrong with it."""
    good = (torch.zeros(2, 4, dtype=torch.bfloat16, device='cuda'), torch.zeros(3, dtype=torch.int32, device='cuda'))
    look, fill = _lib.tensor_args().addresses, _lib.tensor_args().layer_addresses
    addresses = [t.data_ptr() for t in good]
    numels = [(8,), (8, 3, 1), [8, 3], (None, 3), (1 << 70, 3), (8.0, 3), (7, 3), (8, 4), None]
    devices = [None, 1, -1, 0.0, 1 << 70, torch.device('cuda:0')]
    specs = [SPEC[:1], SPEC * 2, list(SPEC), (SPEC[0], SPEC[1][:2]), (SPEC[0], list(SPEC[1])), (SPEC[0], (1, 'b', -1)),
             (SPEC[0], (torch.int64, 'b', -1)), (SPEC[0], (torch.int32, 'b', 2)), (SPEC[0], (torch.int32, 'b', None)), None]

    args = (SPEC, good, (8, 3), 0)
    assert list(look(*args)) == addresses
    for broken in with_one_changed(args, {0: specs, 1: [good[:1], list(good), good + good, None], 2: numels, 3: devices}):
        assert look(*broken) is None, broken

    table = torch.full((5, 2), -7, dtype=torch.int64)
    args = (table, 1, [good, good], SPEC, (8, 3), 0)
    assert fill(*args) is True
    assert table.tolist() == [[-7, -7], [addresses[0]] * 2, [addresses[1]] * 2, [-7, -7], [-7, -7]]
    assert fill(table, 3, *args[2:]) is True and table[3:].tolist() == table[1:3].tolist()      # the last rows
    table.fill_(-7)
    wide = torch.full((5, 4), -7, dtype=torch.int64)
    other = [table.int(), table.double(), table.view(-1), table[None], wide, wide[:, ::2], table.cuda(), table.as_subclass(Wrapped),
             table[:2], None]
    layers = [(good, good), [good], [good] * 3, [good, good[:1]], [good, list(good)], [good, good + good], [good, None], None]
    for broken in with_one_changed(args, {0: other, 1: [4, 5, 1 << 40, (1 << 63) - 1, -1, None, 1.0], 2: layers, 3: specs, 4: numels, 5: devices}):
        assert fill(*broken) is False, broken
    assert (wide == -7).all() and (table[0] == -7).all() and (table[3:] == -7).all()


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
