"""Operator module with the surface of the reference's `sub1_cuda` extension
(reference sub1_cuda.cpp:56-59): `sub1matvec` and `sub1pack`, same positional
arguments, tensors in, launched on torch's current stream.  Underneath is the C
ABI of libsub1_hip.so; torch supplies device memory, the stream and, through the
extension _tensor_args, the tensors' addresses.

    import qmoe_amd.sub1_hip as sub1_cuda      # drop-in for `import sub1_cuda`

Additions the reference does not have: argument checking (the reference casts
raw pointers unchecked and silently ignores unsupported shapes,
sub1_cuda_kernel.cu:78-87), `sub1matvec_tokens`, `sub1decode`, and the grouped
expert launch `ExpertStack.forward`.
"""
import ctypes

import torch

from . import _lib

DICT_ENTRIES = _lib.DICT_ENTRIES
PREPARED_MAX_WIDTH = _lib.PREPARED_MAX_WIDTH
Sub1Fault = _lib.Sub1Fault
check_faults = _lib.check_faults


def clear_faults():
    """Reset the library's fault flags once the work that raised them has
    ended (synchronise first).  The stacks zero their workspaces again before
    their next launch, and the static scratch of the launch that does not
    allocate is zeroed here, on the current stream."""
    _lib.clear_faults(_stream())


def _stream():
    """torch's current stream on the current device, as the C ABI takes it."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


class _on_device:
    """`with _on_device(dev):` makes dev the current device for the launch; a
    device that already is costs two cheap calls instead of torch's guard."""

    def __init__(self, device):
        self.want = device.index if device.index is not None else torch._C._cuda_getDevice()
        self.guard = None

    def __enter__(self):
        if torch._C._cuda_getDevice() != self.want:
            self.guard = torch.cuda.device(self.want)
            self.guard.__enter__()

    def __exit__(self, *exc):
        if self.guard is not None:
            self.guard.__exit__(*exc)
        return False


def _launch(device, function, *args):
    """function(*args, torch's current stream there) with `device` as the current one."""
    if torch._C._cuda_getDevice() == device.index:
        status = function(*args, torch._C._cuda_getCurrentRawStream(device.index))
    else:
        with torch.cuda.device(device):
            status = function(*args, _stream())
    _lib.check(status)


def _need(t, dtype, name, device=None, numel=None, dim=None):
    if not isinstance(t, torch.Tensor):
        raise TypeError('%s must be a torch.Tensor' % name)
    if t.dtype != dtype:
        raise TypeError('%s must be %s, got %s' % (name, dtype, t.dtype))
    if not t.is_cuda:
        raise ValueError('%s must live on the GPU' % name)
    if device is not None and t.device != device:
        raise ValueError('%s is on %s, expected %s' % (name, t.device, device))
    if not t.is_contiguous():
        raise ValueError('%s must be contiguous' % name)
    if numel is not None and t.numel() != numel:
        raise ValueError('%s must hold %d elements, got %d' % (name, numel, t.numel()))
    if dim is not None and t.dim() != dim:
        raise ValueError('%s must be %d-D' % (name, dim))
    return t.data_ptr()


def _addresses(spec, tensors, numels, device):
    """Addresses of the tensors, each looked over as _need does: spec holds (dtype,
    name, dimensions or -1), numels the elements or -1.  Plain tensors in order are
    looked over in C++; anything else goes through _need, for its error."""
    got = _lib.tensor_args().addresses(spec, tensors, numels, getattr(device, 'index', None))
    if got is None:
        got = [_need(t, dtype, name, device, None if n < 0 else n, None if dim < 0 else dim)
               for t, (dtype, name, dim), n in zip(tensors, spec, numels)]
    return got


_MATRIX = ((torch.int32, 'dec', -1), (torch.int16, 'w_comp', -1), (torch.int32, 'row_off', -1),
           (torch.bfloat16, 'ter_minmax', -1))
_MATVEC = _MATRIX + ((torch.bfloat16, 'x', -1), (torch.bfloat16, 'y', -1))
_MATVEC_TOKENS = _MATRIX + ((torch.bfloat16, 'x', 2), (torch.bfloat16, 'y', 2))
_ROUTED = ((torch.bfloat16, 'x', 2), (torch.int32, 'token_expert', -1))


def route_from_mask(router_mask):
    """(route int32 [T], expert_index int64 shaped like the mask without its
    last dimension) from a top-1 router's mask [..., E] in one launch:
    expert_index = argmax over the experts (reference sub1.py:311), route the
    same with -1 for a token whose row is all zero (dropped by the router's
    capacity limit: it keeps its input, reference sub1.py:312-318)."""
    if not isinstance(router_mask, torch.Tensor) or not router_mask.is_cuda:
        raise ValueError('router_mask must be a tensor on the GPU')
    size = {torch.int64: 8, torch.int32: 4, torch.uint8: 1, torch.bool: 1}.get(router_mask.dtype)
    if size is None:
        raise TypeError('router_mask must be int64, int32, uint8 or bool, got %s' % router_mask.dtype)
    mask = router_mask.contiguous()
    experts = mask.shape[-1]
    tokens = mask.numel() // experts if experts else 0
    route = torch.empty(tokens, dtype=torch.int32, device=mask.device)
    index = torch.empty(mask.shape[:-1], dtype=torch.int64, device=mask.device)
    if tokens == 0:
        return route, index
    _launch(mask.device, _lib.load().sub1_route_from_mask, mask.data_ptr(), size, tokens, experts,
            route.data_ptr(), index.data_ptr())
    return route, index


def build_tables():
    """(dec int32 [131072], trie int32 [65537, 9]) on the CPU: the fixed
    dictionary of reference sub1.py:29-102, built by the library (C++)."""
    dec = torch.empty(_lib.DEC_WORDS, dtype=torch.int32)
    trie = torch.empty((_lib.TRIE_ROWS, 9), dtype=torch.int32)
    _lib.check(_lib.load().sub1_build_tables(dec.data_ptr(), trie.data_ptr()))
    return dec, trie


def sub1matvec(dec, w_comp, row_off, ter_minmax, x, y):
    """y += W x for one compressed matrix; height = y.numel(), width =
    x.numel() (reference sub1_cuda_kernel.cu:78-79).  Any shape, in place."""
    dev = dec.device if isinstance(dec, torch.Tensor) else None
    _lib.check_faults()
    height, width = y.numel(), x.numel()
    args = _addresses(_MATVEC, (dec, w_comp, row_off, ter_minmax, x, y),
                      (_lib.DEC_WORDS, -1, height + 1, 2 * height, -1, -1), dev)
    _launch(dev, _lib.load().sub1_matvec, *args, height, width)


def sub1matvec_tokens(dec, w_comp, row_off, ter_minmax, x, y):
    """y[t] += W x[t] for x [T, W], y [T, H] in one launch."""
    dev = dec.device if isinstance(dec, torch.Tensor) else None
    args = _addresses(_MATVEC_TOKENS, (dec, w_comp, row_off, ter_minmax, x, y),
                      (_lib.DEC_WORDS, -1, -1, -1, -1, -1), dev)
    tokens, width = x.shape
    height = row_off.numel() - 1
    if y.shape != (tokens, height) or ter_minmax.numel() != 2 * height:
        raise ValueError('y must be [%d, %d] and ter_minmax [%d]' % (tokens, height, 2 * height))
    _launch(dev, _lib.load().sub1_matvec_tokens, *args, height, width, tokens, width, height)


def sub1pack(trie, w_tern, row_off):
    """Greedy dictionary encode of w_tern (int32 [H, W] symbols, CLOBBERED);
    row_off (int32 [H+1]) is overwritten with the cumulative code counts and
    the int16 code stream is returned (reference sub1_cuda_kernel.cu:92-126)."""
    dev = trie.device if isinstance(trie, torch.Tensor) else None
    p_trie = _need(trie, torch.int32, 'trie', numel=_lib.TRIE_ROWS * 9)
    p_w = _need(w_tern, torch.int32, 'w_tern', dev, dim=2)
    height, width = w_tern.shape
    p_ro = _need(row_off, torch.int32, 'row_off', dev, numel=height + 1)
    lib = _lib.load()
    with _on_device(dev):
        _lib.check(lib.sub1_pack_count(p_trie, p_w, p_ro, height, width, _stream()))
        total = int(row_off[height].item())      # the one host sync, as in the reference
        w_comp = torch.empty(total, dtype=torch.int16, device=dev)
        _lib.check(lib.sub1_pack_emit(p_w, p_ro, w_comp.data_ptr(), height, width, _stream()))
    return w_comp


def sub1pack_weights(w):
    """(w_comp int16 [C], row_off int32 [H+1], ter_minmax bf16 [2H]) of dense
    bf16 weights [H, W] whose rows take the values {row min, 0, row max}, by the
    fixed dictionary: what sub1pack gives for their symbols (reference
    sub1.py:145-159)."""
    p_w = _need(w, torch.bfloat16, 'w', dim=2)
    height, width = w.shape
    dev = w.device
    lib = _lib.load()
    row_off = torch.empty(height + 1, dtype=torch.int32, device=dev)
    minmax = torch.empty(2 * height, dtype=torch.bfloat16, device=dev)
    codes = torch.empty((height, (width + 1) // 2), dtype=torch.int16, device=dev)
    with _on_device(dev):
        total = ctypes.c_int32()      # the one wait for the GPU, as in the reference
        _lib.check(lib.sub1_pack_weights_total(p_w, codes.data_ptr(), minmax.data_ptr(), row_off.data_ptr(),
                                               ctypes.byref(total), height, width, _stream()))
        w_comp = torch.empty(total.value, dtype=torch.int16, device=dev)
        _lib.check(lib.sub1_pack_weights_emit(codes.data_ptr(), row_off.data_ptr(), w_comp.data_ptr(),
                                              height, width, _stream()))
    return w_comp, row_off, minmax


def sub1decode(dec, w_comp, row_off, ter_minmax, width, want_tern=True, want_w=True):
    """Decode without multiplying: (symbols uint8 [H, W] or None, weights bf16
    [H, W] or None, number of rows whose codes do not cover the width).  Waits
    for the GPU: the outputs are complete when it returns, on any stream."""
    dev = dec.device if isinstance(dec, torch.Tensor) else None
    height = row_off.numel() - 1
    if ter_minmax is None:
        p_dec, p_wc, p_ro = _addresses(_MATRIX[:3], (dec, w_comp, row_off), (_lib.DEC_WORDS, -1, -1), dev)
        p_mm = None
    else:
        p_dec, p_wc, p_ro, p_mm = _addresses(_MATRIX, (dec, w_comp, row_off, ter_minmax),
                                             (_lib.DEC_WORDS, -1, -1, 2 * height), dev)
    tern = torch.empty((height, width), dtype=torch.uint8, device=dev) if want_tern else None
    w = torch.empty((height, width), dtype=torch.bfloat16, device=dev) if want_w else None
    bad = ctypes.c_int32()
    _launch(dev, _lib.load().sub1_decode_counted, p_dec, p_wc, p_ro, p_mm, tern.data_ptr() if want_tern else None,
            w.data_ptr() if want_w else None, ctypes.byref(bad), height, width)
    return tern, w, bad.value


def _workspace(stack, tokens):
    """The launch's scratch memory (control words and h), one buffer per
    stream: launches on different streams may run at once, launches on one
    stream run in order and share theirs.  Zeroed when it is made; the
    launches leave its control words at zero again, except that a wait which
    gave up may not: once such a fault has been cleared (clear_faults moves
    fault_epoch on), every buffer made before that is zeroed again at its next
    use.  A buffer that has to grow is replaced; the old one goes back to
    torch's allocator, which hands it out again only in the order of the stream
    it was allocated on."""
    need = _lib.load().sub1_moe_workspace_bytes(tokens, stack.d_ff)
    key = _stream()
    epoch = _lib.fault_epoch()
    ws = stack._ws.get(key)
    if ws is None or ws.numel() < need:
        with _on_device(stack.device):
            ws = torch.zeros(need, dtype=torch.uint8, device=stack.device)
        stack._ws[key] = ws
        stack._seen[key] = (0, 0)
        stack._ws_epoch[key] = epoch
    elif stack._ws_epoch.get(key) != epoch:
        ws.zero_()
        stack._seen[key] = (0, 0)
        stack._ws_epoch[key] = epoch
    return ws


def _arguments(stack, x, token_expert):
    """(address of x, of token_expert, tokens) of a forward."""
    p_x, p_te = _addresses(_ROUTED, (x, token_expert), (-1, -1), stack.device)
    tokens, width = x.shape
    if width != stack.d_model:
        raise ValueError('x must be [T, %d]' % stack.d_model)
    if token_expert.numel() != tokens:
        raise ValueError('token_expert must hold %d elements, got %d' % (tokens, token_expert.numel()))
    return p_x, p_te, tokens


def _result(y, x, device):
    """(y, its address): what the caller gave, looked over, or a new tensor like x."""
    if y is None:
        y = torch.empty_like(x)
        return y, y.data_ptr()
    return y, _need(y, torch.bfloat16, 'y', device, numel=x.numel()) if x.shape[0] else None


def _fault_delta(stack, tokens):
    # words 1 and 2 of the workspace count over all launches; report what is new
    key = _stream()
    ctrl = stack.workspace(tokens)[:16].view(torch.int32).tolist()
    before = stack._seen.get(key, (0, 0))
    stack._seen[key] = (ctrl[1], ctrl[2])
    return (ctrl[1] - before[0]) & 0xffffffff, (ctrl[2] - before[1]) & 0xffffffff


class ExpertStack:
    """The Sub1Linear buffers of all experts of one MoE layer, back to back in
    one set of tensors, and the one-launch forward over them.

    wi[e], wo[e] are (w_comp int16 [C], row_off int32 [H+1], ter_minmax bf16
    [2H]) triples as Sub1Linear holds them; wi has H = d_ff, wo has H = d_model.
    """

    def __init__(self, dec, w_comp, wi_code_base, wo_code_base, wi_row_off, wo_row_off,
                 wi_minmax, wo_minmax, d_model, d_ff):
        dev = dec.device
        experts = wi_code_base.numel()
        self.dec, self.w_comp = dec, w_comp
        self.wi_code_base, self.wo_code_base = wi_code_base, wo_code_base
        self.wi_row_off, self.wo_row_off = wi_row_off, wo_row_off
        self.wi_minmax, self.wo_minmax = wi_minmax, wo_minmax
        self.experts, self.d_model, self.d_ff = experts, d_model, d_ff
        self.device = dev
        self._c = _lib.MoeStack(
            _need(dec, torch.int32, 'dec', numel=_lib.DEC_WORDS),
            _need(w_comp, torch.int16, 'w_comp', dev),
            _need(wi_code_base, torch.int64, 'wi_code_base', dev, numel=experts),
            _need(wo_code_base, torch.int64, 'wo_code_base', dev, numel=experts),
            _need(wi_row_off, torch.int32, 'wi_row_off', dev, numel=experts * (d_ff + 1)),
            _need(wo_row_off, torch.int32, 'wo_row_off', dev, numel=experts * (d_model + 1)),
            _need(wi_minmax, torch.bfloat16, 'wi_minmax', dev, numel=experts * 2 * d_ff),
            _need(wo_minmax, torch.bfloat16, 'wo_minmax', dev, numel=experts * 2 * d_model),
            experts, d_model, d_ff)
        self._ws = {}
        self._ws_epoch = {}  # per workspace: fault_epoch() when it was last zeroed
        self._seen = {}      # per workspace: the fault counts launch_faults() last returned from

    @classmethod
    def from_layers(cls, dec, wi_layers, wo_layers):
        """Stack per-expert (w_comp, row_off, ter_minmax) triples."""
        dev = dec.device
        d_ff = wi_layers[0][1].numel() - 1
        d_model = wo_layers[0][1].numel() - 1
        sizes = [t[0].numel() for t in wi_layers] + [t[0].numel() for t in wo_layers]
        bases = torch.zeros(len(sizes) + 1, dtype=torch.int64)
        bases[1:] = torch.tensor(sizes, dtype=torch.int64).cumsum(0)
        n = len(wi_layers)
        w_comp = torch.cat([t[0] for t in wi_layers] + [t[0] for t in wo_layers])
        return cls(dec, w_comp, bases[:n].to(dev), bases[n:2 * n].to(dev),
                   torch.cat([t[1] for t in wi_layers]), torch.cat([t[1] for t in wo_layers]),
                   torch.cat([t[2] for t in wi_layers]), torch.cat([t[2] for t in wo_layers]),
                   d_model, d_ff)

    def compressed_bytes(self):
        """Bytes of the stack a full sweep reads: codes, row offsets, min/max."""
        return (2 * self.w_comp.numel() + 4 * self.wi_row_off.numel()
                + 4 * self.wo_row_off.numel() + 2 * self.wi_minmax.numel()
                + 2 * self.wo_minmax.numel())

    workspace = _workspace
    _arguments = _arguments

    def forward(self, x, token_expert, y=None, matrix_cores=False):
        """y[t] = wo_e(relu(wi_e(x[t]))), e = token_expert[t]; tokens with a
        negative expert keep their input.  x bf16 [T, d_model], token_expert
        int32 [T].  (matrix_cores: see PreparedStack.forward; this layout has
        one form.)"""
        dev = self.device
        _lib.check_faults()       # what earlier launches reported (host memory, no sync)
        p_x, p_te, tokens = self._arguments(x, token_expert)
        y, p_y = _result(y, x, dev)
        if tokens == 0:
            return y
        ws = self.workspace(tokens)
        _launch(dev, _lib.load().sub1_moe_grouped, ctypes.byref(self._c), p_te, p_x, p_y, tokens,
                ws.data_ptr(), ws.numel())
        return y

    def can_prepare(self):
        """Whether the fast layout takes these shapes (it also wants the fixed
        dictionary, which prepare() itself checks)."""
        return max(self.d_model, self.d_ff) <= PREPARED_MAX_WIDTH

    def prepare(self):
        """The fast form of this stack (see PreparedStack); the stack itself
        is left as it is and is not referenced by the result."""
        return PreparedStack(self)

    def launch_faults(self, tokens):
        """(waits that gave up, tokens whose expert id was >= experts and were
        passed through) in the forwards on this stream since the last call of
        this method; both 0 when all is well.  Reads the control words of the
        workspace, synchronising.  A wait that gave up is also reported,
        sticky, by check_faults() and by the next forward()."""
        return _fault_delta(self, tokens)

    check_faults = staticmethod(_lib.check_faults)


class PreparedStack:
    """An ExpertStack decoded once into the form the GPU streams at full width:
    every row's non-zero weights as 7-bit gap entries, rows ordered by length,
    64-row slices, entries interleaved 8 bytes per lane; the kernels keep only
    the activations in LDS.  `forward` has the semantics of
    ExpertStack.forward; a row's fp32 sum is taken in the stream's own order,
    so outputs agree with it to rounding, not to the bit."""

    def __init__(self, stack):
        lib = _lib.load()
        self._make(stack.device, stack.experts, stack.d_model, stack.d_ff,
                   lambda *a: lib.sub1_moe_prepare_layout(ctypes.byref(stack._c), *a),
                   lambda *a: lib.sub1_moe_prepare_codes(ctypes.byref(stack._c), *a))

    @classmethod
    def from_layers(cls, dec, wi_layers, wo_layers):
        """Prepared straight from per-expert (w_comp, row_off, ter_minmax)
        triples, as the experts' Sub1Linear modules hold them: nothing is
        stacked first, the triples are only read."""
        lib = _lib.load()
        dev = dec.device
        experts = len(wi_layers)
        if experts < 1 or len(wo_layers) != experts:
            raise ValueError('as many wi as wo layers, at least one')
        d_ff = wi_layers[0][1].numel() - 1
        d_model = wo_layers[0][1].numel() - 1
        # the tables of addresses, from pinned memory: the copy waits for nothing
        table = torch.empty((6, experts), dtype=torch.int64, device='cpu', pin_memory=True)
        for row, layers, rows in ((0, wi_layers, d_ff), (3, wo_layers, d_model)):
            numels = (-1, rows + 1, 2 * rows)
            if not _lib.tensor_args().layer_addresses(table, row, list(layers), _MATRIX[1:], numels, dev.index):
                codes, offsets, minmax = zip(*layers)
                for tensors, (dtype, name, _), n in zip((codes, offsets, minmax), _MATRIX[1:], numels):
                    table[row] = torch.tensor([_need(t, dtype, name, dev, None if n < 0 else n) for t in tensors],
                                              device='cpu')
                    row += 1
        tables = table.to(dev, non_blocking=True)
        wi_c, wi_r, wi_m, wo_c, wo_r, wo_m = (tables.data_ptr() + 8 * experts * i for i in range(6))
        c_layers = _lib.MoeLayers(_need(dec, torch.int32, 'dec', numel=_lib.DEC_WORDS), wi_c, wo_c,
                                  wi_r, wo_r, wi_m, wo_m, experts, d_model, d_ff)
        self = cls.__new__(cls)
        self._make(dev, experts, d_model, d_ff,
                   lambda *a: lib.sub1_moe_prepare_layout_from_layers(ctypes.byref(c_layers), *a),
                   lambda *a: lib.sub1_moe_prepare_codes_from_layers(ctypes.byref(c_layers), *a))
        return self

    def entry_counts(self):
        """(entries a sweep of all experts walks, entries of the rows
        themselves): the difference is what the stream spends on padding rows
        to the length of their slice."""
        walked, in_rows = ctypes.c_int64(), ctypes.c_int64()
        with _on_device(self.device):
            _lib.check(_lib.load().sub1_moe_prepared_entry_counts(
                ctypes.byref(self._c), ctypes.byref(walked), ctypes.byref(in_rows), _stream()))
        return walked.value, in_rows.value

    def _make(self, dev, experts, d_model, d_ff, layout, codes):
        lib = _lib.load()
        self.device = dev
        self.experts, self.d_model, self.d_ff = experts, d_model, d_ff
        self.batch_tokens = max(128, 8 * experts)     # batch_pays for none below
        meta_bytes = lib.sub1_moe_prepared_meta_bytes(experts, d_model, d_ff)
        if meta_bytes <= 0:
            raise ValueError('bad stack dimensions')
        self.meta = torch.empty(meta_bytes, dtype=torch.uint8, device=dev)
        self._c = _lib.MoePrepared()
        with _on_device(dev):
            _lib.check(layout(self.meta.data_ptr(), meta_bytes, ctypes.byref(self._c), _stream()))
            self.code_bytes = self._c.code_bytes
            self.stream_bytes = self._c.total_chunks * 512     # without the checkpoints
            self.codes = torch.empty(max(self.code_bytes, 256), dtype=torch.uint8, device=dev)
            self._c.codes = self.codes.data_ptr()
            _lib.check(codes(ctypes.byref(self._c), _stream()))
        self._ws = {}
        self._ws_epoch = {}  # per workspace: fault_epoch() when it was last zeroed
        self._seen = {}      # per workspace: the fault counts launch_faults() last returned from

    workspace = _workspace
    _arguments = _arguments

    def forward(self, x, token_expert, y=None, matrix_cores=False):
        """As ExpertStack.forward.  matrix_cores: a batch for which batch_pays
        goes through forward_batch (asked for here, where it costs a small batch
        a comparison)."""
        dev = self.device
        _lib.check_faults()       # what earlier launches reported (host memory, no sync)
        p_x, p_te, tokens = self._arguments(x, token_expert)
        if matrix_cores and tokens >= self.batch_tokens and self.batch_pays(tokens):
            return self.forward_batch(x, token_expert, y)
        y, p_y = _result(y, x, dev)
        if tokens == 0:
            return y
        ws = self.workspace(tokens)
        _launch(dev, _lib.load().sub1_moe_grouped_prepared, ctypes.byref(self._c), p_te, p_x, p_y, tokens,
                ws.data_ptr(), ws.numel())
        return y

    def batch_pays(self, tokens):
        """Whether forward_batch is estimated to be the faster one (it never is
        below 8 tokens an expert, nor with more than 1024 experts: a batch runs in
        pieces of up to 8192 tokens, each of which expands its experts anew)."""
        if tokens < self.batch_tokens:
            return False
        with _on_device(self.device):
            return bool(_lib.load().sub1_moe_batch_pays(ctypes.byref(self._c), tokens))

    def forward_batch(self, x, token_expert, y=None):
        """forward() on the matrix cores, for many tokens per expert: results
        agree with it to rounding, not to the bit, and a token's do not depend
        on the other tokens.  Scratch memory comes from torch's allocator for
        the call: an expert's tokens take whole blocks of 32 slots, at most
        T + 31 (min(T, experts) + 1) of them for T tokens (up to 8192, larger
        batches run in pieces), of 2 d_ff + 2 d_model bytes each and a few more."""
        dev = self.device
        _lib.check_faults()       # what earlier launches reported (host memory, no sync)
        lib = _lib.load()
        p_x, p_te, tokens = self._arguments(x, token_expert)
        y, p_y = _result(y, x, dev)
        if tokens == 0:
            return y
        ws = self.workspace(tokens)
        need = lib.sub1_moe_batch_scratch_bytes(ctypes.byref(self._c), tokens)
        if need <= 0:
            raise ValueError('shapes that forward_batch does not take')
        with _on_device(dev):
            scratch = torch.empty(need, dtype=torch.uint8, device=dev)
            _lib.check(lib.sub1_moe_batch_prepared(
                ctypes.byref(self._c), p_te, p_x, p_y, tokens, ws.data_ptr(), ws.numel(),
                scratch.data_ptr(), need, _stream()))
        return y

    def launch_faults(self, tokens):
        """As ExpertStack.launch_faults."""
        return _fault_delta(self, tokens)

    check_faults = staticmethod(_lib.check_faults)

    def decode(self, expert, projection):
        """uint8 [rows, width]: the symbols of one matrix (projection 0 = wi,
        1 = wo) read back from the prepared stream."""
        rows, width = (self.d_ff, self.d_model) if projection == 0 else (self.d_model, self.d_ff)
        out = torch.empty(rows, width, dtype=torch.uint8, device=self.device)
        with _on_device(self.device):
            _lib.check(_lib.load().sub1_moe_prepared_decode(
                ctypes.byref(self._c), expert, projection, out.data_ptr(), _stream()))
        return out


class PreparedMatrix:
    """Compressed matrices of one shape copied into the fast layout;
    `matvec_tokens(x, y)` does y[t] += W x[t] like sub1matvec_tokens, in one
    launch over the prepared stream.

    One matrix: the three buffers of a Sub1Linear.  Several: pass lists of
    equally shaped buffers (or stacked tensors plus `code_base`, int64 [count],
    the first codeword of each matrix in `w_comp`); `matvec_tokens` then takes
    `token_matrix`, int32 [T], the matrix each token uses."""

    def __init__(self, dec, w_comp, row_off, ter_minmax, width, code_base=None):
        lib = _lib.load()
        dev = dec.device
        if isinstance(w_comp, (list, tuple)):
            sizes = torch.tensor([0] + [t.numel() for t in w_comp], dtype=torch.int64)
            code_base = sizes.cumsum(0)[:-1].to(dev)
            w_comp, row_off, ter_minmax = (torch.cat(list(v)) for v in (w_comp, row_off, ter_minmax))
        count = 1 if code_base is None else code_base.numel()
        if row_off.numel() % count:
            raise ValueError('row_off does not hold %d equal parts' % count)
        height = row_off.numel() // count - 1
        self.device, self.count, self.height, self.width = dev, count, height, width
        src = _lib.MatrixSet(
            _need(dec, torch.int32, 'dec', numel=_lib.DEC_WORDS),
            _need(w_comp, torch.int16, 'w_comp', dev),
            None if code_base is None else _need(code_base, torch.int64, 'code_base', dev),
            _need(row_off, torch.int32, 'row_off', dev, numel=count * (height + 1)),
            _need(ter_minmax, torch.bfloat16, 'ter_minmax', dev, numel=count * 2 * height),
            count, height, width)
        meta_bytes = lib.sub1_matrix_prepared_meta_bytes(count, height, width)
        if meta_bytes <= 0:
            raise ValueError('bad matrix dimensions')
        self.meta = torch.empty(meta_bytes, dtype=torch.uint8, device=dev)
        self._c = _lib.MatrixPrepared()
        with _on_device(dev):
            _lib.check(lib.sub1_matrix_prepare_layout(ctypes.byref(src), self.meta.data_ptr(),
                                                      meta_bytes, ctypes.byref(self._c), _stream()))
            self.codes = torch.empty(max(self._c.code_bytes, 256), dtype=torch.uint8, device=dev)
            self._c.codes = self.codes.data_ptr()
            _lib.check(lib.sub1_matrix_prepare_codes(ctypes.byref(src), ctypes.byref(self._c),
                                                     _stream()))

    def matvec_tokens(self, x, y, token_matrix=None):
        dev = self.device
        p_x = _need(x, torch.bfloat16, 'x', dev, dim=2)
        p_y = _need(y, torch.bfloat16, 'y', dev, dim=2)
        tokens = x.shape[0]
        if x.shape[1] != self.width or y.shape != (tokens, self.height):
            raise ValueError('x must be [T, %d] and y [T, %d]' % (self.width, self.height))
        if token_matrix is None and self.count > 1:
            raise ValueError('token_matrix is required with %d matrices' % self.count)
        p_tm = None if token_matrix is None else _need(token_matrix, torch.int32, 'token_matrix',
                                                       dev, numel=tokens)
        if tokens == 0:
            return
        with _on_device(dev):
            _lib.check(_lib.load().sub1_matvec_prepared(
                ctypes.byref(self._c), p_tm, p_x, self.width, p_y, self.height, tokens, _stream()))

    def product_tokens(self, x):
        """W x[t] for all tokens of x [T, width] into a new tensor: what
        matvec_tokens adds onto zeros, without the fill.  One matrix."""
        p_x = _need(x, torch.bfloat16, 'x', self.device, dim=2)
        tokens = x.shape[0]
        if x.shape[1] != self.width:
            raise ValueError('x must be [T, %d]' % self.width)
        if self.count > 1:
            raise ValueError('token_matrix is required with %d matrices' % self.count)
        y = torch.empty((tokens, self.height), dtype=torch.bfloat16, device=self.device)
        if tokens:
            _launch(self.device, _lib.load().sub1_product_prepared, ctypes.byref(self._c), p_x, self.width,
                    y.data_ptr(), self.height, tokens)
        return y

    def decode(self, matrix=0):
        """uint8 [height, width]: the symbols of one matrix read back from the
        prepared stream."""
        out = torch.empty(self.height, self.width, dtype=torch.uint8, device=self.device)
        with _on_device(self.device):
            _lib.check(_lib.load().sub1_matrix_prepared_decode(
                ctypes.byref(self._c), matrix, out.data_ptr(), _stream()))
        return out


class TiledMatrix:
    """Compressed matrices of one shape copied into the tile form that the
    matrix cores multiply from; `matvec_tokens(x, y)` does y[t] += W x[t] for
    all tokens of x [T, width] in one launch, the weights decoded once per
    tile of 64 tokens (made for sequences: from a few dozen tokens on it beats
    walking the non-zeros per token; results agree with the other paths to
    rounding, not to the bit).  Arguments as PreparedMatrix."""

    def __init__(self, dec, w_comp, row_off, ter_minmax, width, code_base=None):
        lib = _lib.load()
        dev = dec.device
        if isinstance(w_comp, (list, tuple)):
            sizes = torch.tensor([0] + [t.numel() for t in w_comp], dtype=torch.int64)
            code_base = sizes.cumsum(0)[:-1].to(dev)
            w_comp, row_off, ter_minmax = (torch.cat(list(v)) for v in (w_comp, row_off, ter_minmax))
        count = 1 if code_base is None else code_base.numel()
        if row_off.numel() % count:
            raise ValueError('row_off does not hold %d equal parts' % count)
        height = row_off.numel() // count - 1
        self.device, self.count, self.height, self.width = dev, count, height, width
        src = _lib.MatrixSet(
            _need(dec, torch.int32, 'dec', numel=_lib.DEC_WORDS),
            _need(w_comp, torch.int16, 'w_comp', dev),
            None if code_base is None else _need(code_base, torch.int64, 'code_base', dev),
            _need(row_off, torch.int32, 'row_off', dev, numel=count * (height + 1)),
            _need(ter_minmax, torch.bfloat16, 'ter_minmax', dev, numel=count * 2 * height),
            count, height, width)
        meta_bytes = lib.sub1_tiles_meta_bytes(count, height, width)
        if meta_bytes <= 0:
            raise ValueError('bad matrix dimensions')
        self.meta = torch.empty(meta_bytes, dtype=torch.uint8, device=dev)
        self._c = _lib.Tiles()
        with _on_device(dev):
            _lib.check(lib.sub1_tiles_layout(ctypes.byref(src), self.meta.data_ptr(), meta_bytes,
                                             ctypes.byref(self._c), _stream()))
            self.entries = torch.empty(max(self._c.entry_bytes, 256), dtype=torch.uint8, device=dev)
            self._c.entries = self.entries.data_ptr()
            _lib.check(lib.sub1_tiles_entries(ctypes.byref(src), ctypes.byref(self._c), _stream()))

    def matvec_tokens(self, x, y, matrix=0):
        dev = self.device
        p_x = _need(x, torch.bfloat16, 'x', dev, dim=2)
        p_y = _need(y, torch.bfloat16, 'y', dev, dim=2)
        tokens = x.shape[0]
        if x.shape[1] != self.width or y.shape != (tokens, self.height):
            raise ValueError('x must be [T, %d] and y [T, %d]' % (self.width, self.height))
        if tokens == 0:
            return
        with _on_device(dev):
            _lib.check(_lib.load().sub1_matvec_tiles(
                ctypes.byref(self._c), matrix, p_x, self.width, p_y, self.height, tokens, _stream()))

    def product_tokens(self, x, matrix=0):
        """W x[t] for all tokens of x [T, width] into a new tensor: what
        matvec_tokens adds onto zeros, without the fill."""
        p_x = _need(x, torch.bfloat16, 'x', self.device, dim=2)
        tokens = x.shape[0]
        if x.shape[1] != self.width:
            raise ValueError('x must be [T, %d]' % self.width)
        y = torch.empty((tokens, self.height), dtype=torch.bfloat16, device=self.device)
        if tokens:
            _launch(self.device, _lib.load().sub1_product_tiles, ctypes.byref(self._c), matrix, p_x, self.width,
                    y.data_ptr(), self.height, tokens)
        return y

    def decode(self, matrix=0):
        """uint8 [height, width]: the symbols of one matrix read back from the
        tile form."""
        out = torch.empty(self.height, self.width, dtype=torch.uint8, device=self.device)
        with _on_device(self.device):
            _lib.check(_lib.load().sub1_tiles_decode(ctypes.byref(self._c), matrix, out.data_ptr(),
                                                     _stream()))
        return out
