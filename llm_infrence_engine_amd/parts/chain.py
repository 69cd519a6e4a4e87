"""A decode step of a narrow model in few launches.

Between two attentions lie four products (output projection, gate/up, down, the next layer's q/k/v) with two norms.  For up to
8 tokens each is over in a few microseconds, most of which are a launch and the wait for weights, so one kernel runs all four
(``ops.decode_chain``): a layer takes two launches instead of five.  Where contexts are short and the attention is the plain one
(heads of 64, no window, sink, cap or slopes, one cache group), that is in the kernel too, and all layers of the step are two launches
(``ops.decode_first``, ``ops.decode_layers``).  Either needs a workspace that outlives the step and belongs to one batch size:
every captured decode graph has its own (``engine/graph.py``), and a runner one for every batch size of the steps that it
launches kernel by kernel (``engine/runner.py``).
"""
from __future__ import annotations

from typing import Optional

import torch

from ..kernels import ops
from .attention import GQAttention
from .blocks import PreNormResidual
from .feed_forward import SwiGLU
from .norms import RMSNorm
from .positions import RotaryHalf


def _sizes(layer) -> Optional[tuple]:
    """(heads, key/value heads, head size, width, intermediate size) of a layer that is made of exactly the parts whose
    arithmetic the chain has; None: it is not."""
    if type(layer) is not PreNormResidual:
        return None
    m, f = layer.mixer, layer.feed_forward
    if type(m) is not GQAttention or type(f) is not SwiGLU or type(m.position) is not RotaryHalf:
        return None
    if type(layer.mixer_norm) is not RMSNorm or type(layer.feed_forward_norm) is not RMSNorm:
        return None
    if m.gate or m.value_blend or m.out_bias or m.value_dim != m.head_dim or m.position.rotary_dim != m.head_dim:
        return None
    if not layer.mixer_norm.size == layer.feed_forward_norm.size == m.hidden_size == f.hidden_size:
        return None
    return m.num_heads, m.num_kv_heads, m.head_dim, m.hidden_size, f.intermediate_size


def _plain_attention(m) -> bool:
    return m.window is None and m.sink_w is None and not m.softcap and m.slopes is None and m.out_scale == 1.0


def _pays(n_tokens: int, sizes: tuple, whole: bool) -> bool:
    """Whether a chain of ``n_tokens`` tokens (``whole``: all layers in two launches) beats the parts one by one.  It saves launches
    and waits, and reads its inputs' words once for every block; of narrow layers that outweighs it from 5 tokens on, whose words are
    twice as many.  The lines are drawn from captured steps of 24 layers of 41 sizes, 64 to 1,024 wide, 33 to 1,100 keys (the chain's
    time over the parts'; values: the weights of a layer):

    chain, up to 4 tokens   0.4M to 0.84M values 0.96 to 1.04; 1.05M 0.94 to 0.98; 4.6M 0.89 to 0.94; 15M 0.75 to 0.85
    chain, 5 to 8           0.4M to 0.84M 1.07 to 1.22; 2.3M 1.03 to 1.09; 3.8M 1.03 to 1.12; 5.77M 0.96 to 1.07; 5.9M to 6.3M 0.92 to
                            1.00 (6.9M and 7.3M up to 1.03 and 1.02, once each); 13M 0.89 to 0.96; 15M 0.81 to 0.85
    whole, up to 4          0.07M 0.77 to 0.87; 1M 0.66 to 0.73; 15M 0.57 to 0.64
    whole, 5 to 8           0.07M 0.85 to 1.02; 0.25M 0.86 to 1.05; 0.44M 0.82 to 0.91; 15M 0.66 to 0.73
    whole, 5 to 8, by tokens x key/value heads, of which each is four blocks that read its keys, beyond 64 more than the CUs: up to 64
                            0.68 to 0.93 at 33 keys, 0.62 to 0.97 at 1,000; 65 to 128 0.77 to 1.02 and 0.92 to 1.10

    A captured step is told no bound of its contexts below 1,024 keys, so what loses at 1,000 is left to the chain.  With these lines no
    measured step takes more than 1.03 of the parts' time (1,128 of them, 0.84 on average)."""
    nh, nkv, d, H, I = sizes
    values = 3 * H * I + 2 * H * d * (nh + nkv)
    if whole:
        return n_tokens * nkv <= 64 and (n_tokens <= 4 or values >= 400_000)
    return values >= (1_000_000 if n_tokens <= 4 else 5_800_000)


def _own_pages(caches, dtype) -> bool:
    """Whether every run stores its keys and values in pages of its own, of ``dtype``."""
    return all(c.kv is not None and c.kv.store and c.kv.k_pages.dtype == dtype for c in caches)


def _plain_layers(model, caches) -> bool:
    """Whether all runs have plain attention of one scale over one group's pages."""
    kv = caches[0].kv
    mixers = [model.layers[run.layer].mixer for run in model.spec.order]
    return (all(_plain_attention(m) and m.scale == mixers[0].scale for m in mixers)
            and all(c.kv.block_table is kv.block_table and c.kv.slot_mapping is kv.slot_mapping and c.kv.window is None
                    and c.kv.v_transposed == kv.v_transposed and c.kv.stride == 1 for c in caches))


def _pages(caches):
    return [t for c in caches for t in (c.kv.k_pages, c.kv.v_pages)]


def _parts(l) -> tuple:
    return l, l.mixer, l.mixer.position, l.feed_forward, l.mixer_norm, l.feed_forward_norm


def _weights(l) -> tuple:
    m, f = l.mixer, l.feed_forward
    return l.mixer_norm.weight, m.w_qkv, m.b_qkv, m.position.inv_freq, m.w_o, l.feed_forward_norm.weight, f.w_gate_up, f.w_down


def _readable(model, align: int) -> bool:
    """Whether the weights are whole rows, and on ``align`` bytes those that are read in pieces (all but biases and frequencies).
    Weights may be views of a larger buffer; the parts' own kernels take them as they come."""
    for run in model.spec.order:
        l = model.layers[run.layer]
        m, f = l.mixer, l.feed_forward
        if any(not t.is_contiguous() or t.data_ptr() % align for t in (m.w_qkv, m.w_o, f.w_gate_up, f.w_down, l.mixer_norm.weight,
                                                                         l.feed_forward_norm.weight)):
            return False
        if not m.position.inv_freq.is_contiguous() or m.b_qkv is not None and not m.b_qkv.is_contiguous():
            return False
    return True


class _Addresses:
    """The parts that a chain runs and the tensors whose addresses a record of them holds: kept alive, and compared with the
    model's and the caches' own before the chain runs again, so that weights loaded anew and layers put in are not missed."""

    def __init__(self, model, caches):
        layers = [model.layers[run.layer] for run in model.spec.order]
        self.parts = [_parts(l) for l in layers]
        self.weights = [t for l in layers for t in _weights(l)]
        self.places = [0 if t is None else t.data_ptr() for t in self.weights]
        self.pages = _pages(caches)

    def hold_weights(self, model) -> bool:
        order, layers = model.spec.order, model.layers
        if len(order) != len(self.parts):
            return False
        now = []
        for run, (layer, mixer, position, feed_forward, mixer_norm, feed_forward_norm) in zip(order, self.parts):
            l = layers[run.layer]
            if (l is not layer or l.mixer is not mixer or mixer.position is not position or l.feed_forward is not feed_forward
                    or l.mixer_norm is not mixer_norm or l.feed_forward_norm is not feed_forward_norm):
                return False
            now += _weights(l)
        return all(a is b and (a is None or a.data_ptr() == place) for a, b, place in zip(now, self.weights, self.places))

    def hold(self, model, caches) -> bool:
        return self.hold_weights(model) and all(a.data_ptr() == b.data_ptr() and a.shape == b.shape
                                                for a, b in zip(self.pages, _pages(caches)))


class FloatLayers:
    """The layers of a step in float32, launched kernel by kernel, by one call (``ops.float_layers``): the kernels that the parts
    would launch one by one, in their order, or, up to 8 tokens of up to 2,048 values, five a layer that take several of them together, to the
    same bits."""

    def __init__(self, model, sizes: tuple, caches):
        self.sizes, self.layers = sizes, [model.layers[run.layer] for run in model.spec.order]
        self.addresses = _Addresses(model, caches)
        nh, nkv, d, _, _ = sizes
        self.records = ops.float_layer_records(
            [dict(norm1=l.mixer_norm.weight, eps1=l.mixer_norm.eps, w_qkv=l.mixer.w_qkv, b_qkv=l.mixer.b_qkv,
                  inv_freq=l.mixer.position.inv_freq, w_o=l.mixer.w_o, norm2=l.feed_forward_norm.weight, eps2=l.feed_forward_norm.eps,
                  w_gate_up=l.feed_forward.w_gate_up, w_down=l.feed_forward.w_down, k_pages=c.kv.k_pages, v_pages=c.kv.v_pages)
             for l, c in zip(self.layers, caches)], nh, nkv, d)

    @classmethod
    def of(cls, model, caches) -> Optional["FloatLayers"]:
        """None where a layer is not of the parts whose kernels these are."""
        runs = model.spec.order
        if model.rt.dtype != torch.float32 or model.pass_entry is not None or any(run.opens_pass is not None for run in runs):
            return None
        sizes = {_sizes(model.layers[run.layer]) for run in runs}
        if len(sizes) != 1 or None in sizes or not _own_pages(caches, torch.float32) or not _plain_layers(model, caches):
            return None
        if not _readable(model, 4):
            return None
        return cls(model, sizes.pop(), caches)

    def takes(self, model, caches) -> bool:
        """Whether these are the weights and the caches that the records were made of."""
        return (len(caches) == len(self.layers) and _own_pages(caches, torch.float32) and self.addresses.hold(model, caches)
                and all(c.kv.slot_mapping is caches[0].kv.slot_mapping for c in caches))

    def check(self) -> None:
        """(Its kernels wait for nothing.)"""

    def forward(self, x, ctx, caches):
        nh, nkv, _, _, I = self.sizes
        kv = caches[0].kv
        return x, ops.float_layers(self.records, len(self.layers), x, ctx.positions, ctx.token_req, kv.slot_mapping, kv.block_table,
                                   kv.table_rows, ctx.n_live_tokens, kv.k_pages, kv.v_transposed, nh, nkv, I, self.layers[0].mixer.scale)


class DecodeChain:
    """The chains of one batch size, with their workspace; ``table``: what ``ops.decode_layers`` reads, where the step's layers
    go in two launches, else None."""

    def __init__(self, model, sizes: tuple, n_bytes: int, caches):
        self.sizes, self.runs = sizes, len(model.spec.order)
        self.layers = [model.layers[run.layer] for run in model.spec.order]
        self.workspace = torch.zeros(n_bytes, dtype=torch.uint8, device=model.rt.device)
        self.table, self.addresses = None, _Addresses(model, caches)
        self.told = torch.zeros(1, dtype=torch.int32)      # not 0: a launch waited in vain (the GPU writes it)
        if self.workspace.is_cuda:
            self.told = self.told.pin_memory()
        self._told = self.told.numpy()
        self.broken_off = False      # a step ended with an exception between its launches, or a launch waited in vain

    @classmethod
    def where_it_pays(cls, model, ctx, caches) -> Optional["DecodeChain"]:
        """``of``, and None also where the parts one by one are as fast or faster (``_pays``)."""
        return cls.of(model, ctx, caches, _pays)

    @classmethod
    def of(cls, model, ctx, caches, pays=lambda n_tokens, sizes, whole: True) -> Optional["DecodeChain"]:
        """For decode steps like ``ctx``, of as many tokens and of contexts on the same side of ``ops.DECODE_KEYS``, from
        ``caches``; None where the kernels do not take the model or the size, or it does not pay."""
        runs, n = model.spec.order, ctx.num_tokens
        if model.rt.dtype != torch.bfloat16 or model.pass_entry is not None or not 2 <= len(runs) <= 1024 or n != ctx.num_requests:
            return None
        if any(run.opens_pass is not None for run in runs):
            return None
        sizes = {_sizes(model.layers[run.layer]) for run in runs}
        if len(sizes) != 1 or None in sizes or not cls._stores(caches) or not _readable(model, 16):
            return None
        sizes = sizes.pop()
        nh, nkv, d, H, I = sizes
        if ctx.max_context_len <= ops.DECODE_KEYS and cls._one_group(model, caches) and pays(n, sizes, True):
            n_bytes = ops.decode_chain_workspace(n, H, nh, nkv, d, I, len(runs))
            if n_bytes:
                chain = cls(model, sizes, n_bytes, caches)
                chain._lay_out(caches)
                return chain
        if not pays(n, sizes, False):
            return None
        n_bytes = ops.decode_chain_workspace(n, H, nh, nkv, d, I)
        return cls(model, sizes, n_bytes, caches) if n_bytes else None

    @classmethod
    def _stores(cls, caches) -> bool:
        return _own_pages(caches, torch.bfloat16)

    @staticmethod
    def _one_group(model, caches) -> bool:
        """Whether the pages are laid out as the kernel reads them, beside ``_plain_layers``."""
        page_size = caches[0].kv.k_pages.shape[2]
        return _plain_layers(model, caches) and caches[0].kv.v_transposed and page_size >= 16 and page_size & (page_size - 1) == 0

    def _lay_out(self, caches):
        rows = []
        for i, (layer, c) in enumerate(zip(self.layers, caches)):
            m, f = layer.mixer, layer.feed_forward
            row = dict(w_o=m.w_o, w_gate_up=f.w_gate_up, w_down=f.w_down, norm2=layer.feed_forward_norm.weight,
                       eps2=layer.feed_forward_norm.eps, k_pages=c.kv.k_pages, v_pages=c.kv.v_pages)
            if i + 1 < len(self.layers):
                then, kv = self.layers[i + 1], caches[i + 1].kv
                row.update(w_front=then.mixer.w_qkv, norm1=then.mixer_norm.weight, eps1=then.mixer_norm.eps, b_front=then.mixer.b_qkv,
                           inv_freq=then.mixer.position.inv_freq, front_k=kv.k_pages, front_v=kv.v_pages)
            rows.append(row)
        self.table = ops.decode_layer_table(rows, self.workspace.device)

    def takes(self, model, caches) -> bool:
        """Whether these are the layers, the weights and the caches that the chain was made for (or, where it reads no table of
        their pages, any caches like them)."""
        if len(caches) != self.runs or not self._stores(caches):
            return False
        return self.addresses.hold_weights(model) if self.table is None else self.addresses.hold(model, caches)

    def check(self) -> None:
        """Raises if a step's launch waited in vain, on the GPU, for what another one should have left: its results are void.  To
        be asked when a step's results have come."""
        if self._told[0]:
            self._told[0], self.broken_off = 0, True
            raise RuntimeError("a decode step's launch waited in vain for its inputs and was broken off; the step's results are void")

    def ready(self) -> None:
        """Before a step's first launch, also a replayed one: its launches count each other up, so behind a step that did not run
        to its end they start over."""
        self.check()
        if self.broken_off:
            ops.decode_chain_start_over(self.workspace)
            self.broken_off = False

    def forward(self, x, ctx, caches):
        """All runs of the order on the embedded tokens ``x`` [N, H], in place; returns x and what is left to add to it (nothing)."""
        self.ready()
        self.broken_off = True
        (self._layer_by_layer if self.table is None else self._whole)(x, ctx, caches)
        self.broken_off = False
        return x, None

    def _whole(self, x, ctx, caches):
        nh, nkv, d, _, I = self.sizes
        first, kv = self.layers[0], caches[0].kv
        m, norm = first.mixer, first.mixer_norm
        ops.decode_first(x, norm.weight, norm.eps, m.w_qkv, m.b_qkv, ctx.positions, m.position.inv_freq, kv.slot_mapping,
                         kv.k_pages, kv.v_pages, nh, nkv, d, I, self.runs, self.workspace)
        ops.decode_layers(self.table, x, ctx.positions, kv.slot_mapping, ctx.context_lens, kv.block_table, kv.table_rows, m.scale,
                          nh, nkv, d, I, kv.k_pages.shape[2], self.runs, self.workspace, self.told, ctx.max_context_len)

    def _layer_by_layer(self, x, ctx, caches):
        nh, nkv, d, _, _ = self.sizes
        layers = self.layers
        q = layers[0].mixer.project_and_store(layers[0].mixer_norm.lazy(x), ctx, caches[0].kv)
        for i, layer in enumerate(layers):
            m, f = layer.mixer, layer.feed_forward
            out = m.attend(q, ctx, caches[i].kv)
            front = None
            if i + 1 < len(layers):
                then, kv = layers[i + 1], caches[i + 1].kv
                front = (then.mixer_norm.weight, then.mixer_norm.eps, then.mixer.w_qkv, then.mixer.b_qkv, ctx.positions,
                         then.mixer.position.inv_freq, kv.slot_mapping, kv.k_pages, kv.v_pages, kv.v_transposed)
            q = ops.decode_chain(out, m.w_o, x, layer.feed_forward_norm.weight, layer.feed_forward_norm.eps, f.w_gate_up,
                                 f.w_down, nh, nkv, d, self.workspace, i, self.runs, front, self.told)
