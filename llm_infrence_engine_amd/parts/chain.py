"""A decode step of a narrow model as attentions and the chains between them.

Between two attentions lie four products (output projection, gate/up, down, the next layer's q/k/v) with two norms.  For up to
8 tokens each is over in a few microseconds, most of which are a launch and the wait for weights, so one kernel runs all four
(``ops.decode_chain``): a layer takes two launches instead of five.  It needs a workspace that outlives the step and belongs
to one batch size: every captured decode graph has its own (``engine/graph.py``), and a runner one for every batch size of
the steps that it launches kernel by kernel (``engine/runner.py``).
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


class DecodeChain:
    """The chains of one batch size, with their workspace."""

    def __init__(self, sizes: tuple, launches: int, n_bytes: int, device):
        self.sizes, self.launches = sizes, launches
        self.workspace = torch.zeros(n_bytes, dtype=torch.uint8, device=device)
        self.broken_off = False      # a step ended with an exception between its launches

    @classmethod
    def of(cls, model, n_tokens: int) -> Optional["DecodeChain"]:
        """For decode steps of ``n_tokens`` tokens; None where the kernel does not take the model or the size."""
        runs = model.spec.order
        if model.rt.dtype != torch.bfloat16 or model.pass_entry is not None or not 2 <= len(runs) <= 1024:
            return None
        if any(run.opens_pass is not None for run in runs):
            return None
        sizes = {_sizes(model.layers[run.layer]) for run in runs}
        if len(sizes) != 1 or None in sizes:
            return None
        sizes = sizes.pop()
        nh, nkv, d, H, I = sizes
        n_bytes = ops.decode_chain_workspace(n_tokens, H, nh, nkv, d, I)
        return cls(sizes, len(runs), n_bytes, model.rt.device) if n_bytes else None

    def takes(self, caches) -> bool:
        """Whether every run stores its keys and values in bfloat16 pages of its own."""
        return len(caches) == self.launches and all(c.kv is not None and c.kv.store and c.kv.k_pages.dtype == torch.bfloat16
                                                    for c in caches)

    def forward(self, model, x, ctx, caches):
        """All runs of the order on the embedded tokens ``x`` [N, H], in place; returns x."""
        if self.broken_off:          # its launches did not count each other up: start over
            self.workspace.zero_()
        self.broken_off = True
        nh, nkv, d, _, _ = self.sizes
        layers = [model.layers[run.layer] for run in model.spec.order]
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
                                 f.w_down, nh, nkv, d, self.workspace, i, self.launches, front)
        self.broken_off = False
        return x
