"""Which kernel a call goes to, where that is a rule on sizes in the library: host code alone, so these run without a GPU (the
library then takes the chip to have 256 compute units, as it has)."""
from types import SimpleNamespace

import pytest
import torch


@pytest.fixture(scope="module")
def ops():
    from llm_infrence_engine_amd.kernels import ops

    return ops


@pytest.mark.parametrize("R,N,most,longest,nh,nkv,d,window,exact,kind", [
    # us of the other kernel, wide, narrow, narrow with twice the groups
    (8, 4096, 512, 512, 14, 2, 64, 0, 1, 1),            # 25.8 19.1 22.2 27.0
    (48, 1680, 35, 35, 16, 8, 64, 0, 1, 1),             # 14.8 9.8 11.6 17.9
    (6, 1644, 274, 274, 32, 4, 64, 0, 1, 1),            # 21.9 15.3 16.9 22.5
    (4, 1436, 1013, 4955, 28, 4, 128, 0, 1, 0),         # 69 160 106 74: the longest context belongs to 13 tokens
    (9, 953, 945, 3535, 40, 8, 128, 0, 1, 0),           # 57 112 76 56: to a single token
    (24, 456, 19, 845, 28, 4, 128, 0, 1, 0),            # 27 33 29 35
    (8, 2048, 256, 256, 28, 4, 128, 0, 1, 1),           # 36 20.7 22.9 33
    (64, 1536, 1536, 8192, 32, 4, 64, 0, 0, 2),         # a capture's bounds; 32 portions of 42 tokens: 16.2 11.3 12.4 18.9
    (64, 256, 256, 8192, 14, 2, 64, 0, 0, 2),
    (64, 512, 512, 4096, 28, 4, 128, 0, 0, 0),          # 24 portions of 20 tokens: 9.7 9.3 8.1 12.5
    (16, 768, 768, 4096, 16, 2, 128, 0, 0, 0),          # 607 tokens beside single ones of 4,000 keys: 51 123 83 59
    # as before
    (1, 2048, 2048, 2048, 14, 2, 64, 0, 1, 2), (3, 396, 171, 171, 14, 2, 64, 0, 1, 2), (1, 3910, 3910, 12105, 14, 2, 64, 0, 1, 3),
    (1, 2345, 2345, 10186, 14, 2, 64, 256, 1, 2), (1, 910, 910, 910, 28, 4, 128, 0, 1, 3), (1, 2059, 2059, 2059, 28, 4, 128, 0, 1, 2),
    (1, 3077, 3077, 3077, 28, 4, 128, 0, 1, 1), (30, 60, 2, 2, 14, 2, 64, 0, 1, 0),
    (1, 800, 800, 4000, 28, 4, 128, 0, 1, 2), (1, 100, 400, 400, 14, 2, 64, 0, 1, 2), (3, 100, 90, 100, 7, 2, 64, 0, 1, 0)])
def test_kind_of_prompt_attention(ops, R, N, most, longest, nh, nkv, d, window, exact, kind):
    """Measured on both sides of its lines: even portions that fill the chip once as they are, contexts that say nothing of the
    longest portion, and what a captured step knows of those that will run in it."""
    assert ops._get("ms_attention_prompt_kind")(R, N, most, longest, nh, nkv, d, 16, window, exact) == kind


@pytest.mark.parametrize("captured", [False, True])
def test_a_captured_step_says_that_its_lengths_are_bounds(ops, monkeypatch, captured):
    seen = {}

    def attention(*args):
        seen["exact"] = args[17]

    monkeypatch.setattr(ops, "paged_attention_mfma", attention)
    pages = torch.zeros(2, 2, 16, 64, dtype=torch.bfloat16)
    kv = SimpleNamespace(k_pages=pages, v_pages=pages.transpose(2, 3).contiguous(), v_transposed=True, block_table=None, table_rows=None)
    ctx = SimpleNamespace(q_start=None, context_lens=None, max_q_len=4, max_context_len=16,
                          n_live_tokens=torch.zeros(1, dtype=torch.int32) if captured else None)
    q = torch.zeros(4, 4 * 64, dtype=torch.bfloat16)
    ops.paged_attention(q, kv, ctx, torch.empty_like(q), 4, 0.125)
    assert seen["exact"] is not captured


@pytest.mark.parametrize("M,N,K,gated,relu2", [
    # times of the library and the activation's kernel over the tiled kernel's: silu, squared relu
    (300, 14336, 3584, 0, 0),         # 0.88 0.88: tiles of 128 fill half a round
    (305, 16384, 3072, 0, 0),         # 0.88
    (2305, 11008, 4096, 0, 0),        # 0.93 0.88
    (3072, 5248, 3008, 0, 0),         # 0.71 0.69: 21 tiles of features over 8 XCDs
    (2305, 19200, 4928, 0, 0),        # 0.80 0.80
    (1024, 37888, 3584, 1, 0), (2176, 37888, 3584, 1, 0), (4096, 22016, 2048, 1, 0), (256, 22016, 2048, 1, 0), (3000, 27648, 5120, 1, 0),
    (2048, 8192, 3072, 1, 1), (70, 37888, 3584, 1, 0), (193, 18944, 3072, 0, 0),
    # both as ever: full rounds, short rows; rows that are no multiple of 64, long ones
    (2048, 37888, 3584, 1, 1), (1300, 55296, 5120, 1, 1), (8192, 9728, 896, 1, 1), (65, 7296, 1536, 1, 1), (512, 8192, 2056, 0, 0),
    (4096, 28672, 8192, 0, 0), (256, 15360, 4096, 0, 0)])
def test_where_the_tiled_kernel_takes_products_with_an_activation(ops, M, N, K, gated, relu2):
    assert ops._get("ms_gemm_tiled_pays")(M, N, K) == gated
    assert ops._get("ms_gemm_tiled_relu2_pays")(M, N, K) == relu2
    if M * max(N, K) < 1 << 24:
        a, w = torch.empty(M, K, dtype=torch.bfloat16), torch.empty(N, K, dtype=torch.bfloat16)
        assert ops.gemm_tiled_pays(a, w, ops.EPI_RELU2) == bool(relu2) and ops.gemm_tiled_pays(a, w, ops.EPI_GEGLU) == bool(gated)


@pytest.mark.parametrize("M,N,K,taken", [
    # times of the other way over partial sums
    (300, 2048, 896, 0), (512, 7296, 896, 0), (384, 4096, 4096, 0), # 0.95 0.88 0.94
    (429, 4480, 6784, 0), (261, 6016, 7296, 0), (437, 6400, 8192, 0),   # 0.82 0.84 0.90
    (900, 3072, 8192, 0), (791, 6080, 8448, 0),                         # 0.89 0.90
    (128, 8192, 2048, 1), (256, 896, 896, 1), (240, 5056, 896, 1), (256, 4096, 4096, 1), (512, 896, 896, 1), (390, 896, 4864, 1),
    (512, 2048, 5632, 1), (512, 3584, 18944, 1), (512, 2048, 8192, 1), (1024, 3584, 18944, 1), (900, 5120, 13824, 1),
    (640, 8192, 28672, 1), (2048, 3584, 18944, 1), (1300, 5120, 27648, 1),
    # as ever
    (64, 896, 4864, 0), (200, 1536, 2048, 0), (1024, 896, 4864, 0), (1600, 3584, 18944, 0), (2048, 4096, 28672, 0), (100, 8256, 4096, 0)])
def test_where_products_of_many_rows_leave_partial_sums(ops, M, N, K, taken):
    assert (ops._get("ms_gemm_tiled_sums_parts")(M, N, K) > 0) == bool(taken)


# ---------------------------------------------------------------- who may leave sums undone, and who may be given them
def _block(ops, norm=None, mixer=None, feed_forward=None, block=None):
    from llm_infrence_engine_amd.parts.attention import GQAttention
    from llm_infrence_engine_amd.parts.blocks import PreNormResidual
    from llm_infrence_engine_amd.parts.feed_forward import SwiGLU
    from llm_infrence_engine_amd.parts.norms import RMSNorm

    def of(base, body):
        if body is True:
            return base
        return type("Own", body if isinstance(body, tuple) else (base,), {} if body is None or isinstance(body, tuple) else body)

    norms = [of(RMSNorm, norm)("", 64, 1e-5) for _ in range(2)]
    m = of(GQAttention, mixer)("", None, 64, 2, 2, 32, 0.1)
    f = of(SwiGLU, feed_forward)("", 64, 128)
    return of(PreNormResidual, block)(position=None, mixer_norm=norms[0], mixer=m, feed_forward_norm=norms[1], feed_forward=f)


def test_parts_of_a_programs_own_see_one_addend(ops):
    """Partial sums pass between the parts that were written for them: a class derived from one of these, with a method of its
    own (here or in a class beside it), is handed one addend and leaves one, unless it says that it knows better."""
    from llm_infrence_engine_amd.parts.norms import RMSNorm

    def flags(b):
        return b.takes_sums, b.mixer.hands_on_sums, b.feed_forward.hands_on_sums

    own = lambda self, *a, **k: None     # noqa: E731
    beside = type("Beside", (), {"forward": own})
    assert flags(_block(ops)) == (True, True, True)
    assert flags(_block(ops, norm={"forward": own})) == flags(_block(ops, norm={"lazy": own})) == (False, False, True)
    assert flags(_block(ops, norm=(beside, RMSNorm))) == (False, False, True)
    assert flags(_block(ops, norm={"forward": own, "takes_sums": True})) == (True, True, True)
    assert flags(_block(ops, norm={"other": own})) == (True, True, True)
    assert flags(_block(ops, mixer={"forward_residual": own})) == (True, False, True)
    assert flags(_block(ops, feed_forward={"forward_residual": own})) == (True, True, False)
    assert flags(_block(ops, block={"forward": own})) == (False, False, False)


@pytest.mark.gpu
@pytest.mark.parametrize("reader", ["norm", "own norm", "layer norm", "block", "own block", None])
def test_the_model_adds_up_sums_for_a_reader_that_takes_one_addend(ops, reader):
    """Three partial sums of 5 rows by 64, before each kind of reader and before nobody's (an entry into another pass)."""
    from llm_infrence_engine_amd.parts.model import Model
    from llm_infrence_engine_amd.parts.norms import LayerNorm, RMSNorm

    own = {"forward": lambda self, *a, **k: None}
    r = {"norm": lambda: RMSNorm("", 64, 1e-5), "own norm": lambda: type("Own", (RMSNorm,), own)("", 64, 1e-5),
         "layer norm": lambda: LayerNorm("", 64, 1e-5), "block": lambda: _block(ops), "own block": lambda: _block(ops, norm=own),
         None: lambda: None}[reader]()
    g = torch.Generator().manual_seed(7)
    x0, sums = torch.randn(5, 64, generator=g), torch.randn(3, 5, 64, generator=g)
    x, pending = x0.cuda(), sums.cuda()
    left = Model._settled(x, pending, r)
    if reader in ("norm", "block"):
        assert left is pending and torch.equal(x.cpu(), x0)
    else:
        assert left is None
        torch.testing.assert_close(x.cpu().double(), x0.double() + sums.double().sum(0), atol=2e-6, rtol=2e-6)


def test_chains_take_the_parts_whose_arithmetic_they_have(ops):
    """Layers of exactly the parts that the kernel of a decode step's products stands in for, and no class derived from one;
    whatever it has no place for (a bias behind the heads, gates, blended values, heads turned in part) goes layer by layer."""
    from llm_infrence_engine_amd.parts import chain
    from llm_infrence_engine_amd.parts.attention import GQAttention
    from llm_infrence_engine_amd.parts.positions import RotaryHalf

    exact = dict(norm=True, mixer=True, feed_forward=True, block=True)

    def sizes(turned=32, **attention):
        b = _block(ops, **exact)
        b.mixer = GQAttention("", RotaryHalf("", 32, turned, 1e4), 64, 2, 2, 32, 0.1, **attention)
        return chain._sizes(b)

    assert sizes() == sizes(qkv_bias=False) == sizes(window=8, sink=True) == (2, 2, 32, 64, 128)
    assert sizes(turned=16) is sizes(out_bias=True) is sizes(gate=True) is sizes(value_blend="first") is None
    own = {"other": lambda self: None}
    for part in ("norm", "mixer", "feed_forward", "block"):
        b = _block(ops, **dict(exact, **{part: own}))
        b.mixer.position = RotaryHalf("", 32, 32, 1e4)
        assert chain._sizes(b) is None
    assert chain._sizes(_block(ops, **exact)) is None      # no position encoding

    def of(n=8, runs=2, opens=None, dtype=torch.bfloat16, entry=None, keys=64, store=True, page=16, transposed=True, **attention):
        b = _block(ops, **exact)
        b.mixer = GQAttention("", RotaryHalf("", 64, 64, 1e4), 64, 2, 1, 64, 0.1, **attention)
        b.load = None
        for part, names in ((b.mixer, ("w_o", "w_qkv", "b_qkv", "sink_w")), (b.feed_forward, ("w_gate_up", "w_down")),
                            (b.mixer_norm, ("weight",)), (b.feed_forward_norm, ("weight",)), (b.mixer.position, ("inv_freq",))):
            for name in names:
                setattr(part, name, torch.zeros(1))
        b.mixer.sink_w = torch.zeros(1) if b.mixer.sink else None
        m = SimpleNamespace(spec=SimpleNamespace(order=[SimpleNamespace(layer=0, opens_pass=opens)] * runs), layers=[b],
                            rt=SimpleNamespace(dtype=dtype, device="cpu"), pass_entry=entry)
        table, slots, pages = torch.zeros(1), torch.zeros(1), torch.zeros(1, 1, page, 64, dtype=torch.bfloat16)
        caches = [SimpleNamespace(kv=SimpleNamespace(k_pages=pages.clone(), v_pages=pages.clone(), block_table=table, slot_mapping=slots,
                                                     v_transposed=transposed, window=b.mixer.window, stride=1, store=store))
                  for _ in range(runs)]
        made = chain.DecodeChain.of(m, SimpleNamespace(num_tokens=n, num_requests=n, max_context_len=keys), caches)
        assert made is None or made.takes(m, caches) and not made.workspace.any()
        if made is not None and made.table is not None:      # weights loaded anew, pages elsewhere
            b.feed_forward.w_down = b.feed_forward.w_down.clone()
            assert not made.takes(m, caches)
            b.feed_forward.w_down = made.addresses.weights[-1]
            caches[-1].kv.k_pages = caches[-1].kv.k_pages.clone()
            assert not made.takes(m, caches)
        return None if made is None else "layers" if made.table is None else "step"

    assert of() == of(keys=1024) == of(page=32) == "step"
    assert of(keys=1025) == of(window=8) == of(sink=True) == of(softcap=9.0) == of(page=48) == of(transposed=False) == of(out_scale=2.0) == "layers"
    assert of(9) is of(runs=1) is of(opens=0) is of(dtype=torch.float32) is of(entry=b"") is of(store=False) is None


def _decode_stand_in(ops, keys=64, runs=2):
    """(model, its one layer, caches, what DecodeChain.of says of them now) of parts that chains take; weights are stand-ins."""
    from llm_infrence_engine_amd.parts import chain
    from llm_infrence_engine_amd.parts.attention import GQAttention
    from llm_infrence_engine_amd.parts.positions import RotaryHalf

    b = _block(ops, norm=True, mixer=True, feed_forward=True, block=True)
    b.mixer = GQAttention("", RotaryHalf("", 64, 64, 1e4), 64, 2, 1, 64, 0.1)
    for part, names in ((b.mixer, ("w_o", "w_qkv", "b_qkv")), (b.feed_forward, ("w_gate_up", "w_down")),
                        (b.mixer_norm, ("weight",)), (b.feed_forward_norm, ("weight",)), (b.mixer.position, ("inv_freq",))):
        for name in names:
            setattr(part, name, torch.zeros(4, 4))
    b.mixer.sink_w = None
    m = SimpleNamespace(spec=SimpleNamespace(order=[SimpleNamespace(layer=0, opens_pass=None)] * runs), layers=[b],
                        rt=SimpleNamespace(dtype=torch.bfloat16, device="cpu"), pass_entry=None)
    table, slots, pages = torch.zeros(1), torch.zeros(1), torch.zeros(1, 1, 16, 64, dtype=torch.bfloat16)
    caches = [SimpleNamespace(kv=SimpleNamespace(k_pages=pages.clone(), v_pages=pages.clone(), block_table=table, slot_mapping=slots,
                                                 v_transposed=True, window=None, stride=1, store=True)) for _ in range(runs)]
    return m, b, caches, lambda: chain.DecodeChain.of(m, SimpleNamespace(num_tokens=8, num_requests=8, max_context_len=keys), caches)


@pytest.mark.parametrize("keys", [64, 2000])
def test_chains_leave_weights_they_cannot_read_to_the_parts(ops, keys):
    """Views of a larger buffer, as a reader of weights may hand out: the products have a kernel for any address and any row
    stride, the chains only for whole rows on 16 bytes.  Biases and frequencies are read one by one."""
    from llm_infrence_engine_amd.parts import chain

    m, b, caches, of = _decode_stand_in(ops, keys)
    aside, strided = torch.zeros(17)[1:].view(4, 4), torch.zeros(4, 8)[:, :4]
    assert aside.data_ptr() % 16 and not strided.is_contiguous() and of() is not None
    for part, name in ((b.mixer, "w_o"), (b.mixer, "w_qkv"), (b.feed_forward, "w_gate_up"), (b.feed_forward, "w_down"),
                       (b.mixer_norm, "weight"), (b.feed_forward_norm, "weight")):
        kept = getattr(part, name)
        for other in (aside, strided):
            setattr(part, name, other)
            assert of() is None
        m.rt.dtype = torch.float32      # all layers of a 32-bit step by one call: any address, whole rows
        for c in caches:
            c.kv.k_pages, c.kv.v_pages = c.kv.k_pages.float(), c.kv.v_pages.float()
        assert chain.FloatLayers.of(m, caches) is None
        m.rt.dtype = torch.bfloat16
        for c in caches:
            c.kv.k_pages, c.kv.v_pages = c.kv.k_pages.bfloat16(), c.kv.v_pages.bfloat16()
        setattr(part, name, kept)
    b.mixer.b_qkv = b.mixer.position.inv_freq = aside
    assert of() is not None
    b.mixer.b_qkv = None
    assert of() is not None


@pytest.mark.parametrize("keys", [64, 2000])
def test_a_chain_holds_for_the_layers_and_weights_it_was_made_of(ops, keys):
    """With or without a table of addresses: another storage under the same tensor, another tensor, another part and another
    layer in a model's place are all seen before the chain runs again."""
    m, b, caches, of = _decode_stand_in(ops, keys)
    made = of()
    assert made.takes(m, caches) and (made.table is None) == (keys == 2000)
    kept = b.mixer.w_o.data
    b.mixer.w_o.data = kept.clone()
    assert not made.takes(m, caches)
    b.mixer.w_o.data = kept
    assert made.takes(m, caches)
    other = _decode_stand_in(ops, keys)[1]
    for part in ("mixer", "feed_forward", "mixer_norm", "feed_forward_norm"):
        kept = getattr(b, part)
        setattr(b, part, SimpleNamespace(weight=getattr(kept, "weight", None)))      # (without what the chain reads of it)
        assert not made.takes(m, caches)
        setattr(b, part, kept)
    kept, b.mixer.position = b.mixer.position, other.mixer.position
    assert not made.takes(m, caches)
    b.mixer.position = kept
    m.layers[0] = other
    assert not made.takes(m, caches)
    m.layers[0] = b
    assert made.takes(m, caches)
    m.spec.order = m.spec.order[:1]
    assert not made.takes(m, caches)


@pytest.mark.parametrize("tokens,sizes,keys,kind", [
    # time of a decode step of 24 such layers over the parts' own: layer by layer, all layers in two launches (at 33, 577, 1,000 keys)
    (1, (14, 2, 64, 896, 4864), 1000, "step"),       # 0.85; 0.62 0.59 0.58
    (8, (14, 2, 64, 896, 4864), 1000, "step"),       # 0.84; 0.73 0.70 0.68
    (8, (14, 2, 64, 896, 4864), 2000, "layers"),     # 0.84
    (4, (2, 1, 64, 128, 512), 64, "step"),           # 1.02; 0.79 0.71
    (4, (2, 1, 64, 128, 512), 2000, None),           # 1.02
    (8, (2, 1, 64, 128, 512), 64, None),             # 1.26; 1.05 0.93
    (1, (4, 2, 64, 256, 768), 2000, None),           # 0.99
    (4, (4, 4, 64, 256, 1024), 2000, "layers"),      # 0.97
    (8, (3, 3, 64, 192, 512), 64, "step"),           # 1.22; 0.91 0.82
    (8, (8, 8, 64, 512, 1536), 64, "step"),          # 1.04; 0.84 0.85 0.89
    (8, (8, 8, 64, 512, 1536), 2000, None),          # 1.04
    (8, (4, 4, 128, 512, 1536), 64, None),           # 1.07, heads of 128
    (4, (4, 4, 128, 512, 1536), 64, "layers"),       # 0.97
    (7, (16, 16, 64, 1024, 512), 2000, None),        # 1.06
    (5, (5, 1, 128, 640, 2560), 64, "layers"),       # 0.98
    (4, (16, 16, 64, 1024, 2048), 64, "step"),       # 0.91; 0.76 0.86 0.93
    (7, (16, 16, 64, 1024, 2048), 64, "layers"),     # 1.00; 0.92 1.01 1.09
    (8, (12, 12, 64, 768, 2048), 64, "layers"),      # 0.97; 0.88 0.93 1.04
    (8, (16, 8, 64, 1024, 4096), 64, "step"),        # 0.90; 0.79 0.82 0.88
    (8, (16, 16, 64, 1024, 512), 64, None)])         # 1.01
def test_chains_run_where_they_pay(ops, tokens, sizes, keys, kind):
    """Measured on both sides of the lines, at which the parts' own launches are as fast or faster."""
    from llm_infrence_engine_amd.parts import chain
    from llm_infrence_engine_amd.parts.attention import GQAttention
    from llm_infrence_engine_amd.parts.positions import RotaryHalf

    nh, nkv, d, H, I = sizes
    m, b, caches, of = _decode_stand_in(ops, keys)
    kept = b.mixer
    b.mixer = GQAttention("", RotaryHalf("", d, d, 1e4), H, nh, nkv, d, 0.1)
    b.mixer.w_o, b.mixer.w_qkv, b.mixer.b_qkv, b.mixer.sink_w = kept.w_o, kept.w_qkv, kept.b_qkv, None
    b.mixer.position.inv_freq = kept.position.inv_freq
    b.mixer_norm.size = b.feed_forward_norm.size = b.feed_forward.hidden_size = H
    b.feed_forward.intermediate_size = I
    made = chain.DecodeChain.where_it_pays(m, SimpleNamespace(num_tokens=tokens, num_requests=tokens, max_context_len=keys), caches)
    assert (None if made is None else "layers" if made.table is None else "step") == kind


def test_a_chains_launches_are_refused_out_of_their_turn(ops, monkeypatch):
    """A launch waits for words of the one before it in the step, and their numbers go by how many have run: the next one due on a
    workspace, of the same sizes, or none.  A launch that was refused does not count; a workspace that starts over takes any."""
    launched = []

    def call(name, *args):
        if name == broken[0]:
            raise RuntimeError("refused")
        launched.append(name)

    broken = [None]
    monkeypatch.setattr(ops, "_check", lambda *args, **kw: None)
    monkeypatch.setattr(ops, "_call", call)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    bf = dict(dtype=torch.bfloat16)

    def args(M, H=64, I=64, nh=2, nkv=1, d=64):
        return dict(x=torch.zeros(M, H), norm=torch.ones(H), w_qkv=torch.zeros((nh + 2 * nkv) * d, H, **bf), pos=torch.zeros(M, dtype=torch.int32),
                    f=torch.ones(d // 2), k=torch.zeros(2, nkv, 16, d, **bf), v=torch.zeros(2, nkv, d, 16, **bf), attn=torch.zeros(M, nh * d, **bf),
                    w_o=torch.zeros(H, nh * d, **bf), w_gu=torch.zeros(2 * I, H, **bf), w_down=torch.zeros(H, I, **bf), table=torch.zeros(M, 4, dtype=torch.int32),
                    sizes=(nh, nkv, d, I))

    def first(ws, M=2, L=3):
        a = args(M)
        ops.decode_first(a["x"], a["norm"], 1e-6, a["w_qkv"], None, a["pos"], a["f"], a["pos"], a["k"], a["v"], *a["sizes"], L, ws)

    def layers(ws, M=2, L=3):
        a = args(M)
        records = torch.zeros(L * ops._get("ms_decode_layer_bytes")(), dtype=torch.uint8)
        records.layer_sizes = (2, 1, 64, 64, 64, 16)
        ops.decode_layers(records, a["x"], a["pos"], a["pos"], a["pos"], a["table"], None, 1.0, *a["sizes"], 16, L, ws)

    def chain(ws, launch, launches=3, M=2):
        a = args(M)
        ops.decode_chain(a["attn"], a["w_o"], a["x"], a["norm"], 1e-6, a["w_gu"], a["w_down"], *a["sizes"][:3], ws, launch, launches)

    def refused(run, *which, **sizes):
        n = len(launched)
        with pytest.raises(ValueError, match="turn|sizes"):
            run(*which, **sizes)
        assert len(launched) == n

    new = lambda: torch.zeros(ops.decode_chain_workspace(8, 64, 2, 1, 64, 64, 8), dtype=torch.uint8)     # noqa: E731
    ws = new()
    refused(layers, ws)
    for _ in range(3):
        first(ws)
        refused(first, ws)
        for other in (dict(M=3), dict(L=4)):
            refused(layers, ws, **other)
        layers(ws)
        refused(layers, ws)
        refused(first, ws, M=1)
        refused(chain, ws, 0)
    first(ws)
    broken[0] = "ms_decode_layers"
    with pytest.raises(RuntimeError, match="refused"):
        layers(ws)
    broken[0] = None
    layers(ws)
    first(ws)
    ws[5] = 1
    ops.decode_chain_start_over(ws)
    assert not ws.any()
    first(ws, M=5, L=2)

    ws = new()
    refused(chain, ws, 1)
    for _ in range(2):
        for i in range(3):
            chain(ws, i)
            refused(chain, ws, i)
            refused(chain, ws, (i + 1) % 3, launches=4)
            refused(chain, ws, (i + 1) % 3, M=1)
    assert launched.count("ms_decode_chain") == 6


def test_contexts_that_all_layers_in_two_launches_cannot_read_are_refused(ops, monkeypatch):
    """The kernel reads 1,024 keys of a context and no more: a bound that the caller knows is held against that, else the
    contexts themselves are."""
    launched = []
    monkeypatch.setattr(ops, "_check", lambda *args, **kw: None)
    monkeypatch.setattr(ops, "_call", lambda name, *args: launched.append(name))
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    ints = lambda *v: torch.tensor(v, dtype=torch.int32)     # noqa: E731

    def layers(*contexts, **bound):
        M = len(contexts)
        ws = torch.zeros(ops.decode_chain_workspace(M, 64, 2, 1, 64, 64, 2), dtype=torch.uint8)
        ws.chain_turn = ((M, 64, 2, 1, 64, 64, "layers", 2), 1)
        records = torch.zeros(2 * ops._get("ms_decode_layer_bytes")(), dtype=torch.uint8)
        records.layer_sizes = (2, 1, 64, 64, 64, 16)
        ops.decode_layers(records, torch.zeros(M, 64), ints(*[0] * M), ints(*[0] * M), ints(*contexts), torch.zeros(M, 99, dtype=torch.int32), None,
                          1.0, 2, 1, 64, 64, 16, 2, ws, **bound)
        return len(launched)

    assert layers(1024, 1) == 1 and layers(5, max_context_len=1024) == 2
    for contexts, bound in (((1025,), {}), ((3, 2000, 1), {}), ((5,), dict(max_context_len=1025))):
        with pytest.raises(ops.UnsupportedShape, match="1024 keys"):
            layers(*contexts, **bound)
    assert len(launched) == 2


@pytest.mark.parametrize("keys", [64, 2000])
def test_a_launch_that_waited_in_vain_is_an_error_and_the_next_step_starts_over(ops, keys):
    """What the GPU writes where a launch was broken off is seen when the step's results have come, or before the next launch,
    replayed or not; once: the workspace is zeroed for the step after it."""
    from llm_infrence_engine_amd.engine import ModelRunner
    from llm_infrence_engine_amd.engine.graph import StepGraphs

    m, b, caches, of = _decode_stand_in(ops, keys)
    made, r = of(), ModelRunner.__new__(ModelRunner)
    r.chain = made
    r.check()
    made.told[0] = 1
    made.workspace[:9] = 7
    with pytest.raises(RuntimeError, match="void"):
        r.check()
    r.check()
    made.ready()
    assert not made.workspace.any() and not made.broken_off

    replays, written = [], []
    g = StepGraphs.__new__(StepGraphs)
    g.manager = SimpleNamespace(pending_updates=lambda: 0)
    g.builder = SimpleNamespace(describe=lambda *a: SimpleNamespace(), write=lambda *a: written.append(1))
    bk = SimpleNamespace(layout=SimpleNamespace(n_updates=1), chain=made, graph=SimpleNamespace(replay=lambda: replays.append(made.workspace.any().item())),
                         buf=SimpleNamespace(wait_until_sent=lambda: None, send=lambda: None, np=None))
    g._fill_and_replay(bk, [], 1)
    assert g.chain is made
    made.told[0] = 1
    made.workspace[:9] = 7
    with pytest.raises(RuntimeError, match="void"):
        g._fill_and_replay(bk, [], 1)
    assert len(written) == 1      # (what it takes from the manager, the block tables' changes, is the next replay's to bring)
    g._fill_and_replay(bk, [], 1)
    assert replays == [False, False] and len(written) == 2
    r.chain = None
    r.check()


def test_a_step_asks_for_the_last_ones_results_before_it_takes_anything(ops):
    """A program that reads its logits without asking hears of void ones from the next step, whichever way that goes, while
    requests and pages are still as they were."""
    from llm_infrence_engine_amd.engine import ModelRunner

    made = _decode_stand_in(ops)[3]()
    r = ModelRunner.__new__(ModelRunner)
    r.chain, r.graphs, r.manager = made, SimpleNamespace(chain=None), None      # (nothing to grow: it is not to be reached)
    for step in (lambda: r.step([SimpleNamespace(req_id=0, tokens=[1])]), lambda: r.decode_steps([SimpleNamespace(req_id=0, tokens=[1])], 2)):
        made.told[0] = 1
        with pytest.raises(RuntimeError, match="void"):
            step()
        assert made.broken_off and not made.told[0]


@pytest.mark.parametrize("dtype,chains", [(torch.bfloat16, True), (torch.float32, True), (torch.float32, False)])
def test_a_step_compares_a_chains_weights_once(ops, monkeypatch, dtype, chains):
    """The host looks through the layers' weights and pages before a step's first launch, while the GPU waits: once a step."""
    from llm_infrence_engine_amd.engine import ModelRunner, runner
    from llm_infrence_engine_amd.parts.model import Model

    looked, made, ran = [], [], []

    class Chain:
        def takes(self, model, caches):
            looked.append(self)
            return True

        def check(self):
            pass

        def forward(self, x, ctx, caches):
            ran.append(self)
            return x, None

    def of(kind):
        return classmethod(lambda cls, *args: made.append(kind) or (Chain() if chains and (kind == "float") == (dtype == torch.float32) else None))

    monkeypatch.setattr(runner.DecodeChain, "where_it_pays", of("decode"))
    monkeypatch.setattr(runner.FloatLayers, "of", of("float"))
    x = torch.zeros(1, 4)
    layer = SimpleNamespace(forward=lambda x, pending, *a: pending, takes_sums=False, settles_writes=False)
    model = SimpleNamespace(embedding=SimpleNamespace(forward=lambda ctx: x), pass_entry=None, layers=[layer], final_norm=None,
                            spec=SimpleNamespace(order=[SimpleNamespace(layer=0, opens_pass=None)]), _settled=Model._settled)
    model.forward = lambda ctx, caches: Model.forward_hidden(model, ctx, caches)[0]
    r = ModelRunner.__new__(ModelRunner)
    ctx = lambda: SimpleNamespace(decode_only=True, num_tokens=1, max_context_len=5, chain=None, state_slots=None)     # noqa: E731
    r.model, r.graphs, r.chains, r.chain = model, None, {}, None
    r.manager = SimpleNamespace(has=lambda i: True, grow=lambda *a: None, computed=lambda i: 4, advance=lambda *a: None)
    r.builder = SimpleNamespace(build=lambda entries: SimpleNamespace(ctx=ctx(), slots=[]))
    r.caches = lambda rows, slots: [SimpleNamespace(kv=None, state=None)]
    for _ in range(3):
        r.step([SimpleNamespace(req_id=0, tokens=[1])])
    assert len(looked) == (2 if chains else 0) and len(ran) == (3 if chains else 0)      # (not in the step that makes it)
    assert made == (["decode"] if dtype == torch.bfloat16 else ["decode", "float"])


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [[1, 1, 1], [1, 40, 3]])
def test_float_layers_are_the_parts_one_by_one(ops, tokens):
    """Two layers of a 32-bit step by one call and part by part: the same kernels, so the same bits, in x, in what is left to
    add and in the pages; decoding and portions, a request further on, pages plain."""
    from llm_infrence_engine_amd.engine.batch import StepEntry
    from llm_infrence_engine_amd.config import config_from_dict
    from llm_infrence_engine_amd.engine import ModelRunner
    from llm_infrence_engine_amd.parts import chain
    from llm_infrence_engine_amd.parts.base import Runtime
    from llm_infrence_engine_amd.parts.model import Model

    cfg = config_from_dict({"model_type": "qwen2", "hidden_size": 96, "intermediate_size": 160, "num_hidden_layers": 2,
                            "num_attention_heads": 6, "num_key_value_heads": 2, "vocab_size": 64, "rms_norm_eps": 1e-6,
                            "rope_theta": 10000.0, "tie_word_embeddings": True, "max_position_embeddings": 128})
    g = torch.Generator().manual_seed(3)

    class Weights:
        def check(self, wanted, ignorable=()):
            self.shapes = {s.name: s.shape for s in wanted}

        def get(self, name):
            return torch.randn(self.shapes[name], generator=g).cuda() / 8

        def close(self):
            pass

    model = Model(cfg.to_spec())
    model.config = cfg
    model.load(Weights(), Runtime(torch.device("cuda:0"), torch.float32))
    got = []
    for whole in (True, False):
        r = ModelRunner(model, 16, 24, 4, 96)
        if not whole:
            r.chains["float"] = None
        r.step([StepEntry(0, list(range(20)), [19])])
        before, ff = r.chains["float"], model.layers[0].feed_forward      # weights loaded anew are not missed
        kept, ff.w_down = ff.w_down, ff.w_down * 2
        anew = r.step([StepEntry(1, [3], [0])]).cpu()
        assert (r.chains["float"] is not before) == whole
        ff.w_down = kept
        r.free_request(1)
        out = [r.step([StepEntry(i, [7 + i] * n, [n - 1]) for i, n in enumerate(tokens)]).cpu() for _ in range(2)]
        assert isinstance(r.chains["float"], chain.FloatLayers) == whole
        got.append([anew] + out + [t.cpu() for pages in r.pools.pages for t in pages.values()])
    assert all(torch.equal(a, b) for a, b in zip(*got))


def _small_model(dtype, seed=3, std=None, **sizes):
    """A model of the plain parts on the GPU, with random weights: matrices of ``std`` (None: 1/8)."""
    from llm_infrence_engine_amd.config import config_from_dict
    from llm_infrence_engine_amd.parts.base import Runtime
    from llm_infrence_engine_amd.parts.model import Model

    cfg = config_from_dict(dict({"model_type": "qwen2", "vocab_size": 64, "rms_norm_eps": 1e-6, "rope_theta": 10000.0,
                                 "tie_word_embeddings": True}, **sizes))
    g = torch.Generator().manual_seed(seed)

    class Weights:
        def check(self, wanted, ignorable=()):
            self.specs = {s.name: s for s in wanted}

        def get(self, name):
            s = self.specs[name]
            w = torch.randn(s.shape, generator=g) * (std or 1 / 8)
            return (1 + w if std and s.role == "norm" else w).cuda()

        def close(self):
            pass

    model = Model(cfg.to_spec())
    model.config = cfg
    model.load(Weights(), Runtime(torch.device("cuda:0"), dtype))
    return model


def test_the_scratch_of_32_bit_layers_is_sized_in_one_place(ops):
    """What the library carves up is what it says it needs, every piece from a boundary of 256 bytes on (the products look at
    addresses), and a scratch that is too small is refused before anything is launched."""
    need = lambda *sizes: ops._get("ms_float_layers_work")(*sizes)     # noqa: E731
    N, H, nh, nkv, d, I = 3, 65, 4, 2, 16, 36
    pieces = (N * H, N * H, N * (nh + 2 * nkv) * d, N * nh * d, N * 2 * I, N * I)
    assert need(N, H, nh, nkv, d, I) == sum(-(-p // 64) * 64 for p in pieces)
    assert need(100000, 8192, 64, 8, 128, 28672) > 1 << 31
    there = torch.zeros(64).data_ptr()
    call = lambda floats: ops._get("ms_float_layers")(there, 1, there, there, floats, there, there, there, there, 1, None, None, N, H, I,     # noqa: E731
                                                      nh, nkv, d, 16, 8, 0, 0.25, None)
    assert call(need(N, H, nh, nkv, d, I) - 1) == call(0) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [[1], [1, 1, 1], [2, 7]])
def test_float_layers_of_an_odd_width_are_the_parts_one_by_one(ops, tokens):
    """The scratch's pieces lie where an allocation of their own would: a width that is no multiple of four leaves the other
    products' kernels, and so their bits, as they are."""
    from llm_infrence_engine_amd.engine import ModelRunner
    from llm_infrence_engine_amd.engine.batch import StepEntry
    from llm_infrence_engine_amd.parts import chain

    model = _small_model(torch.float32, hidden_size=65, intermediate_size=132, num_hidden_layers=2, num_attention_heads=4,
                         num_key_value_heads=2, head_dim=48, max_position_embeddings=64)
    got = []
    for whole in (True, False):
        r = ModelRunner(model, 16, 24, 4, 64)
        if not whole:
            r.chains["float"] = None
        got.append([r.step([StepEntry(i, [7 + i] * n, [n - 1]) for i, n in enumerate(tokens)]).cpu() for _ in range(3)])
        assert isinstance(r.chains["float"], chain.FloatLayers) == whole
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [[1], [1] * 4, [3, 2], [1] * 8, [1] * 9])
@pytest.mark.parametrize("sizes", [dict(hidden_size=1280, intermediate_size=200, num_attention_heads=20, num_key_value_heads=4),
                                   dict(hidden_size=2052, intermediate_size=36, num_attention_heads=6, num_key_value_heads=6, head_dim=16),
                                   dict(hidden_size=96, intermediate_size=10, num_attention_heads=2, num_key_value_heads=1, head_dim=24),
                                   dict(hidden_size=128, intermediate_size=2100, num_attention_heads=2, num_key_value_heads=2)])
def test_norms_rotation_and_gate_within_32_bit_products_are_the_parts_one_by_one(ops, sizes, tokens):
    """Up to 8 tokens the norms, the rotation with the cache store and the gate go with the products: the same bits as one by one,
    for norms of more and of fewer threads, a width that the products leave to the parts (2,052), widths of W that are no whole blocks,
    heads whose halves are a few blocks, blocks of 4 and of 8 rows, and 9 tokens, which are the parts again."""
    from llm_infrence_engine_amd.engine import ModelRunner
    from llm_infrence_engine_amd.engine.batch import StepEntry

    model = _small_model(torch.float32, std=0.05, num_hidden_layers=2, max_position_embeddings=64, **sizes)
    got = []
    for whole in (True, False):
        r = ModelRunner(model, 16, 32, 16, 64)
        if not whole:
            r.chains["float"] = None
        out = [r.step([StepEntry(i, [(7 * i + j) % 64 for j in range(n)], [n - 1]) for i, n in enumerate(tokens)]).cpu() for _ in range(3)]
        got.append(out + [t.cpu() for pages in r.pools.pages for t in pages.values()])
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.fixture(scope="module")
def chained_model():
    return _small_model(torch.bfloat16, seed=5, std=0.05, hidden_size=768, intermediate_size=2048, num_hidden_layers=3, num_attention_heads=12,
                        num_key_value_heads=4, max_position_embeddings=2048)


def _prompts(r, lengths):
    from llm_infrence_engine_amd.engine.batch import StepEntry

    for i, n in enumerate(lengths):
        r.step([StepEntry(i, [(5 * j + i) % 64 for j in range(n)], [n - 1])])


def _like(got, want):
    # three layers, each of the two within 1.2e-2 of doubles (queries, heads, probabilities and the middle are rounded to bfloat16)
    assert got.shape == want.shape and got.isfinite().all()
    assert (got.double() - want.double()).norm() <= 2.4e-2 * want.double().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("lengths", [[40], [1022, 7, 300], [3, 1, 16, 511, 64, 200, 33, 1023]])
def test_a_models_chains_are_its_parts_one_by_one(ops, chained_model, monkeypatch, lengths, graphs):
    """Decode steps of a model through its chains and part by part, logits of every step: one request, three (in a graph a row of
    padding) and eight; a context that grows past 1,024 keys, from two launches for all layers to one a layer; steps launched,
    replayed, and replayed several at a time."""
    from llm_infrence_engine_amd.engine import ModelRunner
    from llm_infrence_engine_amd.engine.batch import StepEntry
    from llm_infrence_engine_amd.parts import chain

    make = lambda graphs: ModelRunner(chained_model, 16, 200, 8, 1100, hip_graphs=graphs, graph_portion_tokens=0)     # noqa: E731
    kinds = set()

    def step(r, t):
        out = r.step([StepEntry(i, [(11 * t + i) % 64], [0]) for i in range(len(lengths))]).clone()
        r.check()
        kinds.add(None if r.chain is None else r.chain.table is not None)
        return out

    a = make(graphs)
    _prompts(a, lengths)
    got = [step(a, t) for t in range(4)]
    assert kinds == ({True, False} if max(lengths) > 1000 else {True})
    tokens = a.decode_steps([StepEntry(i, [9 + i]) for i in range(len(lengths))], 4) if graphs else []
    got.append(step(a, 5))
    kinds.clear()
    monkeypatch.setattr(chain.DecodeChain, "where_it_pays", classmethod(lambda *args: None))
    b = make(False)
    _prompts(b, lengths)
    want = [step(b, t) for t in range(4)]
    for row in [[9 + i for i in range(len(lengths))]] + tokens[:-1] if graphs else []:
        b.step([StepEntry(i, [t], [0]) for i, t in enumerate(row)])
    want.append(step(b, 5))
    assert kinds == {None}
    for g, w in zip(got, want):
        _like(g, w)


@pytest.mark.gpu
@pytest.mark.parametrize("length,name,at", [(40, "decode_first", 0), (40, "decode_layers", 0), (1100, "decode_chain", 0), (1100, "decode_chain", 2)])
def test_a_chain_starts_over_behind_a_step_that_broke_off(ops, chained_model, monkeypatch, length, name, at):
    """An exception between a step's launches: the same step again, and those after it, are as they would have been."""
    from llm_infrence_engine_amd.engine import ModelRunner
    from llm_infrence_engine_amd.engine.batch import StepEntry

    got, call = [], getattr(ops, name)
    for breaks in (False, True):
        r = ModelRunner(chained_model, 16, 200, 4, 1200)
        _prompts(r, [length, 5])
        for t in range(3):
            entries = [StepEntry(i, [(7 * t + i) % 64], [0]) for i in range(2)]
            if breaks and t == 1:
                left = [at]

                def broken(*args, **kw):
                    left[0] -= 1
                    if left[0] < 0:
                        raise RuntimeError("broken off here")
                    return call(*args, **kw)

                monkeypatch.setattr(ops, name, broken)
                with pytest.raises(RuntimeError, match="broken off here"):
                    r.step(entries)
                monkeypatch.setattr(ops, name, call)
            got.append(r.step(entries).cpu())
            r.check()
            assert (r.chain.table is not None) == (length < 1000)
    assert all(torch.equal(x, y) for x, y in zip(got[:3], got[3:]))


@pytest.mark.gpu
def test_a_model_whose_weights_lie_anywhere_steps_as_one_whose_do_not(ops):
    """Weights that are views of one buffer, 4 bytes off 16 (as a reader may hand them out on the GPU): no chain, and the logits of
    the same weights in places of their own."""
    from llm_infrence_engine_amd.engine import ModelRunner
    from llm_infrence_engine_amd.engine.batch import StepEntry

    got = []
    for aside in (False, True):
        model = _small_model(torch.bfloat16, seed=6, std=0.05, hidden_size=768, intermediate_size=2048, num_hidden_layers=2,
                             num_attention_heads=12, num_key_value_heads=4, max_position_embeddings=128)
        for l in model.layers if aside else ():
            for part, names in ((l.mixer, ("w_qkv", "w_o")), (l.feed_forward, ("w_gate_up", "w_down"))):
                for n in names:
                    w = getattr(part, n)
                    there = torch.empty(w.numel() + 2, dtype=w.dtype, device=w.device)[2:].view(w.shape)
                    assert there.copy_(w).data_ptr() % 16 == 4
                    setattr(part, n, there)
        r = ModelRunner(model, 16, 24, 4, 96)
        _prompts(r, [20, 3])
        got.append([r.step([StepEntry(i, [7 + i], [0]) for i in range(2)]) for _ in range(2)])
        assert (r.chain is None) == aside
    for a, b in zip(*got):
        _like(b, a)


@pytest.mark.parametrize("M,N,K,parts", [
    # times of the library and the norm over partial sums and the norm
    (640, 896, 4864, 3), (768, 896, 4864, 3), (1000, 896, 4864, 4), (560, 512, 4864, 7), (960, 768, 6912, 5), (700, 2048, 8192, 2),    # 1.18 1.10 1.02 1.10 1.11 1.13
    (900, 1536, 4864, 0), (700, 2048, 4352, 0),        # 0.98 0.97
    # parts by the model of product and norm, times of other parts over them
    (150, 3584, 18944, 4), (512, 3584, 18944, 8), (300, 5120, 27648, 2), (150, 2048, 5632, 5),       # 1.30 1.07 1.13 1.23
    (1001, 896, 4864, 0), (768, 896, 4096, 0), (768, 2176, 8192, 0)])                            # as ever
def test_where_products_leave_partial_sums_and_in_how_many_parts(ops, M, N, K, parts):
    assert ops._get("ms_gemm_tiled_sums_parts")(M, N, K) == parts


@pytest.mark.parametrize("M,N,K,gated", [
    # times of the library and the silu's kernel over the tiled kernel's
    (900, 37888, 3584, 1), (150, 37888, 3584, 1), (200, 16384, 2048, 1), (850, 13824, 2560, 1), (900, 27648, 5120, 1),     # 1.23 1.16 1.30 1.13 1.15
    (542, 37888, 3584, 0), (300, 55296, 5120, 0), (1300, 27648, 5120, 0)])                                                 # 0.86 0.84 0.95
def test_where_the_tiled_kernel_takes_gated_products_by_what_it_is_expected_to_take(ops, M, N, K, gated):
    assert ops._get("ms_gemm_tiled_pays")(M, N, K) == gated


@pytest.mark.parametrize("M,N,K,kind", [
    (193, 37888, 3584, "gated"), (288, 37888, 3584, "gated"), (318, 37888, 3584, "gated"), (385, 37888, 3584, "gated"), (640, 22016, 4096, "gated"),
    (1025, 55296, 5120, "gated"), (1092, 27648, 5120, "gated"), (2210, 2560, 2048, "gated"), (1031, 5632, 3072, "gated"), (2048, 57344, 8192, "gated"),
    (415, 23560, 1600, "relu2"), (338, 23560, 2880, "relu2"), (464, 23560, 5120, "relu2"),
    (387, 4608, 7168, "sums"), (506, 4778, 4352, "sums"), (450, 4480, 5120, "sums"), (1031, 1536, 16512, "sums"), (3727, 512, 16384, "sums")])
def test_products_held_in_32_bits_up_to_their_reader_stay_so(ops, M, N, K, kind):
    """Sizes whose gate and up, whose squared relu's input or whose norm's addend the tiled kernel holds in float, where the library, which rounds
    them to bfloat16, is expected to be as fast or a little faster."""
    rule = {"gated": "ms_gemm_tiled_pays", "relu2": "ms_gemm_tiled_relu2_pays", "sums": "ms_gemm_tiled_sums_parts"}[kind]
    assert ops._get(rule)(M, N, K) > 0


@pytest.mark.parametrize("M,N,K,tile", [
    # us of the tiles of 256 x 256, 128 x 128, 64 x 64, 192 and 160 x 256, 64 x 64 deep, 96 x 128
    (4926, 512, 768, 2), (5069, 472, 768, 2), (4402, 460, 1280, 2),         # 19.3 9.5 9.6 16.2 15.7 12.2 15.2;  23.9 10.7 10.9 .. 15.2;  35.0 15.7 15.7 .. 21.1
    (5370, 1496, 1536, 2),                                                  # as 128 x 256 46.5, as 192 x 256 29.7
    (10455, 980, 128, 2), (8403, 1906, 768, 2), (1188, 12558, 128, 2),      # 21.7 15.4 15.9 22.2 13.2;  62.3 45.6 49.6 47.0 39.7;  28.8 21.0 21.1 27.5 21.2
    (13607, 4864, 1024, 4), (352, 2000, 128, 3),                            # 133 150 276 131 142;  .. 3.99 3.22 .. 3.36
    # the measured range of the model
    (300, 9728, 896, 2), (512, 9728, 896, 7), (2048, 9728, 896, 5), (157, 224, 1280, 6), (4096, 9728, 896, 1), (4096, 37888, 3584, 1)])
def test_tiles_by_the_model_within_what_it_was_measured_at(ops, M, N, K, tile):
    """Beyond 6,143 tokens and below 256 columns the choice is the older tiles'; from 4,096 tokens on rounds are counted as the tiles lie."""
    assert ops._get("ms_gemm_tiled_tile")(M, N, K) == tile


@pytest.mark.parametrize("M,K,heads,d,tile", [
    # time in tiles of 128 x 128 over that in tiles of 64 x 64
    (4096, 896, 18, 64, 3), (8192, 512, 32, 64, 3), (4000, 1024, 32, 64, 3), (11000, 896, 18, 64, 3),            # 1.0 1.1 0.95 1.05
    (8192, 1024, 32, 64, 2), (4096, 1024, 32, 64, 2), (16384, 896, 18, 64, 2), (8192, 768, 32, 64, 2),           # 0.79 0.95 0.92 0.97
    (896, 896, 18, 64, 6), (1024, 896, 18, 64, 11), (1800, 1024, 14, 64, 11), (70, 512, 12, 128, 6), (4096, 1024, 12, 128, 2)])
def test_tiles_of_the_qkv_product(ops, M, K, heads, d, tile):
    assert ops._get("ms_gemm_tiled_qkv_tile")(M, K, heads, d) == tile


@pytest.mark.parametrize("M,N,K,gated", [
    # times of the library and the silu's kernel over the tiled kernel's
    (78, 850, 3584, 0), (192, 512, 3584, 0), (128, 2048, 3584, 0), (160, 1536, 3072, 0), (72, 270, 2560, 0), (192, 512, 2304, 0),     # 0.86 0.75 0.79 0.92 0.98 0.87
    (160, 2048, 3584, 1), (192, 1400, 2816, 1), (65, 3072, 3584, 1), (100, 2560, 3584, 1), (78, 850, 3456, 1), (192, 512, 2688, 1), (256, 1024, 2560, 1),  # 1.24 1.13 1.26 1.23 1.2 1.07 1.08
    (65, 128, 2048, 1), (192, 1024, 2304, 1)])                                                                                  # 1.25 1.15
def test_few_rows_and_tokens_by_long_rows_are_left_to_the_library(ops, M, N, K, gated):
    assert ops._get("ms_gemm_tiled_pays")(M, N, K) == gated


@pytest.mark.parametrize("M,N,K", [(1212, 4694, 3072), (565, 12434, 5120), (1837, 9378, 1600), (608, 10862, 2048)])     # 0.84 0.87 0.88 0.93
def test_squared_relus_that_the_library_is_faster_at(ops, M, N, K):
    assert ops._get("ms_gemm_tiled_relu2_pays")(M, N, K) == 0


@pytest.mark.parametrize("M,N,K,parts", [
    # us by the parts of a model that counts neither the reading of W nor rows of sums that begin anywhere, and by these
    (84, 7327, 11456, 4), (127, 7749, 10240, 2), (402, 827, 9088, 2), (77, 7473, 21248, 4),                  # 123 87; 140 103; 47 38; 151 119
    (123, 8072, 10880, 4), (87, 8192, 7360, 4), (112, 6284, 21888, 5), (69, 6552, 7808, 4), (711, 1710, 7936, 0)])   # 62 57; 43 36; 96 86; 38 34; 54 50
def test_parts_of_sums_by_what_reading_w_and_odd_rows_cost(ops, M, N, K, parts):
    assert ops._get("ms_gemm_tiled_sums_parts")(M, N, K) == parts


@pytest.mark.parametrize("M,N,K,kernel", [
    # us of the first kernel, tiles of 64 and 32, slices of 16, 32 and 48 tokens
    (9, 401, 13188, 1), (16, 896, 9008, 1), (13, 3129, 764, 1),                     # 37.8 .. .. 72.7;  30 .. .. 46;  5.4 .. .. 7.1
    (512, 64000, 512, 2), (1000, 3072, 768, 2), (1000, 20000, 512, 2), (350, 9728, 13188, 2),     # 331 .. 571;  50.3 .. 75.8;  207 .. 348;  990 .. .. 1,587
    (17, 896, 4864, 6), (64, 896, 896, 6), (350, 896, 4864, 8), (24, 9728, 512, 6), (2048, 9728, 896, 2),
    # below 512 columns
    (16, 896, 132, 1), (20, 64000, 256, 3), (100, 64000, 256, 2), (100, 896, 256, 3),
    # up to 8 rows: four steps to a load, slices side by side with 4 and with 8 rows of W a block
    (8, 2563, 2048, 1), (4, 2563, 5120, 1), (4, 4608, 4992, 1), (8, 2048, 2048, 1), (3, 9728, 896, 1), (2, 896, 512, 1),       # 11.4 .. 14.2;  25.2 .. 29.9;  41.6 .. 44.6
    (3, 896, 4864, 4), (4, 1024, 18944, 4), (8, 896, 4864, 4), (8, 896, 896, 1), (4, 2048, 4864, 5), (8, 6144, 1536, 5), (4, 4608, 3584, 5)])
def test_kernels_of_32_bit_products(ops, M, N, K, kernel):
    """All of them have the same bits."""
    assert ops._get("ms_gemm_f32_kernel")(M, N, K) == kernel
