"""Each HIP kernel alone against a plain float reference of the same op, at sizes other than the
engine's (odd widths, head sizes in steps of 16, vocabularies that are no power of two)."""
import math

from types import SimpleNamespace

import numpy as np

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from llm_infrence_engine_amd.kernels import ops

    return ops


def tol(dtype):
    # float: sums of a few hundred products; bfloat16: one rounding of the result (2^-8 relative) on top
    return dict(atol=2e-5, rtol=2e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=1.6e-2)


DTYPES = [torch.float32, torch.bfloat16]


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed(ops, dtype):
    g = torch.Generator().manual_seed(0)
    table = torch.randn(331, 72, generator=g).to(dtype).to(DEV)
    ids = torch.randint(0, 331, (13,), generator=g).to(torch.int32).to(DEV)
    out = torch.empty(13, 72, dtype=torch.float32, device=DEV)
    ops.embed(ids, table, out)
    assert torch.equal(out, table[ids.long()].float())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H", [72, 896, 1500, 16384, 20000])
def test_rms_norm(ops, dtype, H):
    g = torch.Generator().manual_seed(1)
    x = (torch.randn(9, H, generator=g) * 3).to(DEV)
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(DEV)
    out = torch.empty(9, H, dtype=dtype, device=DEV)
    ops.rms_norm(x, w, 1e-5, out)
    want = w.double() * (x.double() * torch.rsqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-5))
    torch.testing.assert_close(out.double(), want, **tol(dtype))
    # with the residual sum fused, and rows gathered
    delta = torch.randn(9, H, generator=g).to(dtype).to(DEV)
    x2 = x.clone()
    ops.rms_norm(x2, w, 1e-5, out, delta=delta)
    s = x.double() + delta.double()
    torch.testing.assert_close(x2.double(), s, atol=1e-6, rtol=1e-6)
    want = w.double() * (s * torch.rsqrt((s ** 2).mean(-1, keepdim=True) + 1e-5))
    torch.testing.assert_close(out.double(), want, **tol(dtype))
    rows = torch.tensor([7, 0, 3], dtype=torch.int32, device=DEV)
    out3 = torch.empty(3, H, dtype=dtype, device=DEV)
    ops.rms_norm(x2, w, 1e-5, out3, rows=rows)
    torch.testing.assert_close(out3.double(), want[rows.long()], **tol(dtype))
    # the sum formed but not kept, from two partial sums
    x3 = x.clone()
    halves = torch.stack((delta.float() * 0.25, delta.float() * 0.75)).to(dtype)
    ops.rms_norm(x3, w, 1e-5, out, delta=halves, write_back=False)
    assert torch.equal(x3, x)
    s = x.double() + halves[0].double() + halves[1].double()
    want = w.double() * (s * torch.rsqrt((s ** 2).mean(-1, keepdim=True) + 1e-5))
    torch.testing.assert_close(out.double(), want, **tol(dtype))


def test_rms_norm_eps_inside_root(ops):
    x = torch.full((1, 16), 1e-6, device=DEV)
    out = torch.empty(1, 16, device=DEV)
    ops.rms_norm(x, torch.ones(16, device=DEV), 1e-2, out)
    torch.testing.assert_close(out, x / math.sqrt(1e-12 + 1e-2), rtol=1e-6, atol=0)


@pytest.mark.parametrize("dtype", DTYPES)
def test_silu_mul(ops, dtype):
    g = torch.Generator().manual_seed(2)
    gu = (torch.randn(7, 2 * 200, generator=g) * 2).to(dtype).to(DEV)
    out = torch.empty(7, 200, dtype=dtype, device=DEV)
    ops.silu_mul(gu, out)
    a = gu.double()
    want = torch.nn.functional.silu(a[:, 0::2]) * a[:, 1::2]
    torch.testing.assert_close(out.double(), want, **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 331, 72), (5, 64, 120), (70, 200, 896), (130, 151, 50), (3, 1000, 4864)])
def test_gemm_generic(ops, dtype, M, N, K):
    g = torch.Generator().manual_seed(3)
    a = torch.randn(M, K, generator=g).to(dtype).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dtype).to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T
    out = torch.empty(M, N, dtype=dtype, device=DEV)
    ops.gemm_generic(a, w, out)
    torch.testing.assert_close(out.double(), want, **tol(dtype))
    ops.gemm_generic(a, w, out, bias=bias)
    torch.testing.assert_close(out.double(), want + bias.double(), **tol(dtype))
    acc = torch.randn(M, N, generator=g).to(DEV)
    acc0 = acc.clone()
    ops.gemm_generic(a, w, acc, accumulate=True)  # float result whatever the inputs are
    torch.testing.assert_close(acc.double(), acc0.double() + want, atol=2e-5, rtol=2e-5)


def test_gemm_row_does_not_depend_on_the_batch(ops):
    g = torch.Generator().manual_seed(4)
    a = torch.randn(77, 192, generator=g).to(DEV)
    w = torch.randn(331, 192, generator=g).to(DEV)
    full = torch.empty(77, 331, device=DEV)
    one = torch.empty(1, 331, device=DEV)
    ops.gemm_generic(a, w, full)
    ops.gemm_generic(a[40:41], w, one)
    assert torch.equal(full[40:41], one)


@pytest.mark.parametrize("N,K", [(16, 4), (33, 20), (64, 64), (200, 300), (896, 1028), (9728, 896), (16500, 64), (32801, 36)])
def test_float_product_in_the_same_order_for_any_number_of_rows(ops, N, K):
    """Both kernels of the 32-bit product and both of the tiled one's tiles, at the edges of their tiles, as rows of wider
    matrices: within float rounding of 64 bits, and bit for bit the same row whatever is beside it."""
    g = torch.Generator().manual_seed(31)
    M = 700 if N > 9000 else 130
    a = torch.randn(M, K + 8, generator=g).to(DEV)[:, 4:4 + K]
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T + bias.double()
    # a slice is one chain of at most 16 ceil(K / 256) or 64 sums, then come at most 16 slices and the bias
    chain = max(64, 16 * -(-K // 256)) + 18
    bound = chain * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs())
    full = torch.empty(M, N, device=DEV)
    ops.gemm_generic(a, w, full, bias=bias)
    assert ((full.double() - want).abs() <= bound).all()
    for lo, hi in ((0, 1), (3, 19), (5, 22), (0, 33), (2, 66), (0, 65), (1, 98), (M - 1, M)):
        out = torch.empty(hi - lo, N, device=DEV)
        ops.gemm_generic(a[lo:hi], w, out, bias=bias)
        assert torch.equal(out, full[lo:hi]), (lo, hi)
        ops.gemm_generic(a[lo:hi], w, out, bias=bias, accumulate=True)
        assert torch.equal(out, 2 * full[lo:hi]), (lo, hi)


def rope_reference(x, pos, rot, inv):
    ang = pos.double()[:, None] * inv[None]
    cos, sin = torch.cat((ang, ang), -1).cos()[:, None], torch.cat((ang, ang), -1).sin()[:, None]
    xr = x[..., :rot]
    half = rot // 2
    rotated = xr * cos + torch.cat((-xr[..., half:], xr[..., :half]), -1) * sin
    return torch.cat((rotated, x[..., rot:]), -1)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("vt", [False, True])
@pytest.mark.parametrize("nh,nkv,d,rot", [(4, 2, 16, 16), (5, 1, 48, 48), (6, 3, 80, 32), (3, 1, 20, 20), (2, 2, 24, 12),
                                          (14, 2, 64, 64), (2, 1, 256, 256)])
def test_rope_store(ops, dtype, nh, nkv, d, rot, vt):
    """Sizes that the 16-byte kernel takes and sizes that fall to the element-wise one; values pages plain and
    transposed; with and without a late bias; one token that is not stored."""
    g = torch.Generator().manual_seed(5)
    N, page_size, pages = 11, 4, 9
    qkv = torch.randn(N, (nh + 2 * nkv) * d, generator=g).to(dtype)
    pos = torch.tensor([0, 1, 2, 3, 8191, 5, 100, 7, 4000, 9, 10], dtype=torch.int32)
    slots = torch.randperm(pages * page_size, generator=g)[:N].to(torch.int32)
    slots[3] = -1
    theta = 1e6
    inv_freq = (1.0 / (theta ** (torch.arange(0, rot, 2, dtype=torch.float64) / rot))).float()
    kp = torch.zeros(pages, nkv, page_size, d, dtype=dtype, device=DEV)
    vp = torch.zeros(pages, nkv, d, page_size, dtype=dtype, device=DEV) if vt else torch.zeros_like(kp)
    dev = qkv.to(DEV)
    bias = torch.randn((nh + 2 * nkv) * d, generator=g) if rot != 16 else None   # with and without a late bias
    ops.rope_store(dev, nh, nkv, d, rot, pos.to(DEV), inv_freq.to(DEV), slots.to(DEV), kp, vp, v_transposed=vt,
                   bias=None if bias is None else bias.to(DEV))
    x = qkv.double().view(N, nh + 2 * nkv, d)
    if bias is not None:
        x = x + bias.double().view(1, nh + 2 * nkv, d)
    want_q = rope_reference(x[:, :nh], pos, rot, inv_freq.double())
    want_k = rope_reference(x[:, nh:nh + nkv], pos, rot, inv_freq.double())
    got = dev.double().cpu().view(N, nh + 2 * nkv, d)
    # the angle is a float product of position and frequency: at position 8191 its rounding is ~2.4e-4 rad
    t = dict(atol=2e-3, rtol=0) if dtype == torch.float32 else dict(atol=3e-2, rtol=1.6e-2)
    torch.testing.assert_close(got[:, :nh], want_q, **t)
    torch.testing.assert_close(got[:, nh:nh + nkv], want_k, **t)
    small = pos < 200  # there the float angle is exact to ~1e-5
    torch.testing.assert_close(got[small][:, :nh], want_q[small], **tol(dtype))
    torch.testing.assert_close(got[:, nh + nkv:], x[:, nh + nkv:], **(tol(dtype) if bias is not None else dict(atol=0, rtol=0)))
    for n in range(N):
        s = int(slots[n])
        if s < 0:
            continue
        p, o = divmod(s, page_size)
        assert torch.equal(kp[p, :, o].cpu().double(), got[n, nh:nh + nkv])
        assert torch.equal((vp[p, :, :, o] if vt else vp[p, :, o]).cpu().double(), got[n, nh + nkv:])
    used = torch.zeros(pages * page_size, dtype=torch.bool)
    used[slots[slots >= 0].long()] = True
    assert (kp.cpu().permute(0, 2, 1, 3).reshape(pages * page_size, -1)[~used] == 0).all()


def attention_reference(q, k, v, scale, window=None):
    """q [nh, T, d], k/v [nkv, S, d] with the T queries at the last T of S positions."""
    nh, T, d = q.shape
    S = k.shape[1]
    rep = nh // k.shape[0]
    k, v = k.repeat_interleave(rep, 0), v.repeat_interleave(rep, 0)
    s = torch.einsum("htd,hsd->hts", q, k) * scale
    i = torch.arange(S - T, S)[:, None]
    j = torch.arange(S)[None]
    vis = j <= i
    if window:
        vis = vis & (j > i - window)
    s = s.masked_fill(~vis[None], float("-inf"))
    return torch.einsum("hts,hsd->htd", s.softmax(-1), v)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,page_size,window", [(4, 2, 16, 4, None), (6, 2, 32, 8, None), (5, 1, 48, 16, None),
                                                        (3, 3, 80, 4, 7), (8, 2, 128, 16, 40), (2, 1, 18, 4, None),
                                                        (4, 2, 64, 16, 1100)])
def test_paged_attention_generic(ops, dtype, nh, nkv, d, page_size, window):
    """Three requests in one batch: a whole prompt, a portion after a cached prefix, one decoded token;
    pages handed out in shuffled order and the pool pre-filled with large values that must never be read."""
    g = torch.Generator().manual_seed(6)
    # keys each request holds after this step; behind the widest window so many that every wave has several blocks of 64
    ctx = [70, 513, 1300] if window == 1100 else [70, 133, 201]
    qlen = [70, 9, 1]          # its new tokens
    pages_per = [-(-c // page_size) for c in ctx]
    P = sum(pages_per) + 5
    order = torch.randperm(P - 1, generator=g) + 1
    kp = torch.full((P, nkv, page_size, d), 1e4, dtype=dtype)
    vp = torch.full((P, nkv, page_size, d), -1e4, dtype=dtype)
    table = torch.zeros(3, max(pages_per), dtype=torch.int32)
    scale = 1.0 / math.sqrt(d)
    q_all, req_all, pos_all, want = [], [], [], []
    used = 0
    for r in range(3):
        k = torch.randn(nkv, ctx[r], d, generator=g).to(dtype)
        v = torch.randn(nkv, ctx[r], d, generator=g).to(dtype)
        q = (torch.randn(nh, qlen[r], d, generator=g) * 2).to(dtype)
        # one far key stands out for the last query of each request
        far = 3
        k[:, far] = (q[::nh // nkv, -1].float() * 1.5).to(dtype)
        pages = order[used:used + pages_per[r]]
        used += pages_per[r]
        table[r, :pages_per[r]] = pages.to(torch.int32)
        for j in range(ctx[r]):
            kp[pages[j // page_size], :, j % page_size] = k[:, j]
            vp[pages[j // page_size], :, j % page_size] = v[:, j]
        q_all.append(q.transpose(0, 1).reshape(qlen[r], nh * d))
        req_all += [r] * qlen[r]
        pos_all += list(range(ctx[r] - qlen[r], ctx[r]))
        want.append(attention_reference(q.double(), k.double(), v.double(), scale, window).transpose(0, 1).reshape(qlen[r], nh * d))
    q = torch.cat(q_all).to(DEV)
    N = q.shape[0]
    # q as a row slice of a wider matrix, as in the fused projection
    wide = torch.zeros(N, nh * d + 24, dtype=dtype, device=DEV)
    wide[:, :nh * d] = q
    out = torch.empty(N, nh * d, dtype=dtype, device=DEV)
    ops.paged_attention_generic(wide, kp.to(DEV), vp.to(DEV), table.to(DEV),
                                torch.tensor(req_all, dtype=torch.int32, device=DEV),
                                torch.tensor(pos_all, dtype=torch.int32, device=DEV), out, nh, scale, window)
    torch.testing.assert_close(out.double().cpu(), torch.cat(want), **tol(dtype))


def test_sample_greedy_and_vectors(ops):
    lg = torch.tensor([[0.1, 2.0, 0.5], [3.0, 0.0, 0.0], [1.0, 1.0, 1.0]], device=DEV)
    out = torch.empty(3, dtype=torch.int32, device=DEV)
    ops.sample(lg, out)
    assert out.tolist() == [1, 0, 0]  # first maximum on ties
    g = torch.Generator().manual_seed(7)
    big = torch.randn(5, 151936, generator=g).to(DEV)
    out = torch.empty(5, dtype=torch.int32, device=DEV)
    ops.sample(big, out)
    assert out.tolist() == big.argmax(-1).tolist()


def _draws_of_row(ops, row, n, temperature, top_k, top_p, seed=5, first_draw=0):
    """``n`` draws from one row of logits: the row repeated, each copy with a draw index of its own."""
    V = row.numel()
    lg = row.to(DEV).float().expand(n, V).contiguous()
    out = torch.empty(n, dtype=torch.int32, device=DEV)
    ops.sample(lg, out, torch.full((n,), temperature, device=DEV), torch.full((n,), top_k, dtype=torch.int32, device=DEV),
               torch.full((n,), top_p, device=DEV), torch.full((n,), seed, dtype=torch.int64, device=DEV),
               torch.arange(first_draw, first_draw + n, dtype=torch.int32, device=DEV))
    return out.cpu().long()


@pytest.mark.parametrize("V", [50, 1000, 151936])
@pytest.mark.parametrize("temperature,top_k,top_p", [(0.8, 50, 0.9), (1.3, 0, 0.7), (1.0, 5, 1.0), (1.0, 0, 1.0), (0.5, 7, 0.3)])
def test_sampler_draws_from_the_plain_distribution(ops, V, temperature, top_k, top_p):
    """Draws land only on tokens the plain rule keeps (temperature, top-k, top-p in the reference's order,
    src/miniserve/sampler.py:23-41) and as often as its probabilities say."""
    from tests.plain import qwen2_plain as P

    g = torch.Generator().manual_seed(V + top_k)
    row = torch.randn(V, generator=g) * 2.5
    want = P.logits_to_probs(row[None], temperature, top_k, top_p)[0]
    n = 8192
    got = _draws_of_row(ops, row, n, temperature, top_k, top_p)
    kept = (want > 0).nonzero().flatten()
    assert set(got.tolist()) <= set(kept.tolist()), "a token was drawn that the plain rule drops"
    freq = torch.bincount(got, minlength=V).double() / n
    # the tokens that carry the mass: each within five standard deviations of its probability
    for tok in want.topk(min(20, kept.numel())).indices.tolist():
        pr = float(want[tok])
        assert abs(float(freq[tok]) - pr) < 5 * math.sqrt(pr * (1 - pr) / n) + 2e-4, (tok, pr, float(freq[tok]))
    if kept.numel() <= 64:                                  # few enough that every kept token should appear
        assert (freq[kept] > 0).all() or float(want[kept].min()) * n < 8


def test_sampler_ties_thresholds_and_mixed_rows(ops):
    """Ties at the k-th value are all kept; the token at which the running mass reaches top_p is kept with all its
    equals; top_k = 1 and a tiny top_p are the greedy choice; rows without temperature take the first maximum
    beside rows that draw; and a draw does not depend on the rows beside it (nor on how many blocks a row is
    spread over)."""
    row = torch.tensor([1.0, 3.0, 2.0, 2.0, 0.5, 2.0, -1.0, 3.0])
    got = _draws_of_row(ops, row, 2048, 1.0, 3, 1.0)               # the third largest is 2.0, three times: five tokens stay
    assert set(got.tolist()) == {1, 2, 3, 5, 7}
    got = _draws_of_row(ops, row, 2048, 1.0, 0, 0.59)              # the two 3.0s hold 0.599 of the mass: they stay, nothing else
    assert set(got.tolist()) == {1, 7}
    got = _draws_of_row(ops, row, 2048, 1.0, 0, 0.61)              # a little more: the three 2.0s come in together
    assert set(got.tolist()) == {1, 2, 3, 5, 7}
    assert set(_draws_of_row(ops, row, 256, 2.0, 1, 1.0).tolist()) == {1, 7}      # both maxima tie at k = 1
    g = torch.Generator().manual_seed(3)
    big = torch.randn(151936, generator=g) * 3
    assert set(_draws_of_row(ops, big, 64, 1.5, 1, 1.0).tolist()) == {int(big.argmax())}
    assert set(_draws_of_row(ops, big, 64, 1.0, 0, 1e-6).tolist()) == {int(big.argmax())}
    # mixed rows, and the same draws alone and in company
    rows = torch.stack([big, big.flip(0), big * 0.5, big])
    lg = rows.to(DEV)
    temp = torch.tensor([0.9, 0.0, 1.2, -1.0], device=DEV)
    k = torch.tensor([40, 40, 0, 3], dtype=torch.int32, device=DEV)
    pp = torch.tensor([0.95, 0.5, 0.8, 0.9], device=DEV)
    seeds = torch.tensor([11, 12, 13, 14], dtype=torch.int64, device=DEV)
    draw = torch.tensor([3, 3, 9, 0], dtype=torch.int32, device=DEV)
    out = torch.empty(4, dtype=torch.int32, device=DEV)
    ops.sample(lg, out, temp, k, pp, seeds, draw)
    together = out.tolist()
    assert together[1] == int(rows[1].argmax()) and together[3] == int(rows[3].argmax())
    for r in (0, 2):
        alone = torch.empty(1, dtype=torch.int32, device=DEV)
        ops.sample(lg[r:r + 1].contiguous(), alone, temp[r:r + 1], k[r:r + 1], pp[r:r + 1], seeds[r:r + 1], draw[r:r + 1])
        assert alone.item() == together[r]
        many = torch.empty(200, dtype=torch.int32, device=DEV)          # 200 rows: fewer blocks to a row
        ops.sample(lg[r:r + 1].expand(200, -1).contiguous(), many, temp[r:r + 1].expand(200).contiguous(),
                   k[r:r + 1].expand(200).contiguous(), pp[r:r + 1].expand(200).contiguous(),
                   seeds[r:r + 1].expand(200).contiguous(), draw[r:r + 1].expand(200).contiguous())
        assert set(many.tolist()) == {together[r]}
    # a row that holds nothing to draw from falls back to index 0, like the greedy choice
    nothing = torch.full((1, 5000), float("-inf"), device=DEV)
    ops.sample(nothing, alone, temp[:1], k[:1], pp[:1], seeds[:1], draw[:1])
    assert alone.item() == 0


def test_argmax_in_two_stages(ops):
    """Ties across and inside the slices of the first stage go to the smallest index; a row of -inf or NaN gives
    index 0; vocabularies that are no multiple of the slice count."""
    for V in (1000, 4097, 151936, 200003):
        lg = torch.zeros(6, V, device=DEV)
        lg[0, V - 1] = 1.0
        lg[1, [V // 3, V // 3 + 1, V - 2]] = 2.0            # the first of three equal maxima
        lg[2, :] = -5.0                                      # all equal: index 0
        lg[3, :] = float("-inf")
        lg[4, :] = float("nan")
        lg[5, [7, V // 2]] = torch.tensor([3.0, 3.0], device=DEV)
        out = torch.full((6,), -1, dtype=torch.int32, device=DEV)
        ops.sample(lg, out)
        assert out.tolist() == [V - 1, V // 3, 0, 0, 0, 7], V


@pytest.mark.parametrize("dtype", DTYPES)
def test_bias_add_and_residual_add(ops, dtype):
    g = torch.Generator().manual_seed(12)
    x = torch.randn(7, 331, generator=g).to(dtype).to(DEV)
    b = torch.randn(331, generator=g).to(DEV)
    want = (x.double() + b.double())
    ops.bias_add(x, b)
    torch.testing.assert_close(x.double(), want, **tol(dtype))
    stream = torch.randn(7, 331, generator=g).to(DEV)
    delta = torch.randn(7, 331, generator=g).to(dtype).to(DEV)
    want = stream.double() + delta.double()
    ops.residual_add(stream, delta)
    torch.testing.assert_close(stream.double(), want, atol=1e-6, rtol=1e-6)   # the sum itself is float


@pytest.mark.parametrize("page_size", [4, 16, 48])
@pytest.mark.parametrize("through_rows", [False, True])
def test_decode_advance(ops, page_size, through_rows):
    """Between two decode steps of one launch: live rows move on by one position, take the token just chosen and
    get their slot from their block table (also across a page's edge, in every cache group; the table's row is
    the batch's row or the one ``table_rows`` names); other rows stay."""
    g = torch.Generator().manual_seed(page_size)
    R, width, live = 9, 6, 6
    pos = torch.tensor([0, page_size - 2, page_size - 1, 2 * page_size - 1, 3 * page_size + 1, 5, 7, 8, 9], dtype=torch.int32)
    rows = torch.randperm(R + 4, generator=g)[:R].to(torch.int32) if through_rows else torch.arange(R, dtype=torch.int32)
    tables = [torch.randint(1, 500, (R + 4 if through_rows else R, width), generator=g, dtype=torch.int32) for _ in range(2)]
    prev = torch.randint(0, 1000, (R,), generator=g, dtype=torch.int32)
    toks = torch.randint(0, 1000, (R,), generator=g, dtype=torch.int32)
    ctx = pos + 1
    slots = [torch.full((R,), -7, dtype=torch.int32) for _ in range(2)]
    dev = lambda t: t.clone().to(DEV)
    d_tok, d_pos, d_ctx, d_slots = dev(toks), dev(pos), dev(ctx), [dev(s_) for s_ in slots]
    draws = torch.arange(10, 10 + R, dtype=torch.int32, device=DEV)
    ops.decode_advance(dev(prev), d_tok, d_pos, d_ctx, torch.tensor([live], dtype=torch.int32, device=DEV),
                       dev(rows) if through_rows else None, [dev(t) for t in tables], d_slots, page_size,
                       draws if through_rows else None)
    assert draws.tolist() == [10 + r + (1 if r < live and through_rows else 0) for r in range(R)]
    for r in range(R):
        if r < live:
            p = int(pos[r]) + 1
            assert (int(d_pos[r]), int(d_ctx[r]), int(d_tok[r])) == (p, p + 1, int(prev[r]))
            for t, sl in zip(tables, d_slots):
                assert int(sl[r]) == int(t[int(rows[r]), p // page_size]) * page_size + p % page_size
        else:
            assert (int(d_pos[r]), int(d_ctx[r]), int(d_tok[r])) == (int(pos[r]), int(ctx[r]), int(toks[r]))
            assert all(int(sl[r]) == -7 for sl in d_slots)


def test_table_update_and_zero_rows(ops):
    """The device's block tables take the entries that changed (counts on the device; an index past the table or
    negative is left alone), and state slots are zeroed by row (as many as a device count says)."""
    g = torch.Generator().manual_seed(4)
    tables = [torch.randint(1, 99, (7, 11), generator=g, dtype=torch.int32) for _ in range(3)]
    want = [t.clone() for t in tables]
    U = 300
    index, value, counts = [], [], []
    for gi, t in enumerate(want):
        n = (0, 40, 77)[gi]
        ix = torch.randperm(77, generator=g)[:n].to(torch.int32)
        v = torch.randint(100, 999, (n,), generator=g, dtype=torch.int32)
        t.view(-1)[ix.long()] = v
        pad_i = torch.full((U - n,), -1, dtype=torch.int32)
        pad_i[:3] = torch.tensor([77, 5000, -9])             # would be out of the table: never written
        index.append(torch.cat([ix, pad_i])); value.append(torch.cat([v, torch.full((U - n,), 12345, dtype=torch.int32)]))
        counts.append(n + (3 if gi == 1 else 0))              # group 1 also counts its three bad indices
    dev_tables = [t.to(DEV) for t in tables]
    ops.table_update(dev_tables, [i.to(DEV) for i in index], [v.to(DEV) for v in value],
                     torch.tensor(counts, dtype=torch.int32, device=DEV), U)
    for got, w in zip(dev_tables, want):
        assert torch.equal(got.cpu(), w)
    for dtype, shape in ((torch.float32, (9, 5, 3)), (torch.bfloat16, (9, 6)), (torch.int32, (9,))):
        t = torch.ones(shape, dtype=dtype, device=DEV)
        rows = torch.tensor([7, 2, 4, 0], dtype=torch.int32, device=DEV)
        ops.zero_rows(t, rows, torch.tensor([3], dtype=torch.int32, device=DEV))
        live = t.reshape(9, -1).float().abs().sum(1).cpu() > 0
        assert live.tolist() == [True, True, False, True, False, True, True, False, True]
        ops.zero_rows(t, rows)
        assert float(t.reshape(9, -1)[0].float().abs().sum()) == 0


def _draws(ops, logits, n, temperature=1.0, top_k=0, top_p=1.0, seed=0):
    M = n
    lg = logits.to(DEV).expand(M, -1).contiguous()
    out = torch.empty(M, dtype=torch.int32, device=DEV)
    ops.sample(lg, out, torch.full((M,), temperature, device=DEV), torch.full((M,), top_k, dtype=torch.int32, device=DEV),
               torch.full((M,), top_p, device=DEV), torch.full((M,), seed, dtype=torch.int64, device=DEV),
               torch.arange(M, dtype=torch.int32, device=DEV))
    return out.cpu()


def test_sample_distribution_and_filters(ops):
    # vectors of the reference's tests/test_sampler.py
    assert set(_draws(ops, torch.tensor([[0.1, 2.0, 0.5]]), 20, top_k=1).tolist()) == {1}
    assert set(_draws(ops, torch.tensor([[2.0, 1.0, 0.0, -1.0]]), 300, top_p=0.7).tolist()) == {0, 1}
    assert set(_draws(ops, torch.tensor([[10.0, 0.0, 0.0]]), 50, top_p=1e-4).tolist()) == {0}
    d = _draws(ops, torch.log(torch.tensor([[0.7, 0.2, 0.1]])), 4000, seed=123)
    freq = torch.bincount(d, minlength=3).float() / 4000
    assert torch.allclose(freq, torch.tensor([0.7, 0.2, 0.1]), atol=0.03)
    # temperature sharpens: T = 0.5 squares the odds
    d = _draws(ops, torch.log(torch.tensor([[0.5, 0.5 / 3]])), 4000, temperature=0.5, seed=5)
    assert abs((d == 0).float().mean().item() - 0.9) < 0.03
    # same seed and draw index, same token; top-k = 2 on a wide row leaves two tokens
    row = torch.randn(1, 5000, generator=torch.Generator().manual_seed(8))
    a, b = _draws(ops, row, 64, seed=9), _draws(ops, row, 64, seed=9)
    assert torch.equal(a, b) and len(set(a.tolist())) > 10
    top2 = set(row[0].topk(2).indices.tolist())
    assert set(_draws(ops, row, 200, top_k=2, seed=1).tolist()) == top2


def test_ops_refuse_cpu_tensors_and_wrong_shapes(ops):
    with pytest.raises(RuntimeError, match="no CPU path"):
        ops.silu_mul(torch.zeros(2, 4), torch.zeros(2, 2))
    with pytest.raises(ValueError):
        ops.silu_mul(torch.zeros(2, 4, device=DEV), torch.zeros(2, 3, device=DEV))
    with pytest.raises(RuntimeError, match="unsupported"):
        kp = torch.zeros(2, 1, 4, 260, device=DEV)  # head sizes go up to 256
        ops.paged_attention_generic(torch.zeros(1, 260, device=DEV), kp, kp, torch.zeros(1, 1, dtype=torch.int32, device=DEV),
                                    torch.zeros(1, dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV),
                                    torch.zeros(1, 260, device=DEV), 1, 1.0)


@pytest.mark.parametrize("M", [1, 8, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K", [(1152, 896), (331, 72), (896, 4864), (50, 200), (9728, 104), (17000, 64)])
def test_gemm_skinny(ops, M, N, K):
    g = torch.Generator().manual_seed(M * 1000 + N)
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T
    out = ops.gemm_skinny(a, w, bias)
    torch.testing.assert_close(out.double(), want + bias.double(), **tol(torch.bfloat16))
    f = ops.gemm_skinny(a, w, None, out_dtype=torch.float32)
    assert f.dtype == torch.float32
    torch.testing.assert_close(f.double(), want, atol=2e-5, rtol=2e-5)
    x = torch.randn(M, N, generator=g).to(DEV)
    x0 = x.clone()
    ops.gemm_skinny(a, w, bias, ops.EPI_RESIDUAL, residual=x)
    torch.testing.assert_close(x.double(), x0.double() + want + bias.double(), atol=2e-5, rtol=2e-5)
    if N % 2 == 0:
        act = ops.gemm_skinny(a, w, None, ops.EPI_SWIGLU)
        wantact = torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2]
        torch.testing.assert_close(act.double(), wantact, **tol(torch.bfloat16))
    # a row slice of a wider matrix, and the same row alone: the same bits whatever else is in the batch
    wide = torch.zeros(M, K + 8, dtype=torch.bfloat16, device=DEV)
    wide[:, :K] = a
    assert torch.equal(ops.gemm_skinny(wide[:, :K], w, bias), out)
    assert torch.equal(ops.gemm_skinny(a[M - 1:], w, bias), out[M - 1:])


@pytest.mark.parametrize("M", [3, 40])
@pytest.mark.parametrize("shape", [(4, 4, 0), (4, 8, 0), (3, 4, 0), (3, 8, 0), (2, 8, 0), (2, 16, 0), (1, 8, 0), (1, 16, 0),
                                   (4, 8, 1), (3, 8, 1), (2, 8, 2)])
def test_gemm_skinny_block_shapes(ops, M, shape):
    """Every block shape on offer (tiles per block, waves, token groups per block) gives the same numbers (to
    float rounding of another summation order), also with the gated epilogue and the folded norm.  A forced
    shape also keeps few rows in this kernel; unforced they go to the streaming kernel, which must agree."""
    from llm_infrence_engine_amd.kernels import build

    lib = build.load()
    g = torch.Generator().manual_seed(sum(shape) + M)
    N, K = 1000, 1544
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T + bias.double()
    x0 = torch.randn(M, N, generator=g).to(DEV)
    try:
        lib.ms_gemm_skinny_force(*shape)
        x = x0.clone()
        try:
            ops.gemm_skinny(a, w, bias, ops.EPI_RESIDUAL, residual=x)
        except RuntimeError as e:      # a shape that does not fit LDS with this many token groups is refused
            assert "unsupported" in str(e) and (shape[1] - 1) * shape[0] * (shape[2] or (1 if M <= 16 else 4)) > 60
            return
        torch.testing.assert_close(x.double(), x0.double() + want, atol=3e-5, rtol=3e-5)
        f = ops.gemm_skinny(a, w, bias, out_dtype=torch.float32)
        torch.testing.assert_close(f.double(), want, atol=3e-5, rtol=3e-5)
        # gated epilogue over interleaved rows, norm folded in: against the default shape
        x32 = torch.randn(M, K, generator=g).to(DEV)
        nw = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
        got = ops.gemm_skinny_norm(x32, nw, 1e-6, w, None, ops.EPI_SWIGLU)
        lib.ms_gemm_skinny_force(0, 0, 0)
        ref = ops.gemm_skinny_norm(x32, nw, 1e-6, w, None, ops.EPI_SWIGLU)
        torch.testing.assert_close(got.double(), ref.double(), atol=1e-2, rtol=1e-2)
    finally:
        lib.ms_gemm_skinny_force(0, 0, 0)


@pytest.mark.parametrize("M", [1, 5, 8, 16])
@pytest.mark.parametrize("N,K", [(896, 4864), (1152, 896), (330, 72), (52, 200), (9728, 904), (1000, 9000), (4000, 2056),
                                 (16384, 64)])
def test_gemm_stream(ops, M, N, K):
    """The streaming kernel at every shape it can compute: one or several stages, a last k-step that K fills in
    part, one to four tiles of rows to a block, rows that run out in the last block; every epilogue, the folded
    norm with gathered rows; a row's numbers do not depend on the rest of the batch."""
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T
    out = ops.gemm_stream(a, w, bias)
    torch.testing.assert_close(out.double(), want + bias.double(), **tol(torch.bfloat16))
    f = ops.gemm_stream(a, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(f.double(), want, atol=3e-5, rtol=3e-5)
    x = torch.randn(M, N, generator=g).to(DEV)
    x0 = x.clone()
    ops.gemm_stream(a, w, bias, ops.EPI_RESIDUAL, residual=x)
    torch.testing.assert_close(x.double(), x0.double() + want + bias.double(), atol=3e-5, rtol=3e-5)
    act = ops.gemm_stream(a, w, None, ops.EPI_SWIGLU)
    torch.testing.assert_close(act.double(), torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2], **tol(torch.bfloat16))
    assert torch.equal(ops.gemm_stream(a[M - 1:], w, bias), out[M - 1:])
    # the folded norm over gathered rows of a taller residual stream
    xs = torch.randn(M + 3, K, generator=g).to(DEV)
    nw = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
    rows = torch.randperm(M + 3, generator=g)[:M].to(torch.int32).to(DEV)
    xr = xs[rows.long()].double()
    h = (xr * nw.double()).float().bfloat16().double() * torch.rsqrt((xr * xr).mean(-1, keepdim=True) + 1e-5)
    got = ops.gemm_stream(xs, w, bias, out_dtype=torch.float32, norm_weight=nw, eps=1e-5, rows=rows)
    torch.testing.assert_close(got.double(), h @ w.double().T + bias.double(), atol=2e-4, rtol=2e-4)
    gated = ops.gemm_stream(xs, w, None, ops.EPI_SWIGLU, norm_weight=nw, eps=1e-5, rows=rows)
    hw = h @ w.double().T
    torch.testing.assert_close(gated.double(), torch.nn.functional.silu(hw[:, 0::2]) * hw[:, 1::2], **tol(torch.bfloat16))


@pytest.mark.parametrize("M", [1, 3, 7, 16])
@pytest.mark.parametrize("N,K", [(898, 6136), (898, 2056), (1030, 264), (2040, 1032), (4100, 1000), (898, 1000), (514, 424),
                                 (1030, 584), (2040, 904), (1030, 3080), (2046, 1000), (4100, 904)])
def test_products_in_units_of_four_rows(ops, M, N, K):
    """Few rows and a narrow matrix, on both sides of where it is worth it: one or two units of four rows to a block, 8 and 16
    waves, one to three loads of four k-steps, steps that fill a load in part, a last step that K fills in part, rows that run out inside a unit, strided activations.  A
    row has the same bits alone and among the rows that go to the tiled kernel; an infinite activation stays in its row.
    Tolerance: float sums of K products of unit variance over another order."""
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    a = torch.randn(16, K + 8, generator=g).bfloat16().to(DEV)[:, :K]
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T
    got = ops.gemm_skinny(a[:M], w, out_dtype=torch.float32)
    torch.testing.assert_close(got.double(), want[:M], atol=3e-5, rtol=3e-5)
    assert torch.equal(got, ops.gemm_skinny(a, w, out_dtype=torch.float32)[:M])
    x = torch.randn(16, K, generator=g).to(DEV)
    nw = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
    h = (x.double() * nw.double()).float().bfloat16().double() * torch.rsqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-6)
    got = ops.gemm_skinny_norm(x[:M], nw, 1e-6, w, bias, out_dtype=torch.float32)
    torch.testing.assert_close(got.double(), (h @ w.double().T + bias.double())[:M], atol=2e-4, rtol=2e-4)
    if K < 2048:   # (longer rows with a norm are staged, by as many columns as the rows leave room for)
        assert torch.equal(got, ops.gemm_skinny_norm(x, nw, 1e-6, w, bias, out_dtype=torch.float32)[:M])
    b = a[:M].clone()
    b[0, K - 1] = float("inf")
    torch.testing.assert_close(ops.gemm_skinny(b, w, out_dtype=torch.float32)[1:].double(), want[1:M], atol=3e-5, rtol=3e-5)


@pytest.mark.parametrize("M", [1, 4, 5, 16])
@pytest.mark.parametrize("N,K", [(2, 64), (898, 4872), (1030, 264), (5120, 2056), (9728, 904), (4100, 1000), (16 * 256 * 9 + 6, 136),
                                 (3000, 128), (7168, 2560)])
def test_gemm_ring(ops, M, N, K):
    """W ringed through LDS: blocks of two rows and of 146, tiles of 4, 8, 12 and 16 rows, fewer items than waves, tiles that
    several waves share and waves that hold several tiles, columns that end inside a strip, one strip; every epilogue, the
    folded norm with gathered rows, strided activations; a row's numbers do not depend on the rest of the batch, and what is
    not a number stays in its row.  Tolerances: float sums of K products of unit variance over another order."""
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    a = torch.randn(M, K + 8, generator=g).bfloat16().to(DEV)[:, :K]
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T
    out = ops.gemm_ring(a, w, bias)
    torch.testing.assert_close(out.double(), want + bias.double(), **tol(torch.bfloat16))
    f = ops.gemm_ring(a, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(f.double(), want, atol=3e-5, rtol=3e-5)
    x = torch.randn(M, N, generator=g).to(DEV)
    x0 = x.clone()
    ops.gemm_ring(a, w, bias, ops.EPI_RESIDUAL, residual=x)
    torch.testing.assert_close(x.double(), x0.double() + want + bias.double(), atol=3e-5, rtol=3e-5)
    act = ops.gemm_ring(a, w, None, ops.EPI_SWIGLU)
    torch.testing.assert_close(act.double(), torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2], **tol(torch.bfloat16))
    assert torch.equal(ops.gemm_ring(a[M - 1:], w, bias), out[M - 1:])
    if M > 1:
        b = a.clone()
        b[0, K - 1] = float("nan")
        assert torch.equal(ops.gemm_ring(b, w, bias)[1:], out[1:])
    xs = torch.randn(M + 3, K, generator=g).to(DEV)
    nw = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
    rows = torch.randperm(M + 3, generator=g)[:M].to(torch.int32).to(DEV)
    xr = xs[rows.long()].double()
    h = (xr * nw.double()).float().bfloat16().double() * torch.rsqrt((xr * xr).mean(-1, keepdim=True) + 1e-5)
    if M * K > 46000:
        with pytest.raises(RuntimeError, match="unsupported"):
            ops.gemm_ring(xs, w, bias, norm_weight=nw, eps=1e-5, rows=rows)
        return
    got = ops.gemm_ring(xs, w, bias, out_dtype=torch.float32, norm_weight=nw, eps=1e-5, rows=rows)
    torch.testing.assert_close(got.double(), h @ w.double().T + bias.double(), atol=2e-4, rtol=2e-4)
    gated = ops.gemm_ring(xs, w, None, ops.EPI_SWIGLU, norm_weight=nw, eps=1e-5, rows=rows)
    hw = h @ w.double().T
    torch.testing.assert_close(gated.double(), torch.nn.functional.silu(hw[:, 0::2]) * hw[:, 1::2], **tol(torch.bfloat16))


@pytest.mark.parametrize("M", [1, 4, 9, 16])
def test_a_large_matrix_goes_to_the_ring(ops, M):
    """Both sides of the line on values of W, the activations that only these products have, and the front of an attention
    layer of that size against the separate kernels (values transposed and not)."""
    g = torch.Generator().manual_seed(M)
    for N, K in ((12000, 2000), (11990, 2000)):
        a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
        w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
        f = ops.gemm_skinny(a, w, out_dtype=torch.float32)
        assert torch.equal(f, ops.gemm_ring(a, w, out_dtype=torch.float32)) == (N * K >= 24000000 and M <= 8)
        want = a.double() @ w.double().T
        torch.testing.assert_close(f.double(), want, atol=3e-5, rtol=3e-5)
        torch.testing.assert_close(ops.gemm_skinny(a, w, None, ops.EPI_RELU2).double(), want.clamp(min=0) ** 2, **tol(torch.bfloat16))
        numbers = torch.tensor([1.5, 1.702], device=DEV)
        gate, up = want[:, 0::2].clamp(max=1.5), want[:, 1::2].clamp(-1.5, 1.5)
        torch.testing.assert_close(ops.gemm_skinny(a, w, numbers, ops.EPI_CLAMPED).double(), gate * torch.sigmoid(1.702 * gate) * (up + 1),
                                   **tol(torch.bfloat16))
    if M * 4608 <= 46000:
        _qkv_fused_case(ops, M, 32, 5, 128, 4608, True)
        _qkv_fused_case(ops, M, 72, 5, 64, 4616, False)


@pytest.mark.parametrize("M", [1, 9, 17, 33, 64])
@pytest.mark.parametrize("N,K", [(2, 64), (6, 8), (898, 1032), (1030, 264), (5120, 520), (16 * 256 * 10 + 6, 136), (2560, 9000),
                                 (16 * 256 * 10 * 2 + 20, 72)])
def test_gemm_slab(ops, M, N, K):
    """Slabs of W through LDS: blocks of fewer rows than a unit and of ten tiles, one slab and three to a CU, fewer items than
    waves, waves that begin and end inside a slice, columns that end inside a slice; every epilogue, strided activations;
    a row's numbers do not depend on the rest of the batch, and what is not a number stays in its row.  Tolerances: float sums
    of K products of unit variance over another order."""
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    a = torch.randn(M, K + 8, generator=g).bfloat16().to(DEV)[:, :K]
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T
    out = ops.gemm_slab(a, w, bias)
    torch.testing.assert_close(out.double(), want + bias.double(), **tol(torch.bfloat16))
    f = ops.gemm_slab(a, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(f.double(), want, atol=3e-5, rtol=3e-5)
    x = torch.randn(M, N, generator=g).to(DEV)
    x0 = x.clone()
    ops.gemm_slab(a, w, bias, ops.EPI_RESIDUAL, residual=x)
    torch.testing.assert_close(x.double(), x0.double() + want + bias.double(), atol=3e-5, rtol=3e-5)
    act = ops.gemm_slab(a, w, None, ops.EPI_SWIGLU)
    torch.testing.assert_close(act.double(), torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2], **tol(torch.bfloat16))
    torch.testing.assert_close(ops.gemm_slab(a, w, None, ops.EPI_RELU2).double(), want.clamp(min=0) ** 2, **tol(torch.bfloat16))
    numbers = torch.tensor([1.5, 1.702], device=DEV)
    gate, up = want[:, 0::2].clamp(max=1.5), want[:, 1::2].clamp(-1.5, 1.5)
    torch.testing.assert_close(ops.gemm_slab(a, w, numbers, ops.EPI_CLAMPED).double(), gate * torch.sigmoid(1.702 * gate) * (up + 1),
                               **tol(torch.bfloat16))
    assert torch.equal(ops.gemm_slab(a[max(0, M - 17):], w, bias), out[max(0, M - 17):])
    b = a.clone()
    b[0, K - 1] = float("nan")
    assert torch.equal(ops.gemm_slab(b, w, bias)[1:], out[1:])


@pytest.mark.parametrize("M", [5, 8, 9, 16, 17, 40, 64])
@pytest.mark.parametrize("N,K", [(896, 896), (900, 1000), (3584, 776), (640, 9000), (10240, 768), (10248, 768), (512, 8192)])
def test_few_rows_by_a_large_matrix_go_to_slabs(ops, M, N, K):
    """Both sides of the lines on the size of W and on its rows: partial sums for a reader that adds them up (the RMS norm,
    against the sum and the norm in double), the plain product and the sum into the residual stream."""
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    want = a.double() @ w.double().T
    torch.testing.assert_close(ops.gemm_skinny(a, w, out_dtype=torch.float32).double(), want, atol=3e-5, rtol=3e-5)
    x = torch.randn(M, N, generator=g).to(DEV)
    x0 = x.double()
    ops.gemm_skinny(a, w, None, ops.EPI_RESIDUAL, residual=x)
    torch.testing.assert_close(x.double(), x0 + want, atol=3e-5, rtol=3e-5)
    parts = ops.gemm_sums(a, w)
    assert (parts is not None) == (750000 <= N * K and N <= 10240 and M > (4 if K >= 8192 else 8))
    if parts is None:
        return
    assert parts.shape == (4, M, N)
    torch.testing.assert_close(parts.double().sum(0), want, atol=3e-5, rtol=3e-5)
    x = x0.float()
    nw = (1 + 0.1 * torch.randn(N, generator=g)).to(DEV)
    rows = torch.randperm(M, generator=g)[:M - 3].to(torch.int32).to(DEV)
    total = x0 + want
    normed = total * torch.rsqrt((total * total).mean(-1, keepdim=True) + 1e-6) * nw.double()
    some = ops.rms_norm(x, nw, 1e-6, torch.empty(M - 3, N, dtype=torch.bfloat16, device=DEV), delta=parts, rows=rows, write_back=False)
    torch.testing.assert_close(some.double(), normed[rows.long()], **tol(torch.bfloat16))
    assert torch.equal(x, x0.float())
    h = ops.rms_norm(x, nw, 1e-6, torch.empty(M, N, dtype=torch.bfloat16, device=DEV), delta=parts)
    torch.testing.assert_close(h.double(), normed, **tol(torch.bfloat16))
    torch.testing.assert_close(x.double(), total, atol=3e-5, rtol=3e-5)


@pytest.mark.parametrize("M", [9, 17])
def test_rows_too_far_apart_for_slabs_go_to_the_other_kernels(ops, M):
    """Rows up to 4,194,304 values apart go through slabs, farther ones as before: long rows in partial sums (plain, into the
    residual stream, and for a reader that would have added them up) and a plain product."""
    from llm_infrence_engine_amd.kernels import linear

    far = (1 << 22) + 8
    flat = torch.zeros((M - 1) * far + 8200, dtype=torch.bfloat16, device=DEV)
    g = torch.Generator().manual_seed(M)
    for N, K in ((1040, 8200), (4200, 2000)):
        a = flat.as_strided((M, K), (far, 1))
        a.copy_(torch.randn(M, K, generator=g).bfloat16())
        w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
        want = a.double() @ w.double().T
        near = flat.as_strided((M, K), (far - 8, 1))
        assert ops.splits_columns(near, w) == (K >= 8192) and ops.gemm_sums(a, w) is None and ops.gemm_sums(near, w) is not None
        torch.testing.assert_close(ops.gemm_skinny(a, w, out_dtype=torch.float32).double(), want, atol=5e-5, rtol=5e-5)
        x = torch.zeros(M, N, device=DEV)
        assert linear.linear_residual(a, w, None, x, True) is None
        torch.testing.assert_close(x.double(), want, atol=5e-5, rtol=5e-5)


@pytest.mark.parametrize("M", [5, 9, 16, 17, 48, 64])
@pytest.mark.parametrize("nh,nkv,d,K,v_transposed", [(14, 2, 64, 896, True), (5, 1, 128, 520, False), (3, 3, 6, 72, False), (70, 5, 64, 136, True)])
def test_gemm_slab_qkv_equals_product_rotation_and_store(ops, M, nh, nkv, d, K, v_transposed):
    """The front of an attention layer of 5 to 64 normed rows against a double product and the plain rotation: heads that
    straddle a unit of four rows and blocks, a token that is not stored, pages plain and transposed."""
    g = torch.Generator().manual_seed(M + d + K)
    page_size, pages = 16, 6
    n = nh + 2 * nkv
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(n * d, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(n * d, generator=g).to(DEV)
    pos = torch.randint(0, 3000, (M,), generator=g).to(torch.int32).to(DEV)
    slots = torch.randperm(pages * page_size, generator=g)[:M].to(torch.int32)
    slots[2] = -1
    slots = slots.to(DEV)
    inv_freq = (1.0 / (1e6 ** (torch.arange(0, d, 2, dtype=torch.float64) / d))).float().to(DEV)
    kp = torch.zeros(pages, nkv, page_size, d, dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros((pages, nkv, d, page_size) if v_transposed else (pages, nkv, page_size, d), dtype=torch.bfloat16, device=DEV)
    q = ops.gemm_slab_qkv(a, w, bias, nh, nkv, d, pos, inv_freq, slots, kp, vp, v_transposed)
    exact = (a.double() @ w.double().T + bias.double()).view(M, n, d).cpu()
    rot = rope_reference(exact[:, :nh + nkv], pos.cpu(), d, inv_freq.double().cpu())
    torch.testing.assert_close(q.double().cpu().view(M, nh, d), rot[:, :nh], atol=3e-2, rtol=1.6e-2)
    for t in range(M):
        s = int(slots[t])
        if s < 0:
            continue
        p, o = divmod(s, page_size)
        torch.testing.assert_close(kp[p, :, o].double().cpu(), rot[t, nh:], atol=3e-2, rtol=1.6e-2)
        v = vp[p, :, :, o] if v_transposed else vp[p, :, o]
        torch.testing.assert_close(v.double().cpu(), exact[t, nh + nkv:], atol=3e-2, rtol=1.6e-2)
    untouched = torch.ones(pages * page_size, dtype=torch.bool)
    untouched[slots[slots >= 0].long().cpu()] = False
    assert (kp.permute(0, 2, 1, 3).reshape(pages * page_size, -1)[untouched.to(DEV)] == 0).all()


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,K,parts", [(65, 896, 896, 3), (390, 900, 4864, 5), (1, 2, 64, 1), (257, 258, 192, 3), (700, 2304, 448, 7),
                                         (1025, 130, 1024, 8)])
def test_gemm_tiled_sums(ops, M, N, K, parts, tile):
    """The tiled product in runs of its columns: every tile, runs of different lengths and of one and two steps, blocks that
    deal out unevenly over the XCDs, features and tokens that fill no whole tile; each part against its own columns in double,
    and the norm that adds them up (one part too)."""
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    force = ops._get("ms_gemm_tiled_force")
    force(tile)
    try:
        got = ops.gemm_tiled_sums(a, w, parts)
    finally:
        force(0)
    edges = [K // 64 * p // parts * 64 for p in range(parts + 1)]
    for p in range(parts):
        want = a[:, edges[p]:edges[p + 1]].double() @ w[:, edges[p]:edges[p + 1]].double().T
        torch.testing.assert_close(got[p].double(), want, atol=3e-5, rtol=3e-5)
    x = torch.randn(M, N, generator=g).to(DEV)
    nw = (1 + 0.1 * torch.randn(N, generator=g)).to(DEV)
    total = x.double() + got.double().sum(0)
    normed = total * torch.rsqrt((total * total).mean(-1, keepdim=True) + 1e-6) * nw.double()
    h = ops.rms_norm(x, nw, 1e-6, torch.empty(M, N, dtype=torch.bfloat16, device=DEV), delta=got)
    torch.testing.assert_close(h.double(), normed, **tol(torch.bfloat16))
    torch.testing.assert_close(x.double(), total, atol=3e-5, rtol=3e-5)


@pytest.mark.parametrize("V", [5, 2048, 2049, 40000, 151936])
def test_greedy_rows_among_drawn_ones(ops, V):
    """Rows without temperature in a call that draws others: the first of equal maxima, on either side of a chunk's edge, +0 and
    -0 equal, NaN never, -inf only (the first) and NaN only (0); many rows and few, which are cut into other chunks."""
    g = torch.Generator().manual_seed(V)
    for M in (3, 40):
        x = torch.randn(M, V, generator=g)
        want = torch.empty(M, dtype=torch.int32)
        for r in range(M):
            if r % 8 == 1:
                at = sorted(torch.randperm(V, generator=g)[:3].tolist())
                x[r, at] = 50.0
                x[r, (at[0] + 1) % V if V > 5 and (at[0] + 1) % V not in at else at[0]] = float("nan") if V > 5 else 50.0
            if r % 8 == 2:
                x[r] = -x[r].abs() - 1
                x[r, V // 3], x[r, V // 2] = -0.0, 0.0
            if r % 8 == 3:
                x[r] = -math.inf
            if r % 8 == 4:
                x[r] = float("nan")
            y = torch.where(torch.isnan(x[r]), torch.full_like(x[r], -math.inf), x[r])
            first = int((y == y.max()).nonzero()[0])
            want[r] = 0 if torch.isnan(x[r]).all() else first
        T = torch.zeros(M)
        T[0], T[-1] = 1.0, -1.0
        logits = x.to(DEV)
        out = torch.full((M,), -1, dtype=torch.int32, device=DEV)
        top_k, top_p = torch.full((M,), 3, dtype=torch.int32, device=DEV), torch.full((M,), 0.9, device=DEV)
        ops.sample(logits, out, T.to(DEV), top_k, top_p, torch.arange(M, device=DEV), torch.zeros(M, dtype=torch.int32, device=DEV))
        assert torch.equal(out.cpu()[1:], want[1:])
        assert 0 <= int(out[0]) < V


@pytest.mark.parametrize("delta", [None, "bfloat16", "sums"])
def test_rms_norm_of_rows_at_odd_addresses(ops, delta):
    """Operands that start between two groups of four values are read one value at a time."""
    g = torch.Generator().manual_seed(3)
    N, H = 5, 900
    x = torch.randn(N * H + 1, generator=g).to(DEV)[1:].view(N, H)
    out = torch.zeros(N * H + 1, dtype=torch.bfloat16, device=DEV)[1:].view(N, H)
    nw = (1 + 0.1 * torch.randn(H + 1, generator=g)).to(DEV)[1:]
    d = None
    if delta == "bfloat16":
        d = torch.randn(N * H + 1, generator=g).bfloat16().to(DEV)[1:].view(N, H)
    elif delta == "sums":
        d = torch.randn(3 * N * H + 1, generator=g).to(DEV)[1:].view(3, N, H)
    total = x.double() + (0 if d is None else d.double().view(-1, N, H).sum(0))
    ops.rms_norm(x, nw, 1e-6, out, delta=d)
    want = total * torch.rsqrt((total * total).mean(-1, keepdim=True) + 1e-6) * nw.double()
    torch.testing.assert_close(out.double(), want, **tol(torch.bfloat16))
    torch.testing.assert_close(x.double(), total, atol=3e-6, rtol=3e-6)


def test_gemm_stream_refuses_what_it_cannot_take(ops):
    w = torch.zeros(64, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError, match="unsupported"):
        ops.gemm_stream(torch.zeros(17, 64, dtype=torch.bfloat16, device=DEV), w)            # more than 16 rows
    with pytest.raises(RuntimeError, match="unsupported"):
        ops.gemm_stream(torch.zeros(2, 36, dtype=torch.bfloat16, device=DEV),
                        torch.zeros(8, 36, dtype=torch.bfloat16, device=DEV))                 # K no multiple of 8
    with pytest.raises(RuntimeError, match="unsupported"):                                   # not the shape it is for
        ops.gemm_stream(torch.zeros(2, 64, dtype=torch.bfloat16, device=DEV), w, any_shape=False)


@pytest.mark.parametrize("M", [17, 32, 41, 64])
@pytest.mark.parametrize("N,K", [(7000, 96), (4100, 200), (330, 256), (48, 896), (16 * 256 * 17 + 6, 64), (1000, 1000)])
def test_gemm_panel(ops, M, N, K):
    """The kernel that holds the activations in LDS, at every shape it can compute: blocks of one tile, of a few
    tiles whose k-steps several waves share, and of more tiles than waves; a last k-step that K fills in part;
    rows of W that run out inside the last tile; every epilogue, the folded norm with gathered rows; a row's
    numbers do not depend on the rest of the batch."""
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T
    out = ops.gemm_panel(a, w, bias)
    torch.testing.assert_close(out.double(), want + bias.double(), **tol(torch.bfloat16))
    f = ops.gemm_panel(a, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(f.double(), want, atol=3e-5, rtol=3e-5)
    x = torch.randn(M, N, generator=g).to(DEV)
    x0 = x.clone()
    ops.gemm_panel(a, w, bias, ops.EPI_RESIDUAL, residual=x)
    torch.testing.assert_close(x.double(), x0.double() + want + bias.double(), atol=3e-5, rtol=3e-5)
    act = ops.gemm_panel(a, w, None, ops.EPI_SWIGLU)
    torch.testing.assert_close(act.double(), torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2], **tol(torch.bfloat16))
    assert torch.equal(ops.gemm_panel(a[M - 3:], w, bias), out[M - 3:])
    # the folded norm over gathered rows of a taller residual stream
    xs = torch.randn(M + 3, K, generator=g).to(DEV)
    nw = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
    rows = torch.randperm(M + 3, generator=g)[:M].to(torch.int32).to(DEV)
    xr = xs[rows.long()].double()
    h = (xr * nw.double()).float().bfloat16().double() * torch.rsqrt((xr * xr).mean(-1, keepdim=True) + 1e-5)
    got = ops.gemm_panel(xs, w, bias, out_dtype=torch.float32, norm_weight=nw, eps=1e-5, rows=rows)
    torch.testing.assert_close(got.double(), h @ w.double().T + bias.double(), atol=2e-4, rtol=2e-4)
    gated = ops.gemm_panel(xs, w, None, ops.EPI_SWIGLU, norm_weight=nw, eps=1e-5, rows=rows)
    hw = h @ w.double().T
    torch.testing.assert_close(gated.double(), torch.nn.functional.silu(hw[:, 0::2]) * hw[:, 1::2], **tol(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", [(20, 300, 1200), (33, 4100, 1528), (18, 500, 2040),
                                   (64, 4300, 3584), (40, 700, 5120), (64, 4096 + 16 * 256 * 2, 2600), (17, 90, 4872),
                                   (50, 16 * 256 * 33 + 40, 2400), (40, 16 * 256 * 50, 1840)])
def test_gemm_panel_long_rows(ops, M, N, K):
    """Rows of three and four 512-column parts (with three a quarter of the waves sit the loading out), and rows
    that do not fit LDS whole and go through it in chunks: a last chunk that is shorter, blocks with whole and
    shared tiles, two and three whole tiles to a wave."""
    g = torch.Generator().manual_seed(K)
    xs = torch.randn(M, K, generator=g).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    nw = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
    h = (xs.double() * nw.double()).float().bfloat16().double() * torch.rsqrt((xs.double() ** 2).mean(-1, keepdim=True) + 1e-6)
    got = ops.gemm_panel(xs, w, None, out_dtype=torch.float32, norm_weight=nw, eps=1e-6)
    torch.testing.assert_close(got.double(), h @ w.double().T, atol=2e-4, rtol=2e-4)
    a = xs.bfloat16()
    plain = ops.gemm_panel(a, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(plain.double(), a.double() @ w.double().T, atol=3e-5, rtol=3e-5)


@pytest.mark.parametrize("M,N,K", [(8, 5120, 13824), (64, 3584, 18944), (33, 5120, 27648), (17, 900, 8200), (64, 16, 9000),
                                   (5, 8192, 16384), (64, 3584, 3584), (40, 4608, 3584), (64, 7168, 5120), (33, 3100, 3080)])
def test_gemm_with_the_columns_split_over_blocks(ops, M, N, K):
    """Long rows against few of them: blocks take parts of the columns, a second kernel adds the partial sums in
    order.  Every epilogue that has no gate; a row's numbers do not depend on the rest of the batch; parts of
    uneven length, a vocabulary-free odd N, one tile only."""
    from llm_infrence_engine_amd.kernels import build
    assert build.load().ms_gemm_panel_splitk_parts(M, N, K) > 1
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    want = a.double() @ w.double().T
    out = ops.gemm_skinny(a, w, bias)
    torch.testing.assert_close(out.double(), want + bias.double(), **tol(torch.bfloat16))
    f = ops.gemm_skinny(a, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(f.double(), want, atol=5e-5, rtol=5e-5)
    x = torch.randn(M, N, generator=g).to(DEV)
    x0 = x.clone()
    ops.gemm_skinny(a, w, bias, ops.EPI_RESIDUAL, residual=x)
    torch.testing.assert_close(x.double(), x0.double() + want + bias.double(), atol=5e-5, rtol=5e-5)
    assert torch.equal(ops.gemm_skinny(a[M - 1:], w, bias), out[M - 1:]) or M > 16   # the same kernel for one row
    unsplit = ops.gemm_skinny(a, w, None, out_dtype=torch.float32, split_columns=False)
    torch.testing.assert_close(unsplit.double(), want, atol=5e-5, rtol=5e-5)


def test_columns_are_split_only_where_it_pays(ops):
    from llm_infrence_engine_amd.kernels import build
    parts = build.load().ms_gemm_panel_splitk_parts
    assert parts(8, 896, 4864) == 0          # rows too short
    assert parts(8, 3584, 18944) == 0        # few tokens and a tile for nearly every CU: as well unsplit
    assert parts(8, 37888, 3584) == 0        # and here, with tiles enough for every CU besides
    assert parts(65, 3584, 18944) == 0       # too many tokens
    assert parts(8, 16384, 18944) == 0       # more than two tiles per CU
    assert parts(64, 3584, 3584) == 4 and parts(64, 5120, 5120) == 4   # shorter rows: only with more than 32 tokens ...
    assert parts(32, 3584, 3584) == 0 and parts(64, 2048, 2048) == 0 and parts(64, 896, 4864) == 0   # ... long enough, and a tile to most CUs


def test_gemm_panel_refuses_what_it_cannot_take(ops):
    w = torch.zeros(64, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError, match="unsupported"):
        ops.gemm_panel(torch.zeros(65, 64, dtype=torch.bfloat16, device=DEV), w)             # more than 64 rows
    with pytest.raises(RuntimeError, match="unsupported"):           # in chunks, and too many tiles to a block
        ops.gemm_panel(torch.zeros(64, 2400, dtype=torch.bfloat16, device=DEV),
                       torch.zeros(16 * 256 * 48, 2400, dtype=torch.bfloat16, device=DEV))
    with pytest.raises(RuntimeError, match="unsupported"):                                   # not the shape it is for
        ops.gemm_panel(torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV), w, any_shape=False)


def test_gemm_skinny_refuses_what_it_cannot_take(ops):
    a = torch.zeros(65, 64, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError, match="at most 64 rows"):
        ops.gemm_skinny(a, w)
    with pytest.raises(ValueError, match="multiple of 8"):
        ops.gemm_skinny(a[:4, :60], w[:, :60].contiguous())


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11])
@pytest.mark.parametrize("M,N,K", [(65, 662, 64), (300, 2 * 331, 192), (257, 130, 896), (1000, 2 * 4864, 896), (2051, 1026, 128),
                                   (130, 16, 64), (513, 4100, 1536), (4100, 2 * 331, 64), (6200, 1300, 128), (70, 700, 256),
                                   (390, 258, 320)])
def test_gemm_tiled(ops, M, N, K, tile):
    """The many-rows product and its gated epilogue with every tile shape (256, 128, 64, 192 and 160 features wide and those with
    more steps ahead; 192, 160 and 96 store a lane's results in pieces of 8 and 4 bytes): rows and features that fill no whole tile, rows
    of the result that start at odd addresses, one to five steps of 64 columns and many, and so many tokens that the tiles are
    laid over the XCDs in two and in four rows."""
    force = ops._get("ms_gemm_tiled_force")
    force.restype = None
    g = torch.Generator().manual_seed(M + N)
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    a[M - 1] *= 3.0                                        # the last row is told apart from a repeated one before it
    want = a.double() @ w.double().T
    force(tile)
    try:
        out = ops.gemm_tiled(a, w)
        act = ops.gemm_tiled(a, w, ops.EPI_SWIGLU)
    finally:
        force(0)
    assert out.shape == (M, N) and act.shape == (M, N // 2) and out.dtype == act.dtype == torch.bfloat16
    torch.testing.assert_close(out.double(), want, **tol(torch.bfloat16))
    torch.testing.assert_close(act.double(), torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2], **tol(torch.bfloat16))
    # a row's result does not depend on what else is in the batch
    assert torch.equal(ops.gemm_tiled(a[M - 70:], w), out[M - 70:])


@pytest.mark.parametrize("M,N,K,taken", [(411, 4670, 384, 6), (411, 4674, 384, 2), (146, 19200, 256, 7), (146, 19246, 256, 3), (65, 32640, 64, 3),
                                         (129, 16386, 128, 2), (6143, 1300, 256, 4), (6144, 1300, 256, 2), (640, 6528, 576, 2), (640, 6530, 576, 7)])
def test_gemm_tiled_on_both_sides_of_its_small_tiles(ops, M, N, K, taken):
    """Where the choice goes from deep tiles of 64 x 64 (two a CU) to wider ones, and to shallow ones where these are more; below 256 columns
    from shallow ones to wider (as many tiles of 128 x 128 as CUs); at the ends of the model: the same bits as with either."""
    assert ops._get("ms_gemm_tiled_tile")(M, N, K) == taken
    force = ops._get("ms_gemm_tiled_force")
    force.restype = None
    g = torch.Generator().manual_seed(M + N)
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    out, act = ops.gemm_tiled(a, w), ops.gemm_tiled(a, w, ops.EPI_SWIGLU)
    torch.testing.assert_close(out.double(), a.double() @ w.double().T, **tol(torch.bfloat16))
    for tile in (2, 3, 6):
        force(tile)
        try:
            assert torch.equal(out, ops.gemm_tiled(a, w)) and torch.equal(act, ops.gemm_tiled(a, w, ops.EPI_SWIGLU))
        finally:
            force(0)


def test_gemm_tiled_of_long_rows_is_not_taken_for_small_tiles(ops):
    """A tile of 128 x 128 to nearly every CU, which the library's product is faster than: rows that begin on 8 bytes and
    rows that do not."""
    for n in (15360, 15362):
        assert ops._get("ms_gemm_tiled_tile")(256, n, 4096) == 2
        assert ops._get("ms_gemm_tiled_pays")(256, n, 4096) == 0


def test_gemm_tiled_refuses_what_it_cannot_take_and_linear_goes_on(ops):
    from llm_infrence_engine_amd.kernels import linear

    g = torch.Generator().manual_seed(5)
    a = torch.randn(100, 72, generator=g).bfloat16().to(DEV)
    w = (torch.randn(60, 72, generator=g) / 8).bfloat16().to(DEV)
    with pytest.raises(ops.UnsupportedShape):
        ops.gemm_tiled(a, w)                               # 72 columns: no multiple of 64
    assert not ops.gemm_tiled_pays(a, w)
    with pytest.raises(TypeError):
        ops.gemm_tiled(a.float(), w)
    # the dispatcher: wide enough rows of a narrow model go to the tiled kernel, others to the library
    a2 = torch.randn(200, 128, generator=g).bfloat16().to(DEV)
    w2 = (torch.randn(96, 128, generator=g) / 11).bfloat16().to(DEV)
    assert ops.gemm_tiled_pays(a2, w2)
    got = linear.linear_swiglu(a2, w2)
    ref = a2.double() @ w2.double().T
    torch.testing.assert_close(got.double(), torch.nn.functional.silu(ref[:, 0::2]) * ref[:, 1::2], **tol(torch.bfloat16))
    assert torch.equal(got, ops.gemm_tiled(a2, w2, ops.EPI_SWIGLU))
    assert linear.fallback_count() == 0 or all(k[3] != "tiled gated product" for k in linear.fallbacks)


def test_linear_picks_a_kernel_for_every_shape(ops):
    from llm_infrence_engine_amd.kernels import linear

    g = torch.Generator().manual_seed(11)
    for dtype in DTYPES:
        for M, N, K in [(3, 40, 72), (100, 40, 72), (200, 331, 120), (5, 33, 60), (70, 33, 60)]:
            a = torch.randn(M, K, generator=g).to(dtype).to(DEV)
            w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(dtype).to(DEV)
            b = torch.randn(N, generator=g).to(DEV)
            want = a.double() @ w.double().T + b.double()
            torch.testing.assert_close(linear.linear(a, w, b).double(), want, **tol(dtype))
            lg = linear.linear(a, w, b, out_dtype=torch.float32)
            assert lg.dtype == torch.float32
            torch.testing.assert_close(lg.double(), want, **(tol(torch.float32) if dtype == torch.float32 or M <= 64 else tol(dtype)))
            x = torch.randn(M, N, generator=g).to(DEV)
            x0 = x.clone()
            r = linear.linear_residual(a, w, b, x)
            got = x.double() - x0.double() if r is None else r.double()
            assert (r is None) == (dtype == torch.bfloat16 and M <= 64 and K % 8 == 0)
            torch.testing.assert_close(got, want, **tol(dtype))
        for M in (4, 90):
            a = torch.randn(M, 72, generator=g).to(dtype).to(DEV)
            gate = (torch.randn(50, 72, generator=g) / 8).to(dtype).to(DEV)
            up = (torch.randn(50, 72, generator=g) / 8).to(dtype).to(DEV)
            got = linear.linear_swiglu(a, linear.interleave_rows(gate, up))
            want = torch.nn.functional.silu(a.double() @ gate.double().T) * (a.double() @ up.double().T)
            torch.testing.assert_close(got.double(), want, **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,d,dv,window,transposed", [(3, 1, 20, 20, None, False), (4, 2, 64, 64, None, True), (2, 2, 18, 70, 150, False),
                                                           (2, 1, 128, 256, None, True)])
def test_generic_attention_has_the_same_bits_with_one_wave_and_with_four(ops, dtype, nh, nkv, d, dv, window, transposed):
    """One wave to a (token, head) or four, as the step's size decides: the same runs of keys merged in the same order, at the
    edges of a run's blocks of 64 keys and of the four runs; alone in the step and beside others; against 64 bits."""
    from llm_infrence_engine_amd.kernels import build

    lib = build.load()
    g = torch.Generator().manual_seed(d + dv)
    seen, page = [1, 2, 5, 63, 64, 65, 128, 129, 192, 256, 257, 320, 700], 4
    pages = [-(-n // page) for n in seen]
    N, P = len(seen), sum(pages) + 1
    k, v = torch.randn(P, nkv, page, d, generator=g).to(dtype), torch.randn(P, nkv, page, dv, generator=g).to(dtype)
    k[0] = v[0] = float("nan")
    table = torch.zeros(N, max(pages), dtype=torch.int32)
    q = (torch.randn(N, nh * d, generator=g) * 2).to(dtype)
    want = torch.empty(N, nh, dv, dtype=torch.float64)
    for r, n in enumerate(seen):
        at = torch.arange(pages[r]) + 1 + sum(pages[:r])
        table[r, :pages[r]] = at
        kk, vv = (x[at].transpose(0, 1).reshape(nkv, -1, x.shape[3])[:, :n].double() for x in (k, v))
        want[r] = attention_reference(q[r].reshape(nh, 1, d).double(), kk, vv, d ** -0.5, window)[:, 0]
    vp = (v.transpose(2, 3).contiguous() if transposed else v).to(DEV)
    rows, pos = torch.arange(N, dtype=torch.int32, device=DEV), torch.tensor(seen, dtype=torch.int32, device=DEV) - 1
    q, kp, table = q.to(DEV), k.to(DEV), table.to(DEV)

    def run(waves, lo=0, hi=N):
        out = torch.empty(hi - lo, nh * dv, dtype=dtype, device=DEV)
        lib.ms_attention_generic_force(waves)
        try:
            return ops.paged_attention_generic(q[lo:hi], kp, vp, table, rows[lo:hi], pos[lo:hi], out, nh, d ** -0.5, window,
                                               v_transposed=transposed)
        finally:
            lib.ms_attention_generic_force(0)

    one = run(1)
    torch.testing.assert_close(one.double().cpu(), want.reshape(N, -1), **tol(dtype))
    assert torch.equal(one, run(4)) and torch.equal(one, run(0))
    for r in (0, 4, 9, N - 1):
        assert torch.equal(one[r:r + 1], run(1, r, r + 1)) and torch.equal(one[r:r + 1], run(4, r, r + 1))


def _paged_case(g, dtype, nh, nkv, d, page_size, ctx, qlen, fill):
    """Random requests laid out in shuffled pages (values transposed); returns what the kernels take and
    the plain answer.  Unused slots, the tails of last pages and the null page hold ``fill``."""
    R = len(ctx)
    pages_per = [-(-c // page_size) for c in ctx]
    P = sum(pages_per) + 4
    order = torch.randperm(P - 1, generator=g) + 1
    kp = torch.full((P, nkv, page_size, d), fill, dtype=dtype)
    vt = torch.full((P, nkv, d, page_size), fill, dtype=dtype)
    table = torch.zeros(R, max(pages_per), dtype=torch.int32)
    qs, ks, vs, q_rows, req, pos = [], [], [], [], [], []
    used = 0
    for r in range(R):
        k = torch.randn(nkv, ctx[r], d, generator=g).to(dtype)
        v = torch.randn(nkv, ctx[r], d, generator=g).to(dtype)
        q = (torch.randn(nh, qlen[r], d, generator=g) * 2).to(dtype)
        k[:, min(3, ctx[r] - 1)] = (q[::nh // nkv, -1].float() * 1.5).to(dtype)   # one far key stands out
        pages = order[used:used + pages_per[r]]
        used += pages_per[r]
        table[r, :pages_per[r]] = pages.to(torch.int32)
        for j in range(ctx[r]):
            kp[pages[j // page_size], :, j % page_size] = k[:, j]
            vt[pages[j // page_size], :, :, j % page_size] = v[:, j]
        qs.append(q); ks.append(k); vs.append(v)
        q_rows.append(q.transpose(0, 1).reshape(qlen[r], nh * d))
        req += [r] * qlen[r]
        pos += list(range(ctx[r] - qlen[r], ctx[r]))
    return dict(kp=kp, vt=vt, table=table, q=torch.cat(q_rows), req=req, pos=pos, qs=qs, ks=ks, vs=vs)


@pytest.mark.parametrize("nh,nkv,d,page_size,window", [(14, 2, 64, 16, None), (6, 2, 32, 16, None), (8, 8, 128, 32, None),
                                                        (4, 1, 64, 16, 40), (28, 4, 128, 16, None), (5, 5, 32, 64, 100),
                                                        (6, 2, 64, 48, None)])
@pytest.mark.parametrize("shape", ["mixed", "decode", "long"])
def test_paged_attention_mfma(ops, nh, nkv, d, page_size, window, shape):
    g = torch.Generator().manual_seed(nh * 100 + d)
    if shape == "mixed":
        ctx, qlen = [70, 133, 201, 300], [70, 9, 1, 150]
    elif shape == "decode":
        ctx, qlen = [1, 31, 32, 33, 600, 1000, 64, 17], [1] * 8
    else:   # few requests with long contexts: keys split over blocks and combined
        ctx, qlen = [2500, 1, 300], [1] * 3
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, page_size, ctx, qlen, float("nan"))
    scale = 1.0 / math.sqrt(d)
    assert ops.attention_splits_keys(len(ctx), nkv, nh // nkv, max(qlen), max(ctx)) == (shape == "long")
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), scale, window).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    N = c["q"].shape[0]
    wide = torch.zeros(N, (nh + 2 * nkv) * d, dtype=torch.bfloat16, device=DEV)
    wide[:, :nh * d] = c["q"].to(DEV)
    out = torch.full((N, nh * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    q_start = torch.tensor([0] + list(np.cumsum(qlen)), dtype=torch.int32, device=DEV)
    ops.paged_attention_mfma(wide, c["kp"].to(DEV), c["vt"].to(DEV), c["table"].to(DEV), q_start,
                             torch.tensor(ctx, dtype=torch.int32, device=DEV), out, nh, scale, max(qlen), max(ctx), window)
    torch.testing.assert_close(out.double().cpu(), want, **tol(torch.bfloat16))
    # the generic kernel reads the same transposed pages
    out2 = torch.empty_like(out)
    ops.paged_attention_generic(wide, c["kp"].to(DEV), c["vt"].to(DEV), c["table"].to(DEV),
                                torch.tensor(c["req"], dtype=torch.int32, device=DEV),
                                torch.tensor(c["pos"], dtype=torch.int32, device=DEV), out2, nh, scale, window, v_transposed=True)
    torch.testing.assert_close(out2.double().cpu(), want, **tol(torch.bfloat16))


@pytest.mark.parametrize("nh,nkv,d,page_size,window", [(14, 2, 64, 16, None), (6, 2, 32, 16, 50), (8, 2, 128, 32, None)])
@pytest.mark.parametrize("shape", ["mixed", "decode", "long", "many"])
def test_attention_of_a_padded_batch_through_table_rows(ops, nh, nkv, d, page_size, window, shape):
    """A batch as a captured graph sees it: the block table has a row per request the engine can hold and the
    step's requests name theirs; requests without tokens or keys pad the batch, tokens past the last request's
    belong to nobody and their output rows are left alone; the launch is sized for more and longer portions
    than there are.  Matrix-core and generic kernels alike."""
    g = torch.Generator().manual_seed(nh + d)
    if shape == "mixed":
        ctx, qlen = [70, 133, 201, 300], [70, 9, 1, 150]
    elif shape == "decode":
        ctx, qlen = [1, 31, 600, 1000, 64], [1] * 5
    elif shape == "long":
        ctx, qlen = [2500, 1, 300], [1] * 3
    else:   # more requests than a wave has lanes, most of them short portions: the tile search goes round twice
        ctx = [int(v) for v in torch.randint(5, 90, (70,), generator=g)]
        qlen = [min(c, int(v)) for c, v in zip(ctx, torch.randint(1, 6, (70,), generator=g))]
        qlen[40] = ctx[40] = 77
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, page_size, ctx, qlen, float("nan"))
    scale = 1.0 / math.sqrt(d)
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), scale, window).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    R, N = len(ctx), c["q"].shape[0]
    pad_r, pad_n = 3, (0 if shape in ("decode", "long") else 45)       # a decode graph pads requests, not tokens
    if shape in ("decode", "long"):
        pad_n = pad_r                                                    # ... each padding request's row is a padding token
    rows_total = R + pad_r + 2
    perm = torch.randperm(rows_total - 1, generator=g)[:R]              # the last row stays all null pages
    table = torch.zeros(rows_total, c["table"].shape[1] + 3, dtype=torch.int32)
    table[perm, :c["table"].shape[1]] = c["table"]
    table_rows = torch.cat([perm.to(torch.int32), torch.full((pad_r,), rows_total - 1, dtype=torch.int32)]).to(DEV)
    q = torch.full((N + pad_n, nh * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    q[:N] = c["q"].to(DEV)
    q_start = torch.tensor([0] + list(np.cumsum(qlen)) + [N] * pad_r, dtype=torch.int32, device=DEV)
    ctx_all = torch.tensor(ctx + [0] * pad_r, dtype=torch.int32, device=DEV)
    room = table.shape[1] * page_size                                   # what a request's table row can hold
    cap_q = max(qlen) if shape in ("decode", "long") else min(N + pad_n, room)
    cap_ctx = room
    out = torch.full((N + pad_n, nh * d), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.paged_attention_mfma(q, c["kp"].to(DEV), c["vt"].to(DEV), table.to(DEV), q_start, ctx_all, out, nh, scale,
                             cap_q, cap_ctx, window, table_rows)
    torch.testing.assert_close(out[:N].double().cpu(), want, **tol(torch.bfloat16))
    assert (out[N:] == 7.0).all()
    out2 = torch.full_like(out, 7.0)
    req = torch.tensor(c["req"] + [R + pad_r - 1] * pad_n, dtype=torch.int32, device=DEV)
    pos = torch.tensor(c["pos"] + [0] * pad_n, dtype=torch.int32, device=DEV)
    ops.paged_attention_generic(q, c["kp"].to(DEV), c["vt"].to(DEV), table.to(DEV), req, pos, out2, nh, scale, window,
                                v_transposed=True, table_rows=table_rows, n_live_tokens=q_start[R + pad_r:R + pad_r + 1])
    torch.testing.assert_close(out2[:N].double().cpu(), want, **tol(torch.bfloat16))
    assert (out2[N:] == 7.0).all()


@pytest.mark.parametrize("R,nh,nkv,d,window", [(40, 6, 2, 64, None), (64, 4, 2, 32, None), (21, 8, 4, 128, 700)])
def test_split_decode_attention_of_a_large_uneven_batch(ops, R, nh, nkv, d, window):
    """Many requests whose contexts differ widely, some far beyond the length from which keys are split over
    blocks: few splits per request (a number that is no power of two), short requests that use one of them."""
    g = torch.Generator().manual_seed(R)
    ctx = [int(v) for v in torch.randint(1, 1500, (R,), generator=g)]
    ctx[3], ctx[R - 1] = 2300, 1
    qlen = [1] * R
    assert ops.attention_splits_keys(R, nkv, nh // nkv, 1, max(ctx))
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, 16, ctx, qlen, float("nan"))
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), 1.0 / math.sqrt(d), window).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    torch.testing.assert_close(_run_mfma(ops, c, nh, d, ctx, qlen, window), want, **tol(torch.bfloat16))


@pytest.mark.parametrize("longest,splits_window", [(17000, None), (70000, None), (70000, 30000)])
def test_split_decode_attention_of_very_long_contexts(ops, longest, splits_window):
    """Tens of thousands of keys: more splits than at a few thousand (32 and 128), beside a short request that
    uses one of them."""
    nh, nkv, d = 4, 2, 64
    g = torch.Generator().manual_seed(longest)
    ctx, qlen = [longest, 40], [1, 1]
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, 16, ctx, qlen, float("nan"))
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), 1.0 / math.sqrt(d), splits_window).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    torch.testing.assert_close(_run_mfma(ops, c, nh, d, ctx, qlen, splits_window), want, **tol(torch.bfloat16))


@pytest.mark.parametrize("nh,nkv,d,window", [(4, 2, 64, None), (2, 1, 128, None), (4, 4, 32, None), (4, 2, 64, 700)])
def test_prompt_attention_of_thousands_of_tokens(ops, nh, nkv, d, window):
    """A whole prompt of 3,300 tokens in one step (more column tiles than CUs, late tiles first, every wave of a
    block many key blocks deep) beside a portion of 1,500 tokens behind a prefix of 1,100, with a far key that
    stands out for the last query of each."""
    g = torch.Generator().manual_seed(d + nh)
    ctx, qlen = [3300, 2600], [3300, 1500]
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, 16, ctx, qlen, float("nan"))
    scale = 1.0 / math.sqrt(d)
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), scale, window).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    torch.testing.assert_close(_run_mfma(ops, c, nh, d, ctx, qlen, window), want, **tol(torch.bfloat16))


def _run_mfma(ops, c, nh, d, ctx, qlen, window=None):
    N = c["q"].shape[0]
    out = torch.full((N, nh * d), float("nan"), dtype=torch.bfloat16, device=DEV)
    q_start = torch.tensor([0] + list(np.cumsum(qlen)), dtype=torch.int32, device=DEV)
    ops.paged_attention_mfma(c["q"].to(DEV), c["kp"].to(DEV), c["vt"].to(DEV), c["table"].to(DEV), q_start,
                             torch.tensor(ctx, dtype=torch.int32, device=DEV), out, nh, 1.0 / math.sqrt(d), max(qlen),
                             max(ctx), window)
    return out.double().cpu()


@pytest.mark.parametrize("d,shape", [(32, (4, 4, 1)), (32, (2, 4, 1)), (32, (2, 8, 1)), (32, (1, 8, 1)), (32, (1, 16, 1)),
                                     (64, (4, 4, 1)), (64, (2, 4, 1)), (64, (2, 8, 1)), (64, (1, 4, 1)), (64, (1, 8, 1)),
                                     (64, (1, 16, 1)), (128, (2, 4, 1)), (128, (1, 4, 1)), (128, (1, 8, 1)),
                                     (32, (1, 16, 2)), (64, (1, 16, 2)), (64, (1, 16, 4)), (64, (1, 8, 2)), (64, (1, 8, 4)),
                                     (128, (1, 8, 2)), (128, (1, 8, 4))])
def test_attention_mfma_tile_shapes(ops, d, shape):
    """Every tile width, wave count and number of blocks to a narrow tile on the menu gives the same answer (the
    choice by size picks among them)."""
    from llm_infrence_engine_amd.kernels import build
    nh, nkv = 6, 2
    g = torch.Generator().manual_seed(d + shape[0] * 7 + shape[1] + shape[2] * 1000)
    ctx, qlen = [300, 97, 520], [130, 1, 45]
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, 16, ctx, qlen, float("nan"))
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), 1.0 / math.sqrt(d), None).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    lib = build.load()
    lib.ms_attention_mfma_force(*shape)
    try:
        got = _run_mfma(ops, c, nh, d, ctx, qlen)
    finally:
        lib.ms_attention_mfma_force(0, 0, 0)
    torch.testing.assert_close(got, want, **tol(torch.bfloat16))


@pytest.mark.parametrize("nh,nkv,d,page_size,window", [(14, 2, 64, 16, None), (8, 8, 128, 32, None), (4, 1, 64, 16, 40),
                                                        (28, 4, 128, 16, None), (6, 2, 64, 48, 130), (20, 1, 128, 16, 65)])
def test_attention_of_staged_prompts(ops, nh, nkv, d, page_size, window):
    """The prompt kernel that stages keys and values in LDS: single tokens, portions behind cached keys, prompts whose columns
    fill no tile, a request without a token, rows of the table in no order, at the edges of its tiles of 64 keys; what no
    request owns is NaN.  Against the oracle, and against the kernel that shares nothing."""
    g = torch.Generator().manual_seed(nh * 10 + d)
    ctx, qlen = [70, 133, 64, 65, 300, 1, 500], [70, 9, 64, 1, 150, 1, 257]
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, page_size, ctx, qlen, float("nan"))
    scale = 1.0 / math.sqrt(d)
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), scale, window).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    N, R = c["q"].shape[0], len(ctx) + 1
    wide = torch.zeros(N + 5, (nh + 2 * nkv) * d, dtype=torch.bfloat16, device=DEV)      # five tokens of nobody at the end
    wide[:N, :nh * d] = c["q"].to(DEV)
    perm = torch.randperm(R, generator=g)
    table = torch.zeros(R, c["table"].shape[1], dtype=torch.int32)
    table[perm[:R - 1]] = c["table"]
    kp, vt, table, rows = c["kp"].to(DEV), c["vt"].to(DEV), table.to(DEV), perm.to(torch.int32).to(DEV)
    q_start = torch.tensor([0] + list(np.cumsum(qlen)) + [N], dtype=torch.int32, device=DEV)
    lens = torch.tensor(ctx + [7], dtype=torch.int32, device=DEV)
    out = torch.full((N + 5, nh * d), 3.0, dtype=torch.bfloat16, device=DEV)
    ops._call("ms_attention_prompt", wide.data_ptr(), wide.stride(0), kp.data_ptr(), vt.data_ptr(), table.data_ptr(),
              table.shape[1], rows.data_ptr(), q_start.data_ptr(), lens.data_ptr(), out.data_ptr(), nh * d, R, N + 5, 257, nh,
              nkv, d, page_size, scale, window or 0, ops._stream())
    torch.testing.assert_close(out[:N].double().cpu(), want, **tol(torch.bfloat16))
    assert (out[N:] == 3.0).all()
    other = torch.empty(N, nh * d, dtype=torch.bfloat16, device=DEV)
    ops.paged_attention_mfma(wide[:N], kp, vt, table, q_start, lens, other, nh, scale, 257, 500, window, table_rows=rows)
    torch.testing.assert_close(out[:N].double(), other.double(), **tol(torch.bfloat16))


@pytest.mark.parametrize("nh,nkv,d,lens,past,spread,window", [(6, 2, 64, [130] * 8, 0, 2.0, None), (6, 2, 64, [512, 40], 0, 4.0, None),
                                                              (8, 2, 128, [200] * 4, 0, 2.0, None), (4, 2, 128, [700], 900, 3.0, None),
                                                              (4, 1, 64, [700], 900, 3.0, None), (4, 4, 64, [600], 200, 2.0, 100),
                                                              (4, 4, 128, [600], 200, 2.0, 100)])
def test_staged_prompts_lie_no_farther_from_64_bits_than_the_other_kernel(ops, nh, nkv, d, lens, past, spread, window):
    """Both kernels round probabilities to bfloat16 between the two products; how many of a column's largest ones are
    powers of two, and so lose nothing, depends on how its reference moves.  Errors in the 2-norm over a few hundred
    thousand results: two kernels with the same mean square error differ by under 0.2 %, a reference that stays where the
    first 64 keys put it costs 1.5 to 9 % here."""
    g = torch.Generator().manual_seed(d + past)
    R, N, ctx, page = len(lens), sum(lens), [past + n for n in lens], 16
    pages = [-(-n // page) for n in ctx]
    kp = torch.randn(sum(pages) + 1, nkv, page, d, generator=g).bfloat16().to(DEV)
    vp = torch.randn(sum(pages) + 1, nkv, page, d, generator=g).bfloat16().to(DEV)
    vt = vp.transpose(2, 3).contiguous()
    q = (torch.randn(N, nh * d, generator=g) * spread).bfloat16().to(DEV)
    table = torch.zeros(R, max(pages), dtype=torch.int32)
    for r in range(R):
        table[r, :pages[r]] = torch.arange(pages[r]) + 1 + sum(pages[:r])
    table = table.to(DEV)
    q_start = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device=DEV)
    held = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    want = []
    for r in range(R):
        k, v = (x[table[r, :pages[r]].long()].transpose(1, 2).reshape(-1, nkv, d)[:ctx[r]].transpose(0, 1).double() for x in (kp, vp))
        rows = q[int(q_start[r]):int(q_start[r + 1])].reshape(-1, nh, d).transpose(0, 1).double()
        i, j = torch.arange(past, ctx[r], device=DEV)[:, None], torch.arange(ctx[r], device=DEV)[None]
        hidden = (j > i) | (j <= i - window) if window else j > i
        o = [(rows[h] @ k[h * nkv // nh].t() * d ** -0.5).masked_fill(hidden, -math.inf).softmax(-1) @ v[h * nkv // nh] for h in range(nh)]
        want.append(torch.stack(o, 1).reshape(-1, nh * d))
    want = torch.cat(want)
    staged, other = torch.empty_like(q), torch.empty_like(q)
    ops._call("ms_attention_prompt", q.data_ptr(), nh * d, kp.data_ptr(), vt.data_ptr(), table.data_ptr(), table.shape[1], None,
              q_start.data_ptr(), held.data_ptr(), staged.data_ptr(), nh * d, R, N, max(lens), nh, nkv, d, page, d ** -0.5,
              window or 0, ops._stream())
    ops._call("ms_paged_attention_mfma", q.data_ptr(), nh * d, kp.data_ptr(), vt.data_ptr(), table.data_ptr(), table.shape[1], None,
              q_start.data_ptr(), held.data_ptr(), other.data_ptr(), nh * d, R, N, max(lens), nh, nkv, d, d, page, d ** -0.5,
              window or 0, None, 0.0, None, None, 0, 1, 1.0, ops._stream())
    far = [((x.double() - want).norm() / want.norm()).item() for x in (staged, other)]
    assert far[0] <= 1.005 * far[1], far


@pytest.mark.parametrize("ramp", [0.5, 6.0, 60.0])
def test_attention_mfma_when_the_maximum_keeps_rising(ops, ramp):
    """Scores that grow along the context by ``ramp`` log2 units in all: the running reference of the softmax
    stays (small ramp), moves once or moves at almost every block, and late keys dwarf the early ones."""
    nh, nkv, d = 4, 2, 64
    g = torch.Generator().manual_seed(int(ramp * 10))
    ctx, qlen = [640, 333], [200, 1]
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, 16, ctx, qlen, float("nan"))
    scale = 1.0 / math.sqrt(d)
    # all queries share a direction u; key j carries (j / ctx) * ramp * ln2 / scale along it
    u = torch.zeros(d); u[5] = 1.0
    for r in range(len(ctx)):
        c["qs"][r] = (c["qs"][r].float() * 0.05 + u).to(torch.bfloat16)
        steps = torch.arange(ctx[r]).float() / ctx[r] * ramp * math.log(2.0) / scale
        c["ks"][r] = (c["ks"][r].float() * 0.05 + steps[None, :, None] * u).to(torch.bfloat16)
    # lay the changed keys and queries out again
    rows, p = [], 0
    for r in range(len(ctx)):
        for j in range(ctx[r]):
            c["kp"][c["table"][r, j // 16].item(), :, j % 16] = c["ks"][r][:, j]
        rows.append(c["qs"][r].transpose(0, 1).reshape(qlen[r], nh * d))
    c["q"] = torch.cat(rows)
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), scale, None).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    got = _run_mfma(ops, c, nh, d, ctx, qlen)
    torch.testing.assert_close(got, want, **tol(torch.bfloat16))


@pytest.mark.parametrize("nh,nkv,d", [(7, 1, 64), (4, 2, 64), (3, 1, 128), (4, 4, 128)])
@pytest.mark.parametrize("ramp", [0.5, 6.0, 60.0, -6.0, -60.0])
def test_attention_of_staged_prompts_when_scores_rise_or_fall(ops, nh, nkv, d, ramp):
    """Scores that rise or fall along the context by ``ramp`` log2 units in all: the staged kernel's reference follows its first
    keys up and down, stays, or moves at almost every unit of 32, after several tiles of 64 keys to each group of waves; at 64
    dims the two groups end with references apart, late keys dwarf the early ones or the other way round."""
    g = torch.Generator().manual_seed(int(abs(ramp) * 10) + d + nh)
    ctx, qlen, page = [900, 333, 40], [200, 70, 40], 16
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, page, ctx, qlen, float("nan"))
    scale = 1.0 / math.sqrt(d)
    u = torch.zeros(d); u[5] = 1.0
    for r in range(len(ctx)):
        c["qs"][r] = (c["qs"][r].float() * 0.05 + u).to(torch.bfloat16)
        steps = torch.arange(ctx[r]).float() / ctx[r] * ramp * math.log(2.0) / scale
        c["ks"][r] = (c["ks"][r].float() * 0.05 + steps[None, :, None] * u).to(torch.bfloat16)
        for j in range(ctx[r]):
            c["kp"][c["table"][r, j // page].item(), :, j % page] = c["ks"][r][:, j]
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), scale, None).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    q = torch.cat([x.transpose(0, 1).reshape(-1, nh * d) for x in c["qs"]]).to(DEV)
    kp, vt, table = c["kp"].to(DEV), c["vt"].to(DEV), c["table"].to(DEV)
    q_start = torch.tensor([0] + list(np.cumsum(qlen)), dtype=torch.int32, device=DEV)
    lens, out = torch.tensor(ctx, dtype=torch.int32, device=DEV), torch.empty_like(q)
    ops._call("ms_attention_prompt", q.data_ptr(), nh * d, kp.data_ptr(), vt.data_ptr(), table.data_ptr(), table.shape[1], None,
              q_start.data_ptr(), lens.data_ptr(), out.data_ptr(), nh * d, len(ctx), q.shape[0], max(qlen), nh, nkv, d, page,
              scale, 0, ops._stream())
    torch.testing.assert_close(out.double().cpu(), want, **tol(torch.bfloat16))


def _staged(ops, kind, q, kp, vt, table, q_start, lens, nh, longest, window, rows=None, out=None):
    (P, nkv, page, d), N, R = kp.shape, q.shape[0], lens.numel()
    out = torch.full((N, nh * d), 3.0, dtype=torch.bfloat16, device=DEV) if out is None else out
    ops._call("ms_attention_prompt_as", kind, q.data_ptr(), q.stride(0), kp.data_ptr(), vt.data_ptr(), table.data_ptr(), table.shape[1],
              ops._ptr(rows), q_start.data_ptr(), lens.data_ptr(), out.data_ptr(), nh * d, R, N, longest, nh, nkv, d, page, d ** -0.5,
              window or 0, ops._stream())
    return out


@pytest.mark.parametrize("kind", [2, 3])
@pytest.mark.parametrize("nh,nkv,d,page_size,window", [(14, 2, 64, 16, None), (8, 8, 128, 32, None), (4, 1, 64, 16, 40),
                                                        (28, 4, 128, 16, None), (6, 2, 64, 48, 130), (20, 1, 128, 16, 65)])
def test_narrow_kinds_of_staged_prompts(ops, nh, nkv, d, page_size, window, kind):
    """Blocks of 64 columns, and of more groups of waves that share the keys out (fewer tiles of keys than groups, one more than
    a turn, requests of one token): against the oracle; what no request owns is NaN, and tokens of nobody stay as they are."""
    g = torch.Generator().manual_seed(nh * 10 + d + kind)
    ctx, qlen = [70, 133, 64, 65, 300, 1, 257, 513], [70, 9, 64, 1, 150, 1, 257, 257]
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, page_size, ctx, qlen, float("nan"))
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), d ** -0.5, window).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    N, R = c["q"].shape[0], len(ctx) + 1
    wide = torch.zeros(N + 5, (nh + 2 * nkv) * d, dtype=torch.bfloat16, device=DEV)
    wide[:N, :nh * d] = c["q"].to(DEV)
    perm = torch.randperm(R, generator=g)
    table = torch.zeros(R, c["table"].shape[1], dtype=torch.int32)
    table[perm[:R - 1]] = c["table"]
    q_start = torch.tensor([0] + list(np.cumsum(qlen)) + [N], dtype=torch.int32, device=DEV)
    out = _staged(ops, kind, wide, c["kp"].to(DEV), c["vt"].to(DEV), table.to(DEV), q_start, torch.tensor(ctx + [7], dtype=torch.int32, device=DEV),
                  nh, 257, window, perm.to(torch.int32).to(DEV))
    torch.testing.assert_close(out[:N].double().cpu(), want, **tol(torch.bfloat16))
    assert (out[N:] == 3.0).all()


@pytest.mark.parametrize("kind", [2, 3])
@pytest.mark.parametrize("nh,nkv,d", [(7, 1, 64), (4, 4, 128)])
@pytest.mark.parametrize("ramp", [0.5, 60.0, -6.0, -60.0])
def test_narrow_kinds_when_scores_rise_or_fall(ops, nh, nkv, d, ramp, kind):
    """As for the wide kind: the groups of waves end with references apart, late keys dwarf the early ones or the other way."""
    g = torch.Generator().manual_seed(int(abs(ramp) * 10) + d + nh)
    ctx, qlen, page = [900, 333, 40], [200, 70, 40], 16
    c = _paged_case(g, torch.bfloat16, nh, nkv, d, page, ctx, qlen, float("nan"))
    u = torch.zeros(d); u[5] = 1.0
    for r in range(len(ctx)):
        c["qs"][r] = (c["qs"][r].float() * 0.05 + u).to(torch.bfloat16)
        steps = torch.arange(ctx[r]).float() / ctx[r] * ramp * math.log(2.0) / d ** -0.5
        c["ks"][r] = (c["ks"][r].float() * 0.05 + steps[None, :, None] * u).to(torch.bfloat16)
        for j in range(ctx[r]):
            c["kp"][c["table"][r, j // page].item(), :, j % page] = c["ks"][r][:, j]
    want = torch.cat([attention_reference(q.double(), k.double(), v.double(), d ** -0.5, None).transpose(0, 1).reshape(-1, nh * d)
                      for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
    q = torch.cat([x.transpose(0, 1).reshape(-1, nh * d) for x in c["qs"]]).to(DEV)
    q_start = torch.tensor([0] + list(np.cumsum(qlen)), dtype=torch.int32, device=DEV)
    out = _staged(ops, kind, q, c["kp"].to(DEV), c["vt"].to(DEV), c["table"].to(DEV), q_start, torch.tensor(ctx, dtype=torch.int32, device=DEV), nh, 200, None)
    torch.testing.assert_close(out.double().cpu(), want, **tol(torch.bfloat16))


@pytest.mark.parametrize("kind", [1, 2, 3])
@pytest.mark.parametrize("nh,nkv,d,lens,past,spread", [(6, 2, 64, [130] * 8, 0, 2.0), (6, 2, 64, [512, 40], 0, 4.0), (8, 2, 128, [200] * 4, 0, 2.0),
                                                       (4, 2, 128, [700], 900, 3.0), (4, 1, 64, [700], 900, 3.0), (4, 2, 64, [300], 2200, 1.0),
                                                       (4, 2, 128, [300], 2200, 1.0)])
def test_kinds_of_staged_prompts_lie_no_farther_from_64_bits_than_the_other_kernel(ops, nh, nkv, d, lens, past, spread, kind):
    """As the test of the wide kind above, over the kinds."""
    g = torch.Generator().manual_seed(d + past + 5)
    R, N, ctx, page = len(lens), sum(lens), [past + n for n in lens], 16
    pages = [-(-n // page) for n in ctx]
    kp = torch.randn(sum(pages) + 1, nkv, page, d, generator=g).bfloat16().to(DEV)
    vp = torch.randn(sum(pages) + 1, nkv, page, d, generator=g).bfloat16().to(DEV)
    vt = vp.transpose(2, 3).contiguous()
    q = (torch.randn(N, nh * d, generator=g) * spread).bfloat16().to(DEV)
    table = torch.zeros(R, max(pages), dtype=torch.int32)
    for r in range(R):
        table[r, :pages[r]] = torch.arange(pages[r]) + 1 + sum(pages[:r])
    table = table.to(DEV)
    q_start = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device=DEV)
    held = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    want = []
    for r in range(R):
        k, v = (x[table[r, :pages[r]].long()].transpose(1, 2).reshape(-1, nkv, d)[:ctx[r]].transpose(0, 1).double() for x in (kp, vp))
        rows = q[int(q_start[r]):int(q_start[r + 1])].reshape(-1, nh, d).transpose(0, 1).double()
        hidden = torch.arange(ctx[r], device=DEV)[None] > torch.arange(past, ctx[r], device=DEV)[:, None]
        o = [(rows[h] @ k[h * nkv // nh].t() * d ** -0.5).masked_fill(hidden, -math.inf).softmax(-1) @ v[h * nkv // nh] for h in range(nh)]
        want.append(torch.stack(o, 1).reshape(-1, nh * d))
    want = torch.cat(want)
    staged, other = _staged(ops, kind, q, kp, vt, table, q_start, held, nh, max(lens), None), torch.empty_like(q)
    ops._call("ms_paged_attention_mfma", q.data_ptr(), nh * d, kp.data_ptr(), vt.data_ptr(), table.data_ptr(), table.shape[1], None,
              q_start.data_ptr(), held.data_ptr(), other.data_ptr(), nh * d, R, N, max(lens), nh, nkv, d, d, page, d ** -0.5,
              0, None, 0.0, None, None, 0, 1, 1.0, ops._stream())
    far = [((x.double() - want).norm() / want.norm()).item() for x in (staged, other)]
    print(kind, d, far)
    assert far[0] <= 1.005 * far[1], far


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("R,nkv", [(40, 8), (80, 8)])
def test_the_choice_of_the_staged_prompt_kernel(ops, d, R, nkv):
    """Through the call that chooses: prompts beside single tokens, with the most tokens of a request given as a capacity (as
    a captured step has it) and tokens of nobody behind them; as many blocks as the chip holds at once (40 requests) and more
    (80).  Eagerly, and captured and replayed with other lengths of the same capacity."""
    g = torch.Generator().manual_seed(d + R)
    N, most, nh = 100 * R, 128, nkv
    assert ops._get("ms_attention_prompt_pays")(R, N, most, 160, nh, nkv, d, 16, 0) == 1
    scale = 1.0 / math.sqrt(d)
    cases = []
    for turn in range(2):
        qlen = [1 if r % 5 == turn else 60 + (r * 17 + turn * 11) % 40 for r in range(R)]
        ctx = [n + (r * 7) % 50 for r, n in enumerate(qlen)]
        c = _paged_case(g, torch.bfloat16, nh, nkv, d, 16, ctx, qlen, float("nan"))
        want = torch.cat([attention_reference(q.double(), k.double(), v.double(), scale, None).transpose(0, 1).reshape(-1, nh * d)
                          for q, k, v in zip(c["qs"], c["ks"], c["vs"])])
        cases.append((qlen, ctx, c, want))
    P, T = max(c["kp"].shape[0] for *_, c, _ in cases), 160 // 16
    q, out = torch.zeros(N, nh * d, dtype=torch.bfloat16, device=DEV), torch.zeros(N, nh * d, dtype=torch.bfloat16, device=DEV)
    kp = torch.zeros(P, nkv, 16, d, dtype=torch.bfloat16, device=DEV)
    vt = torch.zeros(P, nkv, d, 16, dtype=torch.bfloat16, device=DEV)
    table = torch.zeros(R, T, dtype=torch.int32, device=DEV)
    q_start, lens = torch.zeros(R + 1, dtype=torch.int32, device=DEV), torch.zeros(R, dtype=torch.int32, device=DEV)

    def put(qlen, ctx, c):
        n = sum(qlen)
        q[:n].copy_(c["q"])
        kp[:c["kp"].shape[0]].copy_(c["kp"])
        vt[:c["vt"].shape[0]].copy_(c["vt"])
        table[:, :c["table"].shape[1]].copy_(c["table"])
        q_start.copy_(torch.tensor([0] + list(np.cumsum(qlen)), dtype=torch.int32))
        lens.copy_(torch.tensor(ctx, dtype=torch.int32))
        out.fill_(3.0)
        return n

    def run():
        ops.paged_attention_mfma(q, kp, vt, table, q_start, lens, out, nh, scale, most, 160)

    eager = []
    for qlen, ctx, c, want in cases:
        n = put(qlen, ctx, c)
        run()
        torch.testing.assert_close(out[:n].double().cpu(), want, **tol(torch.bfloat16))
        assert (out[n:] == 3.0).all()
        eager.append(out.clone())
    graph = torch.cuda.CUDAGraph()
    with torch.inference_mode(), torch.cuda.graph(graph):     # (as the engine captures: the generator keeps the first mode)
        run()
    for turn in (0, 1, 0, 1):
        put(*cases[turn][:3])
        graph.replay()
        assert torch.equal(out, eager[turn])


@pytest.mark.parametrize("R,N,most,longest,nh,nkv,d,window,pays", [
    (13, 1900, 307, 2884, 16, 16, 64, 0, 0), (57, 2143, 69, 839, 8, 8, 64, 0, 0), (16, 1787, 248, 1171, 16, 8, 64, 0, 0),
    (8, 1520, 474, 564, 10, 2, 64, 0, 0), (47, 959, 86, 1191, 16, 16, 64, 0, 0), (1, 7571, 7571, 7571, 8, 2, 64, 0, 0),
    (1, 7777, 7777, 7777, 4, 4, 128, 0, 0), (1, 1880, 1880, 1880, 16, 8, 128, 0, 0), (4, 1902, 1004, 1010, 16, 4, 128, 0, 0),
    (3, 786, 678, 678, 40, 8, 128, 0, 0),
    (42, 1919, 88, 88, 8, 8, 64, 0, 1), (32, 1601, 124, 125, 20, 4, 64, 0, 1), (33, 864, 113, 273, 32, 8, 64, 0, 1),
    (33, 1941, 122, 778, 32, 4, 64, 0, 1), (1, 4096, 4096, 8192, 14, 2, 64, 0, 1), (1, 2048, 2048, 2048, 28, 4, 128, 0, 1),
    (16, 1600, 100, 100, 28, 4, 128, 0, 1), (4, 2048, 512, 512, 28, 4, 128, 0, 1),
    (1, 1880, 1880, 1880, 16, 8, 128, 300, 1), (1, 4319, 4319, 4319, 14, 2, 64, 300, 1), (16, 1787, 248, 1171, 16, 8, 64, 500, 0)])
def test_staged_prompts_are_taken_where_the_step_is_long_beside_its_longest_chain(ops, R, N, most, longest, nh, nkv, d, pays, window):
    """Sizes that the staged kernel was measured on both sides of: those at 0 take 1.05 to 1.3 times as long there."""
    assert ops._get("ms_attention_prompt_pays")(R, N, most, longest, nh, nkv, d, 16, window) == pays


def test_attention_mfma_support_matrix(ops):
    assert ops.attention_mfma_supported(64, 16) and ops.attention_mfma_supported(128, 32)
    assert not ops.attention_mfma_supported(48, 16) and not ops.attention_mfma_supported(64, 8)


@pytest.mark.parametrize("M", [1, 8, 33, 64])
@pytest.mark.parametrize("N,K", [(1152, 896), (330, 72), (50, 200)])
def test_gemm_skinny_with_the_norm_folded_in(ops, M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x = (torch.randn(M + 5, K, generator=g) * 3).to(DEV)
    nw = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn(N, generator=g).to(DEV)
    rows = torch.randperm(M + 5, generator=g)[:M].to(torch.int32).to(DEV)
    xd = x.double()
    h = nw.double() * (xd * torch.rsqrt((xd ** 2).mean(-1, keepdim=True) + 1e-5))
    want = h @ w.double().T + bias.double()
    t = dict(atol=3e-2, rtol=2e-2)   # the operand x * weight is rounded to bfloat16 before the product
    got = ops.gemm_skinny_norm(x[:M].contiguous(), nw, 1e-5, w, bias)
    torch.testing.assert_close(got.double(), want[:M], **t)
    got = ops.gemm_skinny_norm(x, nw, 1e-5, w, bias, out_dtype=torch.float32, rows=rows)
    assert got.dtype == torch.float32
    torch.testing.assert_close(got.double(), want[rows.long()], **t)
    if N % 2 == 0:
        act = ops.gemm_skinny_norm(x, nw, 1e-5, w, None, ops.EPI_SWIGLU, rows=rows)
        p = (h @ w.double().T)[rows.long()]
        torch.testing.assert_close(act.double(), torch.nn.functional.silu(p[:, 0::2]) * p[:, 1::2], **t)
    # against the unfused pair of kernels: the same up to the rounding of the operand
    hb = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    ops.rms_norm(x, nw, 1e-5, hb, rows=rows)
    unfused = ops.gemm_skinny(hb, w, bias, out_dtype=torch.float32)
    torch.testing.assert_close(got, unfused, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("M", [1, 8, 40])
@pytest.mark.parametrize("nh,nkv,d,K,v_transposed", [(14, 2, 64, 896, True), (6, 3, 32, 72, False), (4, 1, 128, 200, True)])
@pytest.mark.parametrize("tiles", ["whole", "8+8"])
def test_qkv_rope_store_fused_equals_the_separate_kernels(ops, M, nh, nkv, d, K, v_transposed, tiles):
    """Both shapes of block: two whole tiles half a head apart, and one tile of 8 + 8 rows whose rotary pairs lie in
    two lanes (the choice between them goes by the number of blocks; here each is forced in turn)."""
    from llm_infrence_engine_amd.kernels import build

    lib = build.load()
    lib.ms_qkv_rope_store_force(0 if tiles == "whole" else 1)
    try:
        _qkv_fused_case(ops, M, nh, nkv, d, K, v_transposed)
    finally:
        lib.ms_qkv_rope_store_force(-1)


@pytest.mark.parametrize("M", [1, 4, 5, 8])
@pytest.mark.parametrize("nh,nkv,d,K,v_transposed", [(14, 2, 64, 896, True), (6, 3, 32, 72, False), (4, 1, 128, 2568, True)])
def test_qkv_rope_store_in_units_of_four_rows(ops, M, nh, nkv, d, K, v_transposed):
    """The blocks of few tokens: two units of two rotary pairs, one or two groups of four tokens, a last group that is
    not full, columns of one piece, of one round and of two."""
    from llm_infrence_engine_amd.kernels import build

    lib = build.load()
    lib.ms_qkv_rope_store_force(2)
    try:
        _qkv_fused_case(ops, M, nh, nkv, d, K, v_transposed)
    finally:
        lib.ms_qkv_rope_store_force(-1)


def _qkv_fused_case(ops, M, nh, nkv, d, K, v_transposed):
    g = torch.Generator().manual_seed(M + d)
    page_size, pages = 16, 12
    x = (torch.randn(M, K, generator=g) * 2).to(DEV)
    nw = (1 + 0.1 * torch.randn(K, generator=g)).to(DEV)
    w = (torch.randn((nh + 2 * nkv) * d, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn((nh + 2 * nkv) * d, generator=g).to(DEV)
    pos = torch.randint(0, 3000, (M,), generator=g).to(torch.int32).to(DEV)
    slots = torch.randperm(pages * page_size, generator=g)[:M].to(torch.int32)
    if M > 2:
        slots[2] = -1
    slots = slots.to(DEV)
    inv_freq = (1.0 / (1e6 ** (torch.arange(0, d, 2, dtype=torch.float64) / d))).float().to(DEV)
    vshape = (pages, nkv, d, page_size) if v_transposed else (pages, nkv, page_size, d)
    kp1, vp1 = torch.zeros(pages, nkv, page_size, d, dtype=torch.bfloat16, device=DEV), torch.zeros(vshape, dtype=torch.bfloat16, device=DEV)
    kp2, vp2 = torch.zeros_like(kp1), torch.zeros_like(vp1)
    q = ops.qkv_rope_store(x, nw, 1e-6, w, bias, nh, nkv, d, pos, inv_freq, slots, kp1, vp1, v_transposed)
    # the separate kernels, in float between them so that only the final rounding differs
    qkv = ops.gemm_skinny_norm(x, nw, 1e-6, w, bias, out_dtype=torch.float32)
    exact = qkv.double().view(M, nh + 2 * nkv, d).cpu()
    rot = rope_reference(exact[:, :nh + nkv], pos.cpu(), d, inv_freq.double().cpu())
    torch.testing.assert_close(q.double().cpu().view(M, nh, d), rot[:, :nh], atol=3e-2, rtol=1.6e-2)
    for n in range(M):
        s = int(slots[n])
        if s < 0:
            continue
        p, o = divmod(s, page_size)
        torch.testing.assert_close(kp1[p, :, o].double().cpu(), rot[n, nh:], atol=3e-2, rtol=1.6e-2)
        v = vp1[p, :, :, o] if v_transposed else vp1[p, :, o]
        torch.testing.assert_close(v.double().cpu(), exact[n, nh + nkv:], atol=3e-2, rtol=1.6e-2)
    untouched = torch.ones(pages * page_size, dtype=torch.bool)
    untouched[slots[slots >= 0].long().cpu()] = False
    assert (kp1.permute(0, 2, 1, 3).reshape(pages * page_size, -1)[untouched.to(DEV)] == 0).all()


@pytest.mark.parametrize("M", [65, 130, 700])
@pytest.mark.parametrize("nh,nkv,d,K,v_transposed,tile", [(14, 2, 64, 896, True, 0), (3, 1, 64, 128, False, 2),
                                                            (5, 5, 64, 192, True, 3), (3, 1, 128, 256, True, 0),
                                                            (2, 2, 128, 64, False, 0)])
def test_gemm_tiled_qkv_equals_product_rotation_and_store(ops, M, nh, nkv, d, K, v_transposed, tile):
    """The many-rows q/k/v product with bias, rotation and cache store as its epilogue, against a double product
    and the plain rotation: every tile shape, tokens and heads that fill no whole tile, one token not stored, pages
    plain and transposed, positions up to thousands."""
    g = torch.Generator().manual_seed(M + d + K)
    page_size = 16
    pages = (M + page_size - 1) // page_size + 3
    a = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn((nh + 2 * nkv) * d, K, generator=g) / math.sqrt(K)).bfloat16().to(DEV)
    bias = torch.randn((nh + 2 * nkv) * d, generator=g).to(DEV) if K != 128 else None
    pos = torch.randint(0, 3000, (M,), generator=g).to(torch.int32).to(DEV)
    slots = torch.randperm(pages * page_size, generator=g)[:M].to(torch.int32)
    slots[2] = -1
    slots = slots.to(DEV)
    inv_freq = (1.0 / (1e6 ** (torch.arange(0, d, 2, dtype=torch.float64) / d))).float().to(DEV)
    vshape = (pages, nkv, d, page_size) if v_transposed else (pages, nkv, page_size, d)
    kp = torch.zeros(pages, nkv, page_size, d, dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros(vshape, dtype=torch.bfloat16, device=DEV)
    assert ops.gemm_tiled_qkv_pays(a, w, d, d, kp)
    assert not ops.gemm_tiled_qkv_pays(a, w, d, d // 2, kp)       # a rotation over part of the head is not taken
    force = ops._get("ms_gemm_tiled_force")
    force(tile)
    try:
        table = ops.rope_table(pos, inv_freq)
        q = ops.gemm_tiled_qkv(a, w, bias, nh, nkv, d, table, slots, kp, vp, v_transposed)
    finally:
        force(0)
    ang = pos.cpu().float()[:, None] * inv_freq.cpu()[None]      # the float product, as the kernel forms it
    torch.testing.assert_close(table.cpu().double(), torch.stack((ang.double().cos(), ang.double().sin()), -1),
                               atol=1e-6, rtol=0)
    exact = a.double().cpu() @ w.double().cpu().T
    if bias is not None:
        exact = exact + bias.double().cpu()
    exact = exact.view(M, nh + 2 * nkv, d)
    rot = rope_reference(exact[:, :nh + nkv], pos.cpu(), d, inv_freq.double().cpu())
    t = dict(atol=3e-2, rtol=1.6e-2)
    torch.testing.assert_close(q.double().cpu().view(M, nh, d), rot[:, :nh], **t)
    sl = slots.cpu()
    stored = sl >= 0
    pg, off = (sl[stored] // page_size).long(), (sl[stored] % page_size).long()
    torch.testing.assert_close(kp.cpu()[pg, :, off].double(), rot[stored][:, nh:], **t)
    v = vp.cpu().permute(0, 1, 3, 2) if v_transposed else vp.cpu()
    torch.testing.assert_close(v[pg, :, off].double(), exact[stored][:, nh + nkv:], **t)
    untouched = torch.ones(pages * page_size, dtype=torch.bool)
    untouched[sl[stored].long()] = False
    assert (kp.cpu().permute(0, 2, 1, 3).reshape(pages * page_size, -1)[untouched] == 0).all()
    assert (v.permute(0, 2, 1, 3).reshape(pages * page_size, -1)[untouched] == 0).all()


# the products of a decode step at the shapes of the published checkpoints: (rows of W, columns) of the packed
# q/k/v, o, interleaved gate/up, down and head matrices
MODEL_PRODUCTS = {
    "0.5b": [(1152, 896), (896, 896), (9728, 896), (896, 4864), (151936, 896)],
    "7b": [(4608, 3584), (3584, 3584), (37888, 3584), (3584, 18944), (152064, 3584)],
    "32b": [(7168, 5120), (5120, 5120), (55296, 5120), (5120, 27648), (152064, 5120)],
}


@pytest.mark.parametrize("shape", sorted(MODEL_PRODUCTS))
def test_every_row_count_of_the_model_products_has_a_kernel(ops, shape):
    """1 to 64 rows against every product of the three model shapes, through ``kernels.linear`` as the parts call it:
    right against a double-precision product, and never by falling back to the vector-ALU kernel."""
    from llm_infrence_engine_amd.kernels import linear

    g = torch.Generator(device=DEV).manual_seed(len(shape))
    before = linear.fallback_count()
    for N, K in MODEL_PRODUCTS[shape]:
        w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
        a = torch.randn(64, K, generator=g, device=DEV).bfloat16()
        want = a.double() @ w.double().T                                    # rows are independent: one reference for all M
        x = torch.randn(64, N, generator=g, device=DEV) if N < 100000 else None
        rows = (range(1, 65) if N < 100000 else (1, 2, 7, 8, 9, 16, 17, 31, 32, 33, 48, 63, 64))
        for M in rows:
            got = linear.linear(a[:M], w, out_dtype=torch.float32)
            err = (got.double() - want[:M]).abs().max().item()
            assert err < 5e-5 * max(1.0, want[:M].abs().max().item()) + 2e-5, (shape, "store", M, N, K, err)
            if x is not None:
                r = x[:M].clone()
                assert linear.linear_residual(a[:M], w, None, r) is None
                err = (r.double() - x[:M].double() - want[:M]).abs().max().item()
                assert err < 1e-4, (shape, "residual", M, N, K, err)
            if N % 2 == 0 and N > K and x is not None:                      # the gated product of gate/up
                act = linear.linear_swiglu(a[:M], w)
                ref = torch.nn.functional.silu(want[:M, 0::2]) * want[:M, 1::2]
                assert (act.double() - ref).abs().max().item() < 0.02 * max(1.0, ref.abs().max().item()), (shape, "gated", M, N, K)
        del w, a, want
    assert linear.fallback_count() == before, linear.fallbacks


def test_random_product_shapes_are_right_whatever_kernel_takes_them(ops):
    """A few hundred random shapes of up to 64 rows: ``kernels.linear`` finds a kernel for each (falling back to the
    vector-ALU kernel where the few-rows kernels have no variant, which is counted, not an error)."""
    from llm_infrence_engine_amd.kernels import linear

    rng = np.random.default_rng(17)
    g = torch.Generator(device=DEV).manual_seed(17)
    for case in range(300):
        M = int(rng.integers(1, 65))
        N = int(rng.choice([rng.integers(1, 64), rng.integers(64, 5000), rng.integers(5000, 40000)]))
        K = int(rng.choice([rng.integers(1, 40), rng.integers(40, 2000), rng.integers(2000, 12000)]))
        if rng.random() < 0.7:
            K = max(8, K // 8 * 8)
        a = torch.randn(M, K, generator=g, device=DEV).bfloat16()
        w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
        b = torch.randn(N, generator=g, device=DEV) if rng.random() < 0.5 else None
        want = a.double() @ w.double().T + (b.double() if b is not None else 0.0)
        got = linear.linear(a, w, b, out_dtype=torch.float32)
        err = (got.double() - want).abs().max().item()
        assert err < 5e-5 * max(1.0, want.abs().max().item()) + 2e-5, (case, M, N, K, err)
        x = torch.randn(M, N, generator=g, device=DEV)
        r = x.clone()
        d = linear.linear_residual(a, w, b, r)
        total = r.double() if d is None else x.double() + d.double()
        assert (total - x.double() - want).abs().max().item() < (1e-4 if d is None else 0.05), (case, M, N, K)


def test_random_gated_products_of_many_rows(ops):
    """Random shapes of more than 64 rows through ``linear_swiglu``: the tiled kernel where it takes the sizes
    (columns in steps of 64) and pays, the library's product and the activation kernel otherwise."""
    from llm_infrence_engine_amd.kernels import linear

    rng = np.random.default_rng(23)
    g = torch.Generator(device=DEV).manual_seed(23)
    tiled = 0
    for case in range(60):
        M = int(rng.choice([rng.integers(65, 300), rng.integers(300, 3000)]))
        inter = int(rng.choice([rng.integers(1, 200), rng.integers(200, 6000)]))
        K = int(rng.choice([64 * rng.integers(1, 40), 8 * rng.integers(1, 300)]))
        a = torch.randn(M, K, generator=g, device=DEV).bfloat16()
        gate = (torch.randn(inter, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
        up = (torch.randn(inter, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
        w = linear.interleave_rows(gate, up)
        tiled += ops.gemm_tiled_pays(a, w)
        got = linear.linear_swiglu(a, w)
        want = torch.nn.functional.silu(a.double() @ gate.double().T) * (a.double() @ up.double().T)
        assert got.shape == (M, inter)
        err = (got.double() - want).abs().max().item()
        # the result is rounded to bfloat16 once; where the library writes the product first, that is rounded too
        assert err < 2.5e-2 * max(1.0, want.abs().max().item()), (case, M, inter, K, err)
    assert 15 < tiled < 60


def test_read_probe_reads_everything_once(ops):
    t = torch.randint(-2 ** 31, 2 ** 31 - 1, (1 << 20,), dtype=torch.int32, device=DEV)
    for n in (1 << 20, 4 * 1000, 4):
        got = np.bitwise_xor.reduce(ops.read_probe(t[:n]).cpu().numpy().view(np.uint32))
        assert got == np.bitwise_xor.reduce(t[:n].cpu().numpy().view(np.uint32))
    with pytest.raises(ValueError, match="16 bytes"):
        ops.read_probe(t[:3])


def _chain_reference(attn, w_o, x, n2, w_gu, w_down, eps):
    """x after the output projection and the gated feed-forward, in double, rounded to bfloat16 where the kernel rounds, and how
    far float sums may lie from it: a product of the middle whose sum falls to the other side of a rounding boundary moves by
    one step of its size, 2^-8 of it at most, and takes w_down's column with it; two of the largest at once, and 1e-4 for the
    float sums of values up to about 5."""
    x = x.double() + attn.double() @ w_o.double().T
    inv = 1 / torch.sqrt((x * x).mean(1, keepdim=True) + eps)
    gu = ((x * n2.double()).bfloat16().double() @ w_gu.double().T) * inv
    act = (torch.nn.functional.silu(gu[:, 0::2]) * gu[:, 1::2]).bfloat16().double()
    return x + act @ w_down.double().T, 2 * act.abs().max().item() / 256 * w_down.abs().max().item() + 1e-4


@pytest.mark.parametrize("limit", [0, 1])
@pytest.mark.parametrize("M", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("H,I,nh,nkv,d,v_transposed", [(896, 4864, 14, 2, 64, True), (1024, 6144, 8, 8, 128, False),
                                                       (64, 32, 2, 1, 32, True), (288, 544, 3, 1, 96, True)])
def test_decode_chain(ops, M, H, I, nh, nkv, d, v_transposed, limit):
    """Two steps of three chains on one workspace, each against double: full and short rows (waves and runs without a
    k-step), tokens that fill a group and not, a token that is not stored, a last chain without a front.  With a limit of one
    look the blocks that wait give their items up and one of them works off the list: the same results to the bit."""
    page_size, pages, eps, n = 16, 8, 1e-6, nh + 2 * nkv

    def run(limit):
        g = torch.Generator().manual_seed(M + H + I)
        x = torch.randn(M, H, generator=g).to(DEV)
        inv_freq = (1.0 / (1e6 ** (torch.arange(0, d, 2, dtype=torch.float64) / d))).float().to(DEV)
        ws = torch.zeros(ops.decode_chain_workspace(M, H, nh, nkv, d, I), dtype=torch.uint8, device=DEV)
        kept = []
        ops.decode_chain_limit(limit)
        try:
            for call in range(6):
                attn = torch.randn(M, nh * d, generator=g).bfloat16().to(DEV)
                w_o = (torch.randn(H, nh * d, generator=g) / math.sqrt(nh * d)).bfloat16().to(DEV)
                n1, n2 = ((1 + 0.1 * torch.randn(H, generator=g)).to(DEV) for _ in range(2))
                w_gu = (torch.randn(2 * I, H, generator=g) / math.sqrt(H)).bfloat16().to(DEV)
                w_down = (torch.randn(H, I, generator=g) / math.sqrt(I)).bfloat16().to(DEV)
                w_qkv = (torch.randn(n * d, H, generator=g) / math.sqrt(H)).bfloat16().to(DEV)
                bias = torch.randn(n * d, generator=g).to(DEV) if call % 2 else None
                pos = torch.randint(0, 3000, (M,), generator=g).to(torch.int32).to(DEV)
                slots = torch.randperm(pages * page_size, generator=g)[:M].to(torch.int32)
                slots[M // 2] = -1 if M > 1 else slots[0]
                slots = slots.to(DEV)
                kp = torch.zeros(pages, nkv, page_size, d, dtype=torch.bfloat16, device=DEV)
                vp = torch.zeros((pages, nkv, d, page_size) if v_transposed else (pages, nkv, page_size, d), dtype=torch.bfloat16, device=DEV)
                want, apart = _chain_reference(attn, w_o, x, n2, w_gu, w_down, eps)
                front = (n1, eps, w_qkv, bias, pos, inv_freq, slots, kp, vp, v_transposed) if call % 3 < 2 else None
                q = ops.decode_chain(attn, w_o, x, n2, eps, w_gu, w_down, nh, nkv, d, ws, call % 3, 3, front)
                assert (x.double() - want).abs().max().item() <= apart
                assert (x.double() - want).square().mean().sqrt().item() <= apart / 8     # (most do not move)
                kept.append(x.clone())
                if front is None:
                    assert q is None
                    continue
                y = ((want * n1.double()) / torch.sqrt((want * want).mean(1, keepdim=True) + eps)) @ w_qkv.double().T
                y = (y + (bias.double() if bias is not None else 0)).view(M, n, d).cpu()
                rot = rope_reference(y[:, :nh + nkv], pos.cpu(), d, inv_freq.double().cpu())
                torch.testing.assert_close(q.double().cpu().view(M, nh, d), rot[:, :nh], atol=4e-2, rtol=1.6e-2)
                for t in range(M):
                    s = int(slots[t])
                    if s < 0:
                        continue
                    p, o = divmod(s, page_size)
                    torch.testing.assert_close(kp[p, :, o].double().cpu(), rot[t, nh:], atol=4e-2, rtol=1.6e-2)
                    v = vp[p, :, :, o] if v_transposed else vp[p, :, o]
                    torch.testing.assert_close(v.double().cpu(), y[t, nh + nkv:], atol=4e-2, rtol=1.6e-2)
                untouched = torch.ones(pages * page_size, dtype=torch.bool)
                untouched[slots[slots >= 0].long().cpu()] = False
                assert (kp.permute(0, 2, 1, 3).reshape(pages * page_size, -1)[untouched.to(DEV)] == 0).all()
                kept += [q, kp, vp]
            assert not ws[:4 * 32768].any()      # nothing is left on the list
        finally:
            ops.decode_chain_limit(0)
        return kept

    got = run(limit)
    if limit:
        assert all(torch.equal(a, b) for a, b in zip(got, run(0)))


@pytest.mark.parametrize("limit", [0, 1])
@pytest.mark.parametrize("contexts", [(1,), (1024,), (17, 600), (32, 33, 2), (513, 64, 1, 1000), (1, 97, 128, 577, 31)])
@pytest.mark.parametrize("H,I,nh,nkv,page_size", [(896, 4864, 14, 2, 16), (96, 64, 16, 1, 64)])
def test_decode_layers(ops, H, I, nh, nkv, page_size, contexts, limit):
    """Three steps of three layers in two launches each against double on what lies in the pages: contexts of one key, of whole
    and of part blocks of 32, of all 1,024; a token that is not stored; pages in no order, with NaN behind the last key.  With
    a limit of one look every waiting block gives its item up, to the same bits."""
    M, d, L, eps, scale, n = len(contexts), 64, 3, 1e-6, 0.125, nh + 2 * nkv
    width = -(-1030 // page_size)

    def run(limit):
        g = torch.Generator().manual_seed(M + H)
        rand = lambda *shape, std=1.0: (torch.randn(*shape, generator=g) * std)     # noqa: E731
        pages = M * width + 1
        table = (torch.randperm(M * width, generator=g) + 1).view(M, width).to(torch.int32)
        rows = torch.randperm(M, generator=g).to(torch.int32)
        inv_freq = (1.0 / (1e6 ** (torch.arange(0, d, 2, dtype=torch.float64) / d))).float().to(DEV)
        layers = []
        for _ in range(L):
            l = dict(w_o=rand(H, nh * d, std=(nh * d) ** -0.5), w_gate_up=rand(2 * I, H, std=H ** -0.5), w_down=rand(H, I, std=I ** -0.5),
                     w_qkv=rand(n * d, H, std=H ** -0.5))
            l = {k: v.bfloat16().to(DEV) for k, v in l.items()}
            l.update(norm1=(1 + rand(H, std=0.1)).to(DEV), norm2=(1 + rand(H, std=0.1)).to(DEV), bias=rand(n * d).to(DEV),
                     k=torch.full((pages, nkv, page_size, d), float("nan"), dtype=torch.bfloat16, device=DEV),
                     v=torch.full((pages, nkv, d, page_size), float("nan"), dtype=torch.bfloat16, device=DEV))
            for m, c in enumerate(contexts):
                for t in range(0, c - 1, page_size):
                    p, w = int(table[rows[m], t // page_size]), min(page_size, c - 1 - t)
                    l["k"][p, :, :w], l["v"][p, :, :, :w] = rand(nkv, w, d).bfloat16().to(DEV), rand(nkv, d, w).bfloat16().to(DEV)
            layers.append(l)
        recs = []
        for i, l in enumerate(layers):
            rec = dict(w_o=l["w_o"], w_gate_up=l["w_gate_up"], w_down=l["w_down"], norm2=l["norm2"], eps2=eps, k_pages=l["k"], v_pages=l["v"])
            if i + 1 < L:
                t = layers[i + 1]
                rec.update(w_front=t["w_qkv"], norm1=t["norm1"], eps1=eps, b_front=t["bias"], inv_freq=inv_freq, front_k=t["k"], front_v=t["v"])
            recs.append(rec)
        records = ops.decode_layer_table(recs, DEV)
        ws = torch.zeros(ops.decode_chain_workspace(M, H, nh, nkv, d, I, L), dtype=torch.uint8, device=DEV)
        kept = []
        ops.decode_chain_limit(limit)
        try:
            for step in range(3):
                lens = [min(c + step, 1024) for c in contexts]
                pos = torch.tensor([c - 1 for c in lens], dtype=torch.int32)
                slot = torch.tensor([int(table[rows[m], (c - 1) // page_size]) * page_size + (c - 1) % page_size for m, c in enumerate(lens)])
                if M > 2 and step == 2:
                    slot[2] = -1
                x = rand(M, H).to(DEV)
                x0 = x.double()
                before = [(l["k"].clone(), l["v"].clone()) for l in layers]
                pos_d, slot_d = pos.to(DEV), slot.to(torch.int32).to(DEV)
                a = layers[0]
                ops.decode_first(x, a["norm1"], eps, a["w_qkv"], a["bias"], pos_d, inv_freq, slot_d, a["k"], a["v"], nh, nkv, d, I, L, ws)
                ops.decode_layers(records, x, pos_d, slot_d, (pos + 1).to(DEV), table.to(DEV), rows.to(DEV), scale, nh, nkv, d, I,
                                  page_size, L, ws)
                y = x0
                for l, (bk, bv) in zip(layers, before):
                    z = ((y * l["norm1"].double()) / torch.sqrt((y * y).mean(1, keepdim=True) + eps)) @ l["w_qkv"].double().T + l["bias"].double()
                    z = z.view(M, n, d).cpu()
                    rot = rope_reference(z[:, :nh + nkv], pos, d, inv_freq.double().cpu())
                    heads = torch.empty(M, nh * d, dtype=torch.float64)
                    for m, c in enumerate(lens):
                        at = [(int(table[rows[m], t // page_size]), t % page_size) for t in range(c - 1)]
                        p, o = [q[0] for q in at], [q[1] for q in at]
                        new_k, new_v = rot[m, nh:], z[m, nh + nkv:]
                        if int(slot[m]) >= 0:      # what was stored is what it should be, and counts as it was rounded
                            sp, so = divmod(int(slot[m]), page_size)
                            torch.testing.assert_close(l["k"][sp, :, so].double().cpu(), new_k, atol=6e-2, rtol=2e-2)
                            torch.testing.assert_close(l["v"][sp, :, :, so].double().cpu(), new_v, atol=6e-2, rtol=2e-2)
                            new_k, new_v = l["k"][sp, :, so].double().cpu(), l["v"][sp, :, :, so].double().cpu()
                        keys = torch.cat([bk[p, :, o].double().cpu(), new_k[None]]).repeat_interleave(nh // nkv, 1)     # [c, nh, d]
                        vals = torch.cat([bv[p, :, :, o].double().cpu(), new_v[None]]).repeat_interleave(nh // nkv, 1)
                        w = (scale * torch.einsum("hd,chd->hc", rot[m, :nh], keys)).softmax(1)
                        heads[m] = torch.einsum("hc,chd->hd", w, vals).reshape(-1)
                    y, _ = _chain_reference(heads.to(DEV), l["w_o"], y, l["norm2"], l["w_gate_up"], l["w_down"], eps)
                # queries, heads, probabilities and the middle are rounded to bfloat16 (2^-9 each) three layers deep
                assert (x.double() - y).norm() < 1.2e-2 * (y - x0).norm()
                for l, (bk, bv) in zip(layers, before):      # nothing else was written
                    for now, was in ((l["k"].permute(0, 2, 1, 3), bk.permute(0, 2, 1, 3)), (l["v"].permute(0, 3, 1, 2), bv.permute(0, 3, 1, 2))):
                        rest = torch.ones(pages * page_size, dtype=torch.bool)
                        rest[slot[slot >= 0]] = False
                        rest = rest.to(DEV)
                        assert torch.equal(now.reshape(pages * page_size, -1)[rest].view(torch.int16), was.reshape(pages * page_size, -1)[rest].view(torch.int16))
                kept += [x.clone()] + [l["k"].clone() for l in layers]
            assert not ws[:4 * 32768].any()
        finally:
            ops.decode_chain_limit(0)
        return kept

    got = run(limit)
    if limit:
        assert all(torch.equal(a.view(torch.int16 if a.dtype == torch.bfloat16 else torch.int32), b.view(torch.int16 if b.dtype == torch.bfloat16 else torch.int32))
                   for a, b in zip(got, run(0)))


def test_a_launch_whose_inputs_never_come_ends(ops):
    """All layers without the launch that goes before them, with the library's own bounds made short: the blocks give up, the one
    that stays stops trying, says so behind the list and to the host, and a launch after it ends, too, with nobody staying.
    Zeroed, the workspace is as good as new."""
    M, H, I, nh, nkv, d, L, page_size = 2, 96, 64, 4, 2, 64, 2, 16
    g = torch.Generator().manual_seed(11)
    n, eps = nh + 2 * nkv, 1e-6
    w = lambda *shape: (torch.randn(*shape, generator=g) / 8).bfloat16().to(DEV)     # noqa: E731
    ones, inv_freq = torch.ones(H, device=DEV), torch.ones(d // 2, device=DEV)
    kv = [torch.zeros(4, nkv, page_size, d, dtype=torch.bfloat16, device=DEV) for _ in range(2 * L)]
    w_qkv = w(n * d, H)
    one = dict(w_o=w(H, nh * d), w_gate_up=w(2 * I, H), w_down=w(H, I), norm2=ones, eps2=eps)
    recs = [dict(one, k_pages=kv[2 * i], v_pages=kv[2 * i + 1].transpose(2, 3).contiguous()) for i in range(L)]
    recs[0].update(w_front=w_qkv, norm1=ones, eps1=eps, b_front=None, inv_freq=inv_freq, front_k=recs[1]["k_pages"], front_v=recs[1]["v_pages"])
    table = ops.decode_layer_table(recs, DEV)
    ints = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)     # noqa: E731
    pos, slots, lens, blocks = ints(3, 0), ints(16 + 3, 32), ints(4, 1), ints(1, 2).view(2, 1)
    x0 = torch.randn(M, H, generator=g).to(DEV)
    new = lambda: torch.zeros(ops.decode_chain_workspace(M, H, nh, nkv, d, I, L), dtype=torch.uint8, device=DEV)     # noqa: E731
    told = torch.zeros(1, dtype=torch.int32).pin_memory()

    def step(ws):
        x = x0.clone()
        ops.decode_first(x, ones, eps, w_qkv, None, pos, inv_freq, slots, recs[0]["k_pages"], recs[0]["v_pages"], nh, nkv, d, I, L, ws)
        return ops.decode_layers(table, x, pos, slots, lens, blocks, None, 0.125, nh, nkv, d, I, page_size, L, ws, told)

    want, ws = step(new()), new()
    x = x0.clone()
    ops.decode_chain_limit(1, 2)
    try:
        for _ in range(2):
            ops._call("ms_decode_layers", table.data_ptr(), x.data_ptr(), H, pos.data_ptr(), slots.data_ptr(), lens.data_ptr(), blocks.data_ptr(),
                      None, 1, 0.125, M, H, I, nh, nkv, d, page_size, L, ws.data_ptr(), told.data_ptr(), ops._stream())
            torch.cuda.synchronize()
            words = ws[:4 * 32768].view(torch.int32)
            assert told[0] == 1 and words[32767] == 1 and 1 < words[0] <= 32767
            listed = int(words[0])
            assert (words[1:listed] > 0).all() and not words[listed:32767].any()
    finally:
        ops.decode_chain_limit(0)
    told.zero_()
    ws.zero_()
    assert torch.equal(step(ws), want) and told[0] == 0 and not ws[:4 * 32768].any()
    with pytest.raises(ValueError, match="pinned"):
        ops.decode_layers(table, x, pos, slots, lens, blocks, None, 0.125, nh, nkv, d, I, page_size, L, ws, torch.zeros(1, dtype=torch.int32))


def test_a_table_of_layers_holds_what_the_kernel_can_read(ops):
    """The kernel reads addresses out of the table and cannot look at them any more: type, shape, layout, device and alignment of
    every tensor are looked at when the table is made, and its sizes when it is used."""
    H, I, nh, nkv, d, page_size = 96, 64, 4, 2, 64, 16
    bf = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16, device=DEV)     # noqa: E731
    f = lambda *shape: torch.zeros(*shape, device=DEV)     # noqa: E731
    pages = lambda: (bf(3, nkv, page_size, d), bf(3, nkv, d, page_size))     # noqa: E731
    kv = [pages(), pages()]

    def rows():
        one = dict(w_o=bf(H, nh * d), w_gate_up=bf(2 * I, H), w_down=bf(H, I), norm2=f(H), eps2=1e-6)
        two = dict(one, k_pages=kv[1][0], v_pages=kv[1][1])
        return [dict(one, k_pages=kv[0][0], v_pages=kv[0][1], w_front=bf((nh + 2 * nkv) * d, H), norm1=f(H), eps1=1e-6, b_front=f((nh + 2 * nkv) * d),
                     inv_freq=f(d // 2), front_k=kv[1][0], front_v=kv[1][1]), two]

    table = ops.decode_layer_table(rows(), DEV)
    assert table.numel() == 2 * ops._get("ms_decode_layer_bytes")()
    r = rows()
    r[0]["b_front"] = None
    ops.decode_layer_table(r, DEV)

    def refused(layer, name, bad, error=(ValueError, TypeError, RuntimeError, KeyError)):
        r = rows()
        if bad is None:
            del r[layer][name]
        else:
            r[layer][name] = bad(r[layer][name])
        with pytest.raises(error):
            ops.decode_layer_table(r, DEV)

    aside = lambda t: torch.zeros(t.numel() + 2, dtype=t.dtype, device=DEV)[2:].view(t.shape)      # 4 or 8 bytes off     # noqa: E731
    strided = lambda t: torch.stack([t, t], -1)[..., 0]     # noqa: E731
    for layer, names in ((0, ("w_o", "w_gate_up", "w_down", "norm2", "w_front", "norm1", "k_pages", "v_pages", "front_k", "front_v")),
                         (1, ("w_o", "w_gate_up", "w_down", "norm2", "k_pages", "v_pages"))):
        for name in names:
            refused(layer, name, lambda t: t.cpu(), RuntimeError)
            refused(layer, name, lambda t: t.half(), TypeError)
            refused(layer, name, strided, ValueError)
            refused(layer, name, lambda t: torch.cat([t, t]) if "pages" not in name and "front_" not in name else t[:, :1].contiguous(), ValueError)
            refused(layer, name, aside, ValueError)
            refused(layer, name, None)
    for name in ("inv_freq", "b_front"):
        refused(0, name, lambda t: t.bfloat16(), TypeError)
        refused(0, name, lambda t: t[1:].clone(), ValueError)
    refused(0, "inv_freq", None)
    refused(0, "v_pages", lambda t: t.transpose(2, 3).contiguous(), ValueError)
    refused(1, "k_pages", lambda t: bf(3, nkv, 2 * page_size, d), ValueError)

    M = 2
    ints = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)     # noqa: E731
    x, blocks = f(M, H), ints(1, 2).view(2, 1)

    def layers(table, nh=nh, nkv=nkv, page_size=page_size, x=x, I=I):
        ws = torch.zeros(ops.decode_chain_workspace(M, x.shape[1], nh, nkv, d, I, 2), dtype=torch.uint8, device=DEV)
        ws.chain_turn = ((M, x.shape[1], nh, nkv, d, I, "layers", 2), 1)
        ops.decode_layers(table, x, ints(3, 0), ints(19, 32), ints(4, 1), blocks, None, 0.125, nh, nkv, d, I, page_size, 2, ws, max_context_len=4)

    for other in (dict(nh=2), dict(nkv=1), dict(page_size=32), dict(x=f(M, 128)), dict(I=32)):
        with pytest.raises(ValueError, match="table"):
            layers(table, **other)
    with pytest.raises(ValueError, match="table"):
        layers(table.clone())


def test_decode_chain_refuses_what_it_cannot_take(ops):
    for sizes in [(9, 896, 14, 2, 64, 4864), (0, 896, 14, 2, 64, 4864), (1, 1056, 14, 2, 64, 4864), (1, 896, 17, 1, 64, 4864),
                  (1, 896, 14, 2, 64, 6176), (1, 896, 14, 2, 64, 4880), (1, 880, 14, 2, 64, 4864), (1, 896, 14, 2, 60, 4864)]:
        assert ops.decode_chain_workspace(*sizes) == 0
    assert ops.decode_chain_workspace(8, 896, 14, 2, 64, 4864) > 0
    for sizes in [(1, 896, 7, 2, 64, 4864, 24), (1, 896, 7, 1, 128, 4864, 24), (1, 1024, 16, 0, 64, 4864, 24), (1, 1024, 32, 1, 32, 64, 2),
                  (1, 896, 14, 2, 64, 4864, 60)]:
        assert ops.decode_chain_workspace(*sizes) == 0
    assert ops.decode_chain_workspace(8, 896, 14, 2, 64, 4864, 24) > 0


@pytest.mark.parametrize("M", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(7, 4), (10, 36), (896, 4864), (1024, 64), (1025, 1040), (2050, 1100), (5001, 1028), (4100, 9000)])
def test_float_products_of_up_to_8_rows_are_those_of_more(ops, M, N, K):
    """Loads that take four k-steps of 4, 8 and 16 rows of W and of up to 4 and 8 tokens: the same bits as the same rows among 16,
    which go one step at a time; slices of one to 36 steps, a last one that is short, a last step that is, rows and columns of
    zeros, infinities and NaN beside others, a bias and a sum in place."""
    g = torch.Generator().manual_seed(N + K)
    a, w = torch.randn(16, K, generator=g), torch.randn(N, K, generator=g)
    a[min(2, M - 1)], w[N // 2] = 0.0, 0.0
    if M > 3:
        a[3, K // 2] = float("inf")
        w[N - 1, K - 1] = float("nan")
    a, w, bias = a.to(DEV), w.to(DEV), torch.randn(N, generator=g).to(DEV)
    base = torch.randn(16, N, generator=g).to(DEV)
    for accumulate in (False, True):
        want = ops.gemm_generic(a, w, base.clone(), bias, accumulate)
        got = ops.gemm_generic(a[:M], w, base[:M].clone(), bias, accumulate)
        assert torch.equal(got.isnan(), want[:M].isnan()) and torch.equal(got.nan_to_num(7.0), want[:M].nan_to_num(7.0))
    exact = a.double() @ w.double().T + bias.double()
    ok = exact[:M].isfinite()
    got = ops.gemm_generic(a[:M], w, torch.empty(M, N, device=DEV), bias)
    assert ((got.double() - exact[:M])[ok].abs() <= 4e-6 * math.sqrt(K) * 4).all()


@pytest.mark.parametrize("keys,cap", [(1, 2048), (257, 2048), (9000, 16384), (9000, 40000), (24001, 70000)])
@pytest.mark.parametrize("nh,nkv,d", [(14, 2, 64), (3, 1, 32), (8, 4, 128)])
def test_splits_are_put_together(ops, nh, nkv, d, keys, cap):
    """One split and many of a row's keys (one, two, 36 of up to 24 or 32, 94 of 128: each wave's share in part, whole, and
    beyond what is asked for ahead), a row that pads the batch, and what lies in the parts nobody wrote."""
    g = torch.Generator().manual_seed(keys + d)
    n = -(-keys // 16)
    kp = torch.randn(n + 1, nkv, 16, d, generator=g).bfloat16().to(DEV)
    vp = torch.randn(n + 1, nkv, d, 16, generator=g).bfloat16().to(DEV)
    table = torch.zeros(2, -(-cap // 16), dtype=torch.int32)
    table[0, :n] = torch.randperm(n, generator=g) + 1
    q = torch.randn(2, nh * d, generator=g).bfloat16().to(DEV)
    out = torch.full_like(q, 7.0)
    junk = torch.full((64 << 20,), float("nan"), device=DEV)
    del junk       # (the parts are likely to lie where this lay)
    ops.paged_attention_mfma(q, kp, vp, table.to(DEV), torch.tensor([0, 1, 1], dtype=torch.int32, device=DEV),
                             torch.tensor([keys, 0], dtype=torch.int32, device=DEV), out, nh, d ** -0.5, 1, cap)
    k = kp[table[0, :n].long()].permute(1, 0, 2, 3).reshape(nkv, n * 16, d)[:, :keys].double()
    v = vp[table[0, :n].long()].permute(1, 0, 3, 2).reshape(nkv, n * 16, d)[:, :keys].double()
    k, v = (t.repeat_interleave(nh // nkv, 0) for t in (k, v))
    w = ((k @ q[0].view(nh, d, 1).double()).squeeze(2) * d ** -0.5).softmax(1)
    want = (w.unsqueeze(1) @ v).reshape(-1)
    # probabilities and result in bfloat16: 2^-9 of the weighted values' size each
    size = (w.unsqueeze(1) @ v.abs()).reshape(-1)
    assert ((out[0].double() - want).abs() <= 2 ** -7 * size + 1e-6).all()
    assert (out[1] == 7.0).all()


@pytest.mark.parametrize("N,K", [(4, 512), (90, 896), (896, 4864), (1031, 1028), (2053, 1100), (1500, 2052), (2048, 16), (1021, 13188)])
def test_32_bit_products_of_up_to_8_rows_have_the_bits_of_the_kernel_for_64(ops, N, K):
    """Blocks of 4 and of 8 rows of W whose instructions hold two or four slices side by side, for one to eight tokens: columns that
    end within a slice, a step or a piece, slices that are not a whole number of instructions, rows past the last; with bias and
    added onto what is there.  The kernel of up to 64 rows sums in the same order, and its own test holds it against 64 bits."""
    from llm_infrence_engine_amd.kernels import build

    lib = build.load()
    g = torch.Generator(device=DEV).manual_seed(N + K)
    a, w = (torch.randn(n, K, generator=g, device=DEV) for n in (8, N))
    bias, there = torch.randn(N, generator=g, device=DEV), torch.randn(8, N, generator=g, device=DEV)

    def run(kind, M, plain):
        lib.ms_gemm_f32_force(kind)
        try:
            out = there[:M].clone()
            return ops.gemm_generic(a[:M], w, out, bias=None if plain else bias, accumulate=not plain)
        finally:
            lib.ms_gemm_f32_force(0)

    for plain in (True, False):
        want = run(1, 8, plain)
        exact = a.double() @ w.double().T + (0 if plain else bias.double() + there.double())
        torch.testing.assert_close(want.double(), exact, atol=K ** 0.5 * 2e-6, rtol=2e-5)      # (sums of K products of about one)
        for kind in (4, 5, 0):
            for M in (1, 2, 3, 4, 5, 8):
                assert torch.equal(run(kind, M, plain), want[:M]), (kind, M, plain)


@pytest.mark.parametrize("tile", [6, 7, 8, 9, 10, 11])
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 384, 448, 896])
@pytest.mark.parametrize("M,N", [(65, 662), (300, 1028), (513, 130)])
def test_gemm_tiled_with_deep_pipelines(ops, M, N, K, tile):
    """The tiles that ask for three to five steps ahead: fewer steps than slots, as many, one more and many; rows and features that
    fill no whole tile.  The same bits as with a tile of two steps ahead (a sum runs over the columns in one order with every tile), and
    right against 64 bits."""
    force = ops._get("ms_gemm_tiled_force")
    force.restype = None
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
    a[M - 1] *= 3.0
    want = a.double() @ w.double().T
    got = []
    for t in (tile, 2):
        force(t)
        try:
            got.append([ops.gemm_tiled(a, w, e) for e in (ops.EPI_STORE, ops.EPI_SWIGLU, ops.EPI_GEGLU, ops.EPI_RELU2)]
                       + [ops.gemm_tiled(a, w, ops.EPI_CLAMPED, 7.0, 1.702)])
        finally:
            force(0)
    torch.testing.assert_close(got[0][0].double(), want, **tol(torch.bfloat16))
    torch.testing.assert_close(got[0][1].double(), torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2], **tol(torch.bfloat16))
    assert all(torch.equal(x, y) for x, y in zip(*got))


@pytest.mark.parametrize("tile", [6, 12])
@pytest.mark.parametrize("M,N,K,parts", [(65, 70, 64, 1), (130, 896, 320, 2), (257, 200, 1216, 3), (513, 132, 4864, 8)])
def test_gemm_tiled_sums_with_deep_pipelines(ops, M, N, K, parts, tile):
    """Runs of one to ten steps on the tiles that ask for four ahead: the bits of the tile that asks for two."""
    force = ops._get("ms_gemm_tiled_force")
    force.restype = None
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
    got = []
    for t in (tile, 3):
        force(t)
        try:
            got.append(ops.gemm_tiled_sums(a, w, parts))
        finally:
            force(0)
    torch.testing.assert_close(got[0].double().sum(0), a.double() @ w.double().T, atol=3e-5, rtol=3e-5)
    assert torch.equal(*got)


@pytest.mark.parametrize("tile", [0, 3, 6, 11])
@pytest.mark.parametrize("nh,nkv,d,K,M,transposed", [(14, 2, 64, 896, 70, True), (3, 1, 64, 64, 129, False), (2, 2, 128, 320, 65, True),
                                                     (5, 1, 128, 128, 200, False), (8, 4, 64, 192, 1200, True)])
def test_gemm_tiled_qkv_with_deep_pipelines(ops, nh, nkv, d, K, M, transposed, tile):
    """The q/k/v product on the tiles of one head (64 and 128 tokens) and as chosen: the bits of the larger tile, whose own test holds it
    against 64 bits; tokens that are not stored, no bias, heads that fill no whole tile."""
    force = ops._get("ms_gemm_tiled_force")
    force.restype = None
    g = torch.Generator(device=DEV).manual_seed(M + K)
    N = (nh + 2 * nkv) * d
    a = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
    pos = torch.arange(M, dtype=torch.int32, device=DEV)
    table = ops.rope_table(pos, 1e4 ** (-torch.arange(0, d, 2, device=DEV).float() / d))
    slots = (pos + 16).int()
    slots[::7] = -1
    got = []
    for bias in (None, torch.randn(N, generator=g, device=DEV)):
        for t in (tile, 2):
            kp = torch.zeros(M // 16 + 3, nkv, 16, d, dtype=torch.bfloat16, device=DEV)
            vp = torch.zeros((M // 16 + 3, nkv, d, 16) if transposed else kp.shape, dtype=torch.bfloat16, device=DEV)
            force(t)
            try:
                got.append((ops.gemm_tiled_qkv(a, w, bias, nh, nkv, d, table, slots, kp, vp, transposed), kp, vp))
            finally:
                force(0)
        assert all(torch.equal(x, y) for x, y in zip(got[-2], got[-1]))
    assert not torch.equal(got[0][0], got[2][0])


@pytest.mark.parametrize("H,G,D,E,ra,rg,pad", [(14, 2, 64, 64, 64, 64, 0), (4, 4, 16, 200, 8, 16, 2), (3, 1, 20, 100, 128, 8, 5),
                                               (6, 2, 100, 32, 72, 128, 0), (2, 1, 128, 7, 40, 24, 1), (2, 2, 33, 64, 8, 8, 3)])
def test_gated_delta_step(ops, H, G, D, E, ra, rg, pad):
    """A decode step of the delta rule in one kernel against 64 bits, with key sizes of one lane to a column and of eight, fewer columns
    than threads, ranks of one piece and of the most, rows of any stride, requests without tokens, and states of others left alone."""
    g = torch.Generator().manual_seed(D + E)
    r = lambda *s: torch.randn(*s, generator=g)     # noqa: E731
    starts = [0, 1, 1, 2, 3, 4, 4]                            # requests 1 and 5 have no token
    N, R = starts[-1], len(starts) - 1
    cw = 2 * G * D + H * E
    qkv = r(N, cw + pad).bfloat16()
    proj = r(N, 3 + ra + rg + H + pad).bfloat16()
    a_at, g_at, b_at = 3, 3 + ra, 3 + ra + rg
    w_a2, w_g2 = (r(H * D, ra) / ra ** 0.5).bfloat16(), (r(H * E, rg) / rg ** 0.5).bfloat16()
    A_log, dt, nw, S = r(H) / 4, r(H * D) / 2 - 2, 1 + r(E) / 8, r(R + 1, H, D, E)
    slots = torch.tensor([3, 0, 5, 1, 6, 2], dtype=torch.int32)
    want_S, want = S.double().clone(), torch.zeros(N, H, E, dtype=torch.float64)
    for q in range(R):
        if starts[q + 1] == starts[q]:
            continue
        n, s = starts[q], int(slots[q])
        x, p = qkv[n].double(), proj[n].double()
        a = (w_a2.double() @ p[a_at:a_at + ra] + dt.double()).view(H, D)
        gate = torch.sigmoid(w_g2.double() @ p[g_at:g_at + rg]).view(H, E)
        for h in range(H):
            k_at = G * D + h // (H // G) * D
            qq, kk, vv = x[h // (H // G) * D:][:D], x[k_at:k_at + D], x[2 * G * D + h * E:][:E]
            qq, kk = qq / torch.sqrt(qq @ qq + 1e-6) / D ** 0.5, kk / torch.sqrt(kk @ kk + 1e-6)
            T = torch.exp(-torch.exp(A_log[h].double()) * torch.nn.functional.softplus(a[h]))[:, None] * want_S[s, h]
            T = T + kk[:, None] * (torch.sigmoid(p[b_at + h]) * (vv - kk @ T))[None]
            want_S[s, h] = T
            o = qq @ T
            want[n, h] = o / torch.sqrt((o * o).mean() + 1e-6) * nw.double() * gate[h]
    ctx = SimpleNamespace(num_requests=R, q_start=torch.tensor(starts, dtype=torch.int32, device=DEV), state_slots=slots.to(DEV), max_q_len=1)
    assert ops.gated_delta_step_ok(proj.to(DEV), w_a2.to(DEV), w_g2.to(DEV), D, E)
    Sd, out = S.to(DEV), torch.empty(N, H * E, dtype=torch.bfloat16, device=DEV)
    ops.gated_delta_step(qkv.to(DEV)[:, :cw], proj.to(DEV), a_at, g_at, b_at, w_a2.to(DEV), w_g2.to(DEV), A_log.to(DEV), dt.to(DEV), nw.to(DEV),
                         1e-6, Sd, ctx, out, H, G, D, E)
    torch.testing.assert_close(Sd.cpu().double(), want_S, atol=2e-5, rtol=2e-5)
    # one rounding to bfloat16 (2^-9), and the float errors of o over its norm
    torch.testing.assert_close(out.cpu().double(), want.view(N, -1), atol=1e-3, rtol=5e-3)
    assert torch.equal(Sd[[0, 2, 4]].cpu(), S[[0, 2, 4]])
    assert not ops._get("ms_gated_delta_step_takes")(130, 8, 8, 8) and not ops._get("ms_gated_delta_step_takes")(64, 65, 8, 8)
    assert not ops._get("ms_gated_delta_step_takes")(64, 64, 12, 8) and not ops._get("ms_gated_delta_step_takes")(64, 64, 8, 136)


@pytest.mark.parametrize("H,taps,delta", [(896, 4, None), (60, 1, "same"), (1028, 8, "same"), (2048, 2, None), (100, 3, "float")])
def test_norm_pair_with_the_convolution_is_the_two_one_after_the_other(ops, H, taps, delta):
    """The same bits in both results, in x and in the states; a token that pads a batch moves no state."""
    g = torch.Generator(device=DEV).manual_seed(H)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)     # noqa: E731
    N, live, dtype = 5, 4, torch.bfloat16
    x, w1, w2, tw = r(N, H), 1 + r(H) / 8, 1 + r(H) / 8, r(H, taps) / 2
    d = None if delta is None else r(N, H).to(torch.float32 if delta == "float" else dtype)
    state = r(7, max(1, taps - 1), H).to(dtype)
    ctx = SimpleNamespace(num_requests=N, token_req=torch.arange(N, dtype=torch.int32, device=DEV), max_q_len=1,
                          q_start=torch.tensor([0, 1, 2, 3, 4, 4], dtype=torch.int32, device=DEV),
                          state_slots=torch.tensor([5, 0, 2, 6, 1], dtype=torch.int32, device=DEV),
                          n_live_tokens=torch.tensor([live], dtype=torch.int32, device=DEV))
    new = lambda: torch.empty(N, H, dtype=dtype, device=DEV)     # noqa: E731
    xa, sa, h, a2 = x.clone(), state.clone(), new(), new()
    ops.rms_norm_pair(xa, w1, w2, 1e-6, h, a2, delta=d)
    a1 = ops.short_conv(h, tw, sa, ctx, new(), ops.CONV_ADD_INPUT)
    xb, sb = x.clone(), state.clone()
    b1, b2 = ops.rms_norm_pair_conv(xb, w1, w2, 1e-6, tw, sb, ctx, new(), new(), delta=d)
    assert torch.equal(sa, sb) and torch.equal(xa[:live], xb[:live])
    assert torch.equal(a1[:live], b1[:live]) and torch.equal(a2[:live], b2[:live])


@pytest.mark.parametrize("M,N,K", [(1, 7296, 896), (4, 7296, 896), (3, 900, 296), (8, 512, 512), (2, 1030, 1000)])
def test_gemm_xielu(ops, M, N, K):
    """The xIELU as the epilogue of the narrow matrices' product, against 64 bits; sizes that another kernel is for are left to it."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * 2 / math.sqrt(K)).bfloat16()
    pq = torch.tensor([0.3, -0.4], device=DEV)
    got = ops.gemm_xielu(a, w, pq)
    z = a.double() @ w.double().T
    p, q = torch.nn.functional.softplus(pq.double())
    want = torch.where(z > 0, p * z * z + z / 2, (0.5 + q) * (torch.expm1(z.clamp(max=0)) - z) + z / 2)
    torch.testing.assert_close(got.double(), want, atol=2e-3, rtol=5e-3)     # one rounding to bfloat16; the product's float error
    assert ops.gemm_xielu(torch.zeros(9, K, device=DEV, dtype=torch.bfloat16), w, pq) is None


@pytest.mark.parametrize("change", ["in place", "another tensor"])
def test_an_xielu_whose_numbers_change_is_the_new_one_for_any_number_of_tokens(ops, change):
    """4 tokens, whose product has the activation as its epilogue, and 16, whose activation is a kernel of its own, before and after."""
    from llm_infrence_engine_amd.parts.base import Runtime
    from llm_infrence_engine_amd.parts.feed_forward import DenseAct

    g = torch.Generator(device=DEV).manual_seed(3)
    tensors = {"up": torch.randn(512, 512, generator=g, device=DEV).bfloat16() / 22, "down": torch.eye(512, device=DEV).bfloat16(),
               "act": torch.tensor([0.3, -0.4], device=DEV)}
    part = DenseAct("", 512, 512)
    part.load(lambda spec: tensors[spec.name], Runtime(torch.device(DEV), torch.bfloat16))
    h = torch.randn(16, 512, generator=g, device=DEV).bfloat16()
    for p, q in ((0.3, -0.4), (1.5, 0.8)):
        if p == 1.5 and change == "in place":
            part.act.copy_(torch.tensor([p, q]))
        elif p == 1.5:
            part.act = torch.tensor([p, q], device=DEV)
        z = h.double() @ tensors["up"].double().T
        ap, an = torch.nn.functional.softplus(torch.tensor([p, q], dtype=torch.float64)) + torch.tensor([0.0, 0.5])
        want = torch.where(z > 0, ap * z * z + z / 2, an * (torch.expm1(z.clamp(max=0)) - z) + z / 2)
        for rows in (4, 16):      # roundings to bfloat16: of the product for 16 rows, by the slope of at most 2 ap |z| + an + 1/2, and of the result
            got = part.forward(h[:rows], None).double()
            assert ((got - want[:rows]).abs() <= 2 ** -8 * 1.02 * ((2 * ap * z.abs() + an + 0.5) * z.abs() + want.abs())[:rows] + 1e-5).all()


@pytest.mark.parametrize("M,N,K", [(17, 41024, 64), (64, 41000, 192), (33, 50001, 896), (40, 41030, 1984)])
def test_logits_of_17_to_64_tokens_by_very_many_rows(ops, M, N, K):
    """A narrow model's head on tiles of 64 x 64: rows that fill no whole tile, results whose rows start on no 16 bytes, one step of columns and
    many; against 64 bits, and a row's bits do not hang on the others."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a = torch.randn(64, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).bfloat16()
    got = ops.gemm_skinny(a[:M], w, out_dtype=torch.float32)
    torch.testing.assert_close(got.double(), a[:M].double() @ w.double().T, atol=3e-5, rtol=3e-5)
    assert torch.equal(got, ops.gemm_skinny(a, w, out_dtype=torch.float32)[:M])
    assert torch.equal(got, ops.gemm_tiled_sums(a[:M], w, 1)[0])


@pytest.mark.parametrize("M,N,K", [(9, 31, 512), (13, 64, 516), (17, 97, 560), (33, 33, 896), (48, 130, 1100), (49, 65, 2052), (97, 896, 4864), (5, 7, 64), (20, 36, 20), (16, 401, 9008), (64, 130, 516), (33, 1026, 692)])
def test_32_bit_products_by_slices_have_the_bits_of_the_tiles(ops, M, N, K):
    """Blocks whose waves have two slices each: one, an odd number and all sixteen of them, columns that end within a slice, a step or a
    piece, tokens and rows of W past the last, rows of C at any address; with bias and added onto what is there.  The tiled kernel sums in
    the same order; both are held against 64 bits, and the choice is one of them."""
    from llm_infrence_engine_amd.kernels import build

    force = build.load().ms_gemm_f32_force
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a, w, bias = (torch.randn(*s, generator=g, device=DEV) for s in ((M, K), (N, K), (N,)))
    there = torch.randn(M, N + 3, generator=g, device=DEV)

    def run(kind, plain, wide):
        force(kind)
        try:
            out = there.clone()[:, :N] if wide else there[:, :N].clone()
            return ops.gemm_generic(a, w, out, bias=None if plain else bias, accumulate=not plain).clone()
        finally:
            force(0)

    for plain in (True, False):
        for wide in (False, True):
            want = run(3, plain, wide)
            exact = a.double() @ w.double().T + (0 if plain else bias.double() + there[:, :N].double())
            torch.testing.assert_close(want.double(), exact, atol=K ** 0.5 * 2e-6, rtol=2e-5)      # (sums of K products of about one)
            for kind in (2, 6, 7, 8, 0):
                assert torch.equal(run(kind, plain, wide), want), (kind, plain, wide)
