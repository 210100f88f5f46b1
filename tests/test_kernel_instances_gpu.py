"""Every kernel instance that is compiled into the library is launched by a test and its result
checked: the products and the attention are templates of which a dispatch picks one by the sizes
of a call, and an instance that only a real model's sizes select would otherwise be unverified
arithmetic (the reference tests its products at model sizes for the same reason:
src/cuda/prefill.cu:1100 `gemv_ref`, src/model.rs:6238-6319).

Each case below names the instances it is meant to select, runs a call of such sizes, checks the
result (against a float64 product, or bit for bit against the unfused kernels, which other cases
check against float64), and asserts that those instances were what the library launched.  The
last test asserts that the cases together cover every instance the library says it contains: a
new instance without a case fails it."""
import math

import pytest
import torch

from axon_amd.kernels import MODE_ADD_F32, MODE_STORE, MODE_STORE_F32, MODE_SWIGLU, kernels
from gpu_helpers import paged_cache, tol
from plain import qwen2_plain as P

pytestmark = pytest.mark.gpu

SEEN = {"bfloat16": set(), "float32": set()}
RAN = set()


def rnd(*shape, seed=0, scale=1.0, device="cpu"):
    g = torch.Generator(device=device).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=device) * scale


def launched(k, dtype, run):
    """What `run()` launched."""
    torch.cuda.synchronize()
    k.reset_instances()
    run()
    torch.cuda.synchronize()
    hit = set(k.instances(launched=True))
    SEEN[dtype] |= hit
    return hit


# --------------------------------------------------------------------------- the checks
def check_gemm(dtype, M, N, K, mode, bias=False):
    """out = epilogue(x w^T + bias) against the float64 product of the rounded operands (on the
    device: the matrices of a real vocabulary are large), and, for packed matrices, the first rows
    bit for bit as a step of those rows alone gives them."""
    k = kernels(dtype)
    td = torch.bfloat16 if dtype == "bfloat16" else torch.float32
    x = rnd(M, K, seed=1, device="cuda").to(td)
    rows_w = 2 * N if mode == MODE_SWIGLU else N
    w = rnd(rows_w, K, seed=2, scale=0.2, device="cuda").to(td)
    b = rnd(N, seed=3, device="cuda") if bias else None
    wp = k.prepare_weight(w, mode == MODE_SWIGLU)
    prod = x.double() @ w.double().T
    if mode == MODE_SWIGLU:
        g, u = prod[:, :N], prod[:, N:]
        want = g / (1 + torch.exp(-g)) * u
    else:
        want = prod if b is None else prod + b.double()
    base = rnd(M, N, seed=4, device="cuda")
    out_dt = td if mode in (MODE_STORE, MODE_SWIGLU) else torch.float32

    def run(m):
        out = base[:m].clone().to(out_dt)
        k.gemm(x[:m], wp, out, b, mode)
        return out
    got = {}
    hit = launched(k, dtype, lambda: got.setdefault("out", run(M)))
    out = got["out"].double()
    if mode == MODE_ADD_F32:
        out = out - base.double()
    loose = mode in (MODE_STORE, MODE_SWIGLU)
    scale = max(1.0, float(want.abs().max()))
    limit = (1e-2 if loose else 2e-5 * math.sqrt(K)) * scale if dtype == "bfloat16" else 2e-6 * math.sqrt(K) * scale
    assert float((out - want).abs().max()) <= limit, (M, N, K, mode)
    for m in sorted({1, min(M, 9), min(M, 17), min(M, 65)}):            # a row's bits do not depend on the step
        assert torch.equal(run(m), got["out"][:m]), (M, N, K, mode, m)
    return hit


def check_then_norm(M, H, F):
    """The product that adds into the rows with the norm behind it written by the kernel that adds
    the segments' sums: bit for bit the product and the norm one after the other."""
    k = kernels("bfloat16")
    a = rnd(M, F, seed=5, device="cuda").bfloat16()
    w = k.prepare_weight(rnd(H, F, seed=6, scale=0.3, device="cuda").bfloat16())
    res = rnd(M, H, seed=7, scale=2.0, device="cuda")
    gain = (1.0 + 0.3 * rnd(H, seed=8, device="cuda")).bfloat16()
    x1 = res.clone()
    k.gemm(a, w, x1, None, MODE_ADD_F32)
    h1 = k.rmsnorm(x1, gain, 1e-5, torch.empty(M, H, dtype=torch.bfloat16, device="cuda"))
    x2, h2 = res.clone(), torch.zeros(M, H, dtype=torch.bfloat16, device="cuda")
    hit = launched(k, "bfloat16", lambda: k.gemm(a, w, x2, None, MODE_ADD_F32, following_norm=(gain, h2, 1e-5)))
    assert torch.equal(x1, x2) and torch.equal(h1, h2)
    return hit


def _qkv_case(M, nh, nkv, hd, hidden, page, seed):
    k = kernels("bfloat16")
    width = (nh + 2 * nkv) * hd
    w = k.pack_matrix(rnd(width, hidden, seed=seed, scale=0.2, device="cuda").bfloat16())
    bias = rnd(width, seed=seed + 1, device="cuda")
    g = torch.Generator().manual_seed(seed + 2)
    n_pages, max_pages = 3 * -(-(M + 8) // page) + 2, -(-(M + 8) // page)
    slots = torch.randperm(3 * max_pages * page, generator=g)[:M]
    seq = (slots // (max_pages * page)).to(torch.int32).cuda()
    pos = (slots % (max_pages * page)).to(torch.int32).cuda()
    pages = torch.randperm(n_pages, generator=g)[:3 * max_pages].view(3, max_pages).to(torch.int32).cuda()
    table = torch.empty(M, hd // 2, 2, dtype=torch.float32, device="cuda")
    k.rope_table(pos, P.rope_freqs(hd, 10000.0).cuda(), table)

    def fresh():
        return (torch.zeros(M, width, dtype=torch.bfloat16, device="cuda"),
                torch.full((n_pages, nkv, page, hd), 7.0, dtype=torch.bfloat16, device="cuda"),
                torch.full((n_pages, nkv, hd, page), 7.0, dtype=torch.bfloat16, device="cuda"))
    return k, w, bias, seq, pos, pages, table, fresh


def check_qkv_rope(M, nh, nkv, hd, hidden, page):
    """The [q; k; v] product with bias, rotation and the store into the pages in its own launches
    against the plain product followed by the rotary kernel: the same bits."""
    k, w, bias, seq, pos, pages, table, fresh = _qkv_case(M, nh, nkv, hd, hidden, page, 20)
    x = rnd(M, hidden, seed=19, device="cuda").bfloat16()
    q1, k1, v1 = fresh()
    k.gemm(x, w, q1, bias, MODE_STORE)
    k.rope_kv_write(q1, table, pos, seq, pages, k1, v1, nh, nkv, hd, hd, page, True)
    q2, k2, v2 = fresh()
    hit = launched(k, "bfloat16", lambda: k.gemm_qkv_rope(x, w, bias, q2, table, pos, seq, pages, k2, v2, nh, nkv, hd, page))
    assert torch.equal(q1[:, :nh * hd], q2[:, :nh * hd]) and torch.equal(k1, k2) and torch.equal(v1, v2)
    return hit


def check_normed_qkv(M, nh, nkv, hd, hidden, page):
    """The same with the RMS norm of the operand inside, against the norm kernel before it."""
    k, w, bias, seq, pos, pages, table, fresh = _qkv_case(M, nh, nkv, hd, hidden, page, 30)
    rows = rnd(M, hidden, seed=29, scale=2.0, device="cuda")
    gain = (1.0 + rnd(hidden, seed=28, device="cuda")).bfloat16()
    assert k.gemm_normed_ok(M, (nh + 2 * nkv) * hd, hidden)
    x = k.rmsnorm(rows, gain, 1e-6, torch.empty(M, hidden, dtype=torch.bfloat16, device="cuda"))
    q1, k1, v1 = fresh()
    k.gemm_qkv_rope(x, w, bias, q1, table, pos, seq, pages, k1, v1, nh, nkv, hd, page)
    q2, k2, v2 = fresh()
    hit = launched(k, "bfloat16", lambda: k.gemm_normed_qkv_rope(rows, gain, 1e-6, w, bias, q2, table, pos, seq, pages, k2, v2,
                                                                  nh, nkv, hd, page))
    assert torch.equal(q1[:, :nh * hd], q2[:, :nh * hd]) and torch.equal(k1, k2) and torch.equal(v1, v2)
    return hit


def check_normed_glu(M, hidden, ffn):
    """The gated product with the RMS norm of its operand inside, against the norm kernel followed by
    the gated product: the same bits."""
    k = kernels("bfloat16")
    assert k.gemm_normed_ok(M, ffn, hidden, gated=True)
    rows = rnd(M, hidden, seed=40, scale=3.0, device="cuda")
    gain = (1.0 + rnd(hidden, seed=41, device="cuda")).bfloat16()
    w = k.pack_matrix(rnd(2 * ffn, hidden, seed=42, scale=0.2, device="cuda").bfloat16())
    x = k.rmsnorm(rows, gain, 1e-5, torch.empty(M, hidden, dtype=torch.bfloat16, device="cuda"))
    want = torch.empty(M, ffn, dtype=torch.bfloat16, device="cuda")
    k.gemm(x, w, want, None, MODE_SWIGLU)
    got = torch.zeros(M, ffn, dtype=torch.bfloat16, device="cuda")
    hit = launched(k, "bfloat16", lambda: k.gemm_normed_glu(rows, gain, 1e-5, w, got))
    assert torch.equal(got, want)
    return hit


def _attention_case(nh, nkv, hd, page, T, window, dtype="bfloat16"):
    td = torch.bfloat16 if dtype == "bfloat16" else torch.float32
    q, kk, vv = (rnd(T, n, hd, seed=s).to(td) for n, s in ((nh, 51), (nkv, 52), (nkv, 53)))
    kc, vc, table = paged_cache(kk.double(), vv.double(), page, dtype, seed=3)
    ref = P.causal_attention(q.double(), kk.double(), vv.double(), window).view(T, nh * hd)
    pos = torch.arange(T, dtype=torch.int32).cuda()
    return q.cuda().view(T, nh * hd), kc, vc, table, pos, torch.zeros(T, dtype=torch.int32).cuda(), ref


def check_attention_rows(dtype, nh, nkv, hd, page, T, window):
    k = kernels(dtype)
    q, kc, vc, table, pos, rows, ref = _attention_case(nh, nkv, hd, page, T, window, dtype)
    out = torch.empty(T, nh * hd, dtype=q.dtype, device="cuda")
    hit = launched(k, dtype, lambda: k.attention(q, nh * hd, kc, vc, table, pos, rows, out, nh, nkv, hd, page, window,
                                                  1.0 / math.sqrt(hd)))
    assert (out.cpu().double() - ref).abs().max() <= tol(dtype, ref, 2e-6, 1e-2)
    # the last tokens alone (few tokens: eight waves each) give the bits they have among all of them
    few = min(T, 1023 // nh, 40)
    alone = torch.empty(few, nh * hd, dtype=q.dtype, device="cuda")
    k.attention(q[T - few:], nh * hd, kc, vc, table, pos[T - few:], rows[T - few:], alone, nh, nkv, hd, page, window,
                1.0 / math.sqrt(hd))
    assert torch.equal(alone, out[T - few:])
    return hit


def check_attention_mfma(nh, nkv, hd, page, T, window, every=1):
    """The prompt kernel over the whole sequence against the plain formula, and every position bit
    for bit as the decoding kernel gives it."""
    k = kernels("bfloat16")
    q, kc, vc, table, pos, rows, ref = _attention_case(nh, nkv, hd, page, T, window)
    scale = 1.0 / math.sqrt(hd)
    tiles = torch.tensor([(a, min(128, T - a)) for a in range(0, T, 128)], dtype=torch.int32).cuda()
    prompt = torch.zeros(T, nh * hd, dtype=torch.bfloat16, device="cuda")
    hit = launched(k, "bfloat16", lambda: k.attention_prefill(q, nh * hd, kc, vc, table, pos, rows, prompt, tiles, nh, nkv, hd,
                                                              page, window, scale))
    assert not torch.isnan(prompt).any()
    assert (prompt.cpu().double() - ref).abs().max() <= tol("bfloat16", ref, bf16=1.5e-2)
    # the decoding kernel for every `every`-th position and the edges of blocks and chunks
    picks = sorted(set(range(0, T, every)) | ({0, 1, 63, 64, 255, 256, 257, T - 2, T - 1} & set(range(T))))
    idx = torch.tensor(picks, dtype=torch.int32).cuda()
    ch = k.attention_decode_chunk
    chunks = max((p - ((max(0, p + 1 - window) if window else 0) // ch * ch)) // ch + 1 for p in picks)
    partial = torch.empty(k.attention_decode_workspace(len(picks), nh, hd, chunks), dtype=torch.float32, device="cuda")
    decoded = torch.zeros(T, nh * hd, dtype=torch.bfloat16, device="cuda")
    hit |= launched(k, "bfloat16", lambda: k.attention_decode(q, nh * hd, kc, vc, table, pos, rows, decoded, idx, partial, chunks,
                                                               nh, nkv, hd, page, window, scale))
    assert torch.equal(decoded[picks], prompt[picks])
    return hit


def check_attention_f32(nh, nkv, hd, page, T, window, last):
    """The float32 build's prompt kernel over the whole sequence and its decoding kernel for the `last` tokens against the
    plain formula, each with the bits of a wave a (token, head)."""
    k = kernels("float32")
    q, kc, vc, table, pos, rows, ref = _attention_case(nh, nkv, hd, page, T, window, "float32")
    sizes = (nh, nkv, hd, page, window, 1.0 / math.sqrt(hd))
    want = k.attention(q, nh * hd, kc, vc, table, pos, rows, torch.empty_like(q), *sizes)
    tiles = torch.tensor([(a, min(128, T - a)) for a in range(0, T, 128)], dtype=torch.int32).cuda()
    prompt = torch.full_like(q, float("nan"))
    hit = launched(k, "float32", lambda: k.attention_prefill(q, nh * hd, kc, vc, table, pos, rows, prompt, tiles, *sizes))
    assert torch.equal(prompt, want)
    assert (prompt.cpu().double() - ref).abs().max() <= tol("float32", ref, 2e-6)
    idx, chunks = torch.arange(T - last, T, dtype=torch.int32).cuda(), -(-T // k.attention_decode_chunk)
    partial = torch.empty(k.attention_decode_workspace(last, nh, hd, chunks), dtype=torch.float32, device="cuda")
    decoded = torch.full_like(q, float("nan"))
    hit |= launched(k, "float32", lambda: k.attention_decode(q, nh * hd, kc, vc, table, pos, rows, decoded, idx, partial, chunks, *sizes))
    assert torch.equal(decoded[T - last:], want[T - last:])
    return hit


def check_rmsnorm(dtype, dim):
    k = kernels(dtype)
    x = rnd(5, dim, seed=60, scale=3.0)
    gain = 1 + 0.3 * rnd(dim, seed=61)
    out = torch.empty(5, dim, dtype=k.dtype, device="cuda")
    hit = launched(k, dtype, lambda: k.rmsnorm(x.cuda(), gain.cuda(), 1e-5, out))
    ref = P.rms_norm(x.double(), gain.double(), 1e-5)
    assert (out.cpu().double() - ref).abs().max() <= tol(dtype, ref, 1e-6, 8e-3)
    return hit


def check_heads_prepare(dtype, T, form, nq):
    """Queries, keys and values of T tokens in one call: the bits of calls of 200 of them.  form: normed head by head, over whole rows,
    not at all, or behind a convolution (single tokens, whose state the calls leave as they find it for the others)."""
    k = kernels(dtype)
    td, nk, dim, page, conv = getattr(torch, dtype), 2, 24, 16, form == "conv"
    W = (nq + 2 * nk) * dim
    proj = rnd(T, W, seed=T, device="cuda")
    freqs, table = P.rope_freqs(dim // 2, 100.0).cuda(), torch.empty(T, dim // 4, 2, device="cuda")
    pos = (torch.arange(T, dtype=torch.int32) % page).cuda()
    seq = (torch.arange(T, dtype=torch.int32) if conv else torch.arange(T, dtype=torch.int32) // page).cuda()
    k.rope_table(pos, freqs, table)
    pages = int(seq.max()) + 1
    block_table = torch.randperm(pages, generator=torch.Generator().manual_seed(1)).int().view(pages, 1).cuda()
    gains = [None, None] if form == "none" else [rnd(n * dim if form == "rows" else dim, seed=n, device="cuda") for n in (nq, nk)]
    w = rnd(W, 3, seed=9, device="cuda").to(td)

    def run(step):
        q = torch.full((T, nq * dim), 3.0, dtype=td, device="cuda")
        cache = torch.full((pages, 1, page, 2 * nk * dim), 3.0, dtype=td, device="cuda")
        state = rnd(pages, 4 * W, seed=8, device="cuda") if conv else None
        for a in range(0, T, step):
            b = min(T, a + step)
            k.heads_prepare(proj[a:b], 0, nq, nq * dim, nk, (nq + nk) * dim, nk * dim, dim, *gains, 1e-6, dim // 2, False, 1.25, table[a:b],
                            pos[a:b], seq[a:b], block_table, cache, page, q[a:b], norm_rows=form == "rows",
                            conv=(w, state, 2 * W, None) if conv else None)
        return q, cache, state
    got = {}
    hit = launched(k, dtype, lambda: got.setdefault("all", run(T)))
    for a, b in zip(got["all"], run(200)):
        assert a is None or torch.equal(a, b)
    assert not bool((got["all"][0] == 3.0).all(1).any())
    return hit


def check_state_conv(dtype, T, C, taps):
    """The convolution of one request's tokens against the same sums of float64."""
    k = kernels(dtype)
    td, copy = getattr(torch, dtype), (taps - 1) * C
    x, w = rnd(T, C, seed=1, device="cuda"), rnd(C, taps, seed=2, device="cuda").to(td)
    bias, state = rnd(C, seed=3, device="cuda"), rnd(1, 2 * copy, seed=4, device="cuda")
    u, pos = torch.empty(T, C, device="cuda"), torch.arange(6, 6 + T, dtype=torch.int32, device="cuda")
    hit = launched(k, dtype, lambda: k.state_conv(x, w, bias, state, copy, 0, pos, torch.zeros_like(pos), u, False))
    rows = torch.cat([state[0, copy:].view(taps - 1, C), x]).double()         # the copy behind position 5
    want = bias.double() + sum(rows[i:i + T] * w[:, i].double() for i in range(taps))
    size = bias.double().abs() + sum((rows[i:i + T] * w[:, i].double()).abs() for i in range(taps))
    assert bool(((u.double() - want).abs() <= (taps + 1) * 2.0 ** -24 * size).all())
    return hit


def check_embed(dtype, T, dim, packed):
    """Rows of a table, widened and scaled."""
    k = kernels(dtype)
    table = rnd(50, dim, seed=dim, device="cuda").to(getattr(torch, dtype))
    tokens = torch.randint(0, 50, (T,), generator=torch.Generator().manual_seed(T), dtype=torch.int32).cuda()
    out = torch.full((T + 1, dim), 7.0, device="cuda")
    held = k.pack_matrix(table) if packed else table
    hit = launched(k, dtype, lambda: k.embed(tokens, held, out[:T], 0.3))
    assert torch.equal(out[:T], table[tokens.long()].float() * torch.tensor(0.3, device="cuda")) and bool((out[T] == 7.0).all())
    return hit


def check_gated_scan(dtype, T):
    """The gated recurrence of one request against a loop of float64."""
    k, C, taps = kernels(dtype), 24, 3
    td = getattr(torch, dtype)
    gates, u = rnd(T, 2 * C, seed=1, device="cuda"), rnd(T, C, seed=2, device="cuda")
    y, x = (rnd(T, C, seed=n, device="cuda").to(td) for n in (3, 4))
    lam, state = rnd(C, seed=5, device="cuda"), rnd(1, 2 * taps * C, seed=6, device="cuda")
    pos, out = torch.arange(T, dtype=torch.int32, device="cuda"), torch.empty(T, C, dtype=td, device="cuda")
    spans, before = torch.tensor([[0, 0, T]], dtype=torch.int32, device="cuda"), state[0, taps * C:].double().cpu()      # behind position -1
    hit = launched(k, dtype, lambda: k.gated_scan(gates, u, y, x, lam, 8.0, state, spans, pos, torch.zeros_like(pos), out, C, taps))
    g, U, Y, L = gates.double().cpu(), u.double().cpu(), y.double().cpu(), lam.double().cpu()
    S, want = before[:C].clone(), []
    for t in range(T):
        log_a = -8.0 * torch.sigmoid(g[t, :C]) * torch.nn.functional.softplus(L)
        S = torch.exp(log_a) * S + torch.sqrt(-torch.expm1(2 * log_a)) * torch.sigmoid(g[t, C:]) * U[t]
        want.append(S * torch.nn.functional.gelu(Y[t], approximate="tanh"))
    want = torch.stack(want)
    limit = 1e-2 if dtype == "bfloat16" else 2e-5
    assert float((out.double().cpu() - want).abs().max()) <= limit * max(1.0, float(want.abs().max()))
    return hit


def check_wide_lists(T, H, F):
    """The gated routed product by tiles of 128 rows: the bits of tiles of 16."""
    k, E, top = kernels("bfloat16"), 5, 2
    P = T * top
    h, wu = rnd(T, H, seed=1, device="cuda").bfloat16(), rnd(E, 2 * F, H, seed=2, scale=0.2, device="cuda").bfloat16()
    chosen = rnd(T, E, seed=3).topk(top, 1).indices.int().contiguous().cuda()

    def run(rows):
        most = k.route_max_tiles(P, E, rows)
        pairs, tokens, tiles, n = (torch.zeros(size, dtype=torch.int32, device="cuda") for size in (P, P, 3 * most, 1))
        k.route_sort(chosen, E, pairs, tokens, tiles, n, tile_rows=rows)
        out = torch.full((P, F), float("nan"), dtype=torch.bfloat16, device="cuda")
        k.grouped_gemm(h, wu, out, x_group_stride=0, out_group_stride=0, glu=(float("inf"), 1.0, 0.0), routed=(tiles, n, most, tokens, pairs, rows), rows=P)
        return out
    got = {}
    hit = launched(k, "bfloat16", lambda: got.setdefault("out", run(128)))
    assert torch.equal(got["out"], run(16)) and not bool(got["out"].isnan().any())
    return hit


def check_masked_blocks(maps, dim, vdim, page, softcap, gated):
    """Single tokens whose blocks of positions run side by side, against the walk of a wave a token (up to the order of the sums), with
    a bend, with gates by head and by dim, in pages of several blocks."""
    k, heads, kv, contexts = kernels("bfloat16"), 6, 2, [0, 63, 64, 200, 413]
    T, need = len(contexts), [c // page + 1 for c in contexts]
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(2)).int().cuda()
    table = torch.zeros(T, max(need), dtype=torch.int32, device="cuda")
    for i, n in enumerate(need):
        table[i, :n] = order[sum(need[:i]):sum(need[:i + 1])]
    cache = rnd(sum(need), 1, page, kv * (maps * dim + vdim), seed=3, device="cuda").bfloat16()
    q = rnd(T, heads * maps * dim, seed=4, device="cuda").bfloat16()
    gate = None if not gated else rnd(T, heads * (vdim if gated == "dims" else 1) + 5, seed=5, device="cuda")[:, :heads * (vdim if gated == "dims" else 1)]
    pos, rows = torch.tensor(contexts, dtype=torch.int32, device="cuda"), torch.arange(T, dtype=torch.int32, device="cuda")

    def attend(span):
        out = torch.full((T, heads * vdim), float("nan"), dtype=torch.bfloat16, device="cuda")
        k.masked_attention(q, cache, table, pos, rows, out, heads, kv, maps, dim, vdim, page, "causal", 0, dim ** -0.5, softcap=softcap, lam=0.3,
                           out_scale=0.7, eps=1e-6, gate=gate, gate_per_head=gated == "heads", span=span)
        return out.double()
    got = {}
    hit = launched(k, "bfloat16", lambda: got.setdefault("out", attend(max(contexts) + 1)))
    walk = attend(0)
    # one rounding of weights to 8 bits and one of the output on either side, over values of a few units
    assert float((got["out"] - walk).abs().max()) <= 2.0 ** -7 * float(walk.abs().max()) * (4 if maps == 2 else 1)
    return hit


# --------------------------------------------------------------------------- the cases
# (names of the instances the case is meant to select, the check, its arguments)
BF, F32 = "bfloat16", "float32"
def check_grouped(dtype, M, G, N, K, glu):
    """A block-diagonal grouped product (gated or plain) against float64."""
    k = kernels(dtype)
    td = torch.bfloat16 if dtype == "bfloat16" else torch.float32
    x = rnd(M, G * K, seed=4).to(torch.bfloat16).float()
    w = rnd(G, (2 if glu else 1) * N, K, seed=5, scale=0.3).to(torch.bfloat16).float()
    out = torch.zeros(M, G * N, dtype=torch.float32, device="cuda")
    hit = launched(k, dtype, lambda: k.grouped_gemm(x.to(td).cuda(), w.to(td).cuda(), out, x_group_stride=K, out_group_stride=N,
                                                    glu=(1.0, 1.702) if glu else None))
    for g in range(G):
        z = x[:, g * K:(g + 1) * K].double() @ w[g].double().T
        if glu:
            gate, up = torch.clamp(z[:, :N], max=1.0), torch.clamp(z[:, N:], -1.0, 1.0)
            z = gate * torch.sigmoid(1.702 * gate) * (up + 1)
        assert float((out[:, g * N:(g + 1) * N].cpu() - z.float()).abs().max()) <= tol(dtype, z.float(), bf16=1e-4)
    return hit


def check_latent(rank, rot, sink):
    """Latent attention of a portion of many tokens against the plain formula (weights and queries rounded as the kernel
    does), and bit for bit as each token alone, a wave a token, gives it."""
    k, T, heads, page = kernels("bfloat16"), 261, 16, 64
    pages = -(-T // page)
    cache = rnd(pages, 1, page, 2 * rank + rot, seed=80, device="cuda").bfloat16()
    table = torch.arange(pages, device="cuda").flip(0).int().view(1, pages)
    q = rnd(T, heads * (rank + rot), seed=81, scale=0.3, device="cuda")
    pos = torch.arange(T, dtype=torch.int32, device="cuda")
    sinks = rnd(heads, seed=82, device="cuda") if sink else None
    scale = (rank + rot) ** -0.5

    def attend(rows, tab):
        out = torch.full((T, heads * rank), float("nan"), device="cuda")
        k.latent_attention(q, cache, tab, pos, rows, out, heads, rank, rot, page, 0, scale, sink=sinks)
        return out
    got = {}
    hit = launched(k, "bfloat16", lambda: got.setdefault("out", attend(torch.zeros(T, dtype=torch.int32, device="cuda"), table)))
    assert torch.equal(got["out"], attend(torch.arange(T, dtype=torch.int32, device="cuda"), table.expand(T, pages).contiguous()))
    lat, at = cache[table[0].long(), 0].reshape(pages, -1), torch.arange(T, device="cuda")
    key = lat[:, :page * (rank + rot)].reshape(pages * page, rank + rot)[:T].double()
    val = lat[:, page * (rank + rot):].reshape(pages, rank, page).transpose(1, 2).reshape(pages * page, rank)[:T].double()
    s = torch.matmul(q.view(T, heads, -1).bfloat16().double().transpose(0, 1), key.T.contiguous()) * scale
    s = s.masked_fill(at[None, :] > at[:, None], float("-inf"))
    m = s.amax(-1, keepdim=True) if sinks is None else torch.maximum(s.amax(-1, keepdim=True), sinks.double()[:, None, None])
    w = torch.exp(s - m)
    want = torch.matmul(w, val) / (w.sum(-1, keepdim=True) + (0 if sinks is None else torch.exp(sinks.double()[:, None, None] - m)))
    # the weights are rounded to 8 bits: each off by at most 2^-9 of itself
    bound = 2.0 ** -8 * float(val.abs().max())
    assert float((got["out"].view(T, heads, rank).transpose(0, 1).double() - want).abs().max()) <= bound
    few = torch.full((3, heads * rank), float("nan"), device="cuda")              # the last tokens' blocks of positions side by side
    rows = torch.zeros(3, dtype=torch.int32, device="cuda")
    hit |= launched(k, "bfloat16", lambda: k.latent_attention(q[T - 3:], cache, table, pos[T - 3:], rows, few, heads, rank, rot, page, 0, scale,
                                                              sink=sinks, span=T))
    assert float((few.view(3, heads, rank).transpose(0, 1).double() - want[:, T - 3:]).abs().max()) <= bound
    return hit


def check_conv(dtype, T, C):
    """The short causal convolution of one request that goes on, and of the tokens behind it, one request each."""
    k = kernels(dtype)
    td = torch.bfloat16 if dtype == "bfloat16" else torch.float32
    taps, long_one = 4, T - 5
    x = rnd(T, C, seed=70, device="cuda").to(td)
    w, bias = rnd(C, taps, seed=71, device="cuda").to(td), rnd(C, seed=72, device="cuda")
    state = rnd(6, 2 * taps * C, seed=73, device="cuda")
    seq = torch.tensor([0] * long_one + [1, 2, 3, 4, 5], dtype=torch.int32).cuda()
    pos = torch.tensor(list(range(9, 9 + long_one)) + [8, 9, 10, 11, 12], dtype=torch.int32).cuda()
    u = torch.empty(T, C, device="cuda")
    hit = launched(k, dtype, lambda: k.causal_conv(x, w, bias, state, pos, seq, u))
    for first, n, slot, start in [(0, long_one, 0, 9)] + [(long_one + i, 1, 1 + i, 8 + i) for i in range(5)]:
        before = (start - 1) & 1                             # the copy behind the position before the request's first
        kept = state[slot, before * taps * C + C:(before + 1) * taps * C].view(taps - 1, C)
        rows = torch.cat([kept.double(), x[first:first + n].double()])
        want = bias.double() + sum(rows[i:i + n] * w.double()[:, i] for i in range(taps))
        # four products and a bias, each sum rounded by at most half a unit of what it holds
        bound = 6 * 2.0 ** -24 * (bias.double().abs() + sum((rows[i:i + n] * w.double()[:, i]).abs() for i in range(taps)))
        assert bool(((u[first:first + n].double() - want).abs() <= bound).all())
    return hit


CASES = [
    # 32-bit FMA products: the float32 build's, and the bfloat16 build's for what cannot be packed
    (F32, ["gemm_fma<16,0>"], check_gemm, (F32, 5, 100, 70, MODE_STORE_F32, True)),
    (F32, ["gemm_fma<64,0>"], check_gemm, (F32, 70, 259, 130, MODE_ADD_F32)),
    (F32, ["gemm_fma<16,1>"], check_gemm, (F32, 9, 96, 70, MODE_SWIGLU)),
    (F32, ["gemm_fma<64,1>"], check_gemm, (F32, 33, 48, 100, MODE_SWIGLU)),
    # (rows of X a block, gated; from 33 to 128 rows by how many tiles there would be)
    *[(d, [f"gemm_fma<{rows},{int(mode == MODE_SWIGLU)}>"], check_gemm, (d, M, N, K, mode)) for d in (F32, BF)
      for rows, M, N, K, mode in ((32, 20, 259, 290, MODE_STORE_F32), (128, 200, 259, 130, MODE_STORE_F32), (128, 40, 16390, 36, MODE_STORE_F32),
                                  (32, 31, 48, 100, MODE_SWIGLU), (128, 129, 48, 100, MODE_SWIGLU), (64, 128, 96, 290, MODE_SWIGLU))],
    (F32, ["gemm_fma_flow<0>"], check_gemm, (F32, 200, 259, 260, MODE_STORE_F32)),
    (F32, ["gemm_fma_flow<1>"], check_gemm, (F32, 129, 48, 292, MODE_SWIGLU)),
    *[(F32, [f"gemm_fma_flow_rows<{rows},0>"], check_gemm, (F32, M, N, K, MODE_STORE_F32))
      for rows, M, N, K in ((32, 129, 2048, 260), (48, 300, 2050, 228), (64, 896, 2048, 292), (80, 626, 2048, 228), (96, 1500, 2048, 644))],
    *[(F32, [f"gemm_fma_flow_rows<{rows},1>"], check_gemm, (F32, M, 1024, K, MODE_SWIGLU))
      for rows, M, K in ((32, 129, 260), (64, 896, 292), (96, 626, 228))],
    # chain by chain: fewer chains than waves, and numbers loaded singly but for one tile of rows and W
    *[(d, [f"gemm_fma_by_chain<{rows},{int(mode == MODE_SWIGLU)},{int(K % 4 == 0)}>"], check_gemm, (d, M, N, K, mode)) for d in (F32, BF)
      for rows, M in ((16, 5), (32, 20), (64, 70)) for N, K, mode in ((259, 100, MODE_STORE_F32), (259, 70, MODE_STORE_F32), (48, 96, MODE_SWIGLU),
                                                                      (48, 290, MODE_SWIGLU))],
    # as many chains as waves, or nearly, asked for ahead
    *[(BF, [f"gemm_fma<{rows},{int(mode == MODE_SWIGLU)}>"], check_gemm, (BF, M, N, 224, mode)) for rows, M in ((16, 5), (32, 20), (64, 70))
      for N, mode in ((259, MODE_STORE_F32), (48, MODE_SWIGLU))],
    (BF, ["gemm_fma<16,0>"], check_gemm, (BF, 5, 100, 70, MODE_STORE, True)),
    (BF, ["gemm_fma<64,0>"], check_gemm, (BF, 70, 259, 130, MODE_STORE_F32)),
    (BF, ["gemm_fma<16,1>"], check_gemm, (BF, 9, 96, 70, MODE_SWIGLU)),
    (BF, ["gemm_fma<64,1>"], check_gemm, (BF, 33, 48, 100, MODE_SWIGLU)),
    (F32, ["rmsnorm<0>"], check_rmsnorm, (F32, 777)),
    (F32, ["rmsnorm<1>"], check_rmsnorm, (F32, 3584)),
    (BF, ["rmsnorm<0>"], check_rmsnorm, (BF, 777)),
    (BF, ["rmsnorm<1>"], check_rmsnorm, (BF, 3584)),
    # eight waves a (token, head) below 1,024 of them, one from there
    (F32, ["attention_rows<0,8>"], check_attention_rows, (F32, 6, 3, 80, 4, 65, 0)),
    (F32, ["attention_rows<0,1>"], check_attention_rows, (F32, 6, 3, 80, 4, 700, 0)),
    (BF, ["attention_rows<1,8>"], check_attention_rows, (BF, 4, 2, 32, 16, 133, 37)),
    (BF, ["attention_rows<1,1>"], check_attention_rows, (BF, 4, 2, 32, 16, 600, 37)),
    # up to 16 rows: a wave a segment of K.  One row tile a block below 16,384 rows of W, two from there
    (BF, ["gemm_stream<1,1,1,0>"], check_gemm, (BF, 3, 100, 128, MODE_STORE, True)),
    (BF, ["gemm_stream<1,1,2,0>"], check_gemm, (BF, 16, 100, 512, MODE_ADD_F32)),
    (BF, ["gemm_stream<1,1,4,0>"], check_gemm, (BF, 8, 3584, 3584, MODE_ADD_F32)),
    (BF, ["gemm_stream<2,1,1,0>"], check_gemm, (BF, 8, 16400, 256, MODE_STORE_F32)),
    (BF, ["gemm_stream<2,1,2,0>"], check_gemm, (BF, 16, 16400, 3584, MODE_STORE_F32)),
    (BF, ["gemm_stream<2,1,1,0>"], check_gemm, (BF, 8, 152064, 3584, MODE_STORE_F32)),      # the head of a real model
    (BF, ["gemm_stream<2,1,1,1>"], check_gemm, (BF, 9, 96, 64, MODE_SWIGLU)),
    (BF, ["gemm_stream<2,1,2,1>"], check_gemm, (BF, 1, 176, 512, MODE_SWIGLU)),
    (BF, ["gemm_stream<2,1,4,1>"], check_gemm, (BF, 16, 320, 1024, MODE_SWIGLU)),
    (BF, ["gemm_stream<2,1,1,2>"], check_qkv_rope, (5, 4, 1, 64, 256, 32)),
    (BF, ["gemm_stream<2,1,2,2>"], check_qkv_rope, (16, 6, 2, 64, 512, 16)),
    (BF, ["gemm_stream<2,1,4,2>"], check_qkv_rope, (8, 28, 4, 128, 3584, 64)),
    # up to 16 rows behind an RMS norm: the norm inside.  (pairs of tiles a wave, segments, epilogue,
    # rows of X in LDS, float4 of a row a lane holds)
    (BF, ["gemm_normed<1,1,1,8,16>"], check_normed_glu, (3, 256, 320)),
    (BF, ["gemm_normed<1,1,1,16,16>"], check_normed_glu, (13, 256, 320)),
    (BF, ["gemm_normed<1,1,1,8,20>"], check_normed_glu, (8, 4352, 12288)),
    (BF, ["gemm_normed<2,1,1,8,16>"], check_normed_glu, (6, 3584, 18944)),                    # a 7B layer's
    (BF, ["gemm_normed<2,1,1,16,16>"], check_normed_glu, (16, 256, 16400)),
    (BF, ["gemm_normed<2,1,1,8,20>"], check_normed_glu, (8, 5120, 27648)),                    # a 32B layer's
    (BF, ["gemm_normed<3,1,1,8,16>"], check_normed_glu, (8, 256, 32784)),
    (BF, ["gemm_normed<3,1,1,16,16>"], check_normed_glu, (9, 256, 32784)),
    (BF, ["gemm_normed<3,1,1,8,20>"], check_normed_glu, (2, 4352, 32784)),
    (BF, ["gemm_normed<1,2,1,8,16>"], check_normed_glu, (8, 512, 320)),
    (BF, ["gemm_normed<1,2,1,16,16>"], check_normed_glu, (16, 768, 4864)),
    (BF, ["gemm_normed<1,2,1,8,20>"], check_normed_glu, (5, 4352, 6144)),
    (BF, ["gemm_normed<2,2,1,8,16>"], check_normed_glu, (8, 512, 8208)),
    (BF, ["gemm_normed<2,2,1,16,16>"], check_normed_glu, (12, 1024, 8208)),
    (BF, ["gemm_normed<2,2,1,8,20>"], check_normed_glu, (7, 5120, 8208)),
    (BF, ["gemm_normed<1,4,1,8,16>"], check_normed_glu, (8, 3584, 2368)),
    (BF, ["gemm_normed<1,4,1,16,16>"], check_normed_glu, (15, 4096, 640)),
    (BF, ["gemm_normed<1,4,1,8,20>"], check_normed_glu, (8, 5120, 1728)),
    (BF, ["gemm_normed<2,4,1,8,16>"], check_normed_glu, (1, 1024, 4112)),
    (BF, ["gemm_normed<2,4,1,16,16>"], check_normed_glu, (10, 1024, 4112)),
    (BF, ["gemm_normed<2,4,1,8,20>"], check_normed_glu, (4, 4352, 4112)),
    (BF, ["gemm_normed<1,1,2,8,16>"], check_normed_qkv, (6, 7, 1, 128, 256, 8)),
    (BF, ["gemm_normed<1,1,2,16,16>"], check_normed_qkv, (11, 4, 2, 64, 256, 16)),
    (BF, ["gemm_normed<1,1,2,8,20>"], check_normed_qkv, (3, 160, 16, 128, 4352, 64)),
    (BF, ["gemm_normed<1,2,2,8,16>"], check_normed_qkv, (7, 3, 3, 96, 512, 4)),
    (BF, ["gemm_normed<1,2,2,16,16>"], check_normed_qkv, (16, 6, 2, 64, 512, 16)),
    (BF, ["gemm_normed<1,2,2,8,20>"], check_normed_qkv, (8, 80, 8, 128, 4352, 64)),
    (BF, ["gemm_normed<1,4,2,8,16>"], check_normed_qkv, (8, 28, 4, 128, 3584, 64)),           # a 7B layer's
    (BF, ["gemm_normed<1,4,2,16,16>"], check_normed_qkv, (12, 28, 4, 128, 3584, 16)),
    (BF, ["gemm_normed<1,4,2,8,20>"], check_normed_qkv, (8, 40, 8, 128, 5120, 64)),           # a 14B layer's
    # 17 to 64 rows: W streamed, X shared through LDS; as many waves a block as give each CU a block.
    # With several segments the sums go through the workspace (gemm_split_reduce<0>).
    (BF, ["gemm_rows<1,4,2,0>"], check_gemm, (BF, 17, 100, 128, MODE_STORE, True)),
    (BF, ["gemm_rows<1,4,3,0>", "gemm_split_reduce<0>"], check_gemm, (BF, 33, 4100, 512, MODE_STORE_F32, True)),
    (BF, ["gemm_rows<1,4,4,0>", "gemm_split_reduce<0>"], check_gemm, (BF, 64, 3584, 1024, MODE_ADD_F32)),
    (BF, ["gemm_rows<1,4,5,0>"], check_gemm, (BF, 40, 4100, 1024, MODE_STORE)),
    (BF, ["gemm_rows<1,4,6,0>"], check_gemm, (BF, 20, 5600, 1024, MODE_STORE_F32)),
    (BF, ["gemm_rows<1,4,7,0>"], check_gemm, (BF, 64, 6400, 1024, MODE_ADD_F32, True)),
    (BF, ["gemm_rows<1,4,8,0>"], check_gemm, (BF, 48, 9600, 1024, MODE_STORE)),
    (BF, ["gemm_rows<2,4,2,0>"], check_gemm, (BF, 17, 16384, 256, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,4,3,0>"], check_gemm, (BF, 64, 16400, 256, MODE_STORE_F32, True)),
    (BF, ["gemm_rows<2,4,4,0>", "gemm_split_reduce<0>"], check_gemm, (BF, 32, 16384, 512, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,4,5,0>", "gemm_split_reduce<0>"], check_gemm, (BF, 17, 16400, 3584, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,4,6,0>"], check_gemm, (BF, 64, 20500, 512, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,4,7,0>"], check_gemm, (BF, 33, 50000, 256, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,4,8,0>"], check_gemm, (BF, 64, 152064, 3584, MODE_STORE_F32)),          # the head of a real model
    (BF, ["gemm_rows<2,4,2,1>"], check_gemm, (BF, 40, 96, 64, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,4,3,1>"], check_gemm, (BF, 17, 8208, 64, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,4,4,1>", "gemm_split_reduce<0>"], check_gemm, (BF, 64, 3584, 1024, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,4,5,1>"], check_gemm, (BF, 64, 18944, 3584, MODE_SWIGLU)),              # a 7B layer's
    (BF, ["gemm_rows<2,4,6,1>"], check_gemm, (BF, 33, 5600, 1024, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,4,7,1>"], check_gemm, (BF, 20, 24592, 64, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,4,8,1>"], check_gemm, (BF, 64, 28688, 64, MODE_SWIGLU)),
    (BF, ["gemm_rows<1,4,2,0>", "gemm_split_reduce<3>"], check_gemm, (BF, 48, 130, 1024, MODE_STORE_F32, True)),   # N % 4 != 0
    (BF, ["gemm_rows<1,4,4,0>", "gemm_split_reduce<1>"], check_then_norm, (64, 3584, 1024)),
    (BF, ["gemm_rows<1,4,5,0>", "gemm_split_reduce<2>"], check_qkv_rope, (64, 28, 4, 128, 3584, 64)),
    (BF, ["gemm_split_reduce<2,8>"], check_qkv_rope, (2056, 36, 4, 128, 512, 16)),
    # 65 to 128 rows: the same kernel with eight tiles of 16 rows of X a step
    (BF, ["gemm_rows<1,8,3,0>"], check_gemm, (BF, 65, 100, 128, MODE_STORE, True)),
    (BF, ["gemm_rows<1,8,3,0>", "gemm_split_reduce<0>"], check_gemm, (BF, 97, 4100, 512, MODE_STORE_F32, True)),
    (BF, ["gemm_rows<1,8,4,0>", "gemm_split_reduce<0>"], check_gemm, (BF, 128, 3584, 1024, MODE_ADD_F32)),
    (BF, ["gemm_rows<1,8,5,0>"], check_gemm, (BF, 100, 4100, 1024, MODE_STORE)),
    (BF, ["gemm_rows<1,8,6,0>"], check_gemm, (BF, 80, 5600, 1024, MODE_STORE_F32)),
    (BF, ["gemm_rows<1,8,7,0>"], check_gemm, (BF, 128, 6400, 1024, MODE_ADD_F32, True)),
    (BF, ["gemm_rows<1,8,8,0>"], check_gemm, (BF, 112, 9600, 1024, MODE_STORE)),
    (BF, ["gemm_rows<2,8,3,0>"], check_gemm, (BF, 65, 16384, 256, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,8,3,0>"], check_gemm, (BF, 128, 16400, 256, MODE_STORE_F32, True)),
    (BF, ["gemm_rows<2,8,4,0>", "gemm_split_reduce<0>"], check_gemm, (BF, 96, 16384, 512, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,8,5,0>", "gemm_split_reduce<0>"], check_gemm, (BF, 66, 16400, 3584, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,8,6,0>"], check_gemm, (BF, 128, 20500, 512, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,8,7,0>"], check_gemm, (BF, 97, 50000, 256, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,8,8,0>"], check_gemm, (BF, 127, 152064, 3584, MODE_STORE_F32)),
    (BF, ["gemm_rows<2,8,3,1>"], check_gemm, (BF, 100, 96, 64, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,8,3,1>"], check_gemm, (BF, 65, 8208, 64, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,8,4,1>", "gemm_split_reduce<0>"], check_gemm, (BF, 128, 3584, 1024, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,8,5,1>"], check_gemm, (BF, 128, 18944, 3584, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,8,6,1>"], check_gemm, (BF, 97, 5600, 1024, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,8,7,1>"], check_gemm, (BF, 80, 24592, 64, MODE_SWIGLU)),
    (BF, ["gemm_rows<2,8,8,1>"], check_gemm, (BF, 128, 28688, 64, MODE_SWIGLU)),
    (BF, ["gemm_rows<1,8,3,0>", "gemm_split_reduce<3>"], check_gemm, (BF, 112, 130, 1024, MODE_STORE_F32, True)),   # N % 4 != 0
    (BF, ["gemm_rows<1,8,4,0>", "gemm_split_reduce<1>"], check_then_norm, (128, 3584, 1024)),
    (BF, ["gemm_rows<1,8,5,0>", "gemm_split_reduce<2>"], check_qkv_rope, (128, 28, 4, 128, 3584, 64)),
    # more than 128 rows: tiles of the output through LDS
    # (129 to 256 rows in no more blocks than CUs: four stages)
    (BF, ["gemm_tile<128,128,2,2,0,4>", "gemm_split_reduce<0>"], check_gemm, (BF, 140, 132, 2048, MODE_STORE, True)),
    (BF, ["gemm_tile<128,128,2,2,0,4>", "gemm_split_reduce<3>"], check_gemm, (BF, 200, 130, 1024, MODE_ADD_F32)),
    (BF, ["gemm_tile<128,128,2,2,1,4>", "gemm_split_reduce<0>"], check_gemm, (BF, 130, 96, 2048, MODE_SWIGLU)),
    (BF, ["gemm_tile<128,128,2,2,0,4>", "gemm_split_reduce<0>"], check_gemm, (BF, 256, 3584, 18944, MODE_ADD_F32)),  # a 7B layer's
    (BF, ["gemm_tile<128,128,2,2,0,2>", "gemm_split_reduce<0>"], check_gemm, (BF, 200, 4608, 3584, MODE_STORE, True)),
    (BF, ["gemm_tile<128,128,2,2,0,2>", "gemm_split_reduce<3>"], check_gemm, (BF, 300, 130, 1024, MODE_ADD_F32)),
    (BF, ["gemm_tile<128,128,2,2,1,2>", "gemm_split_reduce<0>"], check_gemm, (BF, 300, 96, 2048, MODE_SWIGLU)),
    (BF, ["gemm_tile<128,128,2,2,1,2>"], check_gemm, (BF, 200, 8320, 256, MODE_SWIGLU)),
    (BF, ["gemm_tile<256,192,4,2,0,2>"], check_gemm, (BF, 2048, 4608, 192, MODE_STORE, True)),
    (BF, ["gemm_tile<256,256,4,2,0,2>"], check_gemm, (BF, 1100, 9300, 128, MODE_STORE_F32)),
    (BF, ["gemm_tile<256,256,4,2,0,2>", "gemm_split_reduce<0>"], check_gemm, (BF, 2049, 3584, 18944, MODE_ADD_F32)),
    (BF, ["gemm_tile<256,256,4,2,1,2>"], check_gemm, (BF, 2048, 2608, 64, MODE_SWIGLU)),
    (BF, ["gemm_tile<128,128,2,2,0,4>", "gemm_split_reduce<1>"], check_then_norm, (150, 256, 1024)),
    (BF, ["gemm_tile<256,256,4,2,1,2>"], check_gemm, (BF, 200, 18944, 3584, MODE_SWIGLU)),              # a 7B layer's at 200 rows
    (BF, ["gemm_tile<256,256,4,2,0,2>", "gemm_split_reduce<2>"], check_qkv_rope, (1525, 40, 8, 128, 5120, 64)),        # a 14B layer's
    # the segments of K in one block, plain, gated, and with the norm and the rotary store behind
    (BF, ["gemm_kept<0>"], check_gemm, (BF, 2050, 2308, 512, MODE_STORE, True)),
    (BF, ["gemm_kept<0>"], check_gemm, (BF, 1153, 4102, 1088, MODE_ADD_F32, True)),
    (BF, ["gemm_kept<1>"], check_gemm, (BF, 1153, 1040, 1024, MODE_SWIGLU)),
    (BF, ["gemm_kept<0>", "gemm_split_reduce<1>"], check_then_norm, (2049, 2304, 1024)),
    (BF, ["gemm_kept<0>", "gemm_split_reduce<2>"], check_qkv_rope, (2050, 16, 2, 128, 2048, 64)),
    (BF, ["gemm_kept<0>", "gemm_split_reduce<2>"], check_qkv_rope, (2048, 28, 4, 128, 3584, 64)),    # a 7B layer's
    (BF, ["gemm_kept<0>"], check_gemm, (BF, 2049, 3584, 3584, MODE_ADD_F32)),
    # grouped products: (matrix cores or 32-bit FMA, gated epilogue)
    (BF, ["grouped_gemm<4,0>"], check_grouped, (BF, 50, 3, 40, 64, False)),
    (BF, ["grouped_gemm<4,1>"], check_grouped, (BF, 19, 2, 72, 160, True)),
    (BF, ["grouped_gemm<1,0>"], check_grouped, (BF, 50, 3, 40, 288, False)),
    (BF, ["grouped_gemm<1,1>"], check_grouped, (BF, 19, 2, 72, 544, True)),
    (BF, ["grouped_gemm<0,0>"], check_grouped, (BF, 50, 3, 40, 24, False)),
    (BF, ["grouped_gemm<0,1>"], check_grouped, (BF, 19, 2, 72, 40, True)),
    (BF, ["grouped_gemm<3,0>"], check_grouped, (BF, 300, 3, 40, 64, False)),       # many rows: tiles of 64 through LDS
    (BF, ["grouped_gemm<3,1>"], check_grouped, (BF, 270, 2, 72, 160, True)),
    (BF, ["grouped_gemm<2,1>"], check_grouped, (BF, 1030, 16, 200, 96, True)),     # gated, two rounds of large blocks
    (BF, ["grouped_gemm<5,1>"], check_wide_lists, (260, 704, 300)),                # lists of tiles of 128 rows
    (F32, ["grouped_gemm<0,0>"], check_grouped, (F32, 50, 3, 40, 64, False)),
    (F32, ["grouped_gemm<0,1>"], check_grouped, (F32, 19, 2, 72, 160, True)),
    # the short convolution: a thread a (token, channel), and runs of tokens in long steps
    (BF, ["causal_conv<0>"], check_conv, (BF, 256, 2560)),
    (BF, ["causal_conv<1>"], check_conv, (BF, 517, 2564)),
    (F32, ["causal_conv<0>"], check_conv, (F32, 1023, 260)),
    (F32, ["causal_conv<1>"], check_conv, (F32, 2049, 640)),
    # latent attention: many tokens by (tiles of 16 latent dims, chunks of 32 key dims, bounds known when compiled, sink), and
    # the kernels of a wave a token and of its blocks side by side
    *[(BF, [f"latent_prompt<{rt},{qc},1,{sink}>"], check_latent, (16 * rt, 32 * qc - 16 * rt, sink))
      for rt, qcs in ((32, (17, 18, 20)), (16, (9, 10, 12)), (8, (5, 6, 8)), (4, (3, 4, 6))) for qc in qcs for sink in (0, 1)],
    *[(BF, [f"latent_prompt<{rt},{qc},0,{sink}>", f"latent_tokens<{rt},{qc},{sink}>", f"latent_blocks<{rt},{qc}>"], check_latent,
       (rank, rot, sink)) for rt, qc, rank, rot in ((4, 4, 48, 16), (8, 8, 112, 48), (32, 20, 192, 64)) for sink in (0, 1)],
    # the float32 build's attention on the matrix cores: (head size) and (head size, waves a block)
    (F32, ["attention_f32_prefill<64>", "attention_f32_waves<64,2>", "attention_f32_decode<64,1>"], check_attention_f32, (4, 2, 64, 16, 333, 90, 5)),
    (F32, ["attention_f32_prefill<128>", "attention_f32_waves<128,2>", "attention_f32_decode<128,1>"], check_attention_f32, (7, 1, 128, 64, 600, 0, 7)),
    (F32, ["attention_f32_waves<64,1>"], check_attention_f32, (16, 2, 64, 16, 600, 0, 3)),             # more blocks than CUs
    (F32, ["attention_f32_waves<64,1>"], check_attention_f32, (12, 4, 64, 16, 330, 100, 3)),
    (F32, ["attention_f32_waves<128,1>"], check_attention_f32, (16, 1, 128, 16, 800, 0, 3)),
    (F32, ["attention_f32_waves<128,1>"], check_attention_f32, (16, 1, 128, 16, 600, 300, 3)),
    (F32, ["attention_f32_decode<64,4>"], check_attention_f32, (8, 4, 64, 16, 140, 0, 40)),
    (F32, ["attention_f32_decode<128,4>"], check_attention_f32, (8, 4, 128, 32, 150, 60, 33)),
    # decoding attention by blocks of positions (maps, tiles of 16 value dims, chunks of 32 key dims), and what adds them up (value dims a lane)
    *[(BF, [f"masked_blocks<{maps},{dt},{kc}>", f"masked_fold<{maps},{own}>"], check_masked_blocks, (maps, dim, vdim, page, softcap, gated))
      for maps in (1, 2) for dt, own, vdim in ((4, 1, 48), (8, 2, 128), (16, 4, 208))
      for kc, dim, page, softcap, gated in ((2, 40, 64, 0.0, "dims"), (4, 128, 192, 20.0, None), (8, 256, 128, 0.0, "heads"))],
    # the gated recurrence: a thread a channel, or waves that feed the walk
    *[(dtype, [f"gated_scan<{int(T > 4)}>"], check_gated_scan, (dtype, T)) for dtype in (BF, F32) for T in (4, 77)],
    # the embedding: eight numbers a thread, or one (unaligned rows, and many tokens of a packed table)
    *[(dtype, [f"embed<{eights}>"], check_embed, (dtype, T, dim, False)) for dtype in (BF, F32) for T, dim, eights in ((5, 40, 1), (3, 35, 0), (1030, 64, 1))],
    *[(BF, [f"embed<{int(T < 1024)}>"], check_embed, (BF, T, dim, True)) for T, dim in ((1023, 64), (1024, 64), (1100, 192), (7, 2112))],
    # the convolution before a state-space scan: a thread a (token, channel), or runs of tokens
    *[(dtype, [f"state_conv<{runs}>"], check_state_conv, (dtype, T, C, taps))
      for dtype in (BF, F32) for T, C, taps, runs in ((300, 70, 3, 0), (260, 6000, 4, 1), (700, 4436, 2, 1), (2051, 1036, 3, 1))],
    # heads laid out for attention: blocks of four units in steps of up to 1,023 tokens; beyond, one block a token where all would do something
    # again, else of up to eight or sixteen units
    *[(dtype, [f"heads_prepare<{blocks}>"], check_heads_prepare, (dtype, T, form, nq))
      for dtype in (BF, F32) for T, form, nq, blocks in ((1023, "rows", 5, 0), (1024, "rows", 5, 1), (1024, "heads", 5, 2), (1025, "none", 5, 2),
                                                         (1030, "conv", 5, 1), (1024, "heads", 23, 2), (1024, "none", 31, 2), (1100, "heads", 1, 2))],
    # attention on the matrix cores: (head size, query heads a block, pages of 64 positions or more)
    # and (head size, waves a block) (one wave a block in the decoding kernel up to 2,560 blocks of
    # positions, four beyond; two heads a block in the prompt kernel where tiles x heads are more
    # than 256: the long prompts of real models)
    (BF, ["attention_prefill<64,1,0>", "attention_decode<64,1>"], check_attention_mfma, (4, 2, 64, 16, 200, 0)),
    (BF, ["attention_prefill<64,1,1>"], check_attention_mfma, (4, 2, 64, 64, 200, 0)),
    (BF, ["attention_prefill<128,1,1>", "attention_decode<128,1>"], check_attention_mfma, (7, 1, 128, 64, 333, 90)),
    (BF, ["attention_prefill<128,1,0>"], check_attention_mfma, (7, 1, 128, 16, 333, 90)),
    (BF, ["attention_prefill<64,2,1>", "attention_decode<64,4>"], check_attention_mfma, (32, 1, 64, 64, 1700, 0, 5)),
    (BF, ["attention_prefill<64,2,0>"], check_attention_mfma, (64, 2, 64, 16, 800, 0, 3)),
    (BF, ["attention_prefill<128,2,0>", "attention_decode<128,4>"], check_attention_mfma, (14, 2, 128, 16, 3400, 0, 37)),
    (BF, ["attention_prefill<128,2,1>"], check_attention_mfma, (64, 2, 128, 64, 800, 300, 3)),
]
IDS = [f"{dtype[:2]}-{'+'.join(names)}-{i}" for i, (dtype, names, _, _) in enumerate(CASES)]


def run_case(i):
    dtype, names, check, args = CASES[i]
    hit = check(*args)
    RAN.add(i)
    assert set(names) <= hit, f"meant to select {names}, the library launched {sorted(hit)}"
    torch.cuda.empty_cache()


@pytest.mark.parametrize("i", range(len(CASES)), ids=IDS)
def test_the_instance_a_call_selects_gives_the_right_result(i):
    run_case(i)


def test_every_compiled_instance_was_launched_and_checked():
    for i in range(len(CASES)):            # run alone, this test runs the cases itself
        if i not in RAN:
            run_case(i)
    for dtype in (BF, F32):
        known = set(kernels(dtype).instances())
        named = {n for d, names, _, _ in CASES if d == dtype for n in names}
        assert known <= named, f"{dtype}: no case selects {sorted(known - named)}"
        assert known <= SEEN[dtype], f"{dtype}: never launched: {sorted(known - SEEN[dtype])}"
