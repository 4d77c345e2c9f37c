"""Each kernel at the sizes where its tiling or its dispatch turns over: one row or token past an edge, remainders, the
smallest and the largest of a range, against the oracle with the bounds of the other parity tests."""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import parity as P  # noqa: E402

pytestmark = pytest.mark.gpu
F32, BF = torch.float32, torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from mindspeed_mm_amd.ops import _default_ops
    return _default_ops()


@pytest.mark.parametrize("dtype,rows,N", [
    (BF, 1, 128), (BF, 17, 128),                   # one row; one row past a workgroup of the forward kernel
    (BF, 16 * 512 + 1, 128), (BF, 3 * 16 * 512, 128),   # one row past the backward grid; whole trips of it
    (BF, 16 * 768 + 1, 128),                       # one row past the larger backward grid of 16-bit tensors
    (BF, 4 * 512 + 3, 512), (F32, 64 * 512 + 5, 16),    # a row on a whole wave; a row on four lanes
])
@pytest.mark.parametrize("activation", ["silu", "sigmoid"])
def test_rms_norm_gated_edges(ops, dtype, rows, N, activation):
    P.check_rms_norm_gated(ops, "cuda", (rows,), N, dtype, activation=activation)


@pytest.mark.parametrize("activation", ["silu", "sigmoid"])
def test_rms_norm_gated_far_gates(ops, activation):
    """Gates beyond the range of the exponential: the sigmoid is 0 or 1 there, nothing finite becomes inf or NaN, and
    what is not finite stays so."""
    gate = torch.tensor([-1e4, -200.0, -89.0, -88.0, -87.0, 0.0, 87.0, 89.0, 200.0, 1e4], device="cuda", dtype=BF)
    g = gate.repeat(13)[:128].repeat(40, 1)
    x = torch.randn(40, 128, generator=torch.Generator().manual_seed(40)).to("cuda", BF)
    w = torch.ones(128, device="cuda", dtype=BF)
    L = [t.clone().requires_grad_(True) for t in (x, g, w)]
    y = ops.rms_norm_gated(*L, 1e-6, activation)
    y.backward(torch.ones_like(y))
    xn = (x.float() * torch.rsqrt(x.float().square().mean(-1, keepdim=True) + 1e-6)).to(BF).float()
    s = torch.sigmoid(g.double())
    ref = xn.double() * (g.double() * s if activation == "silu" else s)
    # three roundings to bf16 (2^-9 each, the first shared); below -88.7 the exponential overflows and the sigmoid is 0,
    # where in float64 it is at most e^-88.7 = 2.9e-39 (times the gate).  Below bf16's smallest normal number, 2^-126, a
    # rounding moves a value by up to half the spacing there, 2^-134, however small the value is: three of them.
    assert ((y.double() - ref).abs() <= 2.0 ** -7 * ref.abs() + 90 * 2.9e-39 * xn.abs().double() + 3 * 2.0 ** -134).all()
    assert all(torch.isfinite(t.grad.float()).all() for t in L)
    P.check_far_gates(ops, "cuda", activation)


@pytest.mark.parametrize("dtype,B,T,D,W,cu", [
    (BF, 1, 8, 64, 4, None), (BF, 2, 11, 64, 4, None), (BF, 1, 19, 1032, 4, None),   # one tile; its halo; a ragged channel block
    (BF, 1, 600, 64, 4, [0, 3, 16, 19, 24, 24, 300, 303, 600]),       # boundaries on, just past and inside tile edges
    (BF, 1, 41, 64, 4, list(range(42))), (F32, 1, 75, 64, 3, list(range(0, 76, 3))), (BF, 9, 5, 64, 4, None),   # shorter than a window or a tile
    (BF, 3, 64, 72, 4, None), (F32, 1, 257, 64, 3, [0, 128, 257]), (torch.float16, 1, 100, 64, 2, None),
    (BF, 1, 300, 64, 5, [0, 64, 65, 300]), (BF, 1, 200, 64, 8, None),  # windows wider than the straight-line backward tile
    (BF, 1, 16 * 256 + 5, 1024, 4, None),                              # tiles past the first of every backward workgroup
])
def test_conv1d_edges(ops, dtype, B, T, D, W, cu):
    P.check_conv(ops, "cuda", B, T, D, W, dtype, cu=cu, residual=True)
    P.check_conv(ops, "cuda", B, T, D, W, dtype, cu=cu, bias=False, state=False, activation=None)


def test_conv1d_more_work_items_than_a_launch(ops):
    """8 channels: 2^25 workgroups of 128 take 2^28 tokens, and a launch counts fewer than 2^32 work-items."""
    T, D, W, n = (1 << 28) + 1000, 8, 4, 4000
    w = torch.randn(W, D, device="cuda", dtype=BF)
    x = torch.empty(1, T, D, device="cuda", dtype=BF).uniform_(-1, 1)
    with torch.no_grad():
        y, _ = ops.causal_conv1d(x, w, activation="silu")
        for at in (0, T // 2, T - n):
            lo = max(0, at - 8)
            part, _ = ops.causal_conv1d(x[:, lo:at + n].contiguous(), w, activation="silu")
            assert torch.equal(y[:, at:at + n], part[:, at - lo:])


@pytest.mark.parametrize("dtype,W,D", [(BF, 4, 1032), (BF, 1, 8), (BF, 8, 16), (F32, 3, 20)])
@pytest.mark.parametrize("initial", ["none", "given", "in place"])
@pytest.mark.parametrize("cu", [[0, 0, 1, 3, 3, 6, 10, 27, 32, 32], [0, 5], [0, 0, 0, 8]])
def test_conv1d_final_states_of_packed_sequences(ops, dtype, W, D, initial, cu):
    """Empty, shorter than the window, ending on a tile's edge and inside one: the states are copies, bit for bit."""
    from mindspeed_mm_amd._lib import DTYPE_CODE, ptr
    gen = torch.Generator().manual_seed(W)
    T, N = cu[-1], len(cu) - 1
    x, w = torch.randn(T, D, generator=gen).to(dtype), torch.randn(W, D, generator=gen).to(dtype)
    init = None if initial == "none" else torch.randn(N, D, W, generator=gen).to(dtype)
    want = torch.empty(N, D, W, dtype=dtype)
    for n in range(N):
        before = torch.zeros(D, W, dtype=dtype) if init is None else init[n]
        want[n] = torch.cat([before, x[cu[n]:cu[n + 1]].t()], dim=1)[:, -W:]
    xd, wd, cud, h0 = x.cuda(), w.cuda(), torch.tensor(cu).cuda(), None if init is None else init.cuda()
    y, fs = torch.empty_like(xd), h0 if initial == "in place" else torch.empty(N, D, W, dtype=dtype, device="cuda")
    print(f"conv1d packed final states {dtype} W{W} D{D} {initial} {cu}", flush=True)
    ops.lib.check(ops.lib.gdn_conv1d_fwd(ptr(xd), ptr(wd), None, None, ptr(h0), ptr(cud), ptr(y), ptr(fs), 1, T, N, D, W, 0,
                                         DTYPE_CODE[dtype], ops.lib.stream()), "gdn_conv1d_fwd")
    assert torch.equal(fs.cpu(), want)


@pytest.mark.parametrize("dtype,B,T,Hqk,Hv,K,V", [
    (BF, 8, 1, 16, 32, 128, 128), (BF, 9, 1, 16, 32, 128, 128),    # as many states as compute units; more: whole states
    (BF, 17, 1, 16, 32, 128, 128),                                 # states larger than the L2s
    (BF, 129, 1, 16, 32, 128, 128),                                # larger than the memory-side cache
    (F32, 3, 2, 1, 2, 128, 192), (BF, 2, 3, 1, 1, 256, 64), (BF, 140, 2, 1, 2, 256, 128), (BF, 300, 1, 1, 1, 64, 256),
])
def test_recurrent_edges(ops, dtype, B, T, Hqk, Hv, K, V):
    P.check_recurrent(ops, "cuda", B, T, Hqk, Hv, K, V, dtype)


@pytest.mark.parametrize("dtype,K,V,batches", [
    (BF, 128, 128, (1, 9, 17, 129)), (F32, 128, 128, (1, 9)), (BF, 128, 64, (1, 9, 40, 260)), (BF, 64, 128, (1, 33, 258)),
    (BF, 256, 128, (1, 9, 20, 66)), (BF, 256, 256, (1, 33)),
])
def test_recurrent_bits_do_not_depend_on_the_batch(ops, dtype, K, V, batches):
    P.check_recurrent_batch_bits(ops, "cuda", batches, 16, 32, K, V, dtype)


@pytest.mark.parametrize("T,K,V", [(2, 64, 64), (130, 64, 64), (65, 128, 192), (64, 128, 128)])
def test_chunk_fp32_bits_do_not_depend_on_the_batch(ops, T, K, V):
    """The fp32 recurrences give a workgroup 16 or 32 state columns by the size of the call: the same bits either way."""
    x = {n: t.cuda() for n, t in P.gdn_inputs(40, T, 2, 4, K, V, F32, seed=T).items()}

    def call(n):
        leaf = {m: x[m][:n].clone().requires_grad_(True) for m in ("q", "k", "v", "g", "beta", "h0")}
        o, s = ops.chunk_gated_delta_rule(*list(leaf.values())[:5], initial_state=leaf["h0"], output_final_state=True,
                                          use_qk_l2norm_in_kernel=True)
        return [o, s, *torch.autograd.grad([o, s], list(leaf.values()), [x["do"][:n], x["dht"][:n]])]
    for a, b in zip(call(1), call(40)):
        assert torch.equal(a[0], b[0])


@pytest.mark.parametrize("T,Hqk,Hv,K,V,l2,cu", [
    (70, 1, 3, 64, 128, True, None),      # three heads to a group whose sums just fill their place, waves without columns of K
    (65, 1, 2, 128, 192, True, None),     # R in two parts, the second of two V blocks; a last chunk of one token
    (64, 1, 1, 128, 64, False, None),     # one pair of V blocks; no l2 norm
    (33, 1, 2, 64, 64, True, None),       # several heads and V = 64: the four-wave kernel
    (130, 2, 2, 64, 256, False, None),
    (1000, 2, 8, 64, 192, True, [0, 1, 1, 300, 364, 427, 990]),   # chunks of 1, 43, 63 and 64 tokens, rows of no sequence
    (2100, 16, 32, 128, 128, True, [0, 700, 2100]),               # 544 workgroups, where the chip holds 512 at once
])
def test_chunk_local_backward_of_head_groups(ops, T, Hqk, Hv, K, V, l2, cu):
    """The chunk-local kernel where its tiles, its V blocks and the sums over a group's heads end."""
    end = cu[-1] if cu else T
    P.check_chunk(ops, "cuda", 1, end, Hqk, Hv, K, V, BF, l2=l2, cu=cu, backward=True, h0_std=0.1, seed=5)
    if end == T:
        return
    # rows of no sequence: zero gradients, and the others those of the call without them
    x = P.gdn_inputs(1, T, Hqk, Hv, K, V, BF, seed=5, N=len(cu) - 1, l2norm_in_kernel=l2, h0_std=0.1)
    cu_t = torch.tensor(cu, dtype=torch.int64, device="cuda")

    def grads(rows):
        leaf = [x[n][:, :rows].cuda().requires_grad_(True) for n in ("q", "k", "v", "g", "beta")]
        o, _ = ops.chunk_gated_delta_rule(*leaf, initial_state=x["h0"].cuda(), use_qk_l2norm_in_kernel=l2, cu_seqlens=cu_t)
        return torch.autograd.grad([o], leaf, [x["do"][:, :rows].cuda()])
    for a, b in zip(grads(T), grads(end)):
        assert torch.equal(a[:, :end], b) and not a[:, end:].any()


@pytest.mark.parametrize("T,K,V", [(33, 64, 64), (70, 64, 192), (65, 128, 192)])
def test_kda_backward_where_the_sums_over_v_end(ops, T, K, V):
    """One pair of V blocks, R in two parts with the second cut short, waves without columns of K, a last chunk of one token."""
    P.check_kda(ops, "cuda", 1, T, 1, K, V, BF, backward=True, h0_std=0.1, seed=6)


@pytest.mark.parametrize("B,Hv,V", [(2, 32, 64), (3, 22, 64), (1, 24, 192)])
def test_reverse_recurrence_with_two_and_four_loading_waves(ops, B, Hv, V):
    """K = 64: four up to 128 slabs of 32 columns where the recurrence runs alone, else two; the same bits."""
    P.check_chunk(ops, "cuda", B, 300, Hv // 2, Hv, 64, V, BF, backward=True, skip_recompute=True, h0_std=0.1)
    P.check_chunk_recompute_equals_stored(ops, "cuda", B, 300, Hv // 2, Hv, 64, V, BF)


@pytest.mark.parametrize("T,Hqk,Hv,V,cu", [
    (4095, 1, 2, 128, None), (4096, 1, 2, 128, None), (4097, 2, 2, 128, None),   # a token short of being cut; uneven segments
    (4159, 1, 3, 128, None),                                                     # a group of three heads, a short last chunk
    (12400, 1, 2, 128, [0, 130, 130, 12400]),                                    # empty segments, an empty sequence
])
def test_recurrences_in_segments(ops, T, Hqk, Hv, V, cu):
    """Few heads and long sequences: both recurrences run cut into segments.  Rebuilding the forward states in the backward
    pass starts from the segments' saved states and has to give the same bits as keeping them."""
    P.check_chunk(ops, "cuda", 1, T, Hqk, Hv, 128, V, BF, cu=cu, backward=True, h0_std=0.1)
    x = P.gdn_inputs(1, T, Hqk, Hv, 128, V, BF, seed=3, N=len(cu) - 1 if cu else 1)
    cu_t = torch.tensor(cu, dtype=torch.int64, device="cuda") if cu else None
    got = []
    for keep in (True, False):
        leaf = [x[n].cuda().requires_grad_(True) for n in ("q", "k", "v", "g", "beta", "h0")]
        o, ht = ops.chunk_gated_delta_rule(*leaf[:5], initial_state=leaf[5], output_final_state=True,
                                           use_qk_l2norm_in_kernel=True, cu_seqlens=cu_t, skip_recompute=keep)
        got.append((o, ht, *torch.autograd.grad([o, ht], leaf, [x["do"].cuda(), x["dht"].cuda()])))
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T,H,cu", [(4097, 2, None), (12400, 1, [0, 130, 130, 12400])])
def test_kda_recurrences_in_segments(ops, T, H, cu):
    P.check_kda(ops, "cuda", 1, T, H, 128, 128, BF, cu=cu, backward=True)


@pytest.mark.parametrize("T,Hqk,Hv,kda,B,cu", [
    (4097, 1, 2, False, 1, None), (4159, 1, 1, True, 1, None),
    (8192, 4, 8, False, 1, None), (8192, 8, 8, True, 1, None),      # as many slabs as compute units: refill with two to a workgroup
    (4160, 2, 2, False, 2, None), (4160, 2, 2, True, 2, None),      # a dense batch
    (12400, 1, 2, False, 1, [0, 130, 130, 12400]), (12400, 1, 1, True, 1, [0, 130, 130, 12400]),
])
def test_cut_sequences_carry_a_slowly_decaying_state(ops, T, Hqk, Hv, kda, B, cu):
    N = B if cu is None else len(cu) - 1
    P.check_cut_against_uncut(ops, "cuda", T, Hqk, Hv, kda, cu=cu, B=B, tile=-(-24 // (N * Hv)))


def test_cut_sequences_through_the_strided_entry_and_the_norm(ops):
    """The unsplit convolution output and the gated norm in one call, cut: the bits of the separate operators on copies."""
    T, H, K = 4200, 2, 128
    x = P.gdn_inputs(1, T, H, H, K, K, BF, seed=6, a_log=(0.5, 2.0), dt_bias=(-9.0, -8.0))
    d = {n: t.cuda() for n, t in x.items()}
    qkv = torch.cat([d[n].flatten(2) for n in ("q", "k", "v")], -1)
    z, w = torch.randn(1, T, H, K, device="cuda", dtype=BF), torch.rand(K, device="cuda").to(BF)
    with torch.no_grad():
        y, ht = ops.chunk_gated_delta_rule_qkv(qkv, d["g"], d["beta"], H, H, K, K, initial_state=d["h0"],
                                               output_final_state=True, use_qk_l2norm_in_kernel=True, gate=z, norm_weight=w)
        o, ht2 = ops.chunk_gated_delta_rule(d["q"], d["k"], d["v"], d["g"], d["beta"], initial_state=d["h0"],
                                            output_final_state=True, use_qk_l2norm_in_kernel=True)
        assert torch.equal(y, ops.rms_norm_gated(o, z, w)) and torch.equal(ht, ht2)


def test_sequence_bits_alone_and_in_a_batch(ops):
    """Uncut, a sequence's bits do not depend on what is packed with it; a call that is cut has the bits of its own number of
    segments."""
    x = {n: t.cuda() for n, t in P.gdn_inputs(1, 8192, 8, 32, 128, 128, BF, seed=8, N=2).items()}

    def first(T, N, cu):
        with torch.no_grad():
            o, ht = ops.chunk_gated_delta_rule(*(x[n][:, :T].contiguous() for n in ("q", "k", "v", "g", "beta")),
                                               initial_state=x["h0"][:N].contiguous(), output_final_state=True,
                                               use_qk_l2norm_in_kernel=True, cu_seqlens=cu)
        return o[:, :4096], ht[:1]
    alone, packed = first(4096, 1, [0, 4096]), first(8192, 2, [0, 4096, 8192])
    assert torch.equal(alone[0], packed[0]) and torch.equal(alone[1], packed[1])


@pytest.mark.parametrize("N", [1, 64, 65, 256, 257, 520])
def test_chunk_table_of_many_sequences(ops, N):
    """A wave and a workgroup of sequences, one more, several to a thread, empty ones among them: every sequence as in a
    dense batch of its length, bit for bit, and zeros in the rows behind the last one."""
    gen = torch.Generator().manual_seed(N)
    kinds = [0, 1, 64, 65]
    lengths = [kinds[i] for i in torch.randint(0, 4, (N,), generator=gen).tolist()]
    lengths[-1] = 65
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    T, tail, K = cu[-1], 70, 64
    x = P.gdn_inputs(1, T + tail, 1, 1, K, K, BF, seed=N)
    x = {n: t.cuda() for n, t in x.items()}
    print(f"chunk table: {N} sequences, {T} tokens", flush=True)

    def rule(rows, h0, cu_t):
        return ops.chunk_gated_delta_rule(*(rows(x[n]) for n in ("q", "k", "v", "g", "beta")), initial_state=h0,
                                          output_final_state=True, use_qk_l2norm_in_kernel=True, cu_seqlens=cu_t)
    h0 = torch.randn(N, 1, K, K, generator=gen).cuda()
    with torch.no_grad():
        o, ht = rule(lambda t: t, h0, torch.tensor(cu).cuda())
        for L in kinds:
            at = [n for n in range(N) if lengths[n] == L]
            if L == 0 or not at:
                assert all(torch.equal(ht[n], h0[n]) for n in at)
                continue
            idx = torch.tensor([[cu[n] + i for i in range(L)] for n in at]).cuda()
            ob, hb = rule(lambda t: t[0][idx], h0[at], None)
            assert torch.equal(o[0][idx], ob) and torch.equal(ht[at], hb)
    assert not o[0, T:].any()
